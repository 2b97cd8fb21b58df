// A 128-wide block of a training step as two calls, forward and backward: the launches of cf_block_head, the encoding,
// cf_fused_dpa_* and cf_block_tail* on the same operands in the same order, so results are theirs to the bit.
//
// Four operators a block each way, every one with its checks, allocations and an autograd node of its own, took 200 us of host
// time forward and 140 backward; as one node and two calls it is 65 and 85, most of it the launches.  A step of four blocks on
// an ever new batch of 61 crystals, whose kernels take 0.79 ms, waited for the host: 2.44 -> 1.66 ms.
// What is kept for the backward call lies in two pieces of memory, what either call needs for itself in another.
#include "cf_common.h"

namespace {

using namespace cf;

constexpr int64_t W = 128, FF = 512;

struct Carve {
    char *base;
    int64_t at = 0;
    float *take(int64_t bytes)
    {
        float *p = base ? reinterpret_cast<float *>(base + at) : nullptr;
        at += (bytes + 255) / 256 * 256;
        return p;
    }
    float *rows(int64_t n, int64_t width) { return take(n * width * 4); }
};

// What the caller's weight gradients read, rows of whole 256 bytes, and what only the backward call does: two pieces, since the
// first lives on until the weight gradients of all blocks are formed.
struct Saved {
    float *att, *s, *h;
    int64_t bytes;
    float *q, *qs, *k, *v, *a, *alpha_n, *used, *z, *val, *prob;
    int64_t more_bytes;
};
Saved carve_saved(const cf_block_train &f, void *base, void *more)
{
    Saved r{};
    Carve c{(char *)base};
    r.att = c.rows(f.N, W);
    r.s = c.rows(f.N, W);
    r.h = c.rows(f.N, FF);
    r.bytes = c.at;
    Carve m{(char *)more};
    r.q = m.rows(f.N, W);
    r.qs = m.rows(f.N, W);
    r.k = m.rows(f.N, W);
    r.v = m.rows(f.N, W);
    r.a = m.rows(f.N, f.H);
    r.alpha_n = m.rows(f.N, f.H);
    r.used = m.take(8);
    r.z = m.rows(f.E, f.H);
    r.val = f.bins > 0 ? m.rows(f.E, W) : nullptr;
    r.prob = m.rows(f.E, f.H);
    r.more_bytes = m.at;
    return r;
}

struct ForwardScratch {
    float *part;
    void *flags;
    int64_t flag_bytes, bytes;
};
ForwardScratch carve_forward(const cf_block_train &f, void *base)
{
    Carve c{(char *)base};
    ForwardScratch r{};
    r.part = f.normalize ? c.take(cf_gauss_exponents_workspace(f.N, f.H)) : nullptr;
    r.flag_bytes = f.rings && f.cutoff != 0.0 ? cf_real_enc_flag_bytes(f.U, f.H) : 0;
    r.flags = r.flag_bytes ? c.take(r.flag_bytes) : nullptr;
    r.bytes = c.at;
    return r;
}

// gq, gk, gv, gs, gx, gh: what the caller goes on with, at multiples of whole rows.
struct Kept {
    float *gq, *gk, *gv, *gs, *gx, *gh;
    int64_t bytes;
};
Kept carve_kept(const cf_block_train &f, void *base)
{
    Carve c{(char *)base};
    Kept r{};
    r.gq = c.rows(f.N, W);
    r.gk = c.rows(f.N, W);
    r.gv = c.rows(f.N, W);
    r.gs = c.rows(f.N, W);
    r.gx = c.rows(f.N, W);
    r.gh = c.rows(f.N, FF);
    r.bytes = c.at;
    return r;
}

struct BackwardScratch {
    float *gatt, *gqs, *gaij, *gbij, *ga, *g_alpha;
    void *ws;
    int64_t ws_bytes, bytes;
};
BackwardScratch carve_backward(const cf_block_train &f, void *base)
{
    Carve c{(char *)base};
    BackwardScratch r{};
    r.gatt = c.rows(f.N, W);
    r.gqs = c.rows(f.N, W);
    r.gaij = c.rows(f.E, f.H);
    r.gbij = f.bins > 0 ? c.rows(f.E, W) : nullptr;
    r.ga = c.rows(f.N, f.H);
    r.g_alpha = c.rows(f.N, f.H);
    r.ws_bytes = cf_real_enc_bwd_workspace(f.N, f.H, f.E, f.bins, f.bins > 0 ? W / f.H : 0, f.bins > 0 ? 1 : 0, f.want_gw_pe ? 1 : 0);
    r.ws = c.take(r.ws_bytes > 1 ? r.ws_bytes : 1);
    r.bytes = c.at;
    return r;
}

int check_block(const cf_block_train *args, const char *who)
{
    CF_REQUIRE(args, CF_ERR_INVALID_ARGUMENT, "%s: null arguments", who);
    const cf_block_train &f = *args;
    CF_REQUIRE(f.N >= 1 && f.E >= 1 && f.B >= 1 && f.U >= 1 && f.H >= 1 && f.H <= 32 && W % f.H == 0 && W / f.H % 4 == 0 &&
                   f.bins >= 0 && f.bins <= 128, CF_ERR_INVALID_ARGUMENT, "%s: bad sizes", who);
    CF_REQUIRE(2 * f.U == f.E + f.N, CF_ERR_INVALID_ARGUMENT,
               "%s: a pair list over dense crystal blocks has (E+N)/2 = %lld entries, got %lld", who,
               (long long)((f.E + f.N) / 2), (long long)f.U);
    return CF_OK;
}

int check_pointers(const cf_block_train &f, const char *who)
{
    CF_REQUIRE(f.x && f.w_pos && f.rpos && f.tvecs && f.batch && f.edges && f.e_start && f.atom_start &&
                   f.edge_start && f.pairs && f.saved && f.saved_more && f.scratch && (f.bins == 0 || f.w_pe) &&
                   (f.cutoff == 0.0 || f.rvlen), CF_ERR_INVALID_ARGUMENT, "%s: null pointer", who);
    CF_REQUIRE(!cf_get_size_header(), CF_ERR_UNSUPPORTED, "%s: not under a size header", who);
    return CF_OK;
}

}  // namespace

extern "C" int cf_block_train_bytes(const cf_block_train *args, int64_t *bytes_5)
{
    const int rc = check_block(args, "cf_block_train_bytes");
    if (rc) return rc;
    CF_REQUIRE(bytes_5, CF_ERR_INVALID_ARGUMENT, "cf_block_train_bytes: null pointer");
    const Saved b = carve_saved(*args, nullptr, nullptr);
    bytes_5[0] = b.bytes;
    bytes_5[1] = b.more_bytes;
    bytes_5[2] = carve_forward(*args, nullptr).bytes;
    bytes_5[3] = carve_kept(*args, nullptr).bytes;
    bytes_5[4] = carve_backward(*args, nullptr).bytes;
    return CF_OK;
}

extern "C" int cf_block_train_fwd(const cf_block_train *args, void *stream)
{
    int rc = check_block(args, "cf_block_train_fwd");
    if (rc || (rc = check_pointers(*args, "cf_block_train_fwd"))) return rc;
    const cf_block_train &f = *args;
    CF_REQUIRE(f.packed && f.counter && f.gauss_scale && f.y, CF_ERR_INVALID_ARGUMENT, "cf_block_train_fwd: null pointer");
    const Saved b = carve_saved(f, f.saved, f.saved_more);
    const ForwardScratch t = carve_forward(f, f.scratch);
    const int64_t D = W / f.H;
    if ((rc = cf_block_head(f.x, f.N, f.H, f.packed, f.b_in, f.w_pos, f.gauss_scale, (int)f.normalize, (int)f.update_stats,
                            (int)f.positive_func, (float)f.beta, (float)f.lower_bound, (float)f.coef, (float)f.q_scale, t.part,
                            f.counter, b.q, b.qs, b.k, b.v, b.a, b.alpha_n, f.normalize ? b.used : nullptr, stream)))
        return rc;
    const bool boxes = f.cutoff != 0.0;
    rc = f.rings ? cf_real_enc_fwd_rings(b.a, boxes ? f.rpos : nullptr, boxes ? f.tvecs : nullptr, boxes ? f.batch : nullptr,
                                         f.edges, f.pairs, f.U, f.N, f.H, f.E, f.bins, D, f.dist_max, f.wscale, f.w_pe,
                                         boxes ? f.rvlen : nullptr, f.cutoff, (int)f.lattice_range, (int)f.minimum_range,
                                         f.rings, t.flags, t.flag_bytes, b.z, b.val, stream)
                 : cf_real_enc_fwd(b.a, f.rpos, f.tvecs, f.batch, f.edges, f.N, f.H, f.E, f.B, f.bins, f.bins > 0 ? D : 0,
                                   f.dist_max, f.wscale, f.bins > 0 ? f.w_pe : nullptr, f.bins > 0 ? 1 : 0,
                                   boxes ? f.rvlen : nullptr, f.cutoff, (int)f.lattice_range, (int)f.minimum_range, f.pairs,
                                   f.U, f.sched, b.z, b.val, stream);
    if (rc || (rc = cf_fused_dpa_fwd(b.qs, b.k, b.v, b.z, b.val, f.edges, f.e_start, f.N, f.H, f.E, D, D, b.prob, b.att, stream)))
        return rc;
    return cf_block_tail(b.att, f.x, f.N, f.packed, f.bo, f.b1, f.b2, b.s, b.h, f.y, stream);
}

extern "C" int cf_block_train_bwd(const cf_block_train *args, void *stream)
{
    int rc = check_block(args, "cf_block_train_bwd");
    if (rc || (rc = check_pointers(*args, "cf_block_train_bwd"))) return rc;
    const cf_block_train &f = *args;
    CF_REQUIRE(f.packed_bwd && f.gy && f.kept && f.gw_pos && (!f.want_gw_pe || f.gw_pe), CF_ERR_INVALID_ARGUMENT,
               "cf_block_train_bwd: null pointer");
    const Saved b = carve_saved(f, f.saved, f.saved_more);
    const Kept g = carve_kept(f, f.kept);
    const BackwardScratch t = carve_backward(f, f.scratch);
    const int64_t D = W / f.H;
    if ((rc = cf_block_tail_bwd(f.gy, b.h, f.N, f.packed_bwd, g.gh, g.gs, t.gatt, stream))) return rc;
    if ((rc = cf_fused_dpa_bwd(b.qs, b.k, b.v, b.val, f.batch, f.edges, f.e_start, f.atom_start, f.edge_start, f.N, f.H, f.E,
                               f.B, D, D, b.prob, b.att, t.gatt, t.gqs, g.gk, g.gv, t.gaij, t.gbij, stream)))
        return rc;
    float *gw_pe = f.want_gw_pe ? f.gw_pe : nullptr;
    if (f.rings && f.cutoff == 0.0 && f.bins <= 64 && D <= 16)
        rc = cf_real_enc_bwd_rings(b.a, f.rpos, f.tvecs, f.batch, f.edges, f.e_start, b.z, t.gaij, t.gbij, f.N, f.H, f.E, f.B,
                                   f.bins, D, f.dist_max, f.wscale, f.w_pe, (int)f.lattice_range, f.pairs, f.U,
                                   (const float *)f.rings, t.ws, t.ws_bytes, t.ga, gw_pe, stream);
    else
        rc = cf_real_enc_bwd(b.a, f.rpos, f.tvecs, f.batch, f.edges, f.e_start, b.z, t.gaij, t.gbij, f.N, f.H, f.E, f.B, f.bins,
                             f.bins > 0 ? D : 0, f.dist_max, f.wscale, f.bins > 0 ? f.w_pe : nullptr, f.bins > 0 ? 1 : 0,
                             f.cutoff != 0.0 ? f.rvlen : nullptr, f.cutoff, (int)f.lattice_range, (int)f.minimum_range, f.pairs,
                             f.U, t.ws, t.ws_bytes, t.ga, gw_pe, stream);
    if (rc) return rc;
    return cf_block_head_bwd(t.ga, t.gqs, g.gk, g.gv, g.gs, b.q, f.w_pos, b.alpha_n, f.normalize ? b.used : nullptr, f.N, f.H,
                             f.packed_bwd, (int)f.positive_func, (float)f.beta, (float)f.lower_bound, (float)f.coef,
                             (float)f.q_scale, t.g_alpha, g.gq, g.gx, f.gw_pos, stream);
}
