// A whole inference forward of the encoder in one host call: every launch of the blocks issued from
// here, all intermediate tensors carved from one buffer.
//
// Issued operator by operator from Python a forward of the four-block model is about 40 launches at
// some 14 us of host time each, which is what a small batch costs whatever the GPU does (0.65 ms for
// one crystal of 12 atoms whose kernels take 0.20 ms); from here a launch costs 2-3 us.
#include "cf_common.h"
#include "block_rows.h"
#include "real_enc_infer.h"

namespace {

using namespace cf;

struct Carver {
    char *base;
    int64_t used;
    template <typename T>
    T *take(int64_t count)
    {
        used = (used + 255) & ~(int64_t)255;
        T *p = base ? reinterpret_cast<T *>(base + used) : nullptr;
        used += count * (int64_t)sizeof(T);
        return p;
    }
};

struct Buffers {
    float *rvlen, *rpos, *x[2], *h, *q, *k, *v, *qs, *a, *att, *z, *val, *prob, *rings, *pooled, *hidden;
    void *stats, *flags, *units;
    char *weights;
    unsigned *counters, *groups;
    float *packed;
    float *vcell, *recip, *kr, *sumexp;
    int64_t stats_bytes, flag_bytes, words, weight_bytes;
};

// How a block with value bins is encoded: from units staged by real_enc_infer.hip wherever that is served.  Adaptive boxes are
// staged in the box of the weakest exponent the positive map allows, which grows as the lower bound to the power -3/2, while the
// blocks' own boxes hardly do.  Four blocks, staged against not, us a forward by bound (r0 = 1.4 A unless said):
//   128 crystals of up to 64 atoms:          0.1 325 / 392, 0.05 344 / 393, 0.02 369 / 391, 0.01 422 / 389, 0.005 571 / 395
//     with r0 = 3 A:                         0.1 650 / 808, 0.05 694 / 809, 0.03 780 / 810, 0.02 902 / 811
//   4 of 200 to 400 in large skewed cells:   0.5 538 / 633, 0.25 588 / 660, 0.1 669 / 668, 0.07 746 / 675, 0.05 836 / 693
//   16 of them:                              0.5 3390 / 4707, 0.1 4080 / 4706, 0.05 4519 / 4705
// So from a tenth on, where staging is nowhere slower.
bool boxes_of(const cf_forward_args &f, const cf_forward_block &p) { return f.adaptive != 0 && p.cutoff != 0.0; }
int64_t real_heads(const cf_forward_args &f, const cf_forward_block &p) { return p.coef_reci != 0.0 ? f.H / 2 : f.H; }
bool staged_block(const cf_forward_args &f, const cf_forward_block &p)
{
    const bool boxes = boxes_of(f, p);
    return p.bins > 0 && f.staged_rings && (!boxes || (f.adaptive_rings && (p.cutoff > 0.0 || p.lower_bound >= 0.1))) &&
           infer_served(f.N, f.E, real_heads(f, p), p.bins, f.width / f.H, boxes, (int)f.lattice_range, p.weakest,
                        f.unit_limit_bytes);
}

// Whether the other blocks with value bins -- adaptive boxes below that line, and all where a caller leaves the units no room --
// start from staged rings.
bool use_rings(const cf_forward_args &f, int64_t U)
{
    if (!f.staged_rings || U < 1) return false;
    const int64_t edge = 2 * (int64_t)f.lattice_range + 1;
    return edge * edge * edge <= 128 && cf_real_enc_ring_bytes(U) <= f.ring_limit_bytes;
}

// Adaptive boxes from staged rings are three launches, of which the range rule per pair and the two lists cost 8.5 us
// whatever the batch; the pair kernel, which stages for itself, is one.  Against that the rings' rounds are cheaper: 11.2
// for 14.7 us at 4.1 thousand pairs in the fixed cube, 21.7 for 28.4 at 12.7 thousand, and at 29 thousand with nearly all
// pairs in the cube 52 for 61 with everything counted.  So the rings from three rounds of the whole chip on (a unit per
// wavefront, 16 a CU).  The rule does not see how many pairs leave the cube, which only the device knows: where most do the
// pair kernel would stay ahead above that line too, 36.6 for 45.5 us at 12.7 thousand pairs and 486 to 489 for 514 to 522
// in the blocks of the seven-block model with r0 = 3, two thirds of whose pairs leave it.
bool adaptive_rings_pay(int64_t U) { return U > 48 * (int64_t)device_cu_count(); }

// Whether everything between two attentions runs as one launch.
bool use_rows(const cf_forward_args &f) { return block_rows_served(f.width, f.ff, f.H); }

// The head of block l: projections and exponents.
void head_of(RowsArgs &r, const cf_forward_args &f, const cf_forward_block &p, const Buffers &b, int64_t l)
{
    r.packed_head = b.packed + l * SPLIT_BLOCK; r.b_in = p.b_in; r.w_pos = p.w_pos;
    r.gauss_scale = p.gauss_scale;
    r.normalize = (int)p.normalize; r.update_stats = (int)f.update_stats; r.func = (int)p.positive_func;
    r.beta = (float)p.beta; r.lb = (float)p.lower_bound; r.coef = (float)p.coef; r.q_scale = (float)p.q_scale;
    r.split = p.coef_reci != 0.0; r.coef_second = (float)p.coef_reci;
    r.qs = b.qs; r.k = b.k; r.v = b.v; r.a = b.a;
    r.part = (float *)b.stats;
    r.counter = b.counters + l;
    r.groups = b.groups;
}

int64_t carve(const cf_forward_args &f, const cf_forward_block *blocks, char *base, Buffers &b)
{
    Carver c{base, 0};
    const int64_t N = f.N, E = f.E, U = (N + E) / 2, W = f.width;
    bool rings = false, bins = false;
    int64_t units = 0;
    b.weight_bytes = 0;
    for (int64_t l = 0; l < f.layers; l++) {
        const cf_forward_block &p = blocks[l];
        bins = bins || p.bins > 0;
        if (!staged_block(f, p)) {
            rings = rings || p.bins > 0;
            continue;
        }
        const int64_t one = infer_units_bytes(U, boxes_of(f, p), f.unit_limit_bytes),
                      w = infer_weights_bytes(real_heads(f, p), p.bins, W / f.H);
        units = one > units ? one : units;
        b.weight_bytes = w > b.weight_bytes ? w : b.weight_bytes;
    }
    rings = rings && use_rings(f, U);
    const bool rows = use_rows(f);
    b.rvlen = c.take<float>(3 * f.B);
    b.rpos = c.take<float>(3 * E);
    for (int i = 0; i < 2; i++) b.x[i] = c.take<float>(N * W);
    b.h = rows ? nullptr : c.take<float>(N * f.ff);
    b.q = rows ? nullptr : c.take<float>(N * W);
    b.k = c.take<float>(N * W);
    b.v = c.take<float>(N * W);
    b.qs = c.take<float>(N * W);
    b.a = c.take<float>(N * f.H);
    b.att = c.take<float>(N * W);
    b.z = c.take<float>(E * f.H);
    b.prob = dpa_streams(N, f.H, E, W / f.H) ? nullptr : c.take<float>(E * f.H);
    bool reci = false;
    for (int64_t l = 0; l < f.layers; l++) reci = reci || blocks[l].coef_reci != 0.0;
    b.vcell = reci ? c.take<float>(f.B) : nullptr;
    b.recip = reci ? c.take<float>(9 * f.B) : nullptr;
    b.kr = reci ? c.take<float>(3 * E) : nullptr;
    b.sumexp = reci ? c.take<float>(E * (f.H / 2)) : nullptr;
    b.val = bins ? c.take<float>(E * W) : nullptr;
    b.stats_bytes = cf_gauss_exponents_workspace(N, f.H);
    b.stats = c.take<char>(b.stats_bytes);
    b.packed = rows ? c.take<float>(f.layers * SPLIT_BLOCK + W * (W + 1)) : nullptr;
    b.words = f.layers + (N * f.H + 255) / 256;
    b.counters = c.take<unsigned>(b.words);
    b.groups = b.counters + f.layers;
    b.flag_bytes = rings ? cf_real_enc_flag_bytes(U, f.H) : 0;
    b.flags = rings ? c.take<char>(b.flag_bytes) : nullptr;
    b.rings = rings ? c.take<float>(cf_real_enc_ring_bytes(U) / 4) : nullptr;
    b.units = units ? c.take<char>(units) : nullptr;
    b.weights = units ? c.take<char>(f.layers * b.weight_bytes) : nullptr;
    b.pooled = c.take<float>(f.B * W);
    b.hidden = c.take<float>(f.B * (f.hidden > 0 ? f.hidden : 1));
    return c.used;
}

int check_args(const cf_forward_args *f, const cf_forward_block *blocks)
{
    CF_REQUIRE(f && blocks, CF_ERR_INVALID_ARGUMENT, "cf_forward: null arguments");
    CF_REQUIRE(f->N >= 1 && f->E >= f->N && (f->N + f->E) % 2 == 0 && f->B >= 1 && f->layers >= 1, CF_ERR_INVALID_ARGUMENT,
               "cf_forward: bad sizes N=%lld E=%lld B=%lld layers=%lld", (long long)f->N, (long long)f->E,
               (long long)f->B, (long long)f->layers);
    CF_REQUIRE((f->H == 1 || f->H == 2 || f->H == 4 || f->H == 8 || f->H == 16) && f->width % 16 == 0 &&
                   f->ff % 16 == 0 && f->ff >= 16 && f->width >= 16 && f->width % f->H == 0 && f->width / f->H <= 32,
               CF_ERR_UNSUPPORTED, "cf_forward: width %lld, heads %lld, feed-forward %lld not served",
               (long long)f->width, (long long)f->H, (long long)f->ff);
    CF_REQUIRE(!f->w_embed || (use_rows(*f) && f->embed_width >= 1 && f->embed_width <= f->width), CF_ERR_UNSUPPORTED,
               "cf_forward: an embedding of %lld features is not served", (long long)f->embed_width);
    for (int64_t l = 0; l < f->layers; l++)
        CF_REQUIRE(blocks[l].coef_reci == 0.0 ||
                       (use_rows(*f) && f->H % 2 == 0 && dpa_streams(f->N, f->H, f->E, f->width / f->H) && !live_atoms(f->N)),
                   CF_ERR_UNSUPPORTED, "cf_forward: block %lld: two domains not served", (long long)l);
    for (int64_t l = 0; l < f->layers; l++)
        CF_REQUIRE(blocks[l].positive_func >= 0 && blocks[l].positive_func <= 2 && blocks[l].lower_bound < 1.0,
                   CF_ERR_UNSUPPORTED, "cf_forward: block %lld: positive map not served", (long long)l);
    for (int64_t l = 0; l < f->layers; l++)
        CF_REQUIRE(blocks[l].bins >= 0 && blocks[l].bins <= 128 && (blocks[l].bins == 0 || blocks[l].w_pe),
                   CF_ERR_UNSUPPORTED, "cf_forward: block %lld: value bins outside 0..128 or without a projection",
                   (long long)l);
    return CF_OK;
}

}  // namespace

extern "C" int64_t cf_forward_workspace(const cf_forward_args *f, const cf_forward_block *blocks)
{
    if (check_args(f, blocks)) return -1;
    Buffers b;
    return carve(*f, blocks, nullptr, b);
}

extern "C" int64_t cf_forward_staged(const cf_forward_args *f, const cf_forward_block *blocks)
{
    if (check_args(f, blocks)) return -1;
    int64_t count = 0;
    for (int64_t l = 0; l < f->layers; l++) count += staged_block(*f, blocks[l]);
    return count;
}

extern "C" int cf_forward(const cf_forward_args *f_, const cf_forward_block *blocks, void *workspace,
                          int64_t workspace_bytes, void *stream)
{
    int rc = check_args(f_, blocks);
    if (rc) return rc;
    const cf_forward_args &f = *f_;
    Buffers b;
    const int64_t need = carve(f, blocks, (char *)workspace, b);
    CF_REQUIRE(workspace && workspace_bytes >= need, CF_ERR_INVALID_ARGUMENT,
               "cf_forward: workspace of %lld bytes needed", (long long)need);
    CF_REQUIRE(f.x && f.pos && f.tvecs && f.batch && f.atom_start && f.edge_start && f.edges && f.e_start && f.pairs &&
                   f.out && (f.targets == 0 || (f.w_last && (f.hidden == 0 || f.w_head))),
               CF_ERR_INVALID_ARGUMENT, "cf_forward: null pointer");
    const int64_t N = f.N, E = f.E, U = (N + E) / 2, W = f.width, H = f.H, D = W / H;
    const bool adaptive_any = f.adaptive != 0;
    const bool rows = use_rows(f);
    if (rows) {
        for (int64_t first = 0; first < f.layers; first += PACK_BLOCKS) {
            PackArgs a{};
            a.blocks = (int)(f.layers - first < PACK_BLOCKS ? f.layers - first : PACK_BLOCKS);
            for (int i = 0; i < a.blocks; i++) {
                const cf_forward_block &p = blocks[first + i];
                a.block[i] = PackSource{p.wo, p.w1, p.w2, p.wq, p.wk, p.wv};
            }
            a.packed = b.packed + first * SPLIT_BLOCK;
            if (first > 0) {
                if ((rc = launch_forward_prologue(a, PrologueArgs{}, (hipStream_t)stream))) return rc;
                continue;
            }
            if (f.w_embed) {
                a.w_embed = f.w_embed;
                a.embed_width = (int)f.embed_width;
                a.packed_embed = b.packed + f.layers * SPLIT_BLOCK;
            }
            a.zero = b.counters;
            a.words = b.words;
            const PrologueArgs g{f.B, E, f.atom_start, f.edge_start, f.pos, f.tvecs, b.rpos, b.vcell, b.recip, b.rvlen, nullptr};
            if ((rc = launch_forward_prologue(a, g, (hipStream_t)stream))) return rc;
        }
    } else {
        if ((rc = cf_lattice_geometry(f.tvecs, f.B, nullptr, nullptr, b.rvlen, stream))) return rc;
        if ((rc = cf_edge_index(f.atom_start, f.edge_start, f.B, E, f.pos, nullptr, b.rpos, stream))) return rc;
    }
    if (b.kr && (rc = cf_kr_base(b.rpos, b.recip, f.batch, f.edges, E, b.kr, stream))) return rc;
    const cf_forward_block *staged = nullptr;      // the block whose grid the rings in b.rings hold
    int64_t units_until = 0;                       // blocks whose units are in b.units and whose projections are packed
    const float *x = f.x;
    int side = 0;
    if (rows) {
        RowsArgs r{};
        r.N = N; r.H = (int)H; r.x = f.x;
        head_of(r, f, blocks[0], b, 0);
        if (f.w_embed) {
            r.packed_embed = b.packed + f.layers * SPLIT_BLOCK; r.b_embed = f.b_embed; r.embed_width = (int)f.embed_width;
            r.y = b.x[1];
            x = b.x[1];
        }
        if ((rc = launch_block_rows(r, (hipStream_t)stream))) return rc;
    }
    for (int64_t l = 0; l < f.layers; l++) {
        const cf_forward_block &p = blocks[l];
        if (!rows && (rc = cf_linear_rows(x, N, W, p.wq, p.wk, p.wv, 3, W, p.b_in, nullptr, 0, b.q, b.k, b.v, stream)))
            return rc;
        if (!rows && (rc = cf_gauss_exponents(b.q, p.w_pos, p.gauss_scale, N, H, D, p.normalize, f.update_stats, p.positive_func,
                                     (float)p.beta, (float)p.lower_bound, (float)p.coef, (float)p.q_scale, b.stats,
                                     b.stats_bytes, nullptr, b.a, b.qs, stream)))
            return rc;
        const float *rvlen = adaptive_any && p.cutoff != 0.0 ? b.rvlen : nullptr;
        const bool adaptive = rvlen != nullptr;
        const bool split = p.coef_reci != 0.0;                  // real space: the first half of the heads
        const int64_t HR = split ? H / 2 : H;
        if (staged_block(f, p)) {
            const float cutoff = adaptive ? (float)p.cutoff : 0.0f;
            // (blocks of more pairs than fit at once stage slice by slice, each for itself)
            const int64_t slice = infer_slice(U, adaptive, f.unit_limit_bytes);
            const float *w[INFER_WEIGHT_BLOCKS];
            int bins[INFER_WEIGHT_BLOCKS], count = 0;
            bool stage = slice < U;
            if (l >= units_until) {
                // units for this block and those behind it that share them, their projections packed alongside
                stage = true;
                for (units_until = l; units_until < f.layers && count < INFER_WEIGHT_BLOCKS; units_until++, count++) {
                    const cf_forward_block &o = blocks[units_until];
                    if (!staged_block(f, o) || o.weakest != p.weakest || boxes_of(f, o) != adaptive ||
                        (adaptive && o.cutoff != p.cutoff) || real_heads(f, o) != HR)
                        break;
                    w[count] = o.w_pe;
                    bins[count] = (int)o.bins;
                }
            }
            for (int64_t before = 0; before < U && !rc; before += slice, count = 0) {
                const int64_t here = before + slice < U ? slice : U - before;
                if (stage && (rc = launch_infer_stage(b.rpos, f.tvecs, rvlen, f.pairs, U, before, here, p.weakest, cutoff,
                                                      (int)f.lattice_range, (int)f.minimum_range, b.units, count, w, bins, HR,
                                                      D, b.weights + l * b.weight_bytes, b.weight_bytes, (hipStream_t)stream)))
                    return rc;
                rc = launch_real_enc_infer(b.a, b.rpos, f.tvecs, f.pairs, U, before, here, HR, p.bins, D, p.dist_max, p.wscale,
                                           b.weights + l * b.weight_bytes, rvlen, cutoff, (int)f.lattice_range,
                                           (int)f.minimum_range, p.weakest, b.units, b.z, b.val, (hipStream_t)stream);
            }
        } else if (p.bins > 0 && b.rings && (!adaptive || (f.adaptive_rings && HR <= 8 && adaptive_rings_pay(U)))) {
            if (!staged || staged->bins != p.bins || staged->dist_max != p.dist_max || staged->wscale != p.wscale ||
                staged->weakest != p.weakest) {
                if ((rc = cf_real_enc_ring_stage(b.rpos, f.tvecs, f.pairs, U, p.bins, p.dist_max, p.wscale,
                                                 f.lattice_range, p.weakest, b.rings, stream)))
                    return rc;
                staged = &p;
            }
            rc = cf_real_enc_fwd_rings(b.a, adaptive ? b.rpos : nullptr, adaptive ? f.tvecs : nullptr,
                                       adaptive ? f.batch : nullptr, f.edges, f.pairs, U, N, HR, E, p.bins, D, p.dist_max,
                                       p.wscale, p.w_pe, rvlen, p.cutoff, f.lattice_range, f.minimum_range, b.rings,
                                       b.flags, b.flag_bytes, b.z, b.val, stream);
        } else {
            rc = cf_real_enc_fwd(b.a, b.rpos, f.tvecs, f.batch, f.edges, N, HR, E, f.B, p.bins, p.bins > 0 ? D : 0,
                                 p.dist_max, p.wscale, p.bins > 0 ? p.w_pe : nullptr, p.bins > 0 ? 1 : 0, rvlen,
                                 adaptive ? p.cutoff : 0.0, f.lattice_range, f.minimum_range, f.pairs, U, f.sched, b.z,
                                 p.bins > 0 ? b.val : nullptr, stream);
        }
        if (rc) return rc;
        if (split && (rc = cf_reci_enc_fwd(b.a + N * HR, b.kr, b.recip, b.vcell, f.batch, f.e_start, N, HR, E,
                                           (int)f.lattice_range, b.z + E * HR, b.sumexp, stream)))
            return rc;
        const float *val = p.bins > 0 ? b.val : nullptr;
        rc = b.prob ? cf_fused_dpa_fwd(b.qs, b.k, b.v, b.z, val, f.edges, f.e_start, N, H, E, D, D, b.prob, b.att, stream)
                    : launch_dpa_inference(b.qs, b.k, b.v, b.z, split ? E * HR : 0, val, f.edges, f.e_start, N, H, E, D,
                                           b.att, (hipStream_t)stream);
        if (rc) return rc;
        float *y = f.targets == 0 && l + 1 == f.layers ? f.out : b.x[side];
        if (rows) {
            RowsArgs r{};
            r.N = N; r.H = (int)H; r.att = b.att; r.x = x; r.y = y;
            r.packed_tail = b.packed + l * SPLIT_BLOCK; r.bo = p.bo; r.b1 = p.b1; r.b2 = p.b2;
            if (l + 1 < f.layers) head_of(r, f, blocks[l + 1], b, l + 1);
            if ((rc = launch_block_rows(r, (hipStream_t)stream))) return rc;
            x = y;
            side ^= 1;
            continue;
        }
        if ((rc = cf_linear_rows(b.att, N, W, p.wo, nullptr, nullptr, 1, W, p.bo, x, 0, b.qs, nullptr, nullptr, stream)))
            return rc;                              // (the scaled query is spent: its buffer takes the sum)
        if ((rc = cf_linear_rows(b.qs, N, W, p.w1, nullptr, nullptr, 1, f.ff, p.b1, nullptr, 1, b.h, nullptr, nullptr,
                                 stream)))
            return rc;
        if ((rc = cf_linear_rows(b.h, N, f.ff, p.w2, nullptr, nullptr, 1, W, p.b2, b.qs, 0, y, nullptr, nullptr, stream)))
            return rc;
        x = y;
        side ^= 1;
    }
    if (f.targets == 0) return CF_OK;
    if (pool_head_served(W, f.hidden)) {
        const PoolHeadArgs h{x, f.atom_start, f.w_head, f.b_head, f.w_last, f.b_last, f.hidden, f.targets, f.out};
        return launch_pool_head(h, f.B, (hipStream_t)stream);
    }
    if ((rc = cf_irregular_mean_fwd(x, f.atom_start, f.B, W, b.pooled, stream))) return rc;
    const float *top = b.pooled;
    int64_t top_width = W;
    if (f.hidden > 0) {
        if ((rc = cf_linear_rows(b.pooled, f.B, W, f.w_head, nullptr, nullptr, 1, f.hidden, f.b_head, nullptr, 1, b.hidden,
                                 nullptr, nullptr, stream)))
            return rc;
        top = b.hidden;
        top_width = f.hidden;
    }
    return cf_linear_rows(top, f.B, top_width, f.w_last, nullptr, nullptr, 1, f.targets, f.b_last, nullptr, 0, f.out,
                          nullptr, nullptr, stream);
}
