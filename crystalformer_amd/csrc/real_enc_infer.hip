// Real-space periodic encoding of an inference forward: what the kernels of real_enc_mfma.hip and real_enc_ring.hip compute,
// without what a training step's order of summation forbids.  Same unit of work (an unordered atom pair, 16 weight columns:
// 8 heads of i, 8 of j), same rounds of eight units a work-group, same translation sets, same 2^-40 bound on what is left out.
//
// infer_stage_kernel, once per geometry: the translations of every pair that can weigh more than 2^-40 of the leading one
// under the weakest exponent any block can have, ordered by d^2 (in classes), and what a block needs to know of the pair in
// 32 bytes.  real_enc_infer_kernel, once per block: weights, Gaussians, projection.
//
// The pair and ring kernels are bound by the issue of vector and fp32 matrix instructions, which share a SIMD's slots:
// v_mfma_f32_16x16x4_f32 takes 32 cycles in which no vector instruction runs (measured: 32.2 alone, 57.0 beside eight
// v_fma), v_mfma_f32_16x16x16_f16 16 that hide behind them (17.2 alone, 33.7 beside the same eight).  So here
//   * both factors of a matrix product are split in two halves of 11 bits, x 2^15 = hi + lo, and all four products
//     summed in fp32: 22 bits and a sign of each factor.  A split costs two instructions a value.  Weights and Gaussians,
//     none above 1, share one fixed scale: below 2^-17 a factor is off by up to 2^-40, the bound on what is left out;
//   * a translation enters only if its weight exceeds 2^-40 of the leading one in some column, by the block's own
//     exponents (a prefix of the order), and a 16-bin tile only if weight x Gaussian can exceed 2^-40: 17 translations and
//     4.5 tiles of 16 a pair with r0 = 1.4 A where the others evaluate 32 and 16 of 4, 64 and 10 where 98 and 47 with 3 A;
//   * square roots, column lookups and tile tests are made for these only, lane = translation;
//   * nothing about the pair passes through vector registers: its 32 bytes are scalar loads.
// What bounds a block now is the issue of vector instructions: 851 a pair at the largest (52 of them matrix ones) take 86 % of the
// slots, 339 a pair with r0 = 1.4 A in the cube half of them, the rest going on the launch's start, its last round and waits.
// Measured, pair and ring kernels -> this, a block: 28 thousand pairs in the fixed cube 43.5 -> 33.8 us, in boxes 45.4 and 9.4 for
// the lists -> 38.1, 147 thousand (mean of seven blocks) 440 and 15 -> 276, 958 thousand 3060 -> 1540.
//
// Lane roles of the accumulation (q = lane / 16, c = lane % 16): lane (q, c) holds translations 4 q .. 4 q + 3 of a group of
// 16: column c's weights (B operand) and the Gaussians of bin 16 m + c of every tile m in reach (A operand).  Projection
// v = W_h S: normalised column sums exchanged through LDS, 16 bytes at a time, wavefront w multiplies head w's matrix
// (split, scaled by a power of two per row, in registers) with that head's 16 columns.
#include "real_enc_infer.h"
#include "real_enc_pair.h"
#include "split_f16.h"

namespace {

using namespace cf;
using namespace cfpair;

constexpr float SPLIT = 32768.0f;           // values up to 1 are split scaled by it: 22 bits down to 2^-17, off by up to 2^-40 below
constexpr float PAD_D2 = 1e30f;             // d^2 of a slot without a translation: weight 0 and Gaussian 0
constexpr float LEAST_A2 = -1e-25f;         // no decay slower: 1 for every real distance, 0 for PAD_D2
constexpr int CLASSES = 8;                  // of d^2: seven of equal width and one for what lies beyond
constexpr int MOST_STAGED = 832;            // of a pair (fewer than 16 x 64: a lane's share of a class is counted in four bits)
constexpr float CLASSED = 0.55f;            // share of the staged range that the seven cover

// Smallest and largest by the bits: of floats >= 0 the signed order is theirs, of floats < 0 it is turned round.  (As
// floats every step costs a canonicalising instruction and a move beside the one on the DPP path.  A NaN has the largest
// bits among the first and is passed over among the second.)
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ int dpp_min(int v)
{
    return min(v, __builtin_amdgcn_update_dpp(0x7FFFFFFF, v, CTRL, ROW_MASK, 0xF, false));
}
__device__ __forceinline__ float row16_max_negative(float x)
{
    int v = __float_as_int(x);
    v = dpp_min<DPP_QUAD_1032, 0xF>(v);
    v = dpp_min<DPP_QUAD_2301, 0xF>(v);
    v = dpp_min<DPP_ROW_ROR4, 0xF>(v);
    v = dpp_min<DPP_ROW_ROR8, 0xF>(v);
    return __int_as_float(v);
}
__device__ __forceinline__ float wave_min_positive(float x)
{
    int v = __float_as_int(x);
    v = dpp_min<DPP_QUAD_1032, 0xF>(v);
    v = dpp_min<DPP_QUAD_2301, 0xF>(v);
    v = dpp_min<DPP_ROW_ROR4, 0xF>(v);
    v = dpp_min<DPP_ROW_ROR8, 0xF>(v);
    v = dpp_min<DPP_ROW_BCAST15, 0xA>(v);
    v = dpp_min<DPP_ROW_BCAST31, 0xC>(v);
    return __int_as_float(__builtin_amdgcn_readlane(v, 63));
}

__device__ __forceinline__ int lanes_below(unsigned long long mask, int base)
{
    return __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, base));
}

// Where the column sums of a unit are exchanged: 16-byte pieces, head ^ unit so that a writer (one unit, lanes over
// heads) and a reader (one head, lanes over units) both cover all banks.
__device__ __forceinline__ int piece_at(int i, int q, int dir, int unit, int head)
{
    return (((i * 4 + q) * 2 + dir) * WPB + unit) * 8 + (head ^ unit);
}

// What a block needs of a pair.
struct __align__(32) InferUnit {
    unsigned e_ij, e_ji, i, j;
    int count;                              // staged translations (+ CUBE: of the cube only); -1: not staged, the blocks form them themselves
    float least, bound;                     // smallest d^2 staged; an upper bound of every column's smallest
    float keep2;                            // every column has the cube where log2(e) x its weakest exponent is below this
};
__device__ __forceinline__ float class_width(float limit, float least) { return (limit - least) * (CLASSED / (CLASSES - 1)); }
constexpr int CUBE = 1 << 30;
typedef const InferUnit __attribute__((address_space(4))) *InferUnitPtr;
// a scalar load (wave-uniform address of what an earlier launch or the host wrote)
typedef const float __attribute__((address_space(4))) *ConstFloat;
typedef const int64_t __attribute__((address_space(4))) *ConstLong;

// Pairs of a slice that exist.
__device__ __forceinline__ int64_t live_in_slice(const int64_t *live_U, int64_t before, int64_t U)
{
    return min(live_count(live_U, before + U) - before, U);
}

struct StageArgs {
    const float *rpos, *tvecs, *rvlen;
    const int64_t *pairs;                   // this slice's, as units, d2 and n
    int64_t U, before;                      // pairs of the slice, of the slices before it
    const int64_t *live_U;
    float weak_a, cutoff;
    int lattice_range, min_range, capacity;
    InferUnit *units;                       // (U)
    float *d2;                              // (U, capacity)
    unsigned short *n;                      // (U, capacity), n + 16 of the three axes, 5 bits each; null: every box is the cube
};

// The projections of up to WEIGHT_BLOCKS blocks as the blocks read them: per head and 16 rows, HALVES x {hi, lo} pieces of 16
// bytes a lane (rows scaled to 2^14 .. 2^15 and split), and behind all heads the rows' exponents.
constexpr int WEIGHT_BLOCKS = INFER_WEIGHT_BLOCKS;
struct WeightArgs {
    const float *w[WEIGHT_BLOCKS];
    int bins[WEIGHT_BLOCKS];
    int blocks, H, D, heads, DT;            // heads: H rounded up to a multiple of 8
    int64_t stride;                         // int4 per block
    int4_t *out;
};

__host__ __device__ constexpr int tiles_of(int64_t K) { return K <= 16 ? 1 : K <= 32 ? 2 : K <= 64 ? 4 : 8; }
__host__ __device__ constexpr int pieces_of(int NT) { return NT == 1 ? 2 : NT; }

template <int NT>
__device__ __forceinline__ void pack_projection(const WeightArgs &p, int l, int head, int dt, int lane)
{
    constexpr int PIECES = pieces_of(NT);
    const int q = lane >> 4, c = lane & 15, d = 16 * dt + c, K = p.bins[l];
    float zero = 0.f;
    asm volatile("" : "+s"(zero));
    float w[4 * NT], top = 0.f;
#pragma unroll
    for (int s = 0; s < 4 * NT; s++) {
        const int k = proj_bin(s, q);
        w[s] = head < p.H && d < p.D && k < K ? p.w[l][((int64_t)head * p.D + d) * K + k] : 0.f;
        top = fmaxf(top, fabsf(w[s]));
    }
    const int e = __builtin_amdgcn_frexp_expf(rows_max(top));    // (0 for 0, infinity and NaN)
    int4_t piece[PIECES];
    if (NT == 1) piece[0] = piece[PIECES - 1] = int4_t{0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < 4 * NT; s += 2) {
        const Split2 y = split2(ldexpf(w[s], 15 - e), ldexpf(w[s + 1], 15 - e), 1.0f, zero);
        piece[s / 8 * 2][s / 2 % 4] = y.hi;
        piece[s / 8 * 2 + 1][s / 2 % 4] = y.lo;
    }
    int4_t *out = p.out + l * p.stride;
#pragma unroll
    for (int i = 0; i < PIECES; i++) out[((head * p.DT + dt) * PIECES + i) * WAVE + lane] = piece[i];
    // (results are scaled by 2^15 for the row and 2^15 for the sums)
    if (lane < 16) reinterpret_cast<int *>(out + p.heads * p.DT * PIECES * WAVE)[(head * p.DT + dt) * 16 + lane] = e - 30;
}

constexpr int STAGE_WAVES = 4;

// A wavefront per unit, the next unit's cell requested ahead.  LDS per wavefront: capacity + 64 distances and packed n, and 1 KB of places.
// The first work-groups pack the blocks' projections instead.
__global__ __launch_bounds__(STAGE_WAVES * 64) void infer_stage_kernel(StageArgs p, WeightArgs w)
{
    extern __shared__ __align__(16) float lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int packs = w.blocks * w.heads * w.DT, pack_groups = (packs + STAGE_WAVES - 1) / STAGE_WAVES;
    if ((int)blockIdx.x < pack_groups) {
        const int t = (int)blockIdx.x * STAGE_WAVES + wave;
        if (t >= packs) return;
        const int dt = t % w.DT, head = t / w.DT % w.heads, l = t / w.DT / w.heads;
        switch (tiles_of(w.bins[l])) {
            case 1: pack_projection<1>(w, l, head, dt, lane); break;
            case 2: pack_projection<2>(w, l, head, dt, lane); break;
            case 4: pack_projection<4>(w, l, head, dt, lane); break;
            default: pack_projection<8>(w, l, head, dt, lane); break;
        }
        return;
    }
    const int64_t U = live_in_slice(p.live_U, p.before, p.U);
    const int64_t waves = (int64_t)(gridDim.x - pack_groups) * STAGE_WAVES;
    const int64_t first = (int64_t)(blockIdx.x - pack_groups) * STAGE_WAVES + wave;
    if (first >= U) return;
    const int cap = p.capacity;
    float *cand_d2 = lds + wave * (p.n ? 3 : 2) * (cap + WAVE) / 2;
    unsigned short *cand_n = reinterpret_cast<unsigned short *>(cand_d2 + cap + WAVE);
    // (places of a class's next, a column a lane: behind all wavefronts' candidates)
    unsigned short *places = reinterpret_cast<unsigned short *>(lds + STAGE_WAVES * (p.n ? 3 : 2) * (cap + WAVE) / 2) +
                             wave * CLASSES * WAVE;
    struct Ids { int64_t e_ij, e_ji, i, j, n; };
    auto ids_of = [&](int64_t u_) -> Ids {
        const ConstLong d = (ConstLong)p.pairs + (u_ < U ? u_ : U - 1) * PAIR_FIELDS;
        return Ids{d[0], d[1], d[2], d[3], d[4]};
    };
    auto cell_of = [&](const Ids &d) -> Cell {
        const ConstFloat r = (ConstFloat)p.rpos + d.e_ij * 3, t = (ConstFloat)p.tvecs + d.n * 9;
        Cell c_;
        c_.rx = r[0];
        c_.ry = r[1];
        c_.rz = r[2];
#pragma unroll
        for (int x = 0; x < 9; x++) c_.t[x] = t[x];
        return c_;
    };
    BoxDims cube;
    const int lr = p.lattice_range, side = 2 * lr + 1;
    cube.U1 = cube.U2 = cube.U3 = lr;
    cube.S2 = cube.S3 = side;
    cube.plane = side * side;
    cube.T = side * cube.plane;
    cube.inv_plane = 1.0f / (float)cube.plane;
    cube.inv_S3 = 1.0f / (float)side;
    const bool small_cube = cube.T <= 2 * WAVE;
    float pre[2][3];                                             // the cube's translations, decoded once
#pragma unroll
    for (int ch = 0; ch < 2; ch++) {
        int n1, n2, n3;
        decode(cube, min(ch * WAVE + lane, cube.T - 1), n1, n2, n3);
        pre[ch][0] = (float)n1;
        pre[ch][1] = (float)n2;
        pre[ch][2] = (float)n3;
    }
    const float weak_a2 = fminf(p.weak_a * LOG2E, LEAST_A2);
    const float reach = -40.0f / weak_a2;
    // (columns never have less than the cube where the floor says so)
    const bool hold_cube = !p.n || p.min_range >= lr;
    Ids ids = ids_of(first), ids_next = ids_of(first + waves);
    Cell cell = cell_of(ids);
    for (int64_t u = first; u < U; u += waves) {
        const Cell cell_next = cell_of(ids_next);
        const Ids ids_next2 = ids_of(u + 2 * waves);
        BoxDims bx = cube;
        float keep2 = __builtin_inff();
        if (p.n) {
            // (an axis a lane)
            const float rv = p.rvlen[(unsigned)ids.n * 3u + min((unsigned)lane, 2u)];
            const float cut = p.cutoff < 0.f ? sqrtf(-0.5f / p.weak_a) * -p.cutoff : p.cutoff;
            const int R = range_axis(cut, rv, p.min_range);
            bx.U1 = __builtin_amdgcn_readlane(R, 0);
            bx.U2 = __builtin_amdgcn_readlane(R, 1);
            bx.U3 = __builtin_amdgcn_readlane(R, 2);
            bx.S2 = 2 * bx.U2 + 1;
            bx.S3 = 2 * bx.U3 + 1;
            bx.plane = bx.S2 * bx.S3;
            bx.T = (2 * bx.U1 + 1) * bx.plane;
            bx.inv_plane = 1.0f / (float)bx.plane;
            bx.inv_S3 = 1.0f / (float)bx.S3;
            // The exponent below which the rule's quotients stay clear (by 1e-3) of the next whole number on all axes:
            // its columns have the cube if the floor is the cube.  (Those near the line work the rule out.)
            const float top = fmaxf(readlane_f(rv, 0), fmaxf(readlane_f(rv, 1), readlane_f(rv, 2)));
            const float most = ((float)lr - 1.0e-3f) * (2.0f * PI_F) * __builtin_amdgcn_rcpf(top) - 0.01f;
            const bool cube_rule = p.min_range == lr && most > 0.f;
            if (p.cutoff < 0.f) {
                const float t = p.cutoff * __builtin_amdgcn_rcpf(most);
                keep2 = cube_rule ? -0.5f * LOG2E * t * t : -__builtin_inff();
            } else {
                keep2 = cube_rule && p.cutoff <= most ? __builtin_inff() : -__builtin_inff();
            }
        }
        const bool is_cube = bx.U1 == lr && bx.U2 == lr && bx.U3 == lr && small_cube;
        float d2c[2];
        float bound = cell.rx * cell.rx + cell.ry * cell.ry + cell.rz * cell.rz;
        if (small_cube) {
#pragma unroll
            for (int ch = 0; ch < 2; ch++) d2c[ch] = dist2(cell, pre[ch][0], pre[ch][1], pre[ch][2]);
            if (hold_cube) bound = wave_min_positive(fminf(d2c[0], d2c[1]));
        }
        const float limit = bound + reach;
        int count = 0;
        auto keep = [&](float d2, bool valid, float n1, float n2, float n3) {
            const bool alive = valid && !(d2 >= limit);          // (NaN is never beyond)
            const unsigned long long mask = __ballot(alive);
            const int at = lanes_below(mask, count);
            if (alive && at < cap + WAVE) {
                cand_d2[at] = d2;
                if (p.n) cand_n[at] = (unsigned short)(unsigned)(n1 + 32.0f * n2 + 1024.0f * n3 + (16.0f + 512.0f + 16384.0f));
            }
            count += __popcll(mask);
        };
        float least = bound;
        if (is_cube) {
#pragma unroll
            for (int ch = 0; ch < 2; ch++)
                if (ch * WAVE < bx.T)
                    keep(d2c[ch], ch * WAVE + lane < bx.T, pre[ch][0], pre[ch][1], pre[ch][2]);
            if (!hold_cube) least = wave_min_positive(fminf(d2c[0], d2c[1]));
        } else {
            // A lane has a place (two of the three numbers) and walks along the third axis, the one that leaves the fewest
            // steps of 64 places: 15 instructions a step.  (All three numbers of 64 consecutive translations, carried from
            // step to step, took 45: 958 thousand pairs with 132 of them staged 1030 us, so 915, with the ranking below 770.)
            const int S1 = 2 * bx.U1 + 1;
            const int s1 = ((bx.S2 * bx.S3 + 63) >> 6) * S1, s2 = ((S1 * bx.S3 + 63) >> 6) * bx.S2,
                      s3 = ((S1 * bx.S2 + 63) >> 6) * bx.S3;
            const int along = s1 <= s2 && s1 <= s3 ? 0 : s2 <= s3 ? 1 : 2;
            const bool x1 = along == 0, x2 = along == 1;         // the lanes' axes: (2, 3), (1, 3), (1, 2)
            const int Ua = x1 ? bx.U2 : bx.U1, Ub = x1 || x2 ? bx.U3 : bx.U2, Uc = x1 ? bx.U1 : x2 ? bx.U2 : bx.U3;
            const int Sb = 2 * Ub + 1, plane = (2 * Ua + 1) * Sb;
            const int code_a = x1 ? 32 : 1, code_b = x1 || x2 ? 1024 : 32, code_c = x1 ? 1 : x2 ? 32 : 1024;
            float ta[3], tb[3], tc[3];
#pragma unroll
            for (int i = 0; i < 3; i++) {
                ta[i] = x1 ? cell.t[3 + i] : cell.t[i];
                tb[i] = x1 || x2 ? cell.t[6 + i] : cell.t[3 + i];
                tc[i] = x1 ? cell.t[i] : x2 ? cell.t[3 + i] : cell.t[6 + i];
            }
            const float inv_Sb = __builtin_amdgcn_rcpf((float)Sb);
            float closest = PAD_D2;
            for (int p0 = 0; p0 < plane; p0 += WAVE) {
                const bool valid = p0 + lane < plane;
                const unsigned long long there = __ballot(valid);
                const int at_place = min(p0 + lane, plane - 1);
                const int ia = (int)(((float)at_place + 0.5f) * inv_Sb), ib = at_place - ia * Sb;
                const float na = (float)(ia - Ua), nb = (float)(ib - Ub);
                const float bx_ = __builtin_fmaf(na, ta[0], __builtin_fmaf(nb, tb[0], cell.rx));
                const float by_ = __builtin_fmaf(na, ta[1], __builtin_fmaf(nb, tb[1], cell.ry));
                const float bz_ = __builtin_fmaf(na, ta[2], __builtin_fmaf(nb, tb[2], cell.rz));
                int code = (ia - Ua) * code_a + (ib - Ub) * code_b - Uc * code_c + 16 * (1 + 32 + 1024);
                float nc = (float)-Uc;
                int here = __float_as_int(PAD_D2);               // (see dpp_min)
                for (int c_ = -Uc; c_ <= Uc; c_++) {
                    const float vx = __builtin_fmaf(nc, tc[0], bx_), vy = __builtin_fmaf(nc, tc[1], by_),
                                vz = __builtin_fmaf(nc, tc[2], bz_);
                    const float d2 = __builtin_fmaf(vx, vx, __builtin_fmaf(vy, vy, vz * vz));
                    here = min(here, __float_as_int(d2));
                    const bool alive = !(d2 >= limit);           // (NaN is never beyond)
                    const unsigned long long mask = __ballot(alive) & there;
                    if (count <= cap) {                          // (more: the unit isn't staged)
                        const int at = lanes_below(mask, count);
                        if (alive && valid) {
                            cand_d2[at] = d2;
                            cand_n[at] = (unsigned short)code;
                        }
                    }
                    count += __popcll(mask);
                    nc += 1.0f;
                    code += code_c;
                }
                closest = fminf(closest, valid ? __int_as_float(here) : PAD_D2);
            }
            least = fminf(bound, wave_min_positive(closest));
        }
        const bool fits = count <= cap && max(bx.U1, max(bx.U2, bx.U3)) <= 15;
        wave_mem_sync();
        if (fits) {
            const float scale = __builtin_amdgcn_rcpf(class_width(limit, least));
            auto class_of = [&](float d2) -> int { return min(max((int)((d2 - least) * scale), 0), CLASSES - 1); };
            if (count <= WAVE) {
                const bool held = lane < count;
                const float d2 = held ? cand_d2[lane] : 0.f;
                int at = lane;
                if (count > 16) {
                    // ranked in classes by two packed prefix sums over the lanes (a byte a class)
                    const int cls = class_of(d2), shift = 8 * (cls & 3);
                    const int one = held ? 1 << shift : 0;
                    const int low = cls < 4 ? one : 0, high = cls < 4 ? 0 : one;
                    const int upto0 = wave_inclusive_scan_i(low), upto1 = wave_inclusive_scan_i(high);
                    const unsigned t0 = (unsigned)__builtin_amdgcn_readlane(upto0, 63),
                                   t1 = (unsigned)__builtin_amdgcn_readlane(upto1, 63);
                    const unsigned b0 = (t0 << 8) + (t0 << 16) + (t0 << 24), all0 = (t0 * 0x01010101u) >> 24;
                    const unsigned b1 = (t1 << 8) + (t1 << 16) + (t1 << 24) + all0 * 0x01010101u;
                    const unsigned r = (cls < 4 ? (unsigned)(upto0 - low) : (unsigned)(upto1 - high)) + (cls < 4 ? b0 : b1);
                    at = (int)(r >> shift) & 0xFF;
                }
                if (held) {
                    p.d2[u * cap + at] = d2;
                    if (p.n) p.n[u * cap + at] = cand_n[lane];
                }
            } else {
                // More: each lane counts its own (lane, lane + 64, ..) in four bits a class, one prefix sum over the lanes
                // in 16 bits a class says where its first of every class goes, and it counts on from there in LDS.  (A prefix
                // sum for every 64: 60 instructions each where this takes 25.)
                unsigned mine = 0;
                for (int b = lane; b < count; b += WAVE) mine += 1u << (4 * class_of(cand_d2[b]));
                int own[4], upto[4];                             // classes k and k + 4
                unsigned total[CLASSES], start = 0;
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    own[k] = (int)((mine >> (4 * k)) & 0x000F000Fu);
                    upto[k] = wave_inclusive_scan_i(own[k]);
                    const unsigned t = (unsigned)__builtin_amdgcn_readlane(upto[k], 63);
                    total[k] = t & 0xFFFFu;
                    total[k + 4] = t >> 16;
                }
                unsigned first_[CLASSES];
#pragma unroll
                for (int k = 0; k < CLASSES; k++) {
                    first_[k] = start;
                    start += total[k];
                }
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const unsigned from = (unsigned)(upto[k] - own[k]) + (first_[k] | first_[k + 4] << 16);
                    places[k * WAVE + lane] = (unsigned short)from;
                    places[(k + 4) * WAVE + lane] = (unsigned short)(from >> 16);
                }
                for (int b = lane; b < count; b += WAVE) {
                    const float d2 = cand_d2[b];
                    unsigned short *next = places + class_of(d2) * WAVE + lane;
                    const int at = *next;
                    *next = (unsigned short)(at + 1);
                    p.d2[u * cap + at] = d2;
                    if (p.n) p.n[u * cap + at] = cand_n[b];
                }
            }
        }
        if (lane == 0) {
            InferUnit h;
            h.e_ij = (unsigned)ids.e_ij;
            h.e_ji = (unsigned)ids.e_ji;
            h.i = (unsigned)ids.i;
            h.j = (unsigned)ids.j;
            h.count = fits ? count | (is_cube ? CUBE : 0) : -1;
            h.least = least;
            h.bound = bound;
            h.keep2 = keep2;
            p.units[u] = h;
        }
        wave_mem_sync();
        cell = cell_next;
        ids = ids_next;
        ids_next = ids_next2;
    }
}

struct InferArgs {
    const float *a_ik, *rpos, *tvecs, *rvlen;
    const int64_t *pairs;
    const InferUnit *units;
    const float *d2;
    const unsigned short *n;
    const int4_t *weights;                  // this block's, see WeightArgs
    float *z, *v;
    int64_t U, before;                      // as in StageArgs
    const int64_t *live_U;
    int H, D, heads, capacity, lattice_range, min_range, rounds_per_group;
    float cutoff, bin_step, s_scale, inv_bin_step;
    float reach;                            // how far above its bound a unit's d^2 were staged
};

// A work-group is a round: eight units of one group of eight heads.  (Rounds dealt to persistent work-groups left the
// younger of a CU's two to finish alone.)
template <int NT, int DT, bool BOXES>
__global__ __launch_bounds__(512, DT > 1 || NT > 4 ? 6 : 8) void real_enc_infer_kernel(InferArgs x)
{
    constexpr int HALVES = NT == 1 ? 1 : NT / 2;                 // matrix instructions of 32 (or 16) bins
    constexpr int PIECES = pieces_of(NT), WORDS = (BOXES ? 3 : 2) * WAVE;
    __shared__ int4_t xbuf[NT * 4 * 2 * WPB * 8];
    __shared__ __align__(16) float records[WPB][WORDS];
    __shared__ unsigned meta[WPB][2];
    constexpr unsigned NO_EDGE = ~0u;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = lane >> 4, c = lane & 15;
    const int H = x.H, cap = x.capacity;
    const int hg = x.heads == 8 ? 0 : (int)blockIdx.x / x.rounds_per_group;
    const int64_t U = live_in_slice(x.live_U, x.before, x.U);
    const int64_t first = (int64_t)((int)blockIdx.x - hg * x.rounds_per_group) * WPB;
    if (first >= U) return;
    const int64_t u = first + wave < U ? first + wave : first;
    const InferUnitPtr unit = (InferUnitPtr)x.units + u;
    const int staged = unit->count;
    const unsigned e_ij = unit->e_ij, e_ji = unit->e_ji;
    const float least = unit->least, bound = unit->bound;
    const bool unit_on = first + wave < U;
    const int h = hg * 8 + (c & 7);
    const unsigned h_ = (unsigned)min(h, H - 1);
    unsigned i_H = unit->i * (unsigned)H, j_H = unit->j * (unsigned)H;
    asm volatile("" : "+s"(i_H), "+s"(j_H));                    // (else a lane fetches its own of the two)
    const float a_in = x.a_ik[(c < 8 ? i_H : j_H) + h_];
    float d2_here = x.d2[u * cap + lane];
    int n_here = BOXES ? x.n[u * cap + lane] : 0;
    float *rec_d2 = records[wave], *rec_s = rec_d2 + WAVE;
    int *rec_cols = reinterpret_cast<int *>(rec_s + WAVE);       // (BOXES)
    float zero = 0.f;
    asm volatile("" : "+v"(zero));          // (a split reads one scalar register already)
    const bool col_on = unit_on && h < H && (c < 8 || e_ji != e_ij);
    const float a = col_on ? a_in : -1.0f;
    const float a2 = fminf(a * LOG2E, LEAST_A2);
    // A translation beyond `limit` weighs less than 2^-40 of the leading one in every column (the weakest decay counts).
    const float a2_weak = row16_max_negative(col_on ? a2 : -3.0e38f);
    const float limit = bound - 40.0f * __builtin_amdgcn_rcpf(a2_weak);
    float dref = least;                                          // this column's reference: weights are exp(a (d^2 - dref))

    // adaptive boxes, where not every column has the cube: which columns a translation counts for (lane (q, c) works out
    // axis q of column c)
    bool all = true, same_box = true;                            // every staged translation counts / in every column
    int U1 = 0, U2 = 0, U3 = 0;                                  // union over the columns
    ColumnBoxes cbox{0, 0, 0};
    int count = staged & (CUBE - 1);
    const bool formed = BOXES && staged < 0;                     // too many to stage: formed here, in no order
    if (BOXES) {
        // (columns below keep2 have the cube)
        all = staged >= CUBE && __builtin_amdgcn_readfirstlane((int)(a2_weak <= unit->keep2)) != 0;
        if (!all) {
            const int64_t crystal = ((ConstLong)x.pairs)[u * PAIR_FIELDS + 4];
            const ConstFloat rv = (ConstFloat)x.rvlen + crystal * 3;
            const float rvl[3] = {rv[0], rv[1], rv[2]};
            const int Rq = column_axis_range(a, x.cutoff, rvl, x.lattice_range, x.min_range, q, col_on);
            const int Uq = row16_max_i(Rq);
            U1 = __builtin_amdgcn_readlane(Uq, 0);
            U2 = __builtin_amdgcn_readlane(Uq, 16);
            U3 = __builtin_amdgcn_readlane(Uq, 32);
            same_box = __ballot(col_on && q < 3 && Rq != Uq) == 0ull;
            BoxDims bx;
            bx.U1 = U1;
            bx.U2 = U2;
            bx.U3 = U3;
            // (lane l for n = l - 16 where staged, for |n| = l + 1 where not)
            cbox = column_boxes_rows(Rq, bx, formed ? lane : abs(lane - 16) - 1);
            if (!formed && lane == 16) cbox.m1 = cbox.m2 = cbox.m3 = 0xFFFF;
            if (formed) count = (2 * U1 + 1) * (2 * U2 + 1) * (2 * U3 + 1);
        }
    }
    // translations b0 .. b0 + 63 of the unit as seen by the columns: d^2 (PAD_D2 where none has it) and column bits
    auto seen = [&](int b0, float d2, int packed, int &bits) -> float {
        bits = 0xFFFF;
        if (BOXES && !all) {
            if (formed) {
                BoxDims bx;
                bx.U1 = U1;
                bx.U2 = U2;
                bx.U3 = U3;
                asm volatile("" : "+s"(bx.U1), "+s"(bx.U2), "+s"(bx.U3));        // (worked out here, where it is rare)
                bx.S2 = 2 * bx.U2 + 1;
                bx.S3 = 2 * bx.U3 + 1;
                bx.plane = bx.S2 * bx.S3;
                bx.inv_plane = __builtin_amdgcn_rcpf((float)bx.plane);
                bx.inv_S3 = __builtin_amdgcn_rcpf((float)bx.S3);
                int n1, n2, n3;
                decode(bx, min(b0 + lane, count - 1), n1, n2, n3);
                const ConstFloat r = (ConstFloat)x.rpos + (int64_t)e_ij * 3;
                const ConstFloat t = (ConstFloat)x.tvecs + ((ConstLong)x.pairs)[u * PAIR_FIELDS + 4] * 9;
                Cell cell;
                cell.rx = r[0];
                cell.ry = r[1];
                cell.rz = r[2];
#pragma unroll
                for (int i = 0; i < 9; i++) cell.t[i] = t[i];
                d2 = dist2(cell, (float)n1, (float)n2, (float)n3);
                bits = column_bits(cbox, n1, n2, n3);
            } else {
                bits = __shfl(cbox.m1, packed & 31, WAVE) & __shfl(cbox.m2, (packed >> 5) & 31, WAVE) &
                       __shfl(cbox.m3, packed >> 10, WAVE);
            }
            d2 = bits ? d2 : PAD_D2;
        }
        return b0 + lane < count ? d2 : PAD_D2;
    };
    if (BOXES && __builtin_amdgcn_readfirstlane((int)(bound > least))) {
        // One reference serves all columns unless a column's own smallest d^2 could lie so far above it that its weights
        // lose bits; then each column's own is looked for (at most `bound`).
        const float strong = -row16_min(col_on ? a2 : 0.f);
        if (__builtin_amdgcn_readfirstlane((int)!(strong * (bound - least) <= 6.0f))) {
            rec_d2[lane] = bound;                                // (lane c: column c)
#pragma unroll 1
            for (int b0 = 0; b0 < count; b0 += WAVE) {
                const int at = formed ? 0 : min(b0 + lane, count - 1);
                int bits;
                const float d2 = seen(b0, x.d2[u * cap + at], x.n[u * cap + at], bits);
#pragma unroll 1
                for (int col = 0; col < 16; col++) {
                    const float mc = wave_min_positive((bits >> col) & 1 ? d2 : PAD_D2);
                    if (lane == col) rec_d2[lane] = fminf(rec_d2[lane], mc);
                }
            }
            wave_mem_sync();
            dref = rec_d2[c];
            wave_mem_sync();
        }
    }

    float ck[NT];
#pragma unroll
    for (int m = 0; m < NT; m++) ck[m] = x.bin_step * ((float)(c + 1) + (float)(16 * m));
    float4_t acc[NT];
#pragma unroll
    for (int m = 0; m < NT; m++) acc[m] = float4_t{0.f, 0.f, 0.f, 0.f};
    float sum = 0.f;
    if (!unit_on) count = 0;
    for (int b0 = 0; b0 < count; b0 += WAVE) {
        // (more than 16 staged ones are ordered by class: where this one's begins beyond the limit, all that follow are)
        if (b0 > 0 && !formed) {
            float far_ = bound + x.reach;
            asm volatile("" : "+v"(far_));                       // (worked out here, not before the first 64)
            const float edge = fminf(d2_here - class_width(far_, least), least + (far_ - least) * CLASSED);
            if (__builtin_amdgcn_readfirstlane((int)(edge > limit))) break;
        }
        int bits;
        float d2 = seen(b0, d2_here, n_here, bits);
        if (b0 + WAVE < count && !formed) {                      // the next 64 on their way
            const int at = min(b0 + WAVE + lane, count - 1);
            d2_here = x.d2[u * cap + at];
            if (BOXES) n_here = x.n[u * cap + at];
        }
        const float shift = a2 * dref;
        const unsigned long long alive = __ballot(!(d2 >= limit));
        if (alive == 0ull) continue;
        const int n = __popcll(alive);
        {
            // closed up (a lane nobody writes to gets 0), in order
            const int to = ((alive >> lane) & 1 ? lanes_below(alive, 0) : n + lane - lanes_below(alive, 0)) * 4;
            d2 = __int_as_float(__builtin_amdgcn_ds_permute(to, __float_as_int(d2)));
            if (BOXES && !same_box) bits = __builtin_amdgcn_ds_permute(to, bits);
            d2 = lane < n ? d2 : PAD_D2;
        }
        unsigned long long reach[NT];
        {
            const float s = sqrt_hw(d2) * x.s_scale;
            // (weight x Gaussian > 2^-40; the root of a negative number is NaN: no tile)
            const float win = sqrt_hw(40.0f + a2_weak * (d2 - bound)) * x.inv_bin_step;
            const float xb = s * x.inv_bin_step - 1.0f;
            const float hi = xb + win, lo = xb - win;
#pragma unroll
            for (int m = 0; m < NT; m++) reach[m] = __ballot(hi >= (float)(16 * m)) & __ballot(lo <= (float)(16 * m + 15));
            rec_d2[lane] = d2;
            rec_s[lane] = s;
            if (BOXES && !same_box) rec_cols[lane] = bits;
        }
        wave_mem_sync();
        const int groups = (n + 15) >> 4;
#pragma unroll 1
        for (int g = 0; g < groups; g++) {
            const float4_t d2v = *reinterpret_cast<const float4_t *>(rec_d2 + 16 * g + 4 * q);
            const float4_t sv = *reinterpret_cast<const float4_t *>(rec_s + 16 * g + 4 * q);
            float w[4];
#pragma unroll
            for (int r = 0; r < 4; r++) w[r] = exp2_hw(__builtin_fmaf(a2, d2v[r], -shift));
            if (BOXES && !same_box) {
                const int4_t cols = *reinterpret_cast<const int4_t *>(rec_cols + 16 * g + 4 * q);
#pragma unroll
                for (int r = 0; r < 4; r++)
                    w[r] = __int_as_float(__float_as_int(w[r]) & __builtin_amdgcn_sbfe(cols[r], (unsigned)c, 1));
            }
            sum += (w[0] + w[1]) + (w[2] + w[3]);
            const Split2 w01 = split2(w[0], w[1], SPLIT, zero), w23 = split2(w[2], w[3], SPLIT, zero);
            const int2_t wh = {w01.hi, w23.hi}, wl = {w01.lo, w23.lo};
#pragma unroll
            for (int m = 0; m < NT; m++) {
                if ((unsigned)reach[m] & 0xFFFFu) {                                       // wave-uniform
                    float gm[4];
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const float t = ck[m] - sv[r];
                        gm[r] = exp2_hw(-(t * t));
                    }
                    const Split2 g01 = split2(gm[0], gm[1], SPLIT, zero), g23 = split2(gm[2], gm[3], SPLIT, zero);
                    const int2_t gh = {g01.hi, g23.hi}, gl = {g01.lo, g23.lo};
                    acc[m] = mfma16(gl, wl, acc[m]);
                    acc[m] = mfma16(gl, wh, acc[m]);
                    acc[m] = mfma16(gh, wl, acc[m]);
                    acc[m] = mfma16(gh, wh, acc[m]);
                }
                reach[m] >>= 16;
            }
        }
        wave_mem_sync();
    }
    // this wavefront's head of the projection: its operands on their way
    const int hw = hg * 8 + wave;
    const int4_t *wp = x.weights + (int64_t)hw * DT * PIECES * WAVE + lane;
    int4_t W[DT][PIECES], wexp[DT];
#pragma unroll
    for (int dt = 0; dt < DT; dt++) {
#pragma unroll
        for (int i = 0; i < PIECES; i++) W[dt][i] = wp[(dt * PIECES + i) * WAVE];
        wexp[dt] = x.weights[(int64_t)x.heads * DT * PIECES * WAVE + (hw * DT + dt) * 4 + q];
    }
    sum = rows_sum(sum);
    const float inv = __builtin_amdgcn_rcpf(sum) * (1.0f / SPLIT);             // S / sum, scaled by 2^15 (acc: by 2^30)
    // epilogue: lane (q, c) holds S[16 m + 4 q + r][column c]
    {
        int hi[2 * NT], lo[2 * NT];
#pragma unroll
        for (int t = 0; t < 2 * NT; t++) {
            const Split2 s = split2(acc[t / 2][2 * (t & 1)], acc[t / 2][2 * (t & 1) + 1], inv, zero);
            hi[t] = s.hi;
            lo[t] = s.lo;
        }
        if (NT == 1) {
            xbuf[piece_at(0, q, c >> 3, wave, c & 7)] = int4_t{hi[0], hi[1], lo[0], lo[1]};
        } else {
#pragma unroll
            for (int i = 0; i < HALVES; i++) {
                xbuf[piece_at(2 * i, q, c >> 3, wave, c & 7)] = int4_t{hi[4 * i], hi[4 * i + 1], hi[4 * i + 2], hi[4 * i + 3]};
                xbuf[piece_at(2 * i + 1, q, c >> 3, wave, c & 7)] =
                    int4_t{lo[4 * i], lo[4 * i + 1], lo[4 * i + 2], lo[4 * i + 3]};
            }
        }
    }
    const unsigned row = 4u * (unsigned)H * (unsigned)x.D;       // bytes an edge of v
    if (lane == 0) {
        meta[wave][0] = unit_on ? e_ij * row : NO_EDGE;
        meta[wave][1] = unit_on && e_ji != e_ij ? e_ji * row : NO_EDGE;
    }
    unsigned z_ij = e_ij * (unsigned)H, z_ji = e_ji * (unsigned)H;
    asm volatile("" : "+s"(z_ij), "+s"(z_ji));
    if (col_on && q == 0)
        *reinterpret_cast<float *>(reinterpret_cast<char *>(x.z) + 4u * ((c < 8 ? z_ij : z_ji) + (unsigned)h)) =
            (log2_hw(sum) - __builtin_fmaf(a2, dref, -(a2 * dref))) * LN2 + dref * a;        // (the weights' shift is a2 dref rounded)
    __syncthreads();
    // head hw; column j of the product = direction j / 8 of unit j % 8
    const int unit_j = c & 7, dir_j = c >> 3;
    float4_t out[DT];
#pragma unroll
    for (int dt = 0; dt < DT; dt++) out[dt] = float4_t{0.f, 0.f, 0.f, 0.f};
    if (NT == 1) {
        const int4_t s = xbuf[piece_at(0, q, dir_j, unit_j, wave)];
        const int2_t sh = {s[0], s[1]}, sl = {s[2], s[3]};
#pragma unroll
        for (int dt = 0; dt < DT; dt++) {
            const int2_t h2 = {W[dt][0][0], W[dt][0][1]}, l2 = {W[dt][1][0], W[dt][1][1]};
            out[dt] = mfma16(l2, sl, out[dt]);
            out[dt] = mfma16(l2, sh, out[dt]);
            out[dt] = mfma16(h2, sl, out[dt]);
            out[dt] = mfma16(h2, sh, out[dt]);
        }
    } else {
#pragma unroll
        for (int i = 0; i < HALVES; i++) {
            const int4_t sh = xbuf[piece_at(2 * i, q, dir_j, unit_j, wave)];
            const int4_t sl = xbuf[piece_at(2 * i + 1, q, dir_j, unit_j, wave)];
#pragma unroll
            for (int dt = 0; dt < DT; dt++) {
                out[dt] = mfma32(W[dt][2 * i + 1], sl, out[dt]);
                out[dt] = mfma32(W[dt][2 * i + 1], sh, out[dt]);
                out[dt] = mfma32(W[dt][2 * i], sl, out[dt]);
                out[dt] = mfma32(W[dt][2 * i], sh, out[dt]);
            }
        }
    }
    const unsigned e_out = meta[unit_j][dir_j];
    if (e_out != NO_EDGE && hw < H) {
        const int D = x.D;
#pragma unroll
        for (int dt = 0; dt < DT; dt++) {
            const int dbase = 16 * dt + 4 * q;
            float *dst = reinterpret_cast<float *>(reinterpret_cast<char *>(x.v) + (e_out + 4u * (unsigned)(hw * D + dbase)));
            float4_t o;
#pragma unroll
            for (int r = 0; r < 4; r++) o[r] = ldexpf(out[dt][r], wexp[dt][r]);
            if (D == 16 * DT || dbase + 3 < D) {
                *reinterpret_cast<float4_t *>(dst) = o;
            } else {
#pragma unroll
                for (int r = 0; r < 3; r++)
                    if (dbase + r < D) dst[r] = o[r];
            }
        }
    }
}

// Entries a unit may have: all of a small fixed cube, else 832 (what leaves six staging work-groups a CU).  Units under the weakest
// exponent have 31 in the mean with r0 = 1.4 A, 230 with 3 A in small cells (an eighth above 512, two in a thousand above 832),
// 132 and none above 256 in large skewed ones.  The same whatever the batch: a unit that has
// more is formed by the blocks, in another order, and its bits must not depend on what else is in the batch, nor on the capacity
// of a graph that serves it.
constexpr int capacity_of(bool boxes) { return boxes ? MOST_STAGED : 128; }
constexpr int64_t bytes_a_unit(bool boxes) { return (int64_t)sizeof(InferUnit) + capacity_of(boxes) * (boxes ? 6 : 4); }

int64_t align256(int64_t x) { return (x + 255) & ~(int64_t)255; }

struct Carved {
    InferUnit *units;
    float *d2;
    unsigned short *n;
    int64_t bytes;
};
Carved carve_units(void *base, int64_t U, bool boxes)
{
    Carved r;
    char *b = (char *)base;
    int64_t at = 0;
    r.units = (InferUnit *)(b + at);
    at += align256(U * (int64_t)sizeof(InferUnit));
    r.d2 = (float *)(b + at);
    at += align256(U * capacity_of(boxes) * 4);
    r.n = boxes ? (unsigned short *)(b + at) : nullptr;
    if (boxes) at += align256(U * capacity_of(boxes) * 2);
    r.bytes = at;
    return r;
}

int heads_of(int64_t H) { return (int)((H + 7) / 8 * 8); }
int row_tiles_of(int64_t D) { return D > 16 ? 2 : 1; }

}  // namespace

namespace cf {

// Whether a block's units can be staged: boxes that are the fixed cube of up to 128 translations or adaptive, room for a slice
// worth a launch, a shape the kernel has.  The batch's size decides only at 2^30 values of v (8.4 million edges of 128 wide
// blocks), where offsets leave 32 bits and the attention changes its kernel too: below it a graph of any capacity and an eager
// forward agree to the bit.  `weakest` <= 0 bounds the exponents from above.
bool infer_served(int64_t N, int64_t E, int64_t H, int64_t K, int64_t D, bool boxes, int lattice_range, double weakest,
                  int64_t limit)
{
    const int64_t cube = (int64_t)(2 * lattice_range + 1) * (2 * lattice_range + 1) * (2 * lattice_range + 1);
    return N + E >= 2 && K >= 1 && K <= 128 && D >= 1 && D <= 32 && weakest <= 0 && lattice_range >= 0 &&
           lattice_range <= MAX_RANGE && (boxes || cube <= 128) && limit >= INFER_LEAST_SLICE * bytes_a_unit(boxes) &&
           E * H * D < (1ll << 30) && N * H < (1ll << 32);
}

// Units staged at a time: all, or as many whole rounds as `limit` bytes hold.
int64_t infer_slice(int64_t U, bool boxes, int64_t limit)
{
    const int64_t most = limit / bytes_a_unit(boxes) / WPB * WPB;
    return U < most ? U : most;
}

int64_t infer_units_bytes(int64_t U, bool boxes, int64_t limit)
{
    return U < 1 ? 0 : carve_units(nullptr, infer_slice(U, boxes, limit), boxes).bytes;
}

// Packed projection of a block with up to K bins.
int64_t infer_weights_bytes(int64_t H, int64_t K, int64_t D)
{
    const int64_t tiles = (int64_t)heads_of(H) * row_tiles_of(D);
    return align256(tiles * (pieces_of(tiles_of(K)) * WAVE * 16 + 64));
}

// Stages the units of pairs `before` .. `before` + `slice` - 1 of U, and packs the projections of `blocks` blocks (weights:
// (H, D, bins[l]) each) into `packed`, infer_weights_bytes apart.
int launch_infer_stage(const float *rpos, const float *tvecs, const float *rvlen, const int64_t *pairs, int64_t U,
                       int64_t before, int64_t slice, double weakest, float cutoff, int lattice_range, int min_range,
                       void *staged, int blocks, const float *const *weights, const int *bins, int64_t H, int64_t D,
                       void *packed, int64_t packed_bytes, hipStream_t st)
{
    const bool boxes = rvlen && cutoff != 0.0f;
    const Carved m = carve_units(staged, slice, boxes);
    StageArgs p{};
    p.rpos = rpos; p.tvecs = tvecs; p.rvlen = boxes ? rvlen : nullptr; p.pairs = pairs + before * PAIR_FIELDS;
    p.U = slice; p.before = before; p.live_U = live_units(U);
    p.weak_a = (float)weakest; p.cutoff = boxes ? cutoff : 0.0f;
    p.lattice_range = lattice_range; p.min_range = min_range; p.capacity = capacity_of(boxes);
    p.units = m.units; p.d2 = m.d2; p.n = m.n;
    WeightArgs w{};
    w.blocks = blocks; w.H = (int)H; w.D = (int)D; w.heads = heads_of(H); w.DT = row_tiles_of(D);
    w.stride = packed_bytes / 16; w.out = (int4_t *)packed;
    for (int l = 0; l < blocks; l++) {
        w.w[l] = weights[l];
        w.bins[l] = bins[l];
    }
    const int packs = w.blocks * w.heads * w.DT, pack_groups = (packs + STAGE_WAVES - 1) / STAGE_WAVES;
    const size_t lds = (size_t)STAGE_WAVES * ((boxes ? 3 : 2) * (p.capacity + WAVE) * 2 + CLASSES * WAVE * 2);
    const int64_t want = (slice + STAGE_WAVES - 1) / STAGE_WAVES, cap = persistent_grid_cap(lds > 20000 ? 6 : 8);
    infer_stage_kernel<<<pack_groups + (int)(want < cap ? want : cap), STAGE_WAVES * WAVE, lds, st>>>(p, w);
    CF_CHECK_LAUNCH("infer_stage");
    return CF_OK;
}

// The encoding, for the pairs of a slice, of a block whose units were staged with its cutoff and ranges and an exponent none of
// its own exceeds.
int launch_real_enc_infer(const float *a_ik, const float *rpos, const float *tvecs, const int64_t *pairs, int64_t U,
                          int64_t before, int64_t slice, int64_t H, int64_t K, int64_t D, double dist_max, double wscale,
                          const void *packed, const float *rvlen, float cutoff, int lattice_range, int min_range,
                          double weakest, const void *staged, float *z, float *v, hipStream_t st)
{
    const bool boxes = rvlen && cutoff != 0.0f;
    const Carved m = carve_units(const_cast<void *>(staged), slice, boxes);
    InferArgs x{};
    x.a_ik = a_ik; x.rpos = rpos; x.tvecs = tvecs; x.rvlen = rvlen; x.pairs = pairs + before * PAIR_FIELDS;
    x.units = m.units; x.d2 = m.d2; x.n = m.n; x.capacity = capacity_of(boxes);
    x.weights = (const int4_t *)packed; x.z = z; x.v = v;
    x.U = slice; x.before = before; x.live_U = live_units(U);
    x.H = (int)H; x.D = (int)D; x.heads = heads_of(H);
    x.lattice_range = lattice_range; x.min_range = min_range; x.cutoff = cutoff;
    x.bin_step = 1.0f / ((float)wscale * sqrtf(2.0f)) * sqrtf(LOG2E);
    x.s_scale = x.bin_step / ((float)dist_max / (float)K);
    x.inv_bin_step = 1.0f / x.bin_step;
    x.reach = -40.0f / fminf((float)weakest * LOG2E, LEAST_A2);
    x.rounds_per_group = (int)((slice + WPB - 1) / WPB);
    const int blocks = x.rounds_per_group * (x.heads / 8);
#define CF_INFER(NTV, DTV)                                                                  \
    do {                                                                                    \
        if (boxes) real_enc_infer_kernel<NTV, DTV, true><<<blocks, WPB * WAVE, 0, st>>>(x); \
        else real_enc_infer_kernel<NTV, DTV, false><<<blocks, WPB * WAVE, 0, st>>>(x);      \
    } while (0)
#define CF_INFER_NT(NTV) do { if (D <= 16) CF_INFER(NTV, 1); else CF_INFER(NTV, 2); } while (0)
    switch (tiles_of(K)) {
        case 1: CF_INFER_NT(1); break;
        case 2: CF_INFER_NT(2); break;
        case 4: CF_INFER_NT(4); break;
        default: CF_INFER_NT(8); break;
    }
#undef CF_INFER_NT
#undef CF_INFER
    CF_CHECK_LAUNCH("real_enc_infer");
    return CF_OK;
}

}  // namespace cf
