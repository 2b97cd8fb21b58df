// Everything between one block's attention and the next block's that works row by row, in one launch:
//
//   tail   s = att Wo^T + bo + x,  h = relu(s W1^T + b1),  y = h W2^T + b2 + s
//   head   q, k, v = y Wq^T, y Wk^T, y Wv^T (+ b),  a = coef rho(norm(<q, w_pos>)),  q scaled
//
// for the 128-wide blocks with 512 hidden units; the embedding of the atoms can stand in front of the
// first head.  As four linear launches and two for the exponents this was 6.6 and 4.5 us each at the 1.8
// thousand rows of a batch, most of it not arithmetic: 0.7 GFLOP a block take 4.8 us at the fp32 matrix rate.
//
// A work-group of 8 wavefronts owns 16 T rows; the rows and all intermediates stay in LDS, the weights
// (786 KB a block) stream from the L2, a 16-column tile per wavefront, two tiles ahead of their use.  The products
// are split f16 ones (split_f16.h): a column's weights are scaled and split once per forward (forward_prologue_kernel), a
// row's values in LDS in front of each layer, in place, each in pieces of 128 with a scale of their own.  A value 2^-27 of the
// largest of its piece keeps its 22 bits: hidden units 2^26 apart that meet weights as far apart are as close to float64 as any
// (rms 8.3e-8 of an encoder's output, up to 2^28; fp32 products, whose sums round oftener, 1.5e-7), 2^32 apart 2.2e-7, 2^36
// 3.1e-6.  So the matrix cores need 2.7 us for 16 rows, where fp32 ones needed 10 and bound the launch at 4096 rows, and 16 rows
// are the least tile: half the work-groups, and half the weights asked of the L2, that eight fp32 rows had at 1774 rows.  What
// bounds a launch now is the chain of one tile: 16 rows are staged in 2.5 us, each of the twelve units of 128 columns takes
// 0.5, each of the four splits 0.3, output and exponents 0.9.  Without the weights' loads it would be 10.4 us at 12 rows; five
// buffers of weights instead of three: 0.9 us slower.
// Measured, tail and head in a forward, fp32 products -> these: 12 rows 13.7 -> 12.5 us, 1774 rows 17.6 -> 13.7 (0.70 GFLOP: 51
// TFLOP/s), 4096 rows 25.8 -> 16.9, 5.2 thousand rows 40 -> 21.5 (95 TFLOP/s).  One scale a row instead of one a piece, and first
// and second halves scaled alike, made it 12.2, 13.4, 16.8 and 20.0, and lost what lies below 2^-16 of a row's largest.
// Operands of v_mfma_f32_16x16x32_f16, lane (q, c) = (lane / 16, lane % 16), reduction step s of 32:
//   A: 16 bytes of row c at k = 32 s + 8 q, hi or lo;  B: the same of column c's weights;  D: row 4 q + r, column c.
// A row's sums do not depend on T or on the tile it falls in.
#include "cf_common.h"
#include "block_rows.h"
#include "gauss_maps.h"
#include "lattice_geometry.h"
#include "split_f16.h"

#include <math.h>

namespace {

using namespace cf;

constexpr int RW = 128, RF = 512;            // block width, hidden units
constexpr int LDX = RW + 4, LDH = RF + 4;    // LDS row strides: 4 mod 64, so 16 rows' 16-byte reads cover all banks
constexpr int RT = 512;                      // threads

enum Source { ROWS_PLAIN = 0, ROWS_EMBED = 1, ROWS_TAIL = 2 };

struct Weights {
    float4_t w[8];                           // 128 reduction steps of a 16-column tile
};

// `p` is wave-uniform and `off` this lane's byte offset: one address register for all units.
__device__ __forceinline__ void load_weights(Weights &b, const float *__restrict__ p, unsigned off)
{
#pragma unroll
    for (int c = 0; c < 8; c++)
        b.w[c] = *reinterpret_cast<const float4_t *>(reinterpret_cast<const char *>(p + 256 * c) + off);
}

// The rows' values of 128 reduction steps as A operands.
template <int T>
struct Rows {
    int4_t hi[T][4], lo[T][4];
};

template <int T>
__device__ __forceinline__ void read_rows(Rows<T> &a, const float *xs, int ld, int lane)
{
    const float *xr = xs + (lane & 15) * ld + 8 * (lane >> 4);
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
        for (int s = 0; s < 4; s++) {
            a.hi[t][s] = *reinterpret_cast<const int4_t *>(xr + 16 * t * ld + 32 * s);
            a.lo[t][s] = *reinterpret_cast<const int4_t *>(xr + 16 * t * ld + 32 * s + 4);
        }
}

// acc = the 128 steps' products.  (Each kind is summed apart: every addition to the large sum rounds it, and four chains of
// four keep the matrix cores busier than one of sixteen.)
template <int T>
__device__ __forceinline__ void multiply(float4_t (&acc)[T], const Weights &b, const Rows<T> &a)
{
    const float4_t zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < T; t++) {
        float4_t hh = zero, hl = zero, lh = zero, ll = zero;
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const int4_t hi = __builtin_bit_cast(int4_t, b.w[2 * s]), lo = __builtin_bit_cast(int4_t, b.w[2 * s + 1]);
            hh = mfma32(a.hi[t][s], hi, hh);
            hl = mfma32(a.hi[t][s], lo, hl);
            lh = mfma32(a.lo[t][s], hi, lh);
            ll = mfma32(a.lo[t][s], lo, ll);
        }
        acc[t] = sum_of_kinds(hh, hl, lh, ll);
        // (the products belong here: left to itself the compiler moves them to where the sums are used, and keeps
        // every weight until then)
        asm volatile("" : "+v"(acc[t]));
    }
}

// The largest of 8 or 32 adjacent lanes' magnitudes, in each of them.  By the bits: of floats >= 0 the order of the integers is
// theirs (as floats every step costs a canonicalising instruction beside the one on the DPP path).
template <int CTRL>
__device__ __forceinline__ int dpp_max(int v)
{
    return max(v, __builtin_amdgcn_update_dpp(v, v, CTRL, 0xF, 0xF, false));
}
template <int LANES>
__device__ __forceinline__ int lanes_max(int v)
{
    v = dpp_max<DPP_QUAD_1032>(v);
    v = dpp_max<DPP_QUAD_2301>(v);
    if (LANES == 8) return dpp_max<0x141>(v);                   // row_half_mirror: the other four of eight
    v = dpp_max<DPP_ROW_ROR4>(v);
    v = dpp_max<DPP_ROW_ROR8>(v);
    const uint2_cf r = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
    return max((int)r[0], (int)r[1]);
}
__device__ __forceinline__ int magnitude_bits(float x) { return __float_as_int(x) & 0x7FFFFFFF; }

// 4 L values of a piece of 128 columns of a row, whose other values LANES - 1 adjacent lanes hold, scaled by the piece's largest
// magnitude and split (split2_far): of every eight values (32 bytes) the eight his, then the eight los.  v[l] are the columns
// from at(l) on, a multiple of 4; every lane of the piece gives its exponent's place.
template <int L, class Place>
__device__ __forceinline__ void split_piece(float4_t (&v)[L], float *piece, Place at, bool first, int *exp)
{
    constexpr int LANES = RW / (4 * L);
    float zero = 0.f;
    asm volatile("" : "+v"(zero));
    int top = 0;
#pragma unroll
    for (int l = 0; l < L; l++)
#pragma unroll
        for (int i = 0; i < 4; i++) top = max(top, magnitude_bits(v[l][i]));
    top = lanes_max<LANES>(top);
    if (__builtin_expect(__ballot(top >= 0x7F800000) != 0ull, 0)) {              // infinities, or not a number
        float t = 0.f;
#pragma unroll
        for (int l = 0; l < L; l++)
#pragma unroll
            for (int i = 0; i < 4; i++) t = fmaxf(t, finite_magnitude(v[l][i]));
        top = lanes_max<LANES>(__float_as_int(t));
    }
    const int e = __builtin_amdgcn_frexp_expf(__int_as_float(top));              // (0 for 0)
    if (first) *exp = e;
#pragma unroll
    for (int l = 0; l < L; l++) {
#pragma unroll
        for (int i = 0; i < 4; i++) v[l][i] = ldexpf(v[l][i], 26 - e);
        const Split2 a = split2_far(v[l][0], v[l][1], zero), b = split2_far(v[l][2], v[l][3], zero);
        const int c = at(l);
        float *hi = piece + (c & ~7) + (c & 4) / 2;
        *reinterpret_cast<int2_t *>(hi) = int2_t{a.hi, b.hi};
        *reinterpret_cast<int2_t *>(hi + 4) = int2_t{a.lo, b.lo};
    }
}

// The rows of an LDS buffer split in place (the lanes of a piece have read it before any writes), 32 threads a row.
template <int M>
__device__ __forceinline__ void split_rows(float *xs, int *exps)
{
    const int j = threadIdx.x % 32;
#pragma unroll
    for (int r0 = 0; r0 < M; r0 += RT / 32) {
        const int r = r0 + threadIdx.x / 32;
        float4_t v[1] = {*reinterpret_cast<const float4_t *>(xs + r * LDX + 4 * j)};
        split_piece<1>(v, xs + r * LDX, [&](int) { return 4 * j; }, j == 0, exps + r);
    }
}
// The hidden units, four pieces a row with exponents M apart.  Eight lanes a piece, each with four times four columns 32 apart; every
// other piece starts with its second 32, so that 16 lanes' reads cover all banks.
template <int M>
__device__ __forceinline__ void split_hidden(float *hs, int *exps)
{
    const int p = threadIdx.x / 8 % 4, k = threadIdx.x % 8;
    auto at = [&](int l) { return 4 * k + 32 * l + (l % 2 ? -32 : 32) * (p & 1); };
#pragma unroll
    for (int r0 = 0; r0 < M; r0 += RT / 32) {
        const int r = r0 + threadIdx.x / 32;
        float *piece = hs + r * LDH + p * RW;
        float4_t v[4];
#pragma unroll
        for (int l = 0; l < 4; l++) v[l] = *reinterpret_cast<const float4_t *>(piece + at(l));
        split_piece<4>(v, piece, at, k == 0, exps + p * M + r);
    }
}

// Raw exponents on their way to the work-group that finishes them: written through and read past the L2 of an XCD, so that
// no work-group has to write back or invalidate a cache (a fence each cost 35 us a block in all).
__device__ __forceinline__ void put_raw(float *p, float v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float get_raw(const float *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The exponents where no statistics are stored: a holds the raw values, whose statistics are formed as the two
// exponent kernels do -- groups of 256 values, mean first, then the squared deviations, groups merged by Chan's formula
// in the same order.  Up to KEPT groups a wavefront the last work-group to finish holds all values in registers, forms the
// groups' statistics, merges and maps them: 18 us a block at 2048 atoms.  Beyond, the work-group that completes a group
// forms its statistics and the last one only merges: 10 us a block at 8192 atoms with the map, where the last work-group
// took 33 for all of it (forwards of four blocks without value bins 712 for 797 us, 2617 for 2956 at 32768 atoms; 666 and
// 2486 where statistics are stored).
// The map beyond KEPT groups is a launch of its own (apart): it keeps one work-group busy for 28 us at 8192 atoms (39 without
// asking for the next values ahead).  With stored statistics that launch ends at once, 1.8 us a block.  A capacity, whose
// live rows are mostly fewer, takes it from four times that size on (32768 atoms, all live, 2629 us; 3299 with one work-group);
// training, which has stored statistics from its second step on, does without it.
constexpr int KEPT = 8;                      // (all values of 2048 atoms with 8 heads)
constexpr int WAVES = RT / WAVE;

// (a kernel of its own where all values can be kept: the code costs the others 1% of a launch)
__host__ __device__ __forceinline__ bool spread_groups(int64_t total) { return total > 256 * KEPT * WAVES; }

// (count, mean, squared deviations) of group b, one wavefront.
__device__ __forceinline__ void group_statistics(const float (&v)[4], int64_t b, int64_t total, int lane, float (&out)[3])
{
    const float cnt = (float)min((int64_t)256, total - 256 * b);
    float s[4];
#pragma unroll
    for (int u = 0; u < 4; u++) s[u] = wave_sum(v[u]);
    const float mean = (((0.f + s[0]) + s[1]) + s[2] + s[3]) / cnt;
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const float dv = 256 * b + 64 * u + lane < total ? v[u] - mean : 0.f;
        s[u] = wave_sum(dv * dv);
    }
    out[0] = cnt;
    out[1] = mean;
    out[2] = ((0.f + s[0]) + s[1]) + s[2] + s[3];
}

// The raw values of rows row0 .. row0 + rows - 1 are on their way: counts them into the groups they belong to, and forms
// the statistics of those that are complete with them.  A tile's values are one piece (two with split heads) of at most 256
// (launch_block_rows sees to it), so they touch two groups each: one per wavefront.
__device__ void complete_groups(const RowsArgs &p, int64_t N, int64_t row0, int rows)
{
    unsigned tid = threadIdx.x;
    asm volatile("" : "+v"(tid));                               // (worked out here: not kept through the tile loop)
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // this wavefront's raw values have arrived
    __syncthreads();
    if (wave >= (p.split ? 4 : 2)) return;
    const int64_t total = N * p.H;
    const int width = p.split ? p.H / 2 : p.H;
    const int64_t v0 = ((wave >> 1) * N + row0) * width, v1 = v0 + min((int64_t)rows, N - row0) * width;
    const int64_t g = v0 / 256 + (wave & 1), first = 256 * g, last = min(first + 256, total);
    if (first >= v1) return;
    const unsigned mine = (unsigned)(min(v1, last) - max(v0, first));
    unsigned before = 0;
    if (lane == 0) before = atomicAdd(p.groups + g, mine);
    before = __builtin_amdgcn_readfirstlane(before);
    if (before + mine != (unsigned)(last - first)) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    float v[4], out[3];
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const int64_t t = first + 64 * u + lane;
        v[u] = t < total ? get_raw(p.a + t) : 0.f;
    }
    group_statistics(v, g, total, lane, out);
    if (lane == 0) {
#pragma unroll
        for (int i = 0; i < 3; i++) put_raw(p.part + 3 * g + i, out[i]);
        __hip_atomic_store(p.groups + g, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

template <bool SPREAD>
__device__ void finish_exponents(const RowsArgs &p, int64_t total, float *red)
{
    __shared__ float stats[3 * KEPT * WAVES];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t blocks = (total + 255) / 256;
    const bool kept = !spread_groups(total);
    float v[KEPT][4];
    auto fetch = [&](int64_t b0) {                              // this wavefront's groups b0 + wave, + 8, ...: 32 loads in flight
#pragma unroll
        for (int k = 0; k < KEPT; k++)
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int64_t t = 256 * (b0 + wave + WAVES * k) + 64 * u + lane;
                v[k][u] = t < total ? get_raw(p.a + t) : 0.f;
            }
    };
    for (int64_t b0 = 0; b0 < blocks && !(SPREAD && !kept); b0 += KEPT * WAVES) {
        fetch(b0);
#pragma unroll
        for (int k = 0; k < KEPT; k++) {
            const int64_t b = b0 + wave + WAVES * k;
            float out[3];
            if (b < blocks) group_statistics(v[k], b, total, lane, out);
            if (b < blocks && lane == 0) {
                float *to = (kept ? stats : p.part) + 3 * b;
                to[0] = out[0];
                to[1] = out[1];
                to[2] = out[2];
            }
        }
    }
    __syncthreads();
    if (wave == 0) {
        float n, mean, m2;
        if (kept) merge_statistics(stats, (int)blocks, lane, n, mean, m2);
        else if (SPREAD) merge_statistics_of([&](int i) { return get_raw(p.part + i); }, (int)blocks, lane, n, mean, m2);
        else merge_statistics(p.part, (int)blocks, lane, n, mean, m2);
        if (lane == 0) {
            const float scale = 1.0f / sqrtf(m2 / (n - 1.0f));
            red[0] = scale;
            red[1] = -mean;
            if (p.apart) {                                      // (the groups' statistics are merged)
                p.part[0] = scale;
                p.part[1] = -mean;
            }
            if (p.used) {
                p.used[0] = scale;
                p.used[1] = -mean;
            }
            if (p.update_stats) {
                p.gauss_scale[0] = scale;
                p.gauss_scale[1] = -mean;
            }
        }
    }
    if (p.apart) return;
    __syncthreads();
    const float scale = red[0], shift = red[1];
    auto finish = [&](int64_t t, float raw) {
        const float alpha = (raw + shift) * scale;
        if (p.alpha_n) p.alpha_n[t] = alpha;
        p.a[t] = positive_map(alpha, p.func, p.beta, p.lb) * (p.split && 2 * t >= total ? p.coef_second : p.coef);
    };
    if (SPREAD && !kept) fetch(0);
    for (int64_t b0 = 0; b0 < blocks; b0 += KEPT * WAVES) {
        float now[KEPT][4];
        if (SPREAD) {                                           // the next values on their way while these are mapped
#pragma unroll
            for (int k = 0; k < KEPT; k++)
#pragma unroll
                for (int u = 0; u < 4; u++) now[k][u] = v[k][u];
            if (b0 + KEPT * WAVES < blocks) fetch(b0 + KEPT * WAVES);
        } else if (!kept) {
            fetch(b0);
        }
#pragma unroll
        for (int k = 0; k < KEPT; k++)
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int64_t t = 256 * (b0 + wave + WAVES * k) + 64 * u + lane;
                if (t < total) finish(t, SPREAD ? now[k][u] : v[k][u]);
            }
    }
}

// A work-group that had rows (the first `tiles` of the grid) counts itself; the last one finishes the exponents of all.
template <bool SPREAD>
__device__ void finish_if_last(const RowsArgs &p, int64_t N, int64_t tiles, float *red)
{
    const int64_t active = min((int64_t)gridDim.x, tiles);
    if ((int64_t)blockIdx.x >= active) return;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // this wavefront's raw values have arrived
    __syncthreads();
    if (threadIdx.x == 0) red[0] = atomicAdd(p.counter, 1u) + 1u == (unsigned)active ? 1.f : 0.f;
    __syncthreads();
    const bool last = red[0] != 0.f;
    __syncthreads();
    if (last) {
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        finish_exponents<SPREAD>(p, N * p.H, red);
    }
}

constexpr int FINISH_T = 256, FINISH_VALUES = 4 * FINISH_T;
__global__ __launch_bounds__(FINISH_T) void finish_exponents_kernel(RowsArgs p)
{
    if (*p.counter == 0) return;                                // stored statistics: mapped already
    const int64_t total = live_count(p.live_N, p.N) * p.H;
    const float scale = p.part[0], shift = p.part[1];
#pragma unroll
    for (int u = 0; u < 4; u++) {
        const int64_t t = (int64_t)blockIdx.x * FINISH_VALUES + u * FINISH_T + threadIdx.x;
        if (t < total)
            p.a[t] = positive_map((p.a[t] + shift) * scale, p.func, p.beta, p.lb) *
                     (p.split && 2 * t >= total ? p.coef_second : p.coef);
    }
}

// The matrices as a sequence of units, 16 columns a wavefront x 128 reduction steps each:
// 0 output projection, 1-4 hidden units, 5-8 their reduction (or 8 the embedding), 9-11 query, key, value.
constexpr int UNIT_FF1 = 1, UNIT_FF2 = 5, UNIT_EMBED = 8, UNIT_QUERY = 9, UNIT_END = 12, UNIT_FLOATS = RW * RW;

// The weights of up to PACK_BLOCKS blocks in the order the row kernel reads them: per unit and wavefront eight
// 1 KB pieces, one per 16 reduction steps, in lane order.  Read from the matrices themselves every load
// of a wavefront takes 64 bytes of 16 rows, 512 or 2048 bytes apart: 24 us a launch (by the addresses these
// fall into a few of the L2's channels; counters were not taken).
constexpr int PACK_GRID = UNIT_END * UNIT_FLOATS / 1024;       // work-groups of 256 threads a block
__device__ __forceinline__ void pack_weights(const PackArgs &p, int x, int l, bool transposed)
{
    const int u = x / (UNIT_FLOATS / 1024);
    if (p.zero && x == 0 && l == 0 && !transposed)
        for (int64_t t = threadIdx.x; t < p.words; t += 256) p.zero[t] = 0u;
    const int at = 4 * (int)(x % (UNIT_FLOATS / 1024) * 256 + threadIdx.x);             // first of four floats of the unit
    const int wave = at / 2048, k = at / 256 % 8 * 16 + at / 64 % 4 * 4, col = 16 * wave + at / 4 % 16;
    const PackSource &w = p.block[l];
    if (transposed) {                                           // units 0-3 W2, 4-7 W1, 8 Wo, 9-11 Wq, Wk, Wv
        const float *t;
        int ld = RW;
        if (u < 4) t = w.w2 + u * RW, ld = RF;
        else if (u < 8) t = w.w1 + (u - 4) * RW * RW;
        else t = u == 8 ? w.wo : u == 9 ? w.wq : u == 10 ? w.wk : w.wv;
        float4_t v;
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = t[(k + i) * ld + col];
        *reinterpret_cast<float4_t *>(p.packed_bwd + (int64_t)l * PACKED_BLOCK + u * UNIT_FLOATS + at) = v;
        return;
    }
    const float *src;
    if (u == 0) src = w.wo + col * RW + k;
    else if (u < UNIT_FF2) src = w.w1 + ((u - UNIT_FF1) * RW + col) * RW + k;
    else if (u < UNIT_QUERY) src = w.w2 + col * RF + (u - UNIT_FF2) * RW + k;
    else src = (u == UNIT_QUERY ? w.wq : u == UNIT_QUERY + 1 ? w.wk : w.wv) + col * RW + k;
    *reinterpret_cast<float4_t *>(p.packed + (int64_t)l * PACKED_BLOCK + u * UNIT_FLOATS + at) =
        *reinterpret_cast<const float4_t *>(src);
}

// The same weights for the inference kernel: per unit and wavefront four reduction steps of 32, hi and lo, 1 KB each in lane
// order, a column scaled by its largest magnitude in the unit; behind the units the columns' exponents.
constexpr int SPLIT_TILES = UNIT_END * 8, SPLIT_WAVES = 4;      // wavefronts a block, a work-group
__device__ __forceinline__ void pack_split(const PackArgs &p, int x, int l)
{
    const int lane = threadIdx.x & 63, q = lane >> 4, c = lane & 15;
    const int tile = x * SPLIT_WAVES + (int)(threadIdx.x >> 6), u = tile / 8, wave = tile % 8, col = 16 * wave + c;
    if (l == p.blocks && u > 0) return;
    const float *row;
    if (l == p.blocks) {
        row = p.w_embed + col * p.embed_width;
    } else {
        const PackSource &w = p.block[l];
        if (u == 0) row = w.wo + col * RW;
        else if (u < UNIT_FF2) row = w.w1 + ((u - UNIT_FF1) * RW + col) * RW;
        else if (u < UNIT_QUERY) row = w.w2 + col * RF + (u - UNIT_FF2) * RW;
        else row = (u == UNIT_QUERY ? w.wq : u == UNIT_QUERY + 1 ? w.wk : w.wv) + col * RW;
    }
    float4_t w[4][2];
    if (l == p.blocks) {                                        // (an embedding's rows: any width, not aligned)
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const int k = 32 * s + 8 * q + i;
                w[s][i / 4][i % 4] = k < p.embed_width ? row[k] : 0.f;
            }
    } else {
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int i = 0; i < 2; i++) w[s][i] = *reinterpret_cast<const float4_t *>(row + 32 * s + 8 * q + 4 * i);
    }
    float top = 0.f;
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
        for (int i = 0; i < 8; i++) top = fmaxf(top, fabsf(w[s][i / 4][i % 4]));
    top = rows_max(top);
    if (__ballot(top == __builtin_inff()) != 0ull) {
        top = 0.f;
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int i = 0; i < 8; i++) top = fmaxf(top, finite_magnitude(w[s][i / 4][i % 4]));
        top = rows_max(top);
    }
    const int e = __builtin_amdgcn_frexp_expf(top);
    float zero = 0.f;
    asm volatile("" : "+v"(zero));
    float *units = l == p.blocks ? p.packed_embed : p.packed + (int64_t)l * SPLIT_BLOCK;
    int4_t *out = reinterpret_cast<int4_t *>(units + u * UNIT_FLOATS) + wave * 8 * WAVE + lane;
#pragma unroll
    for (int s = 0; s < 4; s++) {
        int4_t hi, lo;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const Split2 y = split2_far(ldexpf(w[s][i / 2][2 * i % 4], 26 - e), ldexpf(w[s][i / 2][2 * i % 4 + 1], 26 - e), zero);
            hi[i] = y.hi;
            lo[i] = y.lo;
        }
        out[2 * s * WAVE] = hi;
        out[(2 * s + 1) * WAVE] = lo;
    }
    int *exps = reinterpret_cast<int *>(units + (l == p.blocks ? UNIT_FLOATS : PACKED_BLOCK)) + u * RW;
    if (lane < 16) exps[col] = e - 30;                          // (a row's and a column's 2^15)
}

__global__ __launch_bounds__(256) void pack_weights_kernel(PackArgs p)
{
    pack_weights(p, blockIdx.x, blockIdx.y, blockIdx.z == 1);
}

// What a forward needs before its first block, none of it depending on the rest, in one launch instead of three of
// 2 to 4 us: the packed weights, the offsets p_j - p_i of the edges and the lattices' geometry.
__global__ __launch_bounds__(256) void forward_prologue_kernel(PackArgs k, PrologueArgs p)
{
    constexpr int GROUPS = SPLIT_TILES / SPLIT_WAVES;
    const int layers = k.blocks + (k.w_embed ? 1 : 0);
    int64_t x = blockIdx.x;
    if (x < (int64_t)layers * GROUPS) {
        if (x == 0)
            for (int64_t t = threadIdx.x; t < k.words; t += 256) k.zero[t] = 0u;
        pack_split(k, (int)(x % GROUPS), (int)(x / GROUPS));
        return;
    }
    x -= (int64_t)layers * GROUPS;
    const int64_t edge_groups = (p.E + 255) / 256;
    if (x < edge_groups) {
        const int64_t e = x * 256 + threadIdx.x;
        if (e >= live_count(p.live_E, p.E)) return;
        const EdgeEnds r = edge_ends(p.atom_start, p.edge_start, p.B, e);
#pragma unroll
        for (int d = 0; d < 3; d++) p.rpos[e * 3 + d] = p.pos[r.j * 3 + d] - p.pos[r.i * 3 + d];
        return;
    }
    const int64_t b = (x - edge_groups) * 256 + threadIdx.x;
    if (b < p.B) lattice_geometry_of(p.trans, b, p.vcell, p.recip, p.rvlen);
}

template <int T, int SRC, bool HEAD, bool SPREAD>
__global__ __launch_bounds__(RT, 2) void block_rows_kernel(RowsArgs p)
{
    constexpr int M = 16 * T;
    constexpr int FIRST = SRC == ROWS_TAIL ? 0 : SRC == ROWS_EMBED ? UNIT_EMBED : UNIT_QUERY;
    constexpr int END = HEAD ? UNIT_END : UNIT_QUERY;
    __shared__ __align__(16) float b0[M * LDX];                 // tail: attention output; then the rows behind it
    __shared__ __align__(16) float b1[M * LDX];                 // tail: block input, then s
    __shared__ __align__(16) float b2[M * LDX];                 // what the coming layer takes, split
    __shared__ __align__(16) float hs[M * LDH];                 // hidden units, then query, key, value
    __shared__ float biases[UNIT_END * RW], w_pos[RW];
    __shared__ int w_exp[UNIT_END * RW];
    __shared__ __align__(16) int x_exp[4 * M];                  // (the reduction's four pieces of a row have their own)
    __shared__ float red[2];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int q = lane >> 4, c = lane & 15;
    const int col = 16 * wave + c;
    const int64_t N = live_count(p.live_N, p.N);
    bool stored = true;
    float scale = 1.f, shift = 0.f;
    if (HEAD && p.normalize) {
        scale = p.gauss_scale[0];
        shift = p.gauss_scale[1];
        stored = scale > 0.f;
    }
    auto unit_weights = [&](int u) -> const float * {
        if (SRC == ROWS_EMBED && u == UNIT_EMBED) return p.packed_embed;
        return (u < UNIT_QUERY ? p.packed_tail : p.packed_head) + u * UNIT_FLOATS;
    };
    // this lane's value of row 16 t + 4 q + r in unit u
    auto value = [&](const float4_t (&acc)[T], int t, int r, int u) -> float {
        const int piece = u >= UNIT_FF2 && u < UNIT_FF2 + 4 && SRC == ROWS_TAIL ? u - UNIT_FF2 : 0;
        const int4_t e = *reinterpret_cast<const int4_t *>(x_exp + piece * M + 16 * t + 4 * q);
        return ldexpf(acc[t][r], e[r] + w_exp[u * RW + col]) + biases[u * RW + col];
    };
    // (one tile per work-group unless the grid was cut short: with a live row count it covers a capacity)
    bool first = true;
    for (int64_t row0 = (int64_t)blockIdx.x * M; row0 < N; row0 += (int64_t)gridDim.x * M) {
        float4_t acc[T];
        // AHEAD + 1 buffers in turn: unit u lies in buffer (u - FIRST) % BUFFERS
        constexpr int BUFFERS = 3;
        Weights w[BUFFERS];
        unsigned woff = (unsigned)(wave * 2048 + lane * 4) * 4u;
        asm volatile("" : "+v"(woff));       // (not a constant of this loop: else a hundred registers hold addresses)
        auto fetch = [&](int u) {
            if (u < END) load_weights(w[(u - FIRST) % BUFFERS], unit_weights(u), woff);
        };
        auto unit = [&](int u) -> Weights & {
            fetch(u + BUFFERS - 1);
            return w[(u - FIRST) % BUFFERS];
        };
        fetch(FIRST);
        // everything the tile needs is asked for before any of it is used
        constexpr int PASSES = M / (RT / 32), EACH = (END - FIRST) * RW / RT;
        const int j = threadIdx.x % 32, k = threadIdx.x % RW;
        float4_t in[PASSES][1], residual[PASSES];
#pragma unroll
        for (int t = 0; t < PASSES; t++) {
            const int64_t row = min(row0 + 16 * t + threadIdx.x / 32, N - 1);
            if (SRC == ROWS_EMBED) {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    in[t][0][i] = 4 * j + i < p.embed_width ? p.x[row * p.embed_width + 4 * j + i] : 0.f;
            } else {
                in[t][0] = *reinterpret_cast<const float4_t *>((SRC == ROWS_TAIL ? p.att : p.x) + row * RW + 4 * j);
            }
            if (SRC == ROWS_TAIL) residual[t] = *reinterpret_cast<const float4_t *>(p.x + row * RW + 4 * j);
        }
        if (first) {
            // unit by unit, four at a time (the reduction's four units share one bias)
            float bias[EACH + 1], wp = 0.f;
            int exps[EACH + 1];
#pragma unroll
            for (int i = 0; i <= EACH; i++) {
                const int u = FIRST + 4 * i + threadIdx.x / RW;
                if (u >= END) break;
                const bool embed = SRC == ROWS_EMBED && u == UNIT_EMBED;
                const float *src = u >= UNIT_QUERY ? p.b_in : embed ? p.b_embed : u == 0 ? p.bo : u < UNIT_FF2 ? p.b1 : p.b2;
                const int from = u >= UNIT_QUERY ? u - UNIT_QUERY : u >= UNIT_FF1 && u < UNIT_FF2 ? u - UNIT_FF1 : 0;
                bias[i] = src && (embed || u <= UNIT_FF2 || u >= UNIT_QUERY) ? src[from * RW + k] : 0.f;
                exps[i] = embed ? reinterpret_cast<const int *>(p.packed_embed + UNIT_FLOATS)[k]
                                : reinterpret_cast<const int *>((u < UNIT_QUERY ? p.packed_tail : p.packed_head) + PACKED_BLOCK)[u * RW + k];
            }
            if (HEAD) wp = p.w_pos[k];
            first = false;
#pragma unroll
            for (int i = 0; i <= EACH; i++) {
                const int u = FIRST + 4 * i + threadIdx.x / RW;
                if (u >= END) break;
                biases[u * RW + k] = bias[i];
                w_exp[u * RW + k] = exps[i];
            }
            if (HEAD && threadIdx.x < RW) w_pos[k] = wp;
        }
#pragma unroll
        for (int u = 1; u < BUFFERS - 1; u++) fetch(FIRST + u);
#pragma unroll
        for (int t = 0; t < PASSES; t++) {
            const int r = 16 * t + threadIdx.x / 32;
            split_piece<1>(in[t], b2 + r * LDX, [&](int) { return 4 * j; }, j == 0, x_exp + r);
            if (SRC == ROWS_TAIL) *reinterpret_cast<float4_t *>(b1 + r * LDX + 4 * j) = residual[t];
        }
        __syncthreads();
        const int at = 4 * q * LDX + col, at_h = 4 * q * LDH + col;          // this lane's results: rows 16 t + 4 q + r
        Rows<T> x;
        if (SRC == ROWS_TAIL) {
            // output projection and residual: s replaces x in place
            read_rows(x, b2, LDX, lane);
            multiply(acc, unit(0), x);
#pragma unroll
            for (int t = 0; t < T; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    float *s = b1 + at + (16 * t + r) * LDX;
                    const float v = *s + value(acc, t, r, 0);
                    *s = v;
                    b0[at + (16 * t + r) * LDX] = v;
                }
            __syncthreads();
            split_rows<M>(b0, x_exp);
            __syncthreads();
            // hidden units, four tiles on one read of the rows
            read_rows(x, b0, LDX, lane);
#pragma unroll
            for (int u = 0; u < 4; u++) {
                multiply(acc, unit(UNIT_FF1 + u), x);
#pragma unroll
                for (int t = 0; t < T; t++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const float v = value(acc, t, r, UNIT_FF1 + u);
                        hs[at_h + (16 * t + r) * LDH + u * RW] = v < 0.f ? 0.f : v;   // (a NaN stays one, as in torch.relu)
                    }
            }
            __syncthreads();
            split_hidden<M>(hs, x_exp);
            __syncthreads();
            float y[T][4];
            Rows<T> ahead;                                      // (read a unit before it is multiplied)
            read_rows(x, hs, LDH, lane);
#pragma unroll
            for (int u = 0; u < 4; u++) {
                Rows<T> &now = u % 2 ? ahead : x;
                if (u < 3) read_rows(u % 2 ? x : ahead, hs + (u + 1) * RW, LDH, lane);
                multiply(acc, unit(UNIT_FF2 + u), now);
                // (a unit's columns have exponents of their own, and a row's pieces)
#pragma unroll
                for (int t = 0; t < T; t++)
#pragma unroll
                    for (int r = 0; r < 4; r++) y[t][r] = (u == 0 ? 0.f : y[t][r]) + value(acc, t, r, UNIT_FF2 + u);
            }
#pragma unroll
            for (int t = 0; t < T; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int i = at + (16 * t + r) * LDX;
                    const float v = y[t][r] + b1[i];
                    b0[i] = v;
                    if (HEAD) b2[i] = v;
                }
            __syncthreads();
        } else if (SRC == ROWS_EMBED) {
            read_rows(x, b2, LDX, lane);
            multiply(acc, unit(UNIT_EMBED), x);
            float v[T][4];
#pragma unroll
            for (int t = 0; t < T; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) v[t][r] = value(acc, t, r, UNIT_EMBED);
            __syncthreads();                                    // (the rows to embed have been read)
#pragma unroll
            for (int t = 0; t < T; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) b0[at + (16 * t + r) * LDX] = b2[at + (16 * t + r) * LDX] = v[t][r];
            __syncthreads();
        }
        if (HEAD) {
            if (SRC != ROWS_PLAIN) {
                split_rows<M>(b2, x_exp);
                __syncthreads();
            }
            read_rows(x, b2, LDX, lane);
#pragma unroll
            for (int u = 0; u < 3; u++) {
                multiply(acc, unit(UNIT_QUERY + u), x);
#pragma unroll
                for (int t = 0; t < T; t++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        hs[at_h + (16 * t + r) * LDH + u * RW] = value(acc, t, r, UNIT_QUERY + u);
            }
        }
        if (HEAD) __syncthreads();
        // results leave LDS in whole rows once the loop has no more loads to wait for
        for (int t = threadIdx.x; t < M * (RW / 4); t += RT) {
            const int r = t / (RW / 4), d = 4 * (t % (RW / 4));
            const int64_t at = (row0 + r) * RW + d;
            if (row0 + r >= N) break;
            if (SRC != ROWS_PLAIN)
                *reinterpret_cast<float4_t *>(p.y + at) = *reinterpret_cast<const float4_t *>(b0 + r * LDX + d);
            if (HEAD) {
                const float *out = hs + r * LDH + d;
                *reinterpret_cast<float4_t *>(p.qs + at) = *reinterpret_cast<const float4_t *>(out) * p.q_scale;
                *reinterpret_cast<float4_t *>(p.k + at) = *reinterpret_cast<const float4_t *>(out + RW);
                *reinterpret_cast<float4_t *>(p.v + at) = *reinterpret_cast<const float4_t *>(out + 2 * RW);
            }
        }
        if (HEAD) {
            const int D = RW / p.H;
            for (int t = threadIdx.x; t < M * p.H; t += RT) {
                const int r = t / p.H, h = t - r * p.H;
                const float *q = hs + r * LDH + h * D, *w = w_pos + h * D;
                float alpha = 0.f;
                for (int d = 0; d < D; d += 4)                  // (the order of the exponent kernel)
                    alpha += (q[d] * w[d] + q[d + 1] * w[d + 1]) + (q[d + 2] * w[d + 2] + q[d + 3] * w[d + 3]);
                if (p.normalize && stored) alpha = (alpha + shift) * scale;
                const int half = p.H >> 1;
                const bool second = p.split && h >= half;
                if (!p.normalize || stored)
                    alpha = positive_map(alpha, p.func, p.beta, p.lb) * (second ? p.coef_second : p.coef);
                if (row0 + r < N) {
                    float *out = p.a + (p.split ? (second ? N : 0) * half + (row0 + r) * half + h - (second ? half : 0)
                                                : (row0 + r) * p.H + h);
                    if (stored) *out = alpha;
                    else put_raw(out, alpha);
                }
            }
        }
        if (SPREAD && !stored && spread_groups(N * p.H)) complete_groups(p, N, row0, M);
        __syncthreads();                                        // the next tile overwrites the rows
    }
    if (HEAD && !stored) finish_if_last<SPREAD>(p, N, (N + M - 1) / M, red);
}

// ---- training ------------------------------------------------------------------
// The same parts with what their backward passes need, and these, on v_mfma_f32_16x16x4_f32 with sixteen rows a
// work-group: every sum of linear_rows_kernel, linear_rows_nn_kernel and the exponent kernels in their order, so that
// a training step is the same to the bit.  (It has to be: after the optimiser's first steps biases come back to zero
// but for rounding, a hidden unit's ReLU then opens or shuts for all atoms at once, and gradients of any other
// order of summation drift apart by 5% within ten steps.)  What bounds a launch is the matrix cores of the CUs that
// have a tile: 7.7 us of a tail.  Measured at 1774 rows: tail 14.1 us forward and 15.0 backward, head 8.2 and 8.7 plus 8.5
// for the gradient of w_pos, 54 us a block where the separate launches took 78.
//   A: lane (q, c) reads 16 bytes of row c at k = 16 s + 4 q;  B: the packed weights as they are;
//   D: lane (q, c), register r: row 4 q + r, column c.
constexpr int TM = 16;
constexpr int TLX = RW + 4, TLH = RF + 4;    // LDS row strides: 4 mod 64, so 16 rows' 16-byte reads cover all banks

__device__ __forceinline__ void multiply16(float4_t &acc, const Weights &b, const float *xs, int ld, int lane)
{
    const float *xr = xs + (lane & 15) * ld + 4 * (lane >> 4);
    float4_t x[8];
#pragma unroll
    for (int c = 0; c < 8; c++) x[c] = *reinterpret_cast<const float4_t *>(xr + 16 * c);
#pragma unroll
    for (int c = 0; c < 8; c++)
#pragma unroll
        for (int s = 0; s < 4; s++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[c][s], b.w[c][s], acc, 0, 0, 0);
    asm volatile("" : "+v"(acc));            // (as in multiply: the products belong here)
}

// rows row0 .. of a (N, 128) matrix into LDS and back: 512 threads are 16 rows x 32 pieces of 16 bytes
__device__ __forceinline__ void stage16(float *dst, const float *__restrict__ src, int64_t row0, int64_t N)
{
    const int r = threadIdx.x / (RW / 4), c = threadIdx.x % (RW / 4);
    *reinterpret_cast<float4_t *>(dst + r * TLX + 4 * c) =
        *reinterpret_cast<const float4_t *>(src + min(row0 + r, N - 1) * RW + 4 * c);
}

__device__ __forceinline__ void unstage16(float *__restrict__ dst, int ld, const float *src, int lds_ld, int64_t row0,
                                          int64_t N)
{
    const int r = threadIdx.x / (RW / 4), c = threadIdx.x % (RW / 4);
    if (row0 + r < N)
        *reinterpret_cast<float4_t *>(dst + (row0 + r) * ld + 4 * c) =
            *reinterpret_cast<const float4_t *>(src + r * lds_ld + 4 * c);
}

__global__ __launch_bounds__(RT) void block_tail_train_kernel(RowsArgs p)
{
    __shared__ __align__(16) float b0[TM * TLX], b1[TM * TLX], hs[TM * TLH];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int q = lane >> 4, col = 16 * wave + (lane & 15);
    const int64_t row0 = (int64_t)blockIdx.x * TM, N = p.N;
    const unsigned woff = (unsigned)(wave * 2048 + lane * 4) * 4u;
    const float *w = p.packed_tail;
    Weights wa, wb, wc;
    load_weights(wa, w, woff);
    stage16(b0, p.att, row0, N);
    stage16(b1, p.x, row0, N);
    const float bo = p.bo ? p.bo[col] : 0.f, b2 = p.b2 ? p.b2[col] : 0.f;
    float bh[4];
#pragma unroll
    for (int u = 0; u < 4; u++) bh[u] = p.b1 ? p.b1[u * RW + col] : 0.f;
    load_weights(wb, w + UNIT_FLOATS, woff);
    __syncthreads();
    const float4_t zero4 = {0.f, 0.f, 0.f, 0.f};
    float4_t acc = zero4;
    load_weights(wc, w + 2 * UNIT_FLOATS, woff);
    multiply16(acc, wa, b0, TLX, lane);
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const float v = acc[r] + bo;
        b1[(4 * q + r) * TLX + col] = v + b1[(4 * q + r) * TLX + col];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; u++) {
        Weights &cur = u % 3 == 0 ? wb : u % 3 == 1 ? wc : wa, &nxt = u % 3 == 0 ? wa : u % 3 == 1 ? wb : wc;
        load_weights(nxt, w + (UNIT_FF1 + 2 + u) * UNIT_FLOATS, woff);
        acc = zero4;
        multiply16(acc, cur, b1, TLX, lane);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float v = acc[r] + bh[u];
            hs[(4 * q + r) * TLH + u * RW + col] = v < 0.f ? 0.f : v;            // (a NaN stays one)
        }
    }
    __syncthreads();
    acc = zero4;
#pragma unroll
    for (int u = 0; u < 4; u++) {
        Weights &cur = u % 3 == 0 ? wc : u % 3 == 1 ? wa : wb, &nxt = u % 3 == 0 ? wb : u % 3 == 1 ? wc : wa;
        if (u < 2) load_weights(nxt, w + (UNIT_FF2 + 2 + u) * UNIT_FLOATS, woff);
        multiply16(acc, cur, hs + u * RW, TLH, lane);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const float v = acc[r] + b2;
        b0[(4 * q + r) * TLX + col] = v + b1[(4 * q + r) * TLX + col];
    }
    __syncthreads();
    unstage16(p.y, RW, b0, TLX, row0, N);
    unstage16(p.s, RW, b1, TLX, row0, N);
#pragma unroll
    for (int u = 0; u < 4; u++) unstage16(p.h + u * RW, RF, hs + u * RW, TLH, row0, N);
}

__global__ __launch_bounds__(RT) void block_head_train_kernel(RowsArgs p)
{
    __shared__ __align__(16) float b0[TM * TLX], out[3][TM * TLX];
    __shared__ float red[2];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int q = lane >> 4, col = 16 * wave + (lane & 15);
    const int64_t row0 = (int64_t)blockIdx.x * TM, N = p.N;
    const unsigned woff = (unsigned)(wave * 2048 + lane * 4) * 4u;
    const float *w = p.packed_head + UNIT_QUERY * UNIT_FLOATS;
    Weights wt[3];
    load_weights(wt[0], w, woff);
    stage16(b0, p.x, row0, N);
    load_weights(wt[1], w + UNIT_FLOATS, woff);
    load_weights(wt[2], w + 2 * UNIT_FLOATS, woff);
    bool stored = true;
    float scale = 1.f, shift = 0.f;
    if (p.normalize) {
        scale = p.gauss_scale[0];
        shift = p.gauss_scale[1];
        stored = scale > 0.f;
        if (p.used && stored && blockIdx.x == 0 && threadIdx.x == 0) {
            p.used[0] = scale;
            p.used[1] = shift;
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 3; u++) {
        const float bias = p.b_in ? p.b_in[u * RW + col] : 0.f;
        float4_t acc = {0.f, 0.f, 0.f, 0.f};
        multiply16(acc, wt[u], b0, TLX, lane);
#pragma unroll
        for (int r = 0; r < 4; r++) out[u][(4 * q + r) * TLX + col] = acc[r] + bias;
    }
    __syncthreads();
    unstage16(p.q, RW, out[0], TLX, row0, N);
    unstage16(p.k, RW, out[1], TLX, row0, N);
    unstage16(p.v, RW, out[2], TLX, row0, N);
    {
        const int r = threadIdx.x / (RW / 4), d = 4 * (threadIdx.x % (RW / 4));
        if (row0 + r < N)
            *reinterpret_cast<float4_t *>(p.qs + (row0 + r) * RW + d) =
                *reinterpret_cast<const float4_t *>(out[0] + r * TLX + d) * p.q_scale;
    }
    const int D = RW / p.H;
    for (int t = threadIdx.x; t < TM * p.H; t += RT) {
        const int r = t / p.H, h = t - r * p.H;
        if (row0 + r >= N) break;
        float alpha = 0.f;
        for (int d = 0; d < D; d += 4) {                        // (the order of the exponent kernel)
            const float4 qv = *reinterpret_cast<const float4 *>(out[0] + r * TLX + h * D + d);
            const float4 wv = *reinterpret_cast<const float4 *>(p.w_pos + h * D + d);
            alpha += (qv.x * wv.x + qv.y * wv.y) + (qv.z * wv.z + qv.w * wv.w);
        }
        const int64_t at = (row0 + r) * p.H + h;
        if (p.normalize && stored) alpha = (alpha + shift) * scale;
        if (!p.normalize || stored) {
            if (p.alpha_n) p.alpha_n[at] = alpha;
            p.a[at] = positive_map(alpha, p.func, p.beta, p.lb) * p.coef;
        } else {
            put_raw(p.a + at, alpha);
        }
    }
    if (!stored) finish_if_last<false>(p, N, (N + TM - 1) / TM, red);
}

// tail: from gy, the gradient behind the block,  gh = (gy W2) where h > 0,  gs = gh W1 + gy,  gatt = gs Wo
__global__ __launch_bounds__(RT) void block_tail_bwd_kernel(TailBwdArgs p)
{
    __shared__ __align__(16) float b0[TM * TLX], b1[TM * TLX], hs[TM * TLH];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int q = lane >> 4, col = 16 * wave + (lane & 15);
    const int64_t row0 = (int64_t)blockIdx.x * TM, N = p.N;
    const unsigned woff = (unsigned)(wave * 2048 + lane * 4) * 4u;
    Weights wa, wb, wc;
    load_weights(wa, p.packed, woff);
    stage16(b0, p.gy, row0, N);
    float open[4][4];                                           // the hidden units of this lane's results
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
        for (int r = 0; r < 4; r++) open[u][r] = p.h[min(row0 + 4 * q + r, N - 1) * RF + u * RW + col];
    load_weights(wb, p.packed + UNIT_FLOATS, woff);
    __syncthreads();
    const float4_t zero4 = {0.f, 0.f, 0.f, 0.f};
    float4_t acc;
#pragma unroll
    for (int u = 0; u < 4; u++) {
        Weights &cur = u % 3 == 0 ? wa : u % 3 == 1 ? wb : wc, &nxt = u % 3 == 0 ? wc : u % 3 == 1 ? wa : wb;
        load_weights(nxt, p.packed + (u + 2) * UNIT_FLOATS, woff);
        acc = zero4;
        multiply16(acc, cur, b0, TLX, lane);
#pragma unroll
        for (int r = 0; r < 4; r++) hs[(4 * q + r) * TLH + u * RW + col] = open[u][r] > 0.f ? acc[r] : 0.f;
    }
    __syncthreads();
    acc = zero4;
#pragma unroll
    for (int u = 0; u < 4; u++) {
        Weights &cur = u % 3 == 0 ? wb : u % 3 == 1 ? wc : wa, &nxt = u % 3 == 0 ? wa : u % 3 == 1 ? wb : wc;
        if (u < 3) load_weights(nxt, p.packed + (6 + u) * UNIT_FLOATS, woff);
        multiply16(acc, cur, hs + u * RW, TLH, lane);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) b1[(4 * q + r) * TLX + col] = acc[r] + b0[(4 * q + r) * TLX + col];
    __syncthreads();
    acc = zero4;
    multiply16(acc, wc, b1, TLX, lane);                         // (unit 8)
#pragma unroll
    for (int r = 0; r < 4; r++) b0[(4 * q + r) * TLX + col] = acc[r];
    __syncthreads();
    unstage16(p.gatt, RW, b0, TLX, row0, N);
    unstage16(p.gs, RW, b1, TLX, row0, N);
#pragma unroll
    for (int u = 0; u < 4; u++) unstage16(p.gh + u * RW, RF, hs + u * RW, TLH, row0, N);
}

// head: g_alpha = ga rho'(alpha_n) coef scale,  gq = g_alpha w_pos + gqs q_scale,  gx = gq Wq + gk Wk + gv Wv + carry
__global__ __launch_bounds__(RT) void block_head_bwd_kernel(HeadBwdArgs p)
{
    __shared__ __align__(16) float b[3][TM * TLX];              // gq, gk, gv
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int q = lane >> 4, col = 16 * wave + (lane & 15);
    const int64_t row0 = (int64_t)blockIdx.x * TM, N = p.N;
    const unsigned woff = (unsigned)(wave * 2048 + lane * 4) * 4u;
    const float *packed = p.packed + UNIT_QUERY * UNIT_FLOATS;
    Weights wt[3];
    load_weights(wt[0], packed, woff);
    const float4_t zero4 = {0.f, 0.f, 0.f, 0.f};
    const int r_ = threadIdx.x / (RW / 4), d = 4 * (threadIdx.x % (RW / 4));
    const bool on = row0 + r_ < N;
    const int64_t row = min(row0 + r_, N - 1), in = row * RW + d;
    const int D = RW / p.H;
    {
        const float4_t sv = p.gqs ? *reinterpret_cast<const float4_t *>(p.gqs + in) : zero4;
        const float4_t wv = *reinterpret_cast<const float4_t *>(p.w_pos + d);
        float g_alpha = 0.f;
        if (p.ga) {
            const int64_t ah = row * p.H + d / D;               // (D is a multiple of 4)
            g_alpha = p.ga[ah] * positive_map_slope(p.alpha_n[ah], p.func, p.beta, p.lb) * p.coef;
            if (p.used) g_alpha *= p.used[0];
            if (on && d % D == 0) p.g_alpha[ah] = g_alpha;
        }
        float4_t gq = sv * p.q_scale;
#pragma unroll
        for (int i = 0; i < 4; i++) gq[i] = fmaf(wv[i], g_alpha, gq[i]);     // (rounded as gauss_exponents_bwd_kernel does)
        *reinterpret_cast<float4_t *>(&b[0][r_ * TLX + d]) = gq;
        if (on) *reinterpret_cast<float4_t *>(p.gq + in) = gq;
        *reinterpret_cast<float4_t *>(&b[1][r_ * TLX + d]) = p.gk ? *reinterpret_cast<const float4_t *>(p.gk + in) : zero4;
        *reinterpret_cast<float4_t *>(&b[2][r_ * TLX + d]) = p.gv ? *reinterpret_cast<const float4_t *>(p.gv + in) : zero4;
    }
    load_weights(wt[1], packed + UNIT_FLOATS, woff);
    load_weights(wt[2], packed + 2 * UNIT_FLOATS, woff);
    __syncthreads();
    float4_t acc = zero4;
#pragma unroll
    for (int u = 0; u < 3; u++) multiply16(acc, wt[u], b[u], TLX, lane);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; r++) b[0][(4 * q + r) * TLX + col] = acc[r];
    __syncthreads();
    if (on) {
        float4_t v = *reinterpret_cast<const float4_t *>(&b[0][r_ * TLX + d]);
        if (p.carry) v += *reinterpret_cast<const float4_t *>(p.carry + in);
        *reinterpret_cast<float4_t *>(p.gx + in) = v;
    }
}

// gw_pos = sum over atoms of g_alpha q: 16 columns a work-group; shares of 256 / H atoms each, 64 side by side, their
// atoms in ascending order, the even and the odd shares added up in order (as the exponent kernels' backward does).
__global__ __launch_bounds__(1024) void head_weight_grad_kernel(const float *__restrict__ g_alpha, const float *__restrict__ q,
                                                                int64_t N, int H, float *__restrict__ gw)
{
#pragma clang fp contract(off)
    __shared__ float run[64][17];
    const int c = threadIdx.x & 15, g = threadIdx.x >> 4, col = blockIdx.x * 16 + c;
    const int h = col / (RW / H);
    const int64_t atoms = 256 / H;
    float s0 = 0.f, s1 = 0.f;
    for (int64_t first = 0; first < N; first += 64 * atoms) {
        const int64_t i0 = first + g * atoms, i1 = min(i0 + atoms, N);
        float s = 0.f;
        int64_t i = i0;
        for (; i + 8 <= i1; i += 8) {        // (sixteen at a time: 15.6 instead of 8.5 us at 1774 atoms)
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = g_alpha[(i + u) * H + h] * q[(i + u) * RW + col];
#pragma unroll
            for (int u = 0; u < 8; u++) s += v[u];
        }
        for (; i < i1; i++) s += g_alpha[i * H + h] * q[i * RW + col];
        __syncthreads();
        run[g][c] = s;                       // (shares past the end: zero)
        __syncthreads();
        if (g == 0) {
            for (int k = 0; k < 64; k += 2) {
                s0 += run[k][c];
                s1 += run[k + 1][c];
            }
        }
    }
    if (g == 0) gw[col] = s0 + s1;
}

// Mean over a crystal's atoms and the regression head, one work-group per crystal: 32 lanes x 16 bytes
// read an atom's row, sixteen atoms side by side; a row of a head matrix is one 512-byte read of half a
// wavefront, requested before the mean so that nothing but the atoms' rows is waited for.  (As a mean and
// two linear launches 17 us at 128 crystals, all latency.)
constexpr int PH_T = 512, PH_G = PH_T / 32;
__global__ __launch_bounds__(PH_T) void pool_head_kernel(PoolHeadArgs p)
{
    __shared__ __align__(16) float part[PH_G][RW];
    __shared__ __align__(16) float top[RW];
    const int64_t b = blockIdx.x;
    const int g = threadIdx.x >> 5, piece = threadIdx.x & 31;
    const int64_t r0 = p.start_n[b], r1 = p.start_n[b + 1];
    float4_t wh[RW / PH_G];
    float bh[RW / PH_G];
    if (p.hidden) {
#pragma unroll
        for (int i = 0; i < RW / PH_G; i++) {
            wh[i] = *reinterpret_cast<const float4_t *>(p.w_head + (i * PH_G + g) * RW + 4 * piece);
            bh[i] = p.b_head ? p.b_head[i * PH_G + g] : 0.f;
        }
    }
    float4_t s[4];
#pragma unroll
    for (int u = 0; u < 4; u++) s[u] = float4_t{0.f, 0.f, 0.f, 0.f};
    int64_t r = r0 + g;
    for (; r + 3 * PH_G < r1; r += 4 * PH_G)
#pragma unroll
        for (int u = 0; u < 4; u++) s[u] += *reinterpret_cast<const float4_t *>(p.x + (r + PH_G * u) * RW + 4 * piece);
#pragma unroll
    for (int u = 0; u < 3; u++)
        if (r + PH_G * u < r1) s[u] += *reinterpret_cast<const float4_t *>(p.x + (r + PH_G * u) * RW + 4 * piece);
    *reinterpret_cast<float4_t *>(&part[g][4 * piece]) = (s[0] + s[1]) + (s[2] + s[3]);
    __syncthreads();
    if (threadIdx.x < RW) {
        float t = part[0][threadIdx.x];
#pragma unroll
        for (int i = 1; i < PH_G; i++) t += part[i][threadIdx.x];
        top[threadIdx.x] = t / (float)(r1 - r0);
    }
    __syncthreads();
    float4_t xv = *reinterpret_cast<const float4_t *>(&top[4 * piece]);
    auto dot = [&](const float4_t wv) {
        float d = (xv[0] * wv[0] + xv[1] * wv[1]) + (xv[2] * wv[2] + xv[3] * wv[3]);
        d += dpp_f<DPP_QUAD_1032, 0xF>(0.f, d);
        d += dpp_f<DPP_QUAD_2301, 0xF>(0.f, d);
        d += dpp_f<DPP_ROW_ROR4, 0xF>(0.f, d);
        d += dpp_f<DPP_ROW_ROR8, 0xF>(0.f, d);
        return d + __shfl_xor(d, 16, 32);
    };
    if (p.hidden) {
        __syncthreads();                                        // everyone holds its piece of the mean
#pragma unroll
        for (int i = 0; i < RW / PH_G; i++) {
            const float v = dot(wh[i]) + bh[i];
            if (piece == 0) top[i * PH_G + g] = v < 0.f ? 0.f : v;
        }
        __syncthreads();
        xv = *reinterpret_cast<const float4_t *>(&top[4 * piece]);
    }
    for (int64_t o = g; o < p.targets; o += PH_G) {
        const float v = dot(*reinterpret_cast<const float4_t *>(p.w_last + o * RW + 4 * piece))
                        + (p.b_last ? p.b_last[o] : 0.f);
        if (piece == 0) p.out[b * p.targets + o] = v;
    }
}

template <int T, bool SPREAD>
void launch_rows(const RowsArgs &p, int source, bool head, unsigned grid, hipStream_t st)
{
    if (source == ROWS_TAIL && head) block_rows_kernel<T, ROWS_TAIL, true, SPREAD><<<grid, RT, 0, st>>>(p);
    else if (source == ROWS_TAIL) block_rows_kernel<T, ROWS_TAIL, false, false><<<grid, RT, 0, st>>>(p);
    else if (source == ROWS_EMBED) block_rows_kernel<T, ROWS_EMBED, true, SPREAD><<<grid, RT, 0, st>>>(p);
    else block_rows_kernel<T, ROWS_PLAIN, true, SPREAD><<<grid, RT, 0, st>>>(p);
}

}  // namespace

namespace cf {

bool block_rows_served(int64_t width, int64_t ff, int64_t H)
{
    return width == RW && ff == RF && H >= 1 && RW % H == 0 && (RW / H) % 4 == 0;
}

int launch_forward_prologue(const PackArgs &k, PrologueArgs p, hipStream_t st)
{
    p.live_E = live_edges(p.E);
    const int64_t grid = (int64_t)(k.blocks + (k.w_embed ? 1 : 0)) * (SPLIT_TILES / SPLIT_WAVES) + (p.E + 255) / 256 + (p.B + 255) / 256;
    CF_REQUIRE(grid < (1ll << 31), CF_ERR_UNSUPPORTED, "forward: too many edges");
    forward_prologue_kernel<<<(unsigned)grid, 256, 0, st>>>(k, p);
    CF_CHECK_LAUNCH("forward: prologue");
    return CF_OK;
}

int launch_block_rows(RowsArgs p, hipStream_t st)
{
    const int source = p.packed_tail ? ROWS_TAIL : (p.packed_embed ? ROWS_EMBED : ROWS_PLAIN);
    const bool head = p.packed_head != nullptr;
    p.live_N = live_atoms(p.N);
    const int64_t cus = device_cu_count();
    // 32 rows a tile beyond one round of 16 (a tile a CU): 257 to 512 tiles of 16 are two rounds, the second short of
    // work, and ask for the weights twice as often.  At 5.2 thousand rows 21.5 us a launch against 28.6; up to one round 16 are
    // better, with all CUs at work (1774 rows: 13.7 us, on 111 of them, and a tile of 32 is the 21.5).
    // (Live rows are somewhere below the capacity; a tile has at most 256 exponents, see complete_groups.)
    const int T = !p.live_N && p.N > 16 * cus && p.H <= 8 ? 2 : 1;
    int64_t grid = (p.N + 16 * T - 1) / (16 * T);
    if (p.live_N && grid > 2 * cus) grid = 2 * cus;             // a capacity: stride over the tiles that exist
    CF_REQUIRE(grid < (1ll << 31), CF_ERR_UNSUPPORTED, "block rows: too many atoms");
    const bool spread = head && p.normalize && spread_groups(p.N * p.H);
    p.apart = spread && (!p.live_N || spread_groups(p.N * p.H / 4));
    if (spread && T == 2) launch_rows<2, true>(p, source, head, (unsigned)grid, st);
    else if (spread) launch_rows<1, true>(p, source, head, (unsigned)grid, st);
    else if (T == 2) launch_rows<2, false>(p, source, head, (unsigned)grid, st);
    else launch_rows<1, false>(p, source, head, (unsigned)grid, st);
    CF_CHECK_LAUNCH("block rows");
    if (p.apart) {
        finish_exponents_kernel<<<(unsigned)((p.N * p.H + FINISH_VALUES - 1) / FINISH_VALUES), FINISH_T, 0, st>>>(p);
        CF_CHECK_LAUNCH("block rows: exponents");
    }
    return CF_OK;
}

bool pool_head_served(int64_t width, int64_t hidden) { return width == RW && (hidden == 0 || hidden == RW); }

int launch_pool_head(const PoolHeadArgs &p, int64_t B, hipStream_t st)
{
    CF_REQUIRE(B >= 1 && B < (1ll << 31), CF_ERR_UNSUPPORTED, "pooling and head: bad crystal count");
    pool_head_kernel<<<(unsigned)B, PH_T, 0, st>>>(p);
    CF_CHECK_LAUNCH("pooling and head");
    return CF_OK;
}

}  // namespace cf

extern "C" int64_t cf_pack_blocks_floats(int64_t blocks) { return blocks < 0 ? -1 : blocks * cf::PACKED_BLOCK; }

extern "C" int cf_pack_blocks(int64_t blocks, const float *const *weights, float *packed, float *packed_bwd,
                              int32_t *zero_words, int64_t words, void *stream)
{
    CF_REQUIRE(blocks >= 0 && words >= 0, CF_ERR_INVALID_ARGUMENT, "cf_pack_blocks: negative size");
    if (blocks == 0) return CF_OK;
    CF_REQUIRE(weights && packed && (words == 0 || zero_words), CF_ERR_INVALID_ARGUMENT, "cf_pack_blocks: null pointer");
    for (int64_t first = 0; first < blocks; first += cf::PACK_BLOCKS) {
        cf::PackArgs a{};
        a.blocks = (int)(blocks - first < cf::PACK_BLOCKS ? blocks - first : cf::PACK_BLOCKS);
        for (int i = 0; i < a.blocks; i++) {
            const float *const *w = weights + 6 * (first + i);
            for (int k = 0; k < 6; k++)
                CF_REQUIRE(w[k], CF_ERR_INVALID_ARGUMENT, "cf_pack_blocks: null weight in block %lld", (long long)(first + i));
            a.block[i] = cf::PackSource{w[0], w[1], w[2], w[3], w[4], w[5]};
        }
        a.packed = packed + first * cf::PACKED_BLOCK;
        a.packed_bwd = packed_bwd ? packed_bwd + first * cf::PACKED_BLOCK : nullptr;
        if (first == 0) {
            a.zero = (unsigned *)zero_words;
            a.words = words;
        }
        const dim3 grid(PACK_GRID, (unsigned)a.blocks, a.packed_bwd ? 2 : 1);
        pack_weights_kernel<<<grid, 256, 0, (hipStream_t)stream>>>(a);
        CF_CHECK_LAUNCH("cf_pack_blocks");
    }
    return CF_OK;
}

extern "C" int cf_block_head(const float *x, int64_t N, int64_t H, const float *packed, const float *b_in,
                             const float *w_pos, float *gauss_scale, int normalize, int update_stats, int positive_func,
                             float beta, float lower_bound, float coef, float q_scale, float *part, int32_t *counter,
                             float *q, float *qs, float *k, float *v, float *a, float *alpha_n, float *used, void *stream)
{
    CF_REQUIRE(N >= 0 && cf::block_rows_served(RW, RF, H), CF_ERR_UNSUPPORTED, "cf_block_head: N=%lld H=%lld not served",
               (long long)N, (long long)H);
    CF_REQUIRE(positive_func >= 0 && positive_func <= 2 && lower_bound < 1.0f, CF_ERR_UNSUPPORTED,
               "cf_block_head: positive map not served");
    if (N == 0) return CF_OK;
    CF_REQUIRE(x && packed && w_pos && q && qs && k && v && a && (!normalize || (gauss_scale && part && counter)),
               CF_ERR_INVALID_ARGUMENT, "cf_block_head: null pointer");
    const int64_t grid = (N + TM - 1) / TM;
    CF_REQUIRE(grid < (1ll << 31), CF_ERR_UNSUPPORTED, "cf_block_head: too many rows");
    cf::RowsArgs r{};
    r.N = N; r.H = (int)H; r.x = x; r.packed_head = packed; r.b_in = b_in; r.w_pos = w_pos; r.gauss_scale = gauss_scale;
    r.normalize = normalize; r.update_stats = update_stats; r.func = positive_func;
    r.beta = beta; r.lb = lower_bound; r.coef = coef; r.q_scale = q_scale;
    r.part = part; r.counter = (unsigned *)counter;
    r.q = q; r.qs = qs; r.k = k; r.v = v; r.a = a; r.alpha_n = alpha_n; r.used = used;
    block_head_train_kernel<<<(unsigned)grid, RT, 0, (hipStream_t)stream>>>(r);
    CF_CHECK_LAUNCH("cf_block_head");
    return CF_OK;
}

extern "C" int cf_block_tail(const float *att, const float *x, int64_t N, const float *packed, const float *bo,
                             const float *b1, const float *b2, float *s, float *h, float *y, void *stream)
{
    CF_REQUIRE(N >= 0, CF_ERR_INVALID_ARGUMENT, "cf_block_tail: negative size");
    if (N == 0) return CF_OK;
    CF_REQUIRE(att && x && packed && s && h && y, CF_ERR_INVALID_ARGUMENT, "cf_block_tail: null pointer");
    const int64_t grid = (N + TM - 1) / TM;
    CF_REQUIRE(grid < (1ll << 31), CF_ERR_UNSUPPORTED, "cf_block_tail: too many rows");
    cf::RowsArgs r{};
    r.N = N; r.H = 1; r.att = att; r.x = x; r.packed_tail = packed; r.bo = bo; r.b1 = b1; r.b2 = b2;
    r.s = s; r.h = h; r.y = y;
    block_tail_train_kernel<<<(unsigned)grid, RT, 0, (hipStream_t)stream>>>(r);
    CF_CHECK_LAUNCH("cf_block_tail");
    return CF_OK;
}

extern "C" int cf_block_tail_bwd(const float *gy, const float *h, int64_t N, const float *packed_bwd, float *gh, float *gs,
                                 float *gatt, void *stream)
{
    CF_REQUIRE(N >= 0, CF_ERR_INVALID_ARGUMENT, "cf_block_tail_bwd: negative size");
    if (N == 0) return CF_OK;
    CF_REQUIRE(gy && h && packed_bwd && gh && gs && gatt, CF_ERR_INVALID_ARGUMENT, "cf_block_tail_bwd: null pointer");
    const cf::TailBwdArgs p{N, gy, h, packed_bwd, gh, gs, gatt};
    const int64_t grid = (N + TM - 1) / TM;
    CF_REQUIRE(grid < (1ll << 31), CF_ERR_UNSUPPORTED, "cf_block_tail_bwd: too many rows");
    block_tail_bwd_kernel<<<(unsigned)grid, RT, 0, (hipStream_t)stream>>>(p);
    CF_CHECK_LAUNCH("cf_block_tail_bwd");
    return CF_OK;
}

extern "C" int cf_block_head_bwd(const float *ga, const float *gqs, const float *gk, const float *gv, const float *carry,
                                 const float *q, const float *w_pos, const float *alpha_n, const float *used, int64_t N,
                                 int64_t H, const float *packed_bwd, int positive_func, float beta, float lower_bound,
                                 float coef, float q_scale, float *g_alpha, float *gq, float *gx, float *gw_pos,
                                 void *stream)
{
    CF_REQUIRE(N >= 0 && cf::block_rows_served(RW, RF, H), CF_ERR_UNSUPPORTED,
               "cf_block_head_bwd: N=%lld H=%lld not served", (long long)N, (long long)H);
    CF_REQUIRE(positive_func >= 0 && positive_func <= 2 && lower_bound < 1.0f, CF_ERR_UNSUPPORTED,
               "cf_block_head_bwd: positive map not served");
    CF_REQUIRE((N == 0 || (w_pos && packed_bwd && gq && gx)) && (!ga || (q && alpha_n && g_alpha && gw_pos)),
               CF_ERR_INVALID_ARGUMENT, "cf_block_head_bwd: null pointer");
    if (N == 0) return CF_OK;
    hipStream_t st = (hipStream_t)stream;
    const int64_t grid = (N + TM - 1) / TM;
    CF_REQUIRE(grid < (1ll << 31), CF_ERR_UNSUPPORTED, "cf_block_head_bwd: too many rows");
    const cf::HeadBwdArgs p{N, (int)H, positive_func, beta, lower_bound, coef, q_scale, ga, gqs, gk, gv, carry, w_pos,
                            alpha_n, used, packed_bwd, g_alpha, gq, gx};
    block_head_bwd_kernel<<<(unsigned)grid, RT, 0, st>>>(p);
    CF_CHECK_LAUNCH("cf_block_head_bwd");
    if (ga) {
        head_weight_grad_kernel<<<RW / 16, 1024, 0, st>>>(g_alpha, q, N, (int)H, gw_pos);
        CF_CHECK_LAUNCH("cf_block_head_bwd: weight gradient");
    }
    return CF_OK;
}
