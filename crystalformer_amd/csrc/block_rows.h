// Arguments and launchers that cf_forward uses beside the C entry points: block_rows.hip and parts of others.
#pragma once
#include "cf_common.h"

namespace cf {

struct RowsArgs {
    int64_t N;
    int H, embed_width;
    const float *att, *x;                     // attention output; block input (or the rows to embed)
    const float *packed_tail, *packed_head;   // packed weights of the block each belongs to (inference: split), null: no such part
    const float *bo, *b1, *b2;                // tail
    const float *packed_embed, *b_embed;      // null: x is the block input itself
    float *y;                                 // tail or embedding: the rows behind it
    const float *b_in, *w_pos;                // head
    float *gauss_scale;
    int normalize, update_stats, func;
    float beta, lb, coef, q_scale;
    int split;                                // heads from H/2 on: factor coef_second, their exponents behind all
    float coef_second;                        //   of the first half's, (N, H/2) each
    float *qs, *k, *v, *a;
    float *s, *h;                             // training: the sum behind the attention, the hidden units,
    float *q, *alpha_n, *used;                //   the query, the normalised alpha, the (scale, shift) applied
    float *part;                              // statistics without stored ones: 3 floats per 256 values of a
    unsigned *counter;                        // zeroed word
    unsigned *groups;                         // inference: such a word per 256 values, left zero again
    int apart;                                // set by the launcher: such exponents are mapped by a launch of their own
    const int64_t *live_N;                    // set by the launcher
};

constexpr int PACK_BLOCKS = 32;               // blocks per packing launch (48 bytes of kernel arguments each)
constexpr int64_t PACKED_BLOCK = 12 * 128 * 128;   // floats a block
constexpr int64_t SPLIT_BLOCK = PACKED_BLOCK + 12 * 128;   // with its columns' exponents, for cf_forward's row kernel
struct PackSource {
    const float *wo, *w1, *w2, *wq, *wk, *wv;
};
struct PackArgs {
    PackSource block[PACK_BLOCKS];
    int blocks, embed_width;
    const float *w_embed;                     // (128, embed_width <= 128), nullable
    float *packed, *packed_embed;             // blocks x PACKED_BLOCK (the prologue: SPLIT_BLOCK) floats; 128 x 129
    float *packed_bwd;                        // nullable: as packed, for the backward kernels
    unsigned *zero;                           // words to clear, nullable
    int64_t words;
};

struct PrologueArgs {
    int64_t B, E;
    const int64_t *atom_start, *edge_start;
    const float *pos, *trans;
    float *rpos, *vcell, *recip, *rvlen;      // vcell, recip nullable
    const int64_t *live_E;                    // set by the launcher
};
// split packing (packed: blocks x SPLIT_BLOCK floats, packed_embed: 128 x 129), edge offsets (cf_edge_index) and lattice
// geometry (cf_lattice_geometry) at once
int launch_forward_prologue(const PackArgs &k, PrologueArgs p, hipStream_t st);

struct TailBwdArgs {
    int64_t N;
    const float *gy, *h, *packed;
    float *gh, *gs, *gatt;
};

struct HeadBwdArgs {
    int64_t N;
    int H, func;
    float beta, lb, coef, q_scale;
    const float *ga, *gqs, *gk, *gv, *carry;  // nullable each
    const float *w_pos, *alpha_n, *used, *packed;
    float *g_alpha, *gq, *gx;
};

struct PoolHeadArgs {
    const float *x;
    const int64_t *start_n;
    const float *w_head, *b_head, *w_last, *b_last;
    int64_t hidden, targets;
    float *out;
};

bool block_rows_served(int64_t width, int64_t ff, int64_t H);
int launch_block_rows(RowsArgs p, hipStream_t st);
bool pool_head_served(int64_t width, int64_t hidden);
int launch_pool_head(const PoolHeadArgs &p, int64_t B, hipStream_t st);
// fused_dpa.hip: attention whose weights nobody reads.  aij_second != 0: the heads come in two halves with a
// bias (E, H/2) each, the second aij_second floats behind the first, and bij (E, H/2, D) is the first half's.
bool dpa_streams(int64_t N, int64_t H, int64_t E, int64_t D);
int launch_dpa_inference(const float *que, const float *key, const float *val, const float *aij, int64_t aij_second,
                         const float *bij, const int64_t *edges, const int64_t *e_start, int64_t N, int64_t H, int64_t E,
                         int64_t D, float *out, hipStream_t st);

}  // namespace cf
