// The encoding of an inference forward (real_enc_infer.hip): launchers that cf_forward uses.
#pragma once
#include "cf_common.h"

namespace cf {

constexpr int INFER_WEIGHT_BLOCKS = 32;    // blocks per launch_infer_stage
bool infer_served(int64_t N, int64_t E, int64_t H, int64_t K, int64_t D, bool boxes, int lattice_range, double weakest,
                  int64_t limit);
constexpr int64_t INFER_LEAST_SLICE = 4096;     // pairs
int64_t infer_slice(int64_t U, bool boxes, int64_t limit);
int64_t infer_units_bytes(int64_t U, bool boxes, int64_t limit);
int64_t infer_weights_bytes(int64_t H, int64_t K, int64_t D);
int launch_infer_stage(const float *rpos, const float *tvecs, const float *rvlen, const int64_t *pairs, int64_t U,
                       int64_t before, int64_t slice, double weakest, float cutoff, int lattice_range, int min_range,
                       void *staged, int blocks, const float *const *weights, const int *bins, int64_t H, int64_t D,
                       void *packed, int64_t packed_bytes, hipStream_t st);
int launch_real_enc_infer(const float *a_ik, const float *rpos, const float *tvecs, const int64_t *pairs, int64_t U,
                          int64_t before, int64_t slice, int64_t H, int64_t K, int64_t D, double dist_max, double wscale,
                          const void *packed, const float *rvlen, float cutoff, int lattice_range, int min_range,
                          double weakest, const void *staged, float *z, float *v, hipStream_t st);

}  // namespace cf
