// Cell volume, reciprocal vectors and their lengths of a crystal.
#pragma once
#include "cf_common.h"

namespace cf {

// One thread per crystal.  Products and sums are kept un-contracted and in the
// term order of models/indexed_latticeformer_encoder.py:34-44 so the volume is
// the one the stock elementwise expression gives.
__device__ __forceinline__ void lattice_geometry_of(const float *trans, int64_t b, float *vcell, float *recip, float *rvlen)
{
#pragma clang fp contract(off)
    const float *m = trans + b * 9;
    const float m00 = m[0], m01 = m[1], m02 = m[2];
    const float m10 = m[3], m11 = m[4], m12 = m[5];
    const float m20 = m[6], m21 = m[7], m22 = m[8];
    float det = m00 * m11 * m22;
    det = det + m01 * m12 * m20;
    det = det + m02 * m10 * m21;
    det = det - m02 * m11 * m20;
    det = det - m00 * m12 * m21;
    det = det - m01 * m10 * m22;
    if (vcell) vcell[b] = det;
    // b1 = 2 pi (a2 x a3) / V and cyclic (models/indexed_latticeformer_encoder.py:206-212)
    const float s = (1.0f / det) * 6.283185307179586f;
    float c[9];
    c[0] = m11 * m22 - m12 * m21;
    c[1] = m12 * m20 - m10 * m22;
    c[2] = m10 * m21 - m11 * m20;
    c[3] = m21 * m02 - m22 * m01;
    c[4] = m22 * m00 - m20 * m02;
    c[5] = m20 * m01 - m21 * m00;
    c[6] = m01 * m12 - m02 * m11;
    c[7] = m02 * m10 - m00 * m12;
    c[8] = m00 * m11 - m01 * m10;
#pragma unroll
    for (int r = 0; r < 3; r++) {
        const float x = c[3 * r] * s, y = c[3 * r + 1] * s, z = c[3 * r + 2] * s;
        if (recip) {
            recip[b * 9 + 3 * r] = x;
            recip[b * 9 + 3 * r + 1] = y;
            recip[b * 9 + 3 * r + 2] = z;
        }
        if (rvlen) rvlen[b * 3 + r] = sqrtf(x * x + y * y + z * z);
    }
}

}  // namespace cf
