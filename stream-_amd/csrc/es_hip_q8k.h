// es_quantize_q8_K (src/es_q2k.c:102-125) of a 256-element block held by 32 consecutive lanes (aligned at 32), eight consecutive
// elements each: id = 127 / amax, q = lrintf(v * id) clamped to +-127, d = amax / 127, bsums. A zero block is all zeros.
#pragma once
#include "es_hip_common.h"

namespace esq {

__device__ __forceinline__ uint32_t pack_i8(int a, int b, int c, int d) {
    return (uint32_t)(a & 0xff) | (uint32_t)(b & 0xff) << 8 | (uint32_t)(c & 0xff) << 16 | (uint32_t)d << 24;
}

// the maximum magnitude over the lane's eight values and its quad's 32 (a maximum is exact in any order)
__device__ __forceinline__ float amax_quad(const float (&v)[8]) {
    float a = __builtin_fabsf(v[0]);
#pragma unroll
    for (int k = 1; k < 8; k++) a = __builtin_fmaxf(a, __builtin_fabsf(v[k]));
    return group_max<4>(a);
}

// quad: amax_quad(v). lo, hi: the lane's eight codes; bsum: the sum of 16 consecutive codes (this lane's and its pair's); every
// lane of the wave takes part
__device__ __forceinline__ void q8k_from8(const float (&v)[8], float quad, float &d, uint32_t &lo, uint32_t &hi, int &bsum) {
    float a = quad;
    a = __builtin_fmaxf(a, dpp_movf<0x141>(a));   // row_half_mirror, row_mirror: the other quads of the 16 lanes
    a = __builtin_fmaxf(a, dpp_movf<0x140>(a));
    const float amax = __builtin_fmaxf(a, __shfl_xor(a, 16));
    int q[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (amax != 0.0f) {
        const float id = 127.0f / amax;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const int t = static_cast<int>(__builtin_rintf(v[k] * id));   // lrintf: round to nearest even
            q[k] = t > 127 ? 127 : t < -127 ? -127 : t;
        }
    }
    d = amax != 0.0f ? amax / 127.0f : 0.0f;
    lo = pack_i8(q[0], q[1], q[2], q[3]);
    hi = pack_i8(q[4], q[5], q[6], q[7]);
    bsum = group_sum<2>(q[0] + q[1] + q[2] + q[3] + q[4] + q[5] + q[6] + q[7]);
}
__device__ __forceinline__ void q8k_from8(const float (&v)[8], float &d, uint32_t &lo, uint32_t &hi, int &bsum) {
    q8k_from8(v, amax_quad(v), d, lo, hi, bsum);
}

}  // namespace esq
