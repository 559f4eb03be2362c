// The activation quantiser on 32-blocks that lie 4 consecutive values to a lane in 8 adjacent lanes
// (crates/strix-backend-rocm/src/kernels.rs:75-96: d = amax / 127, q = clamp(rint(x / d), -127, 127)).  Every lane of a wave calls these.
#pragma once
#include "detmath.h"
#include "gemv_body.h"

namespace smx {

// The largest of 8 adjacent lanes' values, through DPP (a lane swap through LDS, as __shfl_xor makes, is a round trip each).
__device__ __forceinline__ float max8(float a) {
    a = fmaxf(a, dpp_f<0xB1>(a));
    a = fmaxf(a, dpp_f<0x4E>(a));
    return fmaxf(a, dpp_f<0x141>(a));   // lane 7 - i: the other four
}
struct Quant4 {
    int packed;   // the lane's four quants
    float d;      // the block's scale
    int sum;      // of the lane's four quants
};
__device__ __forceinline__ Quant4 quantize4(float4 v) {
    const float a = max8(fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
    const float d = a / 127.f;
    const float inv = d > 0.f ? 1.f / d : 0.f;
    const int q0 = max(-127, min(127, (int)rintf(v.x * inv)));
    const int q1 = max(-127, min(127, (int)rintf(v.y * inv)));
    const int q2 = max(-127, min(127, (int)rintf(v.z * inv)));
    const int q3 = max(-127, min(127, (int)rintf(v.w * inv)));
    return Quant4{(q0 & 0xff) | ((q1 & 0xff) << 8) | ((q2 & 0xff) << 16) | ((q3 & 0xff) << 24), d, q0 + q1 + q2 + q3};
}
// Item i (4 values; 8 items to a block, the same 8 lanes') out: quants, and by the block's first lane its scale and the packed sums
// of its two 16-element halves (xs may be null).
__device__ __forceinline__ void put_quant4(const Quant4& q, bool live, size_t i, int* xq4, float* xd, int* xs) {
    int s = q.sum + dpp_i<0xB1>(q.sum);
    s += dpp_i<0x4E>(s);
    const int other = dpp_i<0x141>(s);
    if (!live) return;
    xq4[i] = q.packed;
    if ((i & 7) == 0) {
        xd[i >> 3] = q.d;
        if (xs) xs[i >> 3] = (s & 0xffff) | (other << 16);
    }
}

}  // namespace smx
