// Activation quantiser: fp32 rows -> per-32-block Q8 (int8 quants + f32 scale + 16-element sums).
//
// Arithmetic of the reference's device quantisers (crates/strix-backend-rocm/src/kernels.rs:75-96,
// 864-876, 1000-1013): d = amax/127, inv = d > 0 ? 1/d : 0, q = clamp(rint(x*inv), -127, 127).
// Layout differs: quants stay contiguous int8 [m][K]; the block sum the reference keeps per 32
// (kernels.rs:93) is kept as two 16-element sums packed in one dword, which also serves the
// 16-wide sub-blocks of Q6_K.
#include <algorithm>

#include "quant_dev.h"
#include "smx_internal.h"

namespace smx {

// Up to SMX_GEMV_GROUP_MAX rows, each the product of an activation function of one operand and a
// second operand (SwiGLU: silu(a) * b, GeGLU: gelu_tanh(a) * b; kernels.rs:151-226), quantised like
// actquant_kernel below.  Row j goes to xq + j*K, xd / xs + j*K/32.  The arithmetic is the one the
// GEMV staging performs when it runs the producer itself, operation for operation.
struct ProdRows {
    const float4* a[SMX_GEMV_GROUP_MAX];
    const float4* b[SMX_GEMV_GROUP_MAX];
};
__global__ __launch_bounds__(256) void actprod_quant_kernel(const ProdRows R, int kind, int* __restrict__ xq4,
                                                            float* __restrict__ xd, int* __restrict__ xs, int nb32) {
#pragma clang fp contract(off)
    const int j = blockIdx.y;
    const int gid = blockIdx.x * 256 + threadIdx.x;
    const int blk = gid >> 3;
    const bool live = blk < nb32;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f), g = v;
    if (live) {
        v = R.a[j][gid];
        g = R.b[j][gid];
    }
    float4 w;
    if (kind == SMX_ACT_SILU_MUL) {
        w.x = det_silu(v.x) * g.x; w.y = det_silu(v.y) * g.y; w.z = det_silu(v.z) * g.z; w.w = det_silu(v.w) * g.w;
    } else {
        w.x = det_gelu_tanh(v.x) * g.x; w.y = det_gelu_tanh(v.y) * g.y;
        w.z = det_gelu_tanh(v.z) * g.z; w.w = det_gelu_tanh(v.w) * g.w;
    }
    put_quant4(quantize4(w), live, (size_t)j * nb32 * 8 + gid, xq4, xd, xs);
}

// m rmsnorm rows through the quantiser (kernels.rs:101-147 rmsnorm_xquant per row), one workgroup per row.  b: the rmsnorm weight [K] or
// null.  Rows of up to 256 * IT items (4096 values) stay in registers between the two passes over them: 2048 x 3840
// 16.2 -> 13.1 us, and of a dense FFN of 100 tokens (2560 <-> 9728), where the second pass is one more trip to memory, 76.7 -> 74.0.
__global__ __launch_bounds__(256) void rmsnorm_quant_kernel(const float* __restrict__ a, const float* __restrict__ b, float eps,
                                                            int* __restrict__ xq4, float* __restrict__ xd, int* __restrict__ xs, int nb32) {
#pragma clang fp contract(off)
    constexpr int IT = 4;
    __shared__ double red[4];
    const size_t row = blockIdx.x;
    const float* ar = a + row * (size_t)nb32 * 32;
    const int items = nb32 * 8;
    float rs = 1.f;
    const bool held = items <= 256 * IT;
    if (!held) rs = rms_scale((char*)red, ar, nb32 * 32, eps);
    for (int i0 = 0; i0 < items; i0 += 256 * IT) {  // whole 8-lane groups stay together: items % 8 == 0
        float4 v[IT], g[IT];
#pragma unroll
        for (int j = 0; j < IT; j++) {
            const int i = i0 + j * 256 + threadIdx.x;
            v[j] = i < items ? ((const float4*)ar)[i] : make_float4(0.f, 0.f, 0.f, 0.f);
            g[j] = b && i < items ? ((const float4*)b)[i] : make_float4(1.f, 1.f, 1.f, 1.f);
        }
        if (held) rs = rms_scale_held<IT>((char*)red, v, nb32 * 32, eps);
#pragma unroll
        for (int j = 0; j < IT; j++) {
            const int i = i0 + j * 256 + threadIdx.x;
            if (i0 + j * 256 >= items) break;   // the whole workgroup
            const float4 x = v[j], y = g[j];
            const float4 w = make_float4((x.x * rs) * y.x, (x.y * rs) * y.y, (x.z * rs) * y.z, (x.w * rs) * y.w);
            put_quant4(quantize4(w), i < items, row * (size_t)items + i, xq4, xd, xs);
        }
    }
}

int launch_actprod_quant(smx_ctx* c, int kind, const float* const* as, const float* const* bs, int n, size_t K,
                         int8_t* xq, float* xd, int32_t* xs) {
    if (K % 32 != 0 || n < 1 || n > SMX_GEMV_GROUP_MAX) return fail(c, SMX_ERR_ARG, "producer quantiser: %d rows of %zu", n, K);
    if (kind != SMX_ACT_SILU_MUL && kind != SMX_ACT_GEGLU) return fail(c, SMX_ERR_ARG, "producer quantiser: kind %d", kind);
    ProdRows R = {};
    for (int j = 0; j < n; j++) {
        R.a[j] = (const float4*)as[j];
        R.b[j] = (const float4*)bs[j];
    }
    const int nb32 = (int)(K / 32);
    ProfScope ps(c, "actprod_quant");
    hipLaunchKernelGGL(actprod_quant_kernel, dim3((unsigned)((nb32 * 8 + 255) / 256), (unsigned)n), dim3(256), 0, c->stream, R,
                       kind, (int*)xq, xd, (int*)xs, nb32);
    SMX_HIP(c, hipGetLastError());
    return SMX_OK;
}

// The prefill form of the producers (rmsnorm: above; kernels.rs:1174-1187 silu_quant_rows).  The exp-based ones have independent blocks and
// [m][K] operands: their m rows are one long row of actprod_quant_kernel, an item per thread.  Against a workgroup per 512 items of a row
// in a loop over its parts: 2048 x 15360 50.8 -> 45.2 us (283 MB: the memory's rate), 400 x 5888 8.0 -> 6.5, 40 x 3072 3.6 -> 2.9.
int launch_rows_prod_quant(smx_ctx* c, int kind, const float* a, const float* b, size_t m, size_t K, float eps, int8_t* xq,
                           float* xd, int32_t* xs) {
    if (K % 32 != 0 || m == 0 || m > 0x7fffffffu) return fail(c, SMX_ERR_ARG, "producer quantiser: %zu rows of %zu", m, K);
    if (kind != SMX_ACT_RMSNORM && kind != SMX_ACT_SILU_MUL && kind != SMX_ACT_GEGLU)
        return fail(c, SMX_ERR_ARG, "producer quantiser: kind %d", kind);
    ProfScope ps(c, "rows_prod_quant");
    if (kind != SMX_ACT_RMSNORM) {
        if (m * K / 4 > 0x7fffff00u) return fail(c, SMX_ERR_LIMIT, "producer quantiser: %zu rows of %zu exceed the launch limits", m, K);
        ProdRows R = {};
        R.a[0] = (const float4*)a;
        R.b[0] = (const float4*)b;
        hipLaunchKernelGGL(actprod_quant_kernel, dim3((unsigned)((m * K / 4 + 255) / 256)), dim3(256), 0, c->stream, R, kind, (int*)xq, xd, (int*)xs,
                           (int)(m * K / 32));
    } else {
        hipLaunchKernelGGL(rmsnorm_quant_kernel, dim3((unsigned)m), dim3(256), 0, c->stream, a, b, eps, (int*)xq, xd, (int*)xs, (int)(K / 32));
    }
    SMX_HIP(c, hipGetLastError());
    return SMX_OK;
}

// 8 lanes per 32-block, one float4 each: 128-bit loads, 32-bit packed stores.  (Two or four items per thread are no faster.)
__global__ __launch_bounds__(256) void actquant_kernel(const float4* __restrict__ x, int* __restrict__ xq4,
                                                       float* __restrict__ xd, int* __restrict__ xs,
                                                       size_t nblocks) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    const bool live = i < nblocks * 8;
    put_quant4(quantize4(live ? x[i] : make_float4(0.f, 0.f, 0.f, 0.f)), live, i, xq4, xd, xs);
}

int launch_actquant(smx_ctx* c, const float* x, size_t m, size_t K, int8_t* xq, float* xd, int32_t* xs) {
    if (K % 32 != 0) return fail(c, SMX_ERR_ARG, "quantise: row length %zu is not a multiple of 32", K);
    const size_t nblocks = m * (K / 32);
    if (nblocks == 0) return SMX_OK;
    const size_t threads = nblocks * 8;
    const size_t grid = (threads + 255) / 256;
    if (grid > 0x7fffffffu) return fail(c, SMX_ERR_LIMIT, "quantise: %zu blocks exceed the grid limit", nblocks);
    ProfScope ps(c, "actquant");
    hipLaunchKernelGGL(actquant_kernel, dim3((unsigned)grid), dim3(256), 0, c->stream, (const float4*)x, (int*)xq,
                       xd, (int*)xs, nblocks);
    SMX_HIP(c, hipGetLastError());
    return SMX_OK;
}

__global__ __launch_bounds__(256) void copy_kernel(const uint4* __restrict__ src, uint4* __restrict__ dst, size_t n16) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n16; i += (size_t)gridDim.x * 256) dst[i] = src[i];
}

}  // namespace smx

extern "C" int smx_dev_copy(smx_ctx* c, void* dst, const void* src, size_t nbytes) {
    using namespace smx;
    if (!c) return SMX_ERR_ARG;
    if (!dst || !src || nbytes % 16 != 0 || ((uintptr_t)dst | (uintptr_t)src) % 16 != 0)
        return fail(c, SMX_ERR_ARG, "dev_copy: pointers and size must be 16-byte aligned");
    if (nbytes == 0) return SMX_OK;
    const size_t n16 = nbytes / 16;
    const unsigned grid = (unsigned)std::min<size_t>((n16 + 255) / 256, (size_t)c->num_cu * 32);
    ProfScope ps(c, "copy");
    hipLaunchKernelGGL(copy_kernel, dim3(grid), dim3(256), 0, c->stream, (const uint4*)src, (uint4*)dst, n16);
    SMX_HIP(c, hipGetLastError());
    return SMX_OK;
}
