// Q6_K prefill GEMM (also the grouped MoE form): Y[m][N] = Xq . W^T with W kept in its 210-byte superblocks
// (kernels.rs:1688-1735 q6_gemm_moe).
//
// The format scales 16-element sub-blocks: d (f16, one per 256) times sc (int8, one per 16).  Both operands go to the matrix
// cores as f16 (x in [-128, 127] and q - 32 in [-32, 31] are exact there, and so is the fp32 sum of 16 of their products):
//   * v_mfma_f32_32x32x16_f16: K = 16 is one sub-block, its result the exact dot as a float, and
//     acc += dx * (dw0 * I0 + dw1 * I1) takes three VALU operations per output and 32-block.  Bound: these, with the MFMAs
//     (they add up: a SIMD runs both at one power budget).  v_mfma_i32_32x32x16_i8 has the same rate but an integer result,
//     whose exact rescale takes four: 536 against 725 TOPS in a loop of nothing else (the machine floors of bench.py).
//   * The weights are widened to f16 once per workgroup, on their way into LDS (two blocks of a row = 128 bytes); a wave
//     reads its own 32 tokens only, as int8, and widens them itself: 20 operations per block next to 192.
//   * A stage is 4 blocks (half a superblock).  The activations and the scales of a stage are double-buffered, the widened
//     weights by halves of a stage (low nibbles = blocks 0 and 1, high nibbles = 2 and 3), so that two workgroups fit a CU.
//   * NW = 8: a workgroup of 256 tokens, one per CU.  What a stage costs besides its arithmetic is weights: loading, widening and
//     scaling them takes 30 % of the time of the two 128-token workgroups that share a CU (each repeats it), and half as
//     much here.  The barriers cost more (all eight waves meet), most of it given back by the waves' priorities below.
// 2048 tokens x 15360 x 3840: 573 -> 485 us against the integer form, 1000 tokens 318 -> 270 us, 300 tokens x 2560 x 2560 35 -> 29 us.
// 256-token tiles against 128-token ones (same bits): 2048 x 15360 x 3840 501 -> 475 us, 2048 x 3840 x 15360 549 -> 490, 1000 x 15360 x
// 3840 265 -> 241, 512 tokens 138.5 -> 123, 400 x 9728 x 2560 94.4 -> 82; without the priorities 2 % more.
#pragma once
#include "gemm_dev.h"

namespace smx {

typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int Q6_W_BYTES = KB * 128 * 8;   // weight scales of a stage: two floats per row and block
constexpr int q6_lds_bytes(int nw) { return 2 * (nw * 4 * GRP + B_BYTES + Q6_W_BYTES + KB * 32 * nw * 4); }

// four bytes 0..255 -> two pairs of f16 with `off` taken off: 0x6400 | v is the f16 1024 + v
__device__ __forceinline__ void widen_h(unsigned v, _Float16 off, unsigned& lo, unsigned& hi) {
    const v2h o = {off, off};
    lo = __builtin_bit_cast(unsigned, __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, v, 0x04010400u)) - o);
    hi = __builtin_bit_cast(unsigned, __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, v, 0x04030402u)) - o);
}

template <bool DUMP, int NW>
__global__ __launch_bounds__(64 * NW, 2) void gemm_q6_kernel(GemmArgs p) {
    SMX_GEMM_T0;
    constexpr int BM = 32 * NW, A_BYTES = 4 * NW * GRP, Q6_X_BYTES = KB * BM * 4;   // NW 8: a workgroup of 256 tokens, one per CU
    extern __shared__ __align__(16) char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned smem_base = lds_addr(smem);
    const TileAt at = gemm_tile_at(p);
    const WaveRole role = gemm_wave_role(at, wave, NW);
    const int tok0 = at.tok0, row0 = at.row0, M_end = at.M_end, N_end = at.N_end, nt_base = role.nt_base;
    const GemmOperand op = p.op[at.op_i];
    const int s_begin = blockIdx.z * p.stages_per_slice;
    const int s_end = min(p.nb / KB, s_begin + p.stages_per_slice);

    // ---- staging ----
    // activations: global -> LDS directly, as in gemm_i8_kernel
    const int g_rowlo = lane >> 3, g_chunk = ((lane & 7) - g_rowlo) & 7;
    unsigned a_off[4];
#pragma unroll
    for (int ps = 0; ps < 4; ps++) {
        const int ti = min(tok0 + (ps * NW + wave) * 8 + g_rowlo, M_end - 1);
        a_off[ps] = (unsigned)(p.a_rowmap ? p.a_rowmap[ti] : ti) * (unsigned)(p.nb * 32) + g_chunk * 16;
    }
    // quants: thread = [row:7][q:1] reads ql[16q..], ql[32 + 16q..] and qh[16q..] of the stage's half superblock: sub-block q of
    // its four blocks (ggml_quant.rs:417-426).  Scales: thread (row sr, half sh) carries d and the sub-block scales
    // 4 * sh .. 4 * sh + 3 of weight row sr; waves 2 and 3 also the four activation scales of token sr.
    constexpr int QI = 8 / NW;   // 16-byte pieces of ql per thread and stage; blocks of weight scales
    const int q_row = tid / (2 * (NW / 4)), q_p = tid & 1, q_i = NW == 8 ? (tid >> 1) & 1 : 0, sr = tid & 127, sh = tid >> 7;
    const int xr = tid & (BM - 1);
    const unsigned nsb = (unsigned)(p.nb >> 3);   // superblocks of a row (M*K and N*K are below 2^31: launch_gemm, moe_check_shape)
    unsigned q_sb = (unsigned)min(row0 + q_row, N_end - 1) * nsb, s_sb = (unsigned)min(row0 + sr, N_end - 1) * nsb, x_b;
    {
        const int ti = min(tok0 + xr, M_end - 1);
        x_b = (unsigned)(p.a_rowmap ? p.a_rowmap[ti] : ti) * (unsigned)p.nb;
    }
    const bool w_valid = row0 + sr < N_end, x_valid = tok0 + xr < M_end, role_x = wave >= NW / 2;
    uint4 rq0, rq1, rqh, rsx = {0, 0, 0, 0};
    unsigned rsc;
    uint16_t rsd;
    auto issue_a = [&](auto full, int buf, int s) __attribute__((always_inline)) {
        const unsigned sA = __builtin_amdgcn_readfirstlane(smem_base + buf * A_BYTES + wave * GRP);
        const int8_t* xa = p.xq + (size_t)s * (KB * 32);
#pragma unroll
        for (int ps = 0; ps < 4; ps++)   // 8-token groups wholly past the tile's end are not fetched (nothing reads their LDS rows)
            if (decltype(full)::value || (ps * NW + wave) * 8 < role.live_tok) load_to_lds16(xa, a_off[ps], sA, ps * NW * GRP);
    };
    auto issue_w = [&](int s) __attribute__((always_inline)) {
        asm volatile("" : "+v"(q_sb), "+v"(s_sb), "+v"(x_b));   // not hoisted: the address arithmetic is cheaper than registers held across the loop
        const int sb = s >> 1, h = s & 1;
        const char* ql = (const char*)op.wquants + (size_t)sb * 128 + h * 64;
        const unsigned o = q_sb * 128u + q_p * 16 + q_i * 32;
        rq0 = *(const uint4*)(ql + o);
        if constexpr (QI == 2) rq1 = *(const uint4*)(ql + (o + 32u));
        rqh = *(const uint4*)((const char*)op.wqh + (size_t)sb * 64 + h * 32 + (q_sb * 64u + q_p * 16));
        rsd = *(const uint16_t*)((const char*)(op.wscales + sb) + s_sb * 2u);
        const char* psc = (const char*)op.wsc + (size_t)sb * 16 + h * 8 + (s_sb * 16u + sh * (2 * QI));
        if constexpr (QI == 2) rsc = *(const unsigned*)psc;
        else rsc = *(const uint16_t*)psc;
        if (role_x) rsx = *(const uint4*)((const char*)(p.xd + (size_t)s * KB) + x_b * 4u);
    };
    // blocks 2 * h and 2 * h + 1 of the stage, widened; 16-byte chunk c (= block 1b, sub-block 1b, half 1b) of row r at slot (c + r) % 8
    auto write_b = [&](auto hc) __attribute__((always_inline)) {
        constexpr int h = decltype(hc)::value;
        char* b = smem + 2 * A_BYTES + h * B_BYTES + (q_row >> 3) * GRP + (q_row & 7) * 128;
#pragma unroll
        for (int ii = 0; ii < QI; ii++) {
            const int i = QI == 2 ? ii : q_i;
            const uint4 q = ii ? rq1 : rq0;
            const unsigned v[4] = {q.x, q.y, q.z, q.w}, g[4] = {rqh.x, rqh.y, rqh.z, rqh.w};
#pragma unroll
            for (int e = 0; e < 2; e++) {
                uint4 o;
                const int hs = 2 * (2 * h + i);
                const auto bits = [&](int k) {
                    const unsigned hi = QI == 1 ? ((g[k] >> (2 * i)) >> (4 * h)) << 4 : hs < 4 ? g[k] << (4 - hs) : g[k] >> (hs - 4);
                    return ((v[k] >> (4 * h)) & 0x0f0f0f0fu) | (hi & 0x30303030u);
                };
                widen_h(bits(2 * e), (_Float16)1056.f, o.x, o.y);
                widen_h(bits(2 * e + 1), (_Float16)1056.f, o.z, o.w);
                *(uint4*)(b + ((i * 4 + q_p * 2 + e + q_row) & 7) * 16) = o;
            }
        }
    };
    auto write_scales = [&](int buf) __attribute__((always_inline)) {
        float2* sdw = (float2*)(smem + 2 * (A_BYTES + B_BYTES) + buf * Q6_W_BYTES);
        const float d = w_valid ? h2f_(rsd) : 0.f;   // d * sc is exact in fp32 (11 x 8 significant bits)
        const auto sc = [&](int j) { return d * (float)(int)(signed char)(rsc >> (8 * j)); };
#pragma unroll
        for (int j = 0; j < QI; j++) sdw[(QI * sh + j) * 128 + sr] = make_float2(sc(2 * j), sc(2 * j + 1));
        if (role_x) {
            float* sdx = (float*)(smem + 2 * (A_BYTES + B_BYTES + Q6_W_BYTES) + buf * Q6_X_BYTES);
            const unsigned v[4] = {rsx.x, rsx.y, rsx.z, rsx.w};
#pragma unroll
            for (int j = 0; j < KB; j++) sdx[j * BM + xr] = x_valid ? __uint_as_float(v[j]) : 0.f;
        }
    };

    // ---- arithmetic ----
    const int half = lane >> 5, col = lane & 31;
    const int row_off = (col >> 3) * GRP + (col & 7) * 128;
    float acc[4][16];
#pragma unroll
    for (int nt = 0; nt < 4; nt++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[nt][i] = 0.f;
    v8h af[2];       // the tokens' fragments of the block whose MFMAs are being issued, per sub-block
    int2 araw[2];    // the next block's, before widening
    // Activation scales of the 16 tokens this lane accumulates, of the block whose products are being scaled.  (As one per lane,
    // read through a row broadcast, they cost a register and one read instead of four; but a broadcast multiply-add takes a SIMD
    // 4 cycles and keeps the other wave's from issuing beside it, where a plain one takes 2: 1000 x 15360 x 3840 261 -> 254 us.)
    float4 dx[4];
    v4i bf[2][2];    // weight fragments, two units in turn, per sub-block
    float2 dw[4];    // weight scales of this lane's row, four units in turn
    v16f d[2][2];    // products, two units in turn, per sub-block
    // unit g of a stage: row tile g % NT of block g / NT
    auto read_unit = [&](auto ntc, int g, int buf) __attribute__((always_inline)) {
        constexpr int NT = decltype(ntc)::value;
        const int bi = (g / NT) & 3, nt = g % NT;
        if (nt == 0) {
            const char* sA = smem + buf * A_BYTES + role.tw * 4 * GRP + row_off + half * 8;
            araw[0] = *(const int2*)(sA + ((2 * bi + col) & 7) * 16);
            araw[1] = *(const int2*)(sA + ((2 * bi + 1 + col) & 7) * 16);
        }
        const char* sB = smem + 2 * A_BYTES + (bi >> 1) * B_BYTES + (nt_base + nt) * 4 * GRP + row_off;
        bf[g & 1][0] = *(const v4i*)(sB + (((bi & 1) * 4 + half + col) & 7) * 16);
        bf[g & 1][1] = *(const v4i*)(sB + (((bi & 1) * 4 + 2 + half + col) & 7) * 16);
        dw[g & 3] = ((const float2*)(smem + 2 * (A_BYTES + B_BYTES) + buf * Q6_W_BYTES))[bi * 128 + (nt_base + nt) * 32 + col];
    };
    auto read_dx = [&](int bi, int buf) __attribute__((always_inline)) {
        const float* sdx = (const float*)(smem + 2 * (A_BYTES + B_BYTES + Q6_W_BYTES) + buf * Q6_X_BYTES) + bi * BM + role.tw * 32 + half * 4;
#pragma unroll
        for (int g = 0; g < 4; g++) dx[g] = *(const float4*)(sdx + g * 8);
    };
    auto widen_tokens = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            uint4 o;
            widen_h((unsigned)araw[j].x ^ 0x80808080u, (_Float16)1152.f, o.x, o.y);
            widen_h((unsigned)araw[j].y ^ 0x80808080u, (_Float16)1152.f, o.z, o.w);
            af[j] = __builtin_bit_cast(v8h, o);
        }
    };
    auto mfma_unit = [&](int g) __attribute__((always_inline)) {
        const v16f zero = {0.f};
#pragma unroll
        for (int j = 0; j < 2; j++) {
            d[g & 1][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[j], __builtin_bit_cast(v8h, bf[g & 1][j]), zero, 0, 0, 0);
            asm volatile("" : "+v"(d[g & 1][j]));
        }
    };
    // The stages, for a number of row tiles known at compile time; 0: a wave whose 32 tokens all lie past the tile's end only
    // helps with the staging.  A unit's fragments are read two units ahead of its FMAs and its MFMAs issued one ahead, so the
    // two barriers of a stage stand where a read first touches what they publish: in front of block 2 (the second half of
    // the weights) and of the next stage's block 0 (everything else).
    using H0 = std::integral_constant<int, 0>;
    using H1 = std::integral_constant<int, 1>;
    auto main_loop = [&](auto ntc, auto full) __attribute__((always_inline)) {
        constexpr int NT = decltype(ntc)::value, U = KB * NT;
        if (s_begin >= s_end) return;   // (an empty K slice)
        issue_a(full, 0, s_begin);
        issue_w(s_begin);
        auto publish = [&](int s) __attribute__((always_inline)) {   // stage s, and what can be requested behind it
            const int buf = (s - s_begin) & 1;
            write_b(H0());
            write_scales(buf);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            if (s + 1 < s_end) issue_a(full, buf ^ 1, s + 1);
            write_b(H1());
            if (s + 1 < s_end) issue_w(s + 1);
        };
        publish(s_begin);
        if constexpr (NT > 0) {
            read_unit(ntc, 0, 0);
            widen_tokens();
            mfma_unit(0);
            if constexpr (NT == 1) __builtin_amdgcn_sched_barrier(0);
            read_unit(ntc, 1, 0);
        }
        for (int s = s_begin; s < s_end; s++) {
            const int buf = (s - s_begin) & 1;
            if constexpr (NT == 0) {
                __syncthreads();
                if (s + 1 < s_end) publish(s + 1);
            } else {
#pragma unroll
                for (int g = 0; g < U; g++) {
                    if constexpr (NW == 8) {
                        // The two waves of a SIMD meet at every stage's barriers; the elder would issue whenever it can and then
                        // wait there while the other goes on alone, at two thirds of the rate of both.  Priority falls with the way.
                        if (g == 0) __builtin_amdgcn_s_setprio(3);
                        else if (g == U / 4) __builtin_amdgcn_s_setprio(2);
                        else if (g == U / 2) __builtin_amdgcn_s_setprio(1);
                        else if (g == 3 * U / 4) __builtin_amdgcn_s_setprio(0);
                    }
                    if (g % NT == 0) read_dx(g / NT, buf);
                    if ((g + 1) % NT == 0) widen_tokens();
                    mfma_unit(g + 1);   // (behind the last stage: of stale operands, never used)
                    if (g + 2 == U / 2) __syncthreads();
                    if (g + 2 == U && s + 1 < s_end) publish(s + 1);
                    read_unit(ntc, (g + 2) % U, g + 2 < U ? buf : buf ^ 1);
                    __builtin_amdgcn_sched_barrier(0);
                    const int bi = g / NT, nt = g % NT;
                    const v16f d0 = d[g & 1][0], d1 = d[g & 1][1];
                    const float2 w = dw[g & 3];
                    float t[16];
#pragma unroll
                    for (int i = 0; i < 16; i++) t[i] = fmaf(w.x, d0[i], w.y * d1[i]);
                    const float dxr[16] = {dx[0].x, dx[0].y, dx[0].z, dx[0].w, dx[1].x, dx[1].y, dx[1].z, dx[1].w,
                                           dx[2].x, dx[2].y, dx[2].z, dx[2].w, dx[3].x, dx[3].y, dx[3].z, dx[3].w};
#pragma unroll
                    for (int i = 0; i < 16; i++) acc[nt][i] = fmaf(dxr[i], t[i], acc[nt][i]);
#pragma unroll
                    for (int i = 0; i < 16; i++) asm volatile("" : "+v"(acc[nt][i]));   // (not moved between units: they would spill)
                    if constexpr (DUMP) {
                        const int row = row0 + (nt_base + nt) * 32 + col;
#pragma unroll
                        for (int i = 0; i < 16; i++) {
                            const int tok = tok0 + role.tw * 32 + (i >> 2) * 8 + half * 4 + (i & 3);
                            if (tok < M_end && row < N_end) {
                                int* o = p.dump + ((size_t)tok * p.N + row) * (2 * p.nb) + 2 * (s * KB + bi);
                                o[0] = (int)d0[i];
                                o[1] = (int)d1[i];
                            }
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
    };
    using T = std::true_type;
    using F = std::false_type;
    if (role.tw * 32 >= role.live_tok) main_loop(std::integral_constant<int, 0>(), F());
    else if (role.nt_cnt == 4) main_loop(std::integral_constant<int, 4>(), T());
    else if (role.nt_cnt == 3) main_loop(std::integral_constant<int, 3>(), F());   // the 96-row strips
    else if (role.nt_cnt == 2) main_loop(std::integral_constant<int, 2>(), F());
    else main_loop(std::integral_constant<int, 1>(), F());
    gemm_store(p, op, at, role, acc, lane);
    SMX_GEMM_T1(role.live_tok, at.op_i);
}

}  // namespace smx
