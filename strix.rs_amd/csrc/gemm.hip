// int8 W8A8 prefill GEMM on CDNA4 matrix cores: Y[m][N] = Xq . Wq^T with per-32-block fp32 rescale.
//
// Stands in for the reference's WMMA GEMMs (crates/strix-backend-rocm/src/kernels.rs:481-537
// q4_gemm_w, :545-601 q4_gemm_w_sk, :1373-1443 q8w_gemm32) on gfx950:
//   * v_mfma_i32_32x32x32_i8: K = 32 is exactly one quant block, so each MFMA yields the exact
//     i32 block dots of a 32-token x 32-row tile (tokens on the A side, weight rows on the B side:
//     a lane then owns one weight row and 16 tokens, and stores are 128-byte row segments);
//   * workgroup tile 128 tokens x 128 rows, 4 waves, two workgroups per CU; or (NW = 8) 256 tokens, 8 waves, one per CU; each
//     wave 32 tokens x 128 rows;
//   * K advances 4 blocks (128 bytes per row, one full cache line) per stage, double-buffered
//     through LDS in MFMA-fragment order so every fragment read is one conflict-free 128-bit load;
//   * Q4_0 nibbles are widened to signed int8 while being staged (kernels.rs:458-462), to 16 (nibble - 8): three operations per
//     eight of them (nine for nibble - 8); the block scale takes the sixteenth, which is exact.  2048 x 15360 x 3840 319 -> 306 us;
//   * per block and output: acc += dx * (dw * I).  The MFMA accumulates onto the constant
//     0x4B400000 so its i32 result, read as a float, is 12582912 + I exactly; one FMA with the
//     exactly representable -dw*12582912 (dw is an f16 value) gives fl(dw*I) with no int->float
//     conversion, a second FMA applies dx and accumulates: two VALU operations per output per block;
//   * Q6_K weights have a kernel of their own (gemm_q6.h);
//   * split-K: grid.z slices of whole stages write fp32 partials that a second kernel sums in slice
//     order (deterministic, unlike the reference's atomicAdd, kernels.rs:597).
// Bound: 2*M*N*K int8 operations on the matrix cores plus 32 FMAs per MFMA; the two add up (a SIMD runs both at one power
// budget: 17 ns per MFMA, 21 ns per 16 FMAs measured alone, 60 ns per MFMA with its 32 FMAs), which puts the exact rescale's
// ceiling at 1.1 POPS.  What is left is every other instruction a wave issues, so the loop holds no bounds test, no 64-bit
// address and no branch per row tile (see main_loop).  2048 tokens x 15360 x 3840: Q8_0 340 -> 303 us, Q4_0 350 -> 316 us with
// row tiles counted at compile time, scalar stage offsets and the MFMAs issued one row tile ahead.
#include <algorithm>
#include <type_traits>

#include "gemm_dev.h"
#include "gemm_q6.h"
#include "mfma_dev.h"

namespace smx {

constexpr int stage_bytes(int nw) { return 4 * nw * GRP + B_BYTES + KB * 128 * 4 + KB * 32 * nw * 4; }

// Operand fragments on their way from LDS to the matrix cores.  The weight fragments of several row tiles are not
// double-buffered: a row tile's registers are refilled for the next block as soon as its MFMA has been issued (a single row
// tile's MFMA comes too soon after that: it takes b[0] and b[1] in turn).
struct GemmFrag {
    v4i a[2];         // this wave's 32 tokens x 32 k, two blocks in turn; a lane holds 16 k of its token
    float4 dx[2][4];  // activation scales of the 16 tokens this lane accumulates
    v4i b[4];         // 4 x (32 weight rows x 32 k)
    float4 dw[4];     // weight scales of this lane's row in each row tile, the four blocks of the stage
};

template <bool Q4, bool DUMP, int NW>
__global__ __launch_bounds__(64 * NW, 2) void gemm_i8_kernel(GemmArgs p) {
    SMX_GEMM_T0;
    constexpr int BM = 32 * NW, A_BYTES = 4 * NW * GRP, STAGE_BYTES = stage_bytes(NW);
    constexpr int BG = 16 / NW;  // 8-row groups of B each wave stages
    extern __shared__ __align__(16) char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int K = p.nb * 32;
    const unsigned smem_base = lds_addr(smem);

    const TileAt at = gemm_tile_at(p);
    const WaveRole role = gemm_wave_role(at, wave, NW);
    const int tok0 = at.tok0, row0 = at.row0, M_end = at.M_end, N_end = at.N_end;
    const int live_tok = role.live_tok, live_rows = role.live_rows, tw = role.tw, nt_cnt = role.nt_cnt, nt_base = role.nt_base;
    const GemmOperand op = p.op[at.op_i];

    const int nstage_total = (p.nb + KB - 1) / KB;
    const int s_begin = blockIdx.z * p.stages_per_slice;
    const int s_end = min(nstage_total, s_begin + p.stages_per_slice);

    // ---- staging.  int8 operands go global -> LDS directly, one 8-row x 128-byte group per wave
    //      instruction, lane = [row:3][slot:3]: the 8 lanes of a row fetch its whole 128-byte line
    //      (scattered 16-byte fetches run at a fraction of the L2 -> CU rate), and lane (r, slot)
    //      fetches chunk (slot - r) % 8, so that chunk c of the 8 rows of a group lies in 8 different
    //      bank groups and every MFMA fragment read below is a conflict-free 128-bit load.
    //      Rows past the tile's end re-read its last one (clamped addresses), blocks past K read whatever follows the row
    //      (up to 96 bytes of quants behind the last one: weights and activation buffers carry kReadSlack bytes more), and
    //      both are neutralised by zero scales.  Q4_0 weights pass through registers to be widened. ----
    const int g_rowlo = lane >> 3, g_chunk = ((lane & 7) - g_rowlo) & 7;
    const int q_bi = lane & 3, q_rowlo = lane >> 2;   // Q4_0 B: lane = [row:4][block:2], 64 contiguous bytes per row
    constexpr int QG = 8 / NW;  // Q4_0 B: 16-byte blocks per thread per stage
    // byte offsets (of this lane's 16-byte chunk of a row's first stage for the LDS-direct operands; M*K and N*K are below 2^31:
    // launch_gemm, for expert tensors moe_check_shape); a stage's own offset is added to the scalar base
    unsigned a_off[4], b_off[Q4 ? QG : BG];
#pragma unroll
    for (int ps = 0; ps < 4; ps++) {
        const int ti = min(tok0 + (ps * NW + wave) * 8 + g_rowlo, M_end - 1);
        a_off[ps] = (unsigned)(p.a_rowmap ? p.a_rowmap[ti] : ti) * (unsigned)K + g_chunk * 16;
    }
    if constexpr (Q4) {
#pragma unroll
        for (int ps = 0; ps < QG; ps++)
            b_off[ps] = ((unsigned)min(row0 + (ps * NW + wave) * 16 + q_rowlo, N_end - 1) * (unsigned)p.nb + q_bi) * 16u;
    } else {
#pragma unroll
        for (int ps = 0; ps < BG; ps++)
            b_off[ps] = (unsigned)min(row0 + (ps * NW + wave) * 8 + g_rowlo, N_end - 1) * (unsigned)K + g_chunk * 16;
    }
    // scales of a stage (4 blocks): threads 0..127 carry the four f16 scales of weight row tid (8
    // contiguous bytes), threads 128..255 the four fp32 scales of token tid - 128 (16 contiguous bytes): one load per thread.
    const bool role_w = wave < 2, role_x = NW == 4 ? !role_w : wave >= NW / 2;   // scalar: waves 0, 1 carry the weights' scales, the second half the activations'
    const int role_r = NW > 4 && role_w ? tid : tid & (BM - 1);
    const bool x_valid = tok0 + role_r < M_end;
    const unsigned scw_base = (unsigned)min(row0 + role_r, N_end - 1) * (unsigned)p.nb;   // below 2^26
    unsigned scx_base;
    {
        const int ti = min(tok0 + role_r, M_end - 1);
        scx_base = (unsigned)(p.a_rowmap ? p.a_rowmap[ti] : ti) * (unsigned)p.nb;
    }
    uint4 rb[Q4 ? QG : 1];     // Q4_0 quants on their way through registers
    uint4 rsv = {0, 0, 0, 0};  // the thread's four raw scales: f16 pairs in .x .y (weights) or four fp32 (activations)

    // all global reads of stage s (issuing them piecemeal between the blocks measures slower); the register-staged parts are
    // written by finish_stage.  full (waves with all four row tiles): every 8-row group is fetched, those past the tile's end as
    // copies of its last row; of four waves' tiles that is more than 64 live tokens, of eight waves' any number
    auto issue_stage = [&](auto full, int buf, int s) __attribute__((always_inline)) {
        const unsigned sA = __builtin_amdgcn_readfirstlane(smem_base + buf * STAGE_BYTES + wave * GRP);
        const int blk0 = s * KB;
        // 8-token groups wholly past the tile's end are not fetched (nothing reads their LDS rows)
        const int8_t* xa = p.xq + (size_t)blk0 * 32;
#pragma unroll
        for (int ps = 0; ps < 4; ps++)
            if (decltype(full)::value || (ps * NW + wave) * 8 < live_tok) load_to_lds16(xa, a_off[ps], sA, ps * NW * GRP);
        if constexpr (Q4) {
            const char* wb = (const char*)op.wquants + (size_t)blk0 * 16;
#pragma unroll
            for (int ps = 0; ps < QG; ps++) rb[ps] = *(const uint4*)(wb + b_off[ps]);
        } else {
            const int8_t* wb = (const int8_t*)op.wquants + (size_t)blk0 * 32;
#pragma unroll
            for (int ps = 0; ps < BG; ps++)
                if (decltype(full)::value || (ps * NW + wave) * 8 < live_rows) load_to_lds16(wb, b_off[ps], sA, A_BYTES + ps * NW * GRP);
        }
        // unconverted, so that nothing here waits for a load before the MFMA work
        if (role_w) {
            uint2 v;
            __builtin_memcpy(&v, (const char*)(op.wscales + blk0) + scw_base * 2u, 8);   // 2-byte aligned where rows are not whole stages
            rsv.x = v.x; rsv.y = v.y;
        }
        if (role_x) __builtin_memcpy(&rsv, (const char*)(p.xd + blk0) + scx_base * 4u, 16);
    };

    auto finish_stage = [&](int buf, int s) __attribute__((always_inline)) {
        char* sB = smem + buf * STAGE_BYTES + A_BYTES;
        float* sdw = (float*)(sB + B_BYTES);
        float* sdx = sdw + KB * 128;
        const int blk0 = s * KB;
        if constexpr (Q4) {
#pragma unroll
            for (int ps = 0; ps < QG; ps++) {
                const int r = (ps * NW + wave) * 16 + q_rowlo;
                const int off = (r >> 3) * GRP + (r & 7) * 128;  // + slot * 16
                const uint4 q = rb[ps];
                const uint4 lo = make_uint4(nib16(q.x << 4), nib16(q.y << 4), nib16(q.z << 4), nib16(q.w << 4));
                const uint4 hi = make_uint4(nib16(q.x), nib16(q.y), nib16(q.z), nib16(q.w));
                *(uint4*)(sB + off + ((2 * q_bi + r) & 7) * 16) = lo;      // elements 0..15 of the block
                *(uint4*)(sB + off + ((2 * q_bi + 1 + r) & 7) * 16) = hi;  // elements 16..31
            }
        }
        const int live = p.nb - blk0;   // blocks of the stage that lie within K (scalar); the scales of the others are zero
        if (role_w) {   // the four block scales of a row side by side: one 16-byte write here, one 16-byte read per row tile and stage
            const unsigned h[4] = {rsv.x & 0xffffu, rsv.x >> 16, rsv.y & 0xffffu, rsv.y >> 16};
            float v[KB];   // (a row past the tile's end has its last one's; nothing of it is stored)
#pragma unroll
            for (int j = 0; j < KB; j++) v[j] = h2f_((uint16_t)h[j]) * (Q4 ? 0.0625f : 1.f);   // nib16: sixteen times the quants
            if (live < KB) {
#pragma unroll
                for (int j = 1; j < KB; j++) v[j] = j < live ? v[j] : 0.f;
            }
            *(float4*)(sdw + role_r * 4) = make_float4(v[0], v[1], v[2], v[3]);
        }
        if (role_x) {
            float v[KB] = {__uint_as_float(rsv.x), __uint_as_float(rsv.y), __uint_as_float(rsv.z), __uint_as_float(rsv.w)};
            if (live < KB) {
#pragma unroll
                for (int j = 1; j < KB; j++) v[j] = j < live ? v[j] : 0.f;
            }
#pragma unroll
            for (int j = 0; j < KB; j++) sdx[j * BM + role_r] = x_valid ? v[j] : 0.f;   // (zeros cost the matrix loop less power than repeated rows)
        }
    };

    float acc[4][16];
#pragma unroll
    for (int nt = 0; nt < 4; nt++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[nt][i] = 0.f;
    v16i cmagic;
#pragma unroll
    for (int i = 0; i < 16; i++) cmagic[i] = MAGIC_I;
    asm volatile("" : "+v"(cmagic));  // keep the constant in vector registers: re-materialising it costs 8 moves per block

    const int half = lane >> 5, col = lane & 31;
    // fragment (tile, block bi): lane -> row lane % 32 of the tile, k-half lane / 32
    int frag_lane[KB];
#pragma unroll
    for (int bi = 0; bi < KB; bi++) frag_lane[bi] = (col >> 3) * GRP + (col & 7) * 128 + ((2 * bi + half + col) & 7) * 16;
    GemmFrag f;
    // of block bi of the stage in `buf`: the tokens' fragment and scales into slot `slot`
    auto read_tokens = [&](int slot, int buf, int bi) __attribute__((always_inline)) {
        const char* sA = smem + buf * STAGE_BYTES + tw * 4 * GRP;
        const float* sdx = (const float*)(smem + buf * STAGE_BYTES + A_BYTES + B_BYTES) + KB * 128 + bi * BM + tw * 32;
#pragma unroll
        for (int g = 0; g < 4; g++) f.dx[slot][g] = *(const float4*)(sdx + g * 8 + half * 4);
        f.a[slot] = *(const v4i*)(sA + frag_lane[bi]);
    };
    // the fragment of row tile nt into f.b[idx]
    auto read_rows = [&](int idx, int nt, int buf, int bi) __attribute__((always_inline)) {
        f.b[idx] = *(const v4i*)(smem + buf * STAGE_BYTES + A_BYTES + (nt_base + nt) * 4 * GRP + frag_lane[bi]);
    };
    auto read_scales = [&](int nt, int buf) __attribute__((always_inline)) {
        f.dw[nt] = *(const float4*)((const float*)(smem + buf * STAGE_BYTES + A_BYTES + B_BYTES) + ((nt_base + nt) * 32 + col) * 4);
    };
    auto mfma_tile = [&](auto ntc, int slot, int nt) __attribute__((always_inline)) -> v16i {
        return __builtin_amdgcn_mfma_i32_32x32x32_i8(f.a[slot], f.b[decltype(ntc)::value == 1 ? slot : nt], cmagic, 0, 0, 0);
    };
    using T = std::true_type;
    using F = std::false_type;
    v16i d[2];
    // One block (bi of the stage in `buf`) of the wave's NT row tiles.  The MFMA of a row tile is issued in front of the FMAs of
    // the tile before it, across the blocks too: a result is read 32 FMAs after its MFMA was issued, and the fragments of the
    // next block (nbi of nbuf) are requested a block ahead.  The scheduling barriers hold that order; left to itself the
    // compiler issues an MFMA right in front of the FMAs that need it and pads the wait with s_nop.
    auto compute = [&](auto ntc, auto blki, auto last, int s, int nbuf) __attribute__((always_inline)) {
        constexpr int NT = decltype(ntc)::value, bi = decltype(blki)::value, slot = bi & 1, nbi = (bi + 1) & 3;
        constexpr bool LAST = decltype(last)::value;   // the last block of all
        if (!LAST) read_tokens(slot ^ 1, nbuf, nbi);
        if (!LAST && NT == 1) read_rows(slot ^ 1, 0, nbuf, nbi);
        const float dxr[16] = {f.dx[slot][0].x, f.dx[slot][0].y, f.dx[slot][0].z, f.dx[slot][0].w, f.dx[slot][1].x, f.dx[slot][1].y,
                               f.dx[slot][1].z, f.dx[slot][1].w, f.dx[slot][2].x, f.dx[slot][2].y, f.dx[slot][2].z, f.dx[slot][2].w,
                               f.dx[slot][3].x, f.dx[slot][3].y, f.dx[slot][3].z, f.dx[slot][3].w};
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            const int cur = (bi * NT + nt) & 1;
            if (nt + 1 < NT) d[cur ^ 1] = mfma_tile(ntc, slot, nt + 1);
            else if (!LAST) d[cur ^ 1] = mfma_tile(ntc, slot ^ 1, 0);
            if (nt + 1 < NT || !LAST) asm volatile("" : "+v"(d[cur ^ 1]));
            if (!LAST && NT > 1) read_rows(nt, nt, nbuf, nbi);   // the MFMA of the tile's old fragment has been issued
            __builtin_amdgcn_sched_barrier(0);
            const v16i dn = d[cur];
            const float dw = bi == 0 ? f.dw[nt].x : bi == 1 ? f.dw[nt].y : bi == 2 ? f.dw[nt].z : f.dw[nt].w;
            const float ndw = -dw * MAGIC_F;  // exact: dw has 11 significant bits
#pragma unroll
            for (int i = 0; i < 16; i++) acc[nt][i] = fmaf(dxr[i], fmaf(dw, __int_as_float(dn[i]), ndw), acc[nt][i]);
            asm volatile("" : "+v"(acc[nt][0]), "+v"(acc[nt][1]), "+v"(acc[nt][2]), "+v"(acc[nt][3]), "+v"(acc[nt][4]),
                              "+v"(acc[nt][5]), "+v"(acc[nt][6]), "+v"(acc[nt][7]), "+v"(acc[nt][8]), "+v"(acc[nt][9]),
                              "+v"(acc[nt][10]), "+v"(acc[nt][11]), "+v"(acc[nt][12]), "+v"(acc[nt][13]),
                              "+v"(acc[nt][14]), "+v"(acc[nt][15]));
            if constexpr (DUMP) {
                const int blk = s * KB + bi;
                const int row = row0 + (nt_base + nt) * 32 + col;
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const int tok = tok0 + tw * 32 + (i >> 2) * 8 + half * 4 + (i & 3);
                    if (tok < M_end && row < N_end && blk < p.nb) p.dump[((size_t)tok * p.N + row) * p.nb + blk] = (dn[i] - MAGIC_I) / (Q4 ? 16 : 1);
                }
            }
            if (!LAST && bi == 3) read_scales(nt, nbuf);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // The stages, for a number of row tiles known at compile time (tested at run time in front of every row tile it cost a
    // stage of 16 MFMAs some 60 branches and 140 scalar instructions, and a wave issues one instruction at a time);
    // 0: a wave whose 32 tokens all lie past the tile's end (ragged expert groups, M tails) only helps with the staging, its
    // SIMD time goes to the other workgroup on the CU.
    // One barrier per stage, in front of its last block: there every wave holds that block's fragments in registers and
    // its own loads of the next stage have landed (they were requested four blocks earlier), so behind the barrier the
    // stage's buffer takes the loads of the stage after next, and the next stage's first fragments are read under the last
    // block's arithmetic.
    auto main_loop = [&](auto ntc, auto full) __attribute__((always_inline)) {
        constexpr int NT = decltype(ntc)::value;
        using I0 = std::integral_constant<int, 0>;
        using I1 = std::integral_constant<int, 1>;
        using I2 = std::integral_constant<int, 2>;
        using I3 = std::integral_constant<int, 3>;
        if (s_begin >= s_end) return;   // (an empty K slice)
        issue_stage(full, 0, s_begin);
        finish_stage(0, s_begin);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (s_begin + 1 < s_end) issue_stage(full, 1, s_begin + 1);
        if constexpr (NT > 0) {
            read_tokens(0, 0, 0);
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                read_rows(nt, nt, 0, 0);
                read_scales(nt, 0);
            }
            d[0] = mfma_tile(ntc, 0, 0);
            asm volatile("" : "+v"(d[0]));
        }
        // The waves of a workgroup leave the barrier together, and 8 KB of loads per wave queue up in the CU's one address
        // unit (20 cycles per 1 KB load alone, 64 behind three other waves): even waves issue the stage after next's loads
        // right behind the barrier, odd waves one block later.
        const int my_slot = NT > 0 ? wave & 1 : 0;
        for (int s = s_begin; s < s_end; s++) {
            const int buf = (s - s_begin) & 1;
            if constexpr (NT > 0) {
                // eight waves that meet once a stage: of a SIMD's two the one that is behind goes first (see gemm_q6_kernel)
                if constexpr (NW == 8) __builtin_amdgcn_s_setprio(3);
                compute(ntc, I0(), F(), s, buf);
                if constexpr (NW == 8) __builtin_amdgcn_s_setprio(2);
                compute(ntc, I1(), F(), s, buf);
                if constexpr (NW == 8) __builtin_amdgcn_s_setprio(1);
                compute(ntc, I2(), F(), s, buf);
                if constexpr (NW == 8) __builtin_amdgcn_s_setprio(0);
            }
            if (s + 1 == s_end) break;
            finish_stage(buf ^ 1, s + 1);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            const bool more = s + 2 < s_end;
            if (more && my_slot == 0) issue_stage(full, buf, s + 2);
            if constexpr (NT > 0) {
                compute(ntc, I3(), F(), s, buf ^ 1);
                if (more && my_slot == 1) issue_stage(full, buf, s + 2);
            }
        }
        if constexpr (NT > 0) compute(ntc, I3(), T(), s_end - 1, 0);
    };
    // Up to 32 live tokens of a Q8_0 weight in whole stages: the tile is bound by its weight stream (a wave has one MFMA per block), and
    // one stage on its way at a time, 1.6 us per 16 KB, is the trip to memory.  A stage without the empty token slots fits three
    // times, so two are on their way while one is computed; its scales go to LDS directly too (their load through registers would
    // have the compiler wait for everything behind it), the activations' as one per lane, read through a row broadcast.
    // MoE layer, 512 tokens over 64 experts (half the tiles are such): 157.6 -> 149.6 us, 64 tokens 111 -> 98; 150 tokens x 15360 x
    // 3840: 54.9 -> 49.5.  For 33..64 tokens the loop below is ahead (161 us on the first): their tiles are bound by the arithmetic.
    auto sparse_loop = [&]() __attribute__((always_inline)) {
        constexpr int W_AT = 4 * GRP, DW_AT = W_AT + B_BYTES, DX_AT = DW_AT + 128 * 8, BUF = DX_AT + 32 * 16;
        constexpr int LOADS = 7;   // of a wave and stage
        static_assert(3 * BUF <= 2 * STAGE_BYTES, "three stages of 32 tokens");
        unsigned w_off[4];   // this wave's 32 weight rows; of the tokens, a_off[0]
#pragma unroll
        for (int j = 0; j < 4; j++) w_off[j] = (unsigned)min(row0 + wave * 32 + j * 8 + g_rowlo, N_end - 1) * (unsigned)K + g_chunk * 16;
        const unsigned dw_off = (unsigned)min(row0 + wave * 32 + (lane >> 1), N_end - 1) * (unsigned)p.nb * 2u + (lane & 1) * 4;
        const int dt = min(tok0 + (wave & 1) * 16 + (lane >> 2), M_end - 1);   // (waves 2 and 3 write what 0 and 1 write)
        const unsigned dx_off = ((unsigned)(p.a_rowmap ? p.a_rowmap[dt] : dt) * (unsigned)p.nb + (lane & 3)) * 4u;
        auto issue = [&](int buf, int s) __attribute__((always_inline)) {
            const unsigned sb = __builtin_amdgcn_readfirstlane(smem_base + buf * BUF);
            load_to_lds16(p.xq + (size_t)s * (KB * 32), a_off[0], sb + wave * GRP);
            const int8_t* wb = (const int8_t*)op.wquants + (size_t)s * (KB * 32);
#pragma unroll
            for (int j = 0; j < 4; j++) load_to_lds16(wb, w_off[j], sb + W_AT + (wave * 4 + j) * GRP);
            load_to_lds4(op.wscales + s * KB, dw_off, sb + DW_AT + wave * 256);
            load_to_lds4(p.xd + s * KB, dx_off, sb + DX_AT + (wave & 1) * 256);
        };
        const int dx_slot = ((lane & 15) >> 2) * 8 + half * 4 + (lane & 3);   // token of accumulator lane % 16 in this lane half
        if (s_begin >= s_end) return;
        issue(0, s_begin);
        if (s_begin + 1 < s_end) issue(1, s_begin + 1);
        int buf = 0;
        for (int s = s_begin; s < s_end; s++) {
            if (s + 1 < s_end) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"(LOADS) : "memory");
            else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();   // every wave's part of the stage has landed, and the stage before it has been read
            asm volatile("" ::: "memory");
            if (s + 2 < s_end) issue(buf == 0 ? 2 : buf - 1, s + 2);
            const char* sb = smem + buf * BUF;
            const uint2 dwr = *(const uint2*)(sb + DW_AT + (wave * 32 + col) * 8);
            const float4 dx4 = *(const float4*)(sb + DX_AT + dx_slot * 16);
            const unsigned dwh[KB] = {dwr.x & 0xffffu, dwr.x >> 16, dwr.y & 0xffffu, dwr.y >> 16};
            const float dxv[KB] = {dx4.x, dx4.y, dx4.z, dx4.w};
#pragma unroll
            for (int bi = 0; bi < KB; bi++) {
                const v4i fa = *(const v4i*)(sb + frag_lane[bi]), fb = *(const v4i*)(sb + W_AT + wave * 4 * GRP + frag_lane[bi]);
                const v16i dn = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa, fb, cmagic, 0, 0, 0);
                const float dw = h2f_((uint16_t)dwh[bi]), ndw = -dw * MAGIC_F;
                float t[16];
#pragma unroll
                for (int i = 0; i < 16; i++) t[i] = fmaf(dw, __int_as_float(dn[i]), ndw);
                bcast_accumulate(acc[0], t, dxv[bi]);
            }
            buf = buf == 2 ? 0 : buf + 1;
        }
    };
    if constexpr (!Q4 && !DUMP && NW == 4) {
        if (live_tok <= 32 && (p.nb & (KB - 1)) == 0) {   // workgroup-uniform
            sparse_loop();
            gemm_store(p, op, at, role, acc, lane);
            SMX_GEMM_T1(live_tok, at.op_i);
            return;
        }
    }
    if (tw * 32 >= live_tok) main_loop(std::integral_constant<int, 0>(), F());
    else if (nt_cnt == 4) main_loop(std::integral_constant<int, 4>(), T());
    else if (nt_cnt == 2) main_loop(std::integral_constant<int, 2>(), F());
    else if (nt_cnt == 1) main_loop(std::integral_constant<int, 1>(), F());
    else main_loop(std::integral_constant<int, 4>(), F());   // three: there is no loop for them, the fourth is computed and not written

    gemm_store(p, op, at, role, acc, lane);
    SMX_GEMM_T1(live_tok, at.op_i);
}

#ifdef SMX_GEMM_TRACE
// buf: device memory for 8192 x 4 u64 (or null to stop); the launches that follow write their workgroups' records
extern "C" int smx_debug_gemm_trace(void* buf) {
    return hipMemcpyToSymbol(HIP_SYMBOL(g_gemm_trace), &buf, sizeof(buf)) == hipSuccess ? 0 : -1;
}
#endif

// y[i] = sum over slices z (ascending) of part[z][i]
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float4* __restrict__ part, float4* __restrict__ y,
                                                            size_t n4, int Z) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n4) return;
    float4 s = part[i];
    for (int z = 1; z < Z; z++) {
        const float4 v = part[(size_t)z * n4 + i];
        s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
    }
    y[i] = s;
}

// Token tiles that are walked together (see launch_gemm): the largest divisor of their number up to 8.
static int walk_group(int tiles_m) {
    int gm = std::min(tiles_m, 8);
    while (tiles_m % gm != 0) gm--;   // whole groups
    return gm;
}

// Tile height and K slices.  The reference splits only the long-K shapes (in_dim >= 12288, decode.rs:5658) to fill its grid.  Here the
// launch that is estimated to take least, among tiles of 64 (Q8_0, Q4_0), 128 and 256 tokens and every number of whole-stage slices
// whose workgroups fit the chip's slots in ONE round (a second, partly filled round costs more than shorter slices save): a
// workgroup's stages one after the other, at the time a stage takes with the CU to itself or shared with a second
// workgroup and one more for its first loads, plus the launch that adds up the slices' partials, 1.9 us, 0.3 a slice and 5 MB of them per us.
// Tiles that need several rounds: one slice, 128 or 256 tokens, whichever's rounds take less; there the first loads and the stores of
// two workgroups on a CU hide behind each other's arithmetic (half a stage a round, 0.8 of Q6_K's), those of one on its own do not (1.5, 1.2).
// The stage times are measured (us): 64 tokens 1.05 alone / 1.46 shared, 128 tokens 1.55 / 2.7, Q6_K 2.75 / 4.3; 256 tokens (one workgroup
// per CU) 2.35, Q6_K 3.85.  Over 252 shapes of 65..2048 tokens (512..15360 rows and columns) the choice takes 0.7 % more than the best of
// all heights and up to 16 slices, 15 % at worst (Q8_0 180 x 2384 x 15328: 44.0 us, twelve slices of one 256-token tile 38.4).  Constants fitted
// to half of the shapes do no better on the other half.  The choice of 64- and 128-token tiles without the first loads takes 4.9 % more than
// the best; it is ahead of this one by more than 2 % on three of 312 shapes: Q8_0 539 x 1264 x 960 (15.2 against 15.9), Q6_K 592 x 960 x 4096 (31.5 /
// 32.8), Q4_0 134 x 1072 x 14464 (28.0 / 28.7).
struct Tiling { int bm, slices; };
static Tiling pick_tiling(int num_cu, bool q6, int M, int N, int nstages, bool split, int only) {
    Tiling best = {only ? only : 128, 1};
    double least = 1e30;
    for (int bm : {64, 128, 256}) {
        if (only ? bm != only : bm == 64 ? q6 || M <= 64 : bm == 128 ? !q6 && M > 64 && M <= 128 : M <= 128) continue;   // (65..128 tokens: as two rows of tiles)
        const int T = (M + bm - 1) / bm * ((N + BN - 1) / BN), slots = bm == 256 ? num_cu : 2 * num_cu;
        // A last row of tiles of up to 64 tokens that is dispatched behind all others (tiles walked one row after the other, no remap over
        // the XCDs) does not count as their neighbours where the rest fits the CUs: every wave of it has one or two row tiles and the
        // tile is over early.  1536-long rows, 128- against 256-token tiles: Q6_K 13 rows of 20 tiles 46.4 / 55.5 us (last row of 8 tokens), 49.3 /
        // 55.6 (64), 58.7 / 55.8 (128); 11 rows of 25 Q8_0 29.9 / 35.2 (8), 30.1 / 35.4 (64), 37.6 / 35.6 (128).  Walked in groups the row's tiles
        // start among the others: 12 rows of 23 58.5 / 55.0 (8), 3 rows of 86 55.6 / 53.1.
        const int tiles_m = (M + bm - 1) / bm, last = M - (tiles_m - 1) * bm;
        const int light = bm == 128 && tiles_m > 1 && last <= 64 && walk_group(tiles_m) == 1 && T % 8 != 0 && T - T / tiles_m <= num_cu ? T / tiles_m : 0;
        const bool low = bm == 64 || M <= 64;
        const double alone = bm == 256 ? (q6 ? 3.85 : 2.35) : q6 ? 2.75 : low ? 1.05 : 1.55;
        const double shared = bm == 256 ? alone : q6 ? 4.3 : low ? 1.46 : 2.7;
        // a stage of `n` workgroups side by side
        const auto stage = [&](int n) {
            return n == 0 ? 0.0 : n <= num_cu ? alone : std::max(alone, shared * (0.93 + 0.07 * (n - num_cu) / num_cu));
        };
        if (T > slots) {   // whole rounds and the rest
            const double us = (nstages + (q6 ? (bm == 256 ? 1.2 : 0.8) : bm == 256 ? 1.5 : 0.5)) * (T / slots * shared + stage(T % slots));
            if (bm >= 128 && us < least) {
                least = us;
                best = {bm, 1};
            }
            continue;
        }
        const int zmax = split ? std::min(std::min(slots / T, nstages), 16) : 1;
        for (int z = 1; z <= zmax; z++) {
            const int stages = (nstages + z - 1) / z;
            if (z > 1 && stages == (nstages + z - 2) / (z - 1)) continue;   // the same slices as with one fewer
            const double us = (stages + 1) * stage(z == 1 ? T - light : T * z) + (z > 1 ? 1.9 + 0.3 * z + (double)z * M * N * 4 / 5e6 : 0.0);
            if (us < least) {
                least = us;
                best = {bm, z};
            }
        }
    }
    return best;
}

template <class Kernel>
static int launch_gemm_variant(smx_ctx* c, Kernel k, size_t lds, const GemmArgs& p, dim3 grid, int nw) {
    int rc = set_dyn_lds(c, k, lds);
    if (rc != SMX_OK) return rc;
    hipLaunchKernelGGL(k, grid, dim3(64 * nw), lds, c->stream, p);
    SMX_HIP(c, hipGetLastError());
    return SMX_OK;
}
// The kernel of a format and tile height, with or without the block dots written out.
template <int WAVES>
static int launch_gemm_waves(smx_ctx* c, QType type, bool dump, const GemmArgs& p, dim3 grid) {
    const size_t lds = type == kQ6_K ? q6_lds_bytes(WAVES) : 2 * stage_bytes(WAVES);
    const auto go = [&](auto kern) { return launch_gemm_variant(c, kern, lds, p, grid, WAVES); };
    if (type == kQ6_K) return dump ? go(gemm_q6_kernel<true, WAVES>) : go(gemm_q6_kernel<false, WAVES>);
    if (type == kQ4_0) return dump ? go(gemm_i8_kernel<true, true, WAVES>) : go(gemm_i8_kernel<true, false, WAVES>);
    return dump ? go(gemm_i8_kernel<false, true, WAVES>) : go(gemm_i8_kernel<false, false, WAVES>);
}
static int launch_gemm_type(smx_ctx* c, QType type, bool dump, const GemmArgs& p, dim3 grid) {
    return p.tile_m == 256 ? launch_gemm_waves<8>(c, type, dump, p, grid) : launch_gemm_waves<NW>(c, type, dump, p, grid);
}

GemmOperand gemm_operand(const Weight& w, float* out) {
    GemmOperand o = {};
    o.wscales = w.scales;
    o.wquants = w.quants;
    o.out = out;
    o.wqh = w.qh;
    o.wsc = w.sc;
    return o;
}

int launch_gemm(smx_ctx* c, const Weight& w, const int8_t* xq, const float* xd, size_t m, float* y, int32_t* dump) {
    if (w.type != kQ4_0 && w.type != kQ8_0 && w.type != kQ6_K) return fail(c, SMX_ERR_ARG, "gemm: weight type %d not supported", (int)w.type);
    if (m > (size_t(1) << 24) || w.N > (size_t(1) << 24) || w.K > (size_t(1) << 20) || m * w.K >= (size_t(1) << 31) ||
        w.N * w.K >= (size_t(1) << 31))
        return fail(c, SMX_ERR_LIMIT, "gemm: shape m=%zu N=%zu K=%zu exceeds the kernel's index range", m, w.N, w.K);
    GemmArgs p = {};
    p.op[0] = gemm_operand(w, y);
    p.xq = xq;
    p.xd = xd;
    p.a_rowmap = nullptr;
    p.tiles = nullptr;
    p.dump = dump;
    p.M = (int)m;
    p.N = (int)w.N;
    p.ldo = (int)w.N;
    p.nb = (int)(w.K / 32);
    // 128 x 128 tiles, two 4-wave workgroups per CU, or 256 x 128, one 8-wave workgroup per CU.  Loading, widening and scaling weights
    // is what the larger tile does half as often (loads alone cost the Q8_0 kernel 13 % of its time, the scales 5 %, Q4_0's nibbles
    // 4 %); all eight waves meeting at the barriers costs some of it back.  Without the priorities of the main loop the larger
    // tile loses (-7 %).  Per call, 128 -> 256 tokens: 2048 x 15360 x 3840 Q8_0 316 -> 308 us, Q4_0 323 -> 306; 2048 x 3840 x 15360 328 -> 310,
    // 334 -> 304; Q8_0 512 x 15360 x 3840 84.8 -> 79.4, Q4_0 512 x 9728 x 2560 58.1 -> 50.6; but Q8_0 1000 x 9728 x 2560 (304 tiles for
    // 256 CUs) 88 -> 101.  Measured and slower on every shape tried (M 512..4096 of both FFN shapes, grouped MoE tiles): three
    // workgroups per CU with 2-block stages, every operand and scale staged LDS-direct and the LDS reads software-pipelined
    // (-5..-10 %: the third wave per SIMD raises the instruction issue rate, and the clock the chip sustains drops by as much).
    p.tiles_n = (p.N + BN - 1) / BN;
    const int nstages = (p.nb + KB - 1) / KB;
    const bool may_split = dump == nullptr && (m * w.N) % 4 == 0;
    const int only = c->tune_gemm_tile_m;
    const Tiling tiling = pick_tiling(c->num_cu, w.type == kQ6_K, p.M, p.N, nstages, may_split && c->tune_gemm_splitk == 0, only);
    // 65..128 tokens are always two rows of 64-token tiles (in one row of 128 half the waves of a workgroup may idle): Q8_0
    // 2560 x 9728 and 9728 x 2560 at 96 / 128 tokens 28.2 / 29.4 -> 25.4 / 26.7 us and 25.9 / 27.3 -> 22.9 / 24.7 us.
    int bm = tiling.bm;
    if (p.M > 64 && p.M <= 128 && w.type != kQ6_K && only == 0) bm = 64;   // (also when they need several rounds)
    const int slots = c->num_cu * (bm == 256 ? 1 : 2);   // workgroups the chip holds
    p.tile_m = bm;
    p.tiles_m = (p.M + bm - 1) / bm;
    const int T = p.tiles_m * p.tiles_n;
    p.xcd_remap = (T % 8 == 0) ? 1 : 0;
    // Tile walk.  Workgroup t runs on XCD t % 8 and each XCD gets a contiguous eighth of the logical tile order, so the order
    // decides which operand bytes an XCD's 4 MB L2 must see.  Token tiles are taken in groups of walk_gm (up to 8): an XCD then
    // works on walk_gm token tiles x (tiles_n * tiles_m / walk_gm / 8) weight strips instead of all token tiles x an eighth of
    // the strips, whose activations (7.9 MB at M = 2048, K = 3840) it fetched again for every strip.  Measured L2 fills per
    // launch at M = 2048 (rocprofv3 FETCH_SIZE, Q8_0): K 3840 x N 15360 540 -> 341 MB, K 15360 x N 3840 580 -> 366 MB with groups
    // of 8; groups of 4: 360 / 363 MB; of 1 (ffn_down): 947 MB.  The launch time does not move (the kernel is bound by
    // instruction issue, and these fetches are served by the Infinity Cache).
    {
        int gm = walk_group(p.tiles_m);
        if (c->tune_gemm_walk > 0) {
            gm = std::max(1, p.tiles_m / c->tune_gemm_walk);
            while (p.tiles_m % gm != 0) gm--;
        }
        p.walk_gm = gm;
    }
    int Z = !may_split ? 1 : c->tune_gemm_splitk > 0 ? std::min(c->tune_gemm_splitk, nstages) : T <= slots ? std::min(tiling.slices, std::max(1, slots / T)) : 1;
    p.stages_per_slice = (nstages + Z - 1) / Z;
    Z = (nstages + p.stages_per_slice - 1) / p.stages_per_slice;
    // Mixed strips.  When the tiles need several rounds of the chip's workgroup slots and the last round is partly filled,
    // its idle slots cost up to a whole tile's time.  A Q6_K tile of 96 weight rows runs three of the four row tiles (about 0.8
    // of the time), so with the first `narrow` strips of N cut at 96 rows and dispatched last, the last round can be made
    // of shorter tiles on more slots: 15360 rows x 2048 tokens = 960 tiles of 256 tokens = 3.75 rounds of 256 becomes 768 tiles of
    // 128 rows (3 rounds) and one round of 256 tiles of 96.  Chosen by the estimated makespan, taken when it saves 3 %.  What is left
    // of the 128-token tiles, two to a CU, for a last round takes 0.64 of the time if every CU gets one at most: 700 x 15360 x 3840 (208
    // tiles left, 280 narrow ones with strips) 211 us without strips, 241 with; 2048 x 10240 x 2560 237 / 256.  Tiles that end early
    // fill no round: a last row of up to 64 tokens that starts behind others (1680 x 4656 x 1024 53 / 60, 1293 x 6336 x 4096 183 / 206), a
    // last strip of up to 64 rows (1672 x 13984 x 1280 150 / 162), narrow ones of up to 32 tokens (798 x 12912 x 1536 with 98.6 -> 92.3).
    // Where strips are taken: 1650 x 6208 x 4608 258 -> 237, 1871 x 5280 x 4352 248 -> 214, 1073 x 9360 x 768 56 -> 49, 2048 x 15360 x 3840 498
    // -> 490; over 106 shapes of more than one round -3.1 %, 58 gain, four lose 1-5 % (786 x 10432 x 1280 71.5 -> 75.0).  The Q8_0 and Q4_0
    // kernel has no loop for three row tiles and computes the fourth of such a strip as well: no rule for them.  The knob forces any number of strips for any format.
    if (Z == 1 && bm >= 128 && !dump && c->tune_gemm_narrow != 1) {
        int best_b = 0;
        const int last = p.M - (p.tiles_m - 1) * bm, row = T / p.tiles_m;
        if (c->tune_gemm_narrow > 1) {
            best_b = std::min(c->tune_gemm_narrow - 1, p.N / 96);
        } else if (T > slots && w.type == kQ6_K &&
                   !(last <= 64 && p.walk_gm < p.tiles_m && T - (p.walk_gm == 1 ? row : row * 2 / 3) <= T / slots * slots)) {
            const double c96 = 0.80, one = 0.64;   // of a 128-row tile's time: a 96-row tile; either with the CU to itself
            const bool two = bm == 128;            // slots per CU
            const auto part = [&](int n, double len) { return n == 0 ? 0.0 : two && n <= c->num_cu ? one * len : len; };
            const auto makespan = [&](int b) {     // in 128-row tile times
                const int full = (p.N - 96 * b + (b == 0 ? 63 : BN - 1)) / BN * p.tiles_m, nar = b * p.tiles_m;   // nar <= slots
                const int early = last <= 32 && p.walk_gm == p.tiles_m ? b : 0;
                const int q = full / slots, r = full % slots, free = slots - r;
                if (nar == 0) return q + part(r, 1.0);
                if (r == 0) return q + part(nar - early, c96);
                if (nar <= free) return q + part(r + nar, 1.0);
                if (nar <= 2 * free) return q + 1 + part(nar - free, 2 * c96 - 1);   // behind the narrow tiles beside the last full ones
                return q + 1 + part(nar - free - early, c96);
            };
            const double plain = makespan(0);
            double best = plain;
            for (int b = 1; b * p.tiles_m <= slots && 96 * b <= p.N; b++) {
                const double t = makespan(b);
                if (t < best && t <= 0.97 * plain) { best = t; best_b = b; }
            }
        }
        if (best_b > 0) {
            p.narrow = best_b;
            p.tiles_n = best_b + (p.N - 96 * best_b + BN - 1) / BN;
            p.xcd_remap = (((p.tiles_n - best_b) * p.tiles_m) % 8 == 0 ? 1 : 0) | ((best_b * p.tiles_m) % 8 == 0 ? 2 : 0);
        }
    }
    const int T_launch = p.tiles_m * p.tiles_n;
    p.op[0].out = y;
    if (Z > 1) {
        int rc = ensure(c, c->work, (size_t)Z * m * w.N * 4);
        if (rc != SMX_OK) return rc;
        p.op[0].out = (float*)c->work.p;
    }
    const dim3 grid((unsigned)T_launch, 1, (unsigned)Z);
    {
        ProfScope ps(c, w.type == kQ4_0 ? "gemm_i8_q4_0" : w.type == kQ6_K ? "gemm_i8_q6_k" : "gemm_i8_q8_0");
        int rc = launch_gemm_type(c, w.type, dump != nullptr, p, grid);
        if (rc != SMX_OK) return rc;
    }
    if (Z > 1) {
        const size_t n = m * w.N;
        ProfScope ps(c, "splitk_reduce");
        hipLaunchKernelGGL(splitk_reduce_kernel, dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, c->stream,
                           (const float4*)c->work.p, (float4*)y, n / 4, Z);
        SMX_HIP(c, hipGetLastError());
    }
    return SMX_OK;
}

// A grouped launch with fewer workgroups than the chip has slots leaves CUs idle while each workgroup walks its K stages alone:
// K slices, up to four, as long as all workgroups run in about one round.  The number follows from the sizes alone: a row's sums
// must not depend on where the router sent the other rows of the call (taken from the tile table they did).  What tiles to expect:
// the rows in whole tiles and, for the groups' ends, 0.8 tiles a group there may be, 0.5 for Q6_K, whose stages take three times
// as long and gain where a second round has begun; slices of only two stages where a tile for every group fits 7/8 of the slots.
// Over 456 calls (44 layers of 8..64 experts, 512..4096 wide, 256..1536 inner, 4..2000 tokens, Zipf and even routing) against one
// slice: Q8_0 -3.4 %, at worst +1.8 %, Q6_K -11.2 %, +0.2 %; taken from the table -3.8 %, +3.8 % and -10.2 %, 0.  Taken from the
// layer alone, so that calls of every size agreed, +14 % at 2000 tokens: a slice is 8 bytes a row and inner column, written and
// read again.  Q6_K, 22 stages: 72 workgroups 65 -> 25 us; Q8_0, 152 tokens 56 -> 45 a call.
int gemm_grouped_slices(const smx_ctx* c, QType type, size_t K, size_t N, size_t groups, size_t rows, int nops) {
    const size_t stages = (K / 32 + KB - 1) / KB;
    const double ends = (double)std::min(groups, rows), whole = (double)rows / BM, per_tile = (double)((N + BN - 1) / BN) * nops;
    const double slots = 2.0 * c->num_cu;
    const size_t z3 = std::min(stages / 3, (size_t)(slots / ((ends * (type == kQ6_K ? 0.5 : 0.8) + whole) * per_tile)));
    const size_t z2 = std::min(stages / 2, (size_t)(0.875 * slots / ((ends + whole) * per_tile)));
    size_t z = std::max<size_t>(1, std::min<size_t>(4, std::max(z3, z2)));
    if (c->tune_gemm_splitk > 0) z = std::min<size_t>((size_t)c->tune_gemm_splitk, stages);
    const size_t per_slice = (stages + z - 1) / z;
    return (int)((stages + per_slice - 1) / per_slice);   // (no empty slices)
}

// Grouped GEMM over a tile table (MoE prefill): one launch covers every expert; a tile's workgroups serve
// one of `nops` weight/output pairs each that share the activation rows (gate and up).  The caller has
// checked the shape (moe_check_shape: the kernels' offsets into the expert tensors are 32 bits wide).
int launch_gemm_grouped(smx_ctx* c, QType type, const GemmArgs& args, int ntiles, int nops, int slices, const char* name) {
    if (ntiles <= 0) return SMX_OK;
    ProfScope ps(c, name);
    const dim3 grid((unsigned)(ntiles * nops), 1, (unsigned)slices);
    GemmArgs p = args;
    p.nops = nops;
    p.stages_per_slice = ((p.nb + KB - 1) / KB + slices - 1) / slices;
    if (type == kQ6_K || type == kQ8_0) return launch_gemm_type(c, type, false, p, grid);
    return fail(c, SMX_ERR_ARG, "grouped gemm: weight type %d not supported", (int)type);
}

}  // namespace smx
