// Shared by the tiled int8 GEMM kernels: tile geometry, which tile a workgroup works on, which part of it a wave.
#pragma once
#include "mfma_dev.h"
#include "smx_internal.h"

namespace smx {

constexpr int BN = 128, KB = 4;
constexpr int GRP = 1024;                   // 8 rows x 128 B of one stage: row r at r * 128, its 16-byte chunk c at slot (c + r) % 8
constexpr int NW = 4, BM = 32 * NW;         // a workgroup of four waves covers 128 tokens x 128 weight rows, two per CU
constexpr int A_BYTES = 4 * NW * GRP;       // 128 tokens
constexpr int B_BYTES = 16 * GRP;           // 128 weight rows

// Optional per-workgroup timeline (development builds only: -DSMX_GEMM_TRACE; compiled out of the library): start and end of
// every workgroup of a launch on the constant 100 MHz clock, with its live tokens and the hardware unit it ran on.
#ifdef SMX_GEMM_TRACE
__device__ unsigned long long* g_gemm_trace = nullptr;   // [(grouped gate/up launch: 4096) + workgroup][4]
#define SMX_GEMM_T0 const unsigned long long smx_t0 = wall_clock64()
#define SMX_GEMM_T1(LIVE, OP)                                                                                                  \
    do {                                                                                                                        \
        if (threadIdx.x == 0 && g_gemm_trace && blockIdx.x < 4096) {                                                            \
            unsigned long long* o_ = g_gemm_trace + ((size_t)(p.nops > 1 ? 4096 : 0) + blockIdx.x) * 4;                         \
            o_[0] = smx_t0; o_[1] = wall_clock64(); o_[2] = (unsigned long long)(LIVE) | ((unsigned long long)(OP) << 32);      \
            o_[3] = (unsigned long long)__builtin_amdgcn_s_getreg(63492) | ((unsigned long long)__builtin_amdgcn_s_getreg(63508) << 32); \
        }                                                                                                                       \
    } while (0)
#else
#define SMX_GEMM_T0 do { } while (0)
#define SMX_GEMM_T1(LIVE, OP) do { } while (0)
#endif
// Tile of a workgroup.  Consecutive logical tiles share a weight strip, and each XCD (blockIdx % 8) gets a contiguous range of
// logical tiles so its L2 holds few strips.
struct TileAt {
    int tok0, row0, col0, M_end, N_end, op_i;
};
__device__ __forceinline__ TileAt gemm_tile_at(const GemmArgs& p) {
    TileAt r;
    int t = blockIdx.x;
    r.op_i = blockIdx.y;
    if (p.tiles) {  // grouped (MoE): tile table, A rows are slots of one expert, B rows that expert's rows
        // the operands (gate, up) of a tile are neighbours in the launch order, so that the table's order
        // (longest tiles first) holds for all of them
        r.op_i = t % p.nops;
        t /= p.nops;
        const GemmTile tl = p.tiles[t];
        r.tok0 = tl.tok0; r.M_end = tl.tok_end; r.row0 = tl.row0; r.N_end = tl.row_end; r.col0 = tl.col0;
    } else {
        // The first `narrow` strips of N are 96 rows high and dispatched last (see launch_gemm); each part (128-row strips,
        // 96-row strips) is walked on its own.
        const int full_strips = p.tiles_n - p.narrow;
        const int t_full = full_strips * p.tiles_m;
        const bool nar = t >= t_full;   // never without narrow strips
        if (nar) t -= t_full;
        const int ns = nar ? p.narrow : full_strips;
        const int T = ns * p.tiles_m;
        if (p.xcd_remap & (nar ? 2 : 1)) t = (t & 7) * (T >> 3) + (t >> 3);
        // logical order: token-tile group (walk_gm token tiles), weight strip, token tile inside the group
        const int per_group = p.walk_gm * ns;
        const int grp = t / per_group, in_grp = t - grp * per_group;
        const int tn = in_grp / p.walk_gm, tm = grp * p.walk_gm + (in_grp - tn * p.walk_gm);
        r.tok0 = tm * p.tile_m; r.M_end = min(p.M, r.tok0 + p.tile_m);
        r.row0 = nar ? tn * 96 : p.narrow * 96 + tn * BN;
        r.N_end = nar ? r.row0 + 96 : p.N;
        r.col0 = r.row0;
    }
    return r;
}

// Wave roles.  A full tile gives each wave 32 tokens x 128 rows (4 row tiles).  A tile with few live
// tokens (the tail of M, a small expert group) would leave three of the four waves idle, so its waves
// share the token sub-tiles that are live and split the rows: <= 32 tokens: every wave takes the first
// 32 tokens and ONE row tile; <= 64 tokens: two waves per token half, two row tiles each.
struct WaveRole {
    int live_tok, live_rows;
    int tw;        // token sub-tile
    int nt_cnt;    // row tiles of this wave; a tile at the end of N, or a 96-row strip: only those that exist (gemm_i8_kernel computes four for three)
    int nt_base;
};
// A workgroup of eight waves (256 tokens): 32 tokens a wave, all of the row tiles; of a ragged last tile the waves past its end only stage
// (77 live tokens: three of eight waves compute), and its time is that of a whole one (pick_tiling prices it so).
__device__ __forceinline__ WaveRole gemm_wave_role(const TileAt& t, int wave, int nw = NW) {
    WaveRole r;
    r.live_tok = t.M_end - t.tok0;
    r.live_rows = min(t.N_end - t.row0, BN);
    if (nw > NW) {
        r.tw = wave;
        r.nt_cnt = (r.live_rows + 31) >> 5;
        r.nt_base = 0;
        return r;
    }
    r.tw = r.live_tok <= 32 ? 0 : r.live_tok <= 64 ? (wave & 1) : wave;
    r.nt_cnt = r.live_tok <= 32 ? 1 : r.live_tok <= 64 ? 2 : (r.live_rows + 31) >> 5;
    r.nt_base = r.live_tok <= 32 ? wave : r.live_tok <= 64 ? (wave >> 1) * 2 : 0;
    return r;
}

// The wave's results.
__device__ __forceinline__ void gemm_store(const GemmArgs& p, const GemmOperand& op, const TileAt& t, const WaveRole& w, const float (&acc)[4][16],
                                           int lane) {
    const int half = lane >> 5, col = lane & 31;
    float* out = op.out + (size_t)blockIdx.z * p.M * p.ldo;
#pragma unroll
    for (int nt = 0; nt < 4; nt++) {
        if (nt >= w.nt_cnt) break;
        const int r = (w.nt_base + nt) * 32 + col;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int tok = t.tok0 + w.tw * 32 + (i >> 2) * 8 + half * 4 + (i & 3);
            if (tok < t.M_end && t.row0 + r < t.N_end) out[(size_t)tok * p.ldo + t.col0 + r] = acc[nt][i];
        }
    }
}

}  // namespace smx
