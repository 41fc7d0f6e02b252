// Dense BF16 projection for token counts too small for the 256 x 256 tiling:
// decode batches above 64 rows, prompts below 256 tokens, and of longer ones
// gate/up up to 512 tokens and q|k|v at 1281-1536, where that tiling is neither
// full nor split.
//
// y[m, n] = epi(sum_k x[m, k] * W[n, k]).  At these sizes a projection moves
// about as many bytes of activations through each CU as of weights, and both
// far outweigh the arithmetic, so the kernel is built around two streams that
// never wait for each other:
//   * weights go from HBM (row-major, 128 bytes of a row per step of 64 K)
//     straight into MFMA A operands, two to seven steps ahead in registers;
//     each weight row is read by one wave, which holds 16 * NB of them.  An
//     operand is 64 bytes of 16 rows.  With one token tile each weight is read
//     once: a load instruction then takes whole 128-byte lines of eight rows,
//     non-temporal (a plain streaming kernel reads 7.0 TB/s so, 6.1 with plain
//     loads), and two DPP moves per register make operands of two loads.  With
//     several token tiles the weights are shared through L2 and L1: plain loads
//     in operand order, the second instruction of a line finding it in L1;
//     non-temporal ones fetch the line again (gate/up at 16 / 45 / 100 tokens,
//     us, one process: non-temporal half lines 30.1 / 32.5 / 37.4, plain half
//     lines 22.0 / 25.9 / 34.2, whole lines 20.3 / 24.0 / 33.1);
//   * the 16 * MB token rows of a step are filled into LDS by loader waves
//     with direct global-to-LDS loads, STAGES - 1 steps ahead, and feed
//     every compute wave as B operands.  Waves of their own, because vector
//     memory counters retire in order: a compute wave that loaded both would
//     wait for its newest token rows with every weight it needs.
// A workgroup is NW compute waves (16 NB NW weight rows) and the loader waves,
// one barrier per step.
//
// What bounds it: the CU's memory path, which carries the weights' HBM stream
// (5.2 TB/s at 16 tokens on gate/up, launch included) and the token rows from
// L2 beside it.  Copies of the kernel, gate/up at 45 / 100 tokens (24.0 / 33
// us): without the token loads 20.0 / 22.2, without the weight loads past the
// first steps 12.8 / 19.1, without the LDS reads 24.1 / 32.9, without the MFMAs
// 24.3 / 33.5.  Counters agree: waves wait for LDS in 0.9 / 2.5% of their
// cycles, no bank conflicts, MFMA busy 7 / 12%.
//
// Against the register-staged tiles (us, cold weights; where the weights were
// allocated moves gate/up by up to 8%): 45 tokens qkv 36.5 -> 12-13, o 56.7 ->
// 11.3, gate/up 40.4 -> 22-24, down 129.4 -> 23.4; 100 tokens 47.6 -> 14.5, 73.5
// -> 13.2, 50.5 -> 30-33, 169 -> 27.9; 512 tokens gate/up 93.0 -> 88.5; qkv at
// 1400 tokens 85.5 -> 73.3.
#pragma once

#include "q3_common.hpp"
#include "q3_dma.hpp"
#include "q3.h"

namespace q3gemm {

using namespace q3dma;

__device__ __forceinline__ f32x4_t mfma(const u32x4_t& a, const u32x4_t& b, const f32x4_t& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b),
                                                   c, 0, 0, 0);
}

// Four consecutive output columns col..col+3 of token row m (col % 4 == 0).
template <int EPI>
__device__ __forceinline__ void store4(bf16_t* y, int ldy, int m, int col, const f32x4_t& v) {
    if constexpr (EPI == Q3_EPI_SWIGLU) {
        const uint32_t a = pack_bf16x2(v[0], v[1]), b = pack_bf16x2(v[2], v[3]);  // gate, up rounded
        *reinterpret_cast<uint32_t*>(y + (int64_t)m * ldy + (col >> 1)) =
            pack_bf16x2(silu_bf16(bflo(a)) * bfhi(a), silu_bf16(bflo(b)) * bfhi(b));
    } else {
        uint2* p = reinterpret_cast<uint2*>(y + (int64_t)m * ldy + col);
        if constexpr (EPI == Q3_EPI_RESID) {
            const uint2 r = *p;
            const uint32_t a = pack_bf16x2(v[0], v[1]), b = pack_bf16x2(v[2], v[3]);
            *p = make_uint2(pack_bf16x2(bflo(r.x) + bflo(a), bfhi(r.x) + bfhi(a)),
                            pack_bf16x2(bflo(r.y) + bflo(b), bfhi(r.y) + bfhi(b)));
        } else {
            *p = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
        }
    }
}

// Position of 16-byte chunk c of 128-byte row r: c ^ ((r >> 1) & 7).  Measured
// on gfx950: a ds_read_b128 whose 64 lanes read rows r0..r0+15 at one logical
// chunk (four k groups) runs at the linear-read rate; no swizzle is 2.5x slower.
__device__ __forceinline__ int wide_swz(int r) { return (r >> 1) & 7; }

constexpr int MID_BK = 64;     // K elements of a step: 128 bytes of a row
constexpr int MID_LEAD = 4;    // LDS reads ahead of their MFMAs

struct MidArgs {
    const bf16_t* x;
    int ldx;
    const bf16_t* w;
    int M, N, K;
    int epi;
    bf16_t* y;
    int ldy;
    int tm;  // token tiles
};

// Loader waves: one per SIMD where the token rows of a step are most of the
// bytes (an odd count of 16-row blocks does not deal out over four; two instead
// of four measure level, 47.6 us for gate/up at 235 tokens).
template <int MB>
constexpr int MID_LOADERS = MB > 4 ? (MB % 2 ? 2 : 4) : MB > 1 ? 2 : 1;

// Two compute waves of 16 rows keep too few bytes in flight with three steps
// ahead: at 0.6 us of latency a step took 0.2 us whatever the token count.
// Seven ahead (us, three -> seven: o at 9 / 45 / 80 / 128 tokens 14.2 / 13.5 /
// 14.1 / 15.0 -> 10.4 / 11.2 / 12.3 / 14.5; down 30.9 / 28.7 / 29.8 / 31.7 ->
// 21.7 / 23.4 / 25.9 / 30.9; qkv at 9 / 33 tokens 10.8 / 11.6 -> 8.5 / 11.1).
// Wider workgroups are no faster so, or slower (qkv in three waves at 80 tokens
// 14.1 -> 14.5, gate/up in five at 128 34.8 -> 41.5, down in eight splits at 45
// 15.7 -> 16.8), nor are two waves beside five or more token blocks (o at 200
// tokens 17.6 -> 17.7).
constexpr bool mid_deep(int MB, int NB, int NW) { return NB == 1 && NW == 2 && MB <= 4; }

// LDS stages of token rows.
constexpr int mid_stages(int MB, int NB, int NW) { return mid_deep(MB, NB, NW) ? 8 : 6; }

// Register sets of weights, one more than the steps ahead; three where four
// would not fit.
constexpr int mid_ring(int MB, int NB, int NW, bool NT) {
    return mid_deep(MB, NB, NW) ? 8 : NT && MB * NB >= 16 ? 3 : 4;
}

// NT: whole-line, non-temporal weight loads.
template <int MB, int NB, int NW, bool NT>
__global__ __launch_bounds__((NW + MID_LOADERS<MB>) * 64) void gemm_mid_kernel(MidArgs a) {
    constexpr int LW = MID_LOADERS<MB>, PER = 2 * MB / LW, XT = 16 * MB * 128;  // XT: bytes of a stage
    constexpr int STAGES = mid_stages(MB, NB, NW), AHEAD = STAGES - 1;
    static_assert(2 * MB % LW == 0 && PER * AHEAD <= 63, "direct loads in flight exceed the vmcnt range");
    __shared__ __align__(1024) char lds[STAGES * XT];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    // Workgroup b runs on XCD b % 8: give each XCD a contiguous range, token
    // tiles fastest, so the workgroups that share weight rows share an L2.
    const int total = gridDim.x, xcd = blockIdx.x & 7, q = total >> 3, rem = total & 7;
    const int v = xcd * q + min(xcd, rem) + (int)(blockIdx.x >> 3);
    const int nt = v / a.tm, m0 = (v - nt * a.tm) * 16 * MB, n0 = nt * 16 * NB * NW;
    const int nk = a.K / MID_BK;

    if (wave >= NW) {
        // Direct load i of loader wave lw fills rows 8d..8d+7 of the stage, d =
        // lw + LW i: lane l the chunk position l % 8 of row 8d + l / 8.  Rows
        // past M re-read the last row: in bounds, results not stored.
        const int lw = wave - NW;
        const bf16_t* xb = a.x + (int64_t)m0 * a.ldx;
        uint32_t voff[PER];
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int r = 8 * (lw + LW * i) + (lane >> 3);
            voff[i] = (uint32_t)((min(m0 + r, a.M - 1) - m0) * a.ldx + 8 * ((lane & 7) ^ wide_swz(r))) * 2u;
        }
        const uint32_t lbase = lds_address(lds) + 1024 * lw;
        auto issue = [&](int c) {
            const bf16_t* xc = xb + min(c, nk - 1) * MID_BK;
            const uint32_t sbase = lbase + (uint32_t)(c % STAGES) * XT;
#pragma unroll
            for (int i = 0; i < PER; ++i) load_to_lds(xc, voff[i], sbase + 1024 * LW * i);
        };
#pragma unroll
        for (int c = 0; c < AHEAD; ++c) issue(c);
        wait_vmcnt<PER * (AHEAD - 1)>();
        __syncthreads();
        for (int c = 0; c + 1 < nk; ++c) {
            // Stage (c + AHEAD) % STAGES was last read in step c - 1, which
            // every wave finished before the barrier that ended it.
            issue(c + AHEAD);
            wait_vmcnt<PER * (AHEAD - 1)>();  // step c + 1 landed
            __syncthreads();
        }
        wait_vmcnt<0>();  // no direct-to-LDS load may land after the workgroup ends
        return;
    }

    const int g = lane >> 4, n = lane & 15;
    const int row0 = n0 + wave * 16 * NB;
    // Load h of block i: with NT whole lines, lane (g, n) chunk g + 4 (n / 8) of
    // row 16i + 8h + n % 8; else the operand itself, chunk 4h + g of row
    // 16i + n.  Rows past N re-read the last row.
    constexpr int RING = mid_ring(MB, NB, NW, NT);
    const char* wb = reinterpret_cast<const char*>(a.w + (int64_t)row0 * a.K);
    int woff[NB][2];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int row = row0 + 16 * i + (NT ? 8 * h + (n & 7) : n), chunk = NT ? g + 4 * (n >> 3) : 4 * h + g;
            woff[i][h] = 2 * ((min(row, a.N - 1) - row0) * a.K + 8 * chunk);
        }
    u32x4_t wv[RING][NB][2];
    auto load = [&](int c, u32x4_t (&d)[NB][2]) {
        const char* wc = wb + min(c, nk - 1) * MID_BK * 2;
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const u32x4_t* p = reinterpret_cast<const u32x4_t*>(wc + woff[i][h]);
                d[i][h] = NT ? __builtin_nontemporal_load(p) : *p;
            }
    };
    // The A operands of a block's two k halves (row n, chunk 4kk + g) from its
    // two whole-line loads: lanes n >= 8 of the first change places with lanes
    // n < 8 of the second, eight lanes away in the row of 16.
    auto operands = [&](const u32x4_t (&d)[2], u32x4_t (&op)[2]) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            op[0][e] = NT ? __builtin_amdgcn_update_dpp(d[0][e], d[1][e], 0x128, 0xf, 0xc, false) : d[0][e];  // row_ror:8
            op[1][e] = NT ? __builtin_amdgcn_update_dpp(d[1][e], d[0][e], 0x128, 0xf, 0x3, false) : d[1][e];
        }
    };
    f32x4_t acc[NB][MB];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < MB; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    // Token row 16j + n (same swizzle as row n), logical chunk 4kk + g.
    int boff[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) boff[kk] = (n * 8 + ((4 * kk + g) ^ wide_swz(n))) * 16;

#pragma unroll
    for (int c = 0; c < RING - 1; ++c) load(c, wv[c]);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    // LDS reads run MID_LEAD operands ahead of their MFMAs; the compiler's own
    // order waits for each right before its use (gate/up at 235 tokens 48.8 ->
    // 47.6 us; level at 128 and below).
    constexpr int LEAD = MB < MID_LEAD ? MB : MID_LEAD;
    auto step = [&](int c, int u) {
        const char* xp = lds + (c % STAGES) * XT;
        u32x4_t op[NB][2];
#pragma unroll
        for (int i = 0; i < NB; ++i) operands(wv[u][i], op[i]);
        u32x4_t b[2][MB];
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int j = 0; j < MB; ++j) b[kk][j] = *reinterpret_cast<const u32x4_t*>(xp + boff[kk] + j * 16 * 128);
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int j = 0; j < MB; ++j)
#pragma unroll
                for (int i = 0; i < NB; ++i) acc[i][j] = mfma(op[i][kk], b[kk][j], acc[i][j]);
        __builtin_amdgcn_sched_group_barrier(0x100, LEAD, 0);  // LDS reads
#pragma unroll
        for (int q = 0; q < 2 * MB - LEAD; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x008, NB, 0);  // MFMAs
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, LEAD * NB, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    // Groups of RING steps, each step first loading the one RING - 1
    // ahead; the last group (1..RING steps) has its steps in flight but one.
    int c0 = 0;
    for (; nk - c0 > RING; c0 += RING) {
#pragma unroll
        for (int u = 0; u < RING; ++u) {
            load(c0 + u + RING - 1, wv[(u + RING - 1) % RING]);
            // Keep the prefetch here: the scheduler would otherwise sink each
            // load down to its use and the MFMAs would wait for fresh loads.
            __builtin_amdgcn_sched_barrier(0);
            step(c0 + u, u);
            __syncthreads();
        }
    }
    load(c0 + RING - 1, wv[RING - 1]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < RING; ++u) {
        if (c0 + u < nk) step(c0 + u, u);
        if (c0 + u + 1 < nk) __syncthreads();
    }

    // acc[i][j][e] = C[token m0 + 16j + n][column row0 + 16i + 4g + e].
#pragma unroll
    for (int j = 0; j < MB; ++j) {
        const int m = m0 + 16 * j + n;
        if (m >= a.M) continue;
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int col = row0 + 16 * i + 4 * g;
            if (col >= a.N) continue;
            if (a.epi == Q3_EPI_SWIGLU)
                store4<Q3_EPI_SWIGLU>(a.y, a.ldy, m, col, acc[i][j]);
            else if (a.epi == Q3_EPI_RESID)
                store4<Q3_EPI_RESID>(a.y, a.ldy, m, col, acc[i][j]);
            else
                store4<Q3_EPI_STORE>(a.y, a.ldy, m, col, acc[i][j]);
        }
    }
}

// Launch shape: MB token blocks x NB NW weight blocks of 16 per workgroup.
struct MidPlan {
    int mb, nb, nw;
};

inline int64_t mid_tiles(const MidPlan& p, int M, int N) {
    return (int64_t)((M + 16 * p.mb - 1) / (16 * p.mb)) * ((N + 16 * p.nb * p.nw - 1) / (16 * p.nb * p.nw));
}

// The tile shapes that are built, as NB, NW.
constexpr int MID_SHAPES[][2] = {{1, 2}, {1, 3}, {1, 4}, {1, 5}, {2, 3}, {2, 5}, {2, 8}};
constexpr int MID_MAX_MB = 8;

// Picks the plan of least estimated time.  A CU's bytes set it, not its
// arithmetic, so a step costs about 20 ns per 16-row block that the workgroup
// loads (weights or tokens) plus 100 ns of barrier and latency, once per round
// of workgroups over the CUs.  Against a sweep of all shapes at 9-512 tokens on
// the four projections the pick is the fastest or within 3% of it at 93 of 100
// sizes, and 4-15% off at seven that it thinks need a round less than they do
// (down at 255 / 512 tokens 47.4 / 61.3 against 43.0 / 53.4 us, o at 512 27.5
// against 25.3, qkv at 255 23.7 against 21.9).  Fewer tokens can take longer:
// down at 64 tokens is two tiles of 80 workgroups (29.1 us, the fastest of the
// shapes), at 65-80 three (25.8).
inline MidPlan mid_plan(int M, int N, int cus) {
    const int mblocks = (M + 15) / 16, nblocks = (N + 15) / 16;
    MidPlan best{1, 1, 2};
    double best_cost = 1e30;
    for (const auto& sh : MID_SHAPES) {
        const int wb = sh[0] * sh[1];
        for (int mb = mblocks < MID_MAX_MB ? mblocks : MID_MAX_MB; mb >= 1; --mb) {
            const int64_t tiles = (int64_t)((mblocks + mb - 1) / mb) * ((nblocks + wb - 1) / wb);
            const double cost = (5 + wb + mb) * (double)((tiles + cus - 1) / cus);
            if (cost < best_cost) {
                best_cost = cost;
                best = {mb, sh[0], sh[1]};
            }
        }
    }
    return best;
}

template <int MB>
int launch_mid_mb(const MidPlan& p, const MidArgs& a, dim3 grid, hipStream_t stream) {
    switch (p.nb * 10 + p.nw) {
#define Q3_MID(nb, nw)                                                                                           \
    case nb * 10 + nw:                                                                                           \
        if (a.tm == 1)                                                                                           \
            Q3_LAUNCH((gemm_mid_kernel<MB, nb, nw, true>), grid, dim3((nw + MID_LOADERS<MB>) * 64), 0, stream, a); \
        else                                                                                                     \
            Q3_LAUNCH((gemm_mid_kernel<MB, nb, nw, false>), grid, dim3((nw + MID_LOADERS<MB>) * 64), 0, stream, a); \
        return (int)hipGetLastError();
        Q3_MID(1, 2) Q3_MID(1, 3) Q3_MID(1, 4) Q3_MID(1, 5) Q3_MID(2, 3) Q3_MID(2, 5) Q3_MID(2, 8)
#undef Q3_MID
    }
    return (int)hipErrorInvalidValue;
}

// y = epi(x . W^T) under plan p.
inline int launch_mid(const MidPlan& p, const bf16_t* x, int ldx, const bf16_t* w, int M, int N, int K, int epi,
                      bf16_t* y, int ldy, hipStream_t stream) {
    if (epi != Q3_EPI_STORE && epi != Q3_EPI_RESID && epi != Q3_EPI_SWIGLU) return (int)hipErrorInvalidValue;
    const int64_t tiles = mid_tiles(p, M, N);
    if (tiles > (1 << 30)) return (int)hipErrorInvalidValue;
    const MidArgs a{x, ldx, w, M, N, K, epi, y, ldy, (M + 16 * p.mb - 1) / (16 * p.mb)};
    const dim3 grid((unsigned)tiles);
    switch (p.mb) {
        case 1: return launch_mid_mb<1>(p, a, grid, stream);
        case 2: return launch_mid_mb<2>(p, a, grid, stream);
        case 3: return launch_mid_mb<3>(p, a, grid, stream);
        case 4: return launch_mid_mb<4>(p, a, grid, stream);
        case 5: return launch_mid_mb<5>(p, a, grid, stream);
        case 6: return launch_mid_mb<6>(p, a, grid, stream);
        case 7: return launch_mid_mb<7>(p, a, grid, stream);
        case 8: return launch_mid_mb<8>(p, a, grid, stream);
    }
    return (int)hipErrorInvalidValue;
}

}  // namespace q3gemm
