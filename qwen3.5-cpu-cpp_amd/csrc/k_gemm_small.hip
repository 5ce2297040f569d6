// Token-batched projection GEMM for few tokens (short prompts, chat turns, the last block of
// a long prompt): the products of k_gemm.hip on the same operands in the same order, so the
// same bits, cut so that a matrix of a few thousand rows still fills the chip. k_gemm.hip's
// 128 x 128 tiles are 16 to 96 workgroups for such a product, each walking all of K by
// itself: 53 us for any of up to 256 tokens at K = 2048, 150 us at K = 6144.
//
// Split: a workgroup's waves share a (16 MR) x (16 NR) tile and take one 512-deep block of K
// each (the partial sum that k_gemm.hip also accumulates from zero), so W and X go straight
// from memory to the matrix operands, with no barrier in the loop. The partial sums meet in
// LDS and are added in K order by the wave that then stores the 16 x 16 block. Deeper K takes
// several rounds, slot 0 carrying the running total.
//
// What bounds it: the lines a compute unit can have on the way. A compute unit streams
// weights at about 26 GB/s whatever its waves hold ready (32 KB of lines in flight, the size
// of its L1, at the 1.2 us a line takes under load), so the chip's 6.7 TB/s needs every one
// of the 256 busy to the end: 257 column tiles took 1.5 times as long as 256 (11.6 against
// 7.4 us, one token, K = 2048). Hence the tiles here are even shares of the columns and row
// blocks, not multiples of the tile with a ragged rest: 8224 columns are 256 tiles of 32 or
// 36. More tokens add the X lines of every column tile (each reads all X rows of its row
// tile) and the split of X into parts. Measured, weights from beyond the L2, against the
// 128 x 128 tiles: 8224 x 2048 rows of bf16 weights, 77 tokens 54.6 -> 24.9 us, 16 tokens
// 55.1 -> 12.7 us; fp16 parts already split, 32 tokens 37.8 -> 11.7 us; 2048 x 6144 with the
// fp16 split, 32 tokens 128.7 -> 16.1 us, 256 tokens 125.9 -> 40.2 us.
#include <algorithm>
#include <type_traits>

#include "dev_common.hpp"
#include "launch.hpp"

namespace q35k {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int kStep = 32;             // k per matrix instruction
constexpr int kSteps = 16;            // steps per partial sum
constexpr int kBlk = kStep * kSteps;  // K of one partial sum (512, as k_gemm.hip)
static_assert(kBlk == kSmallBlk, "the plan's block of K");

template <int PATH>
using operand = typename std::conditional<PATH == kBf16, bf16x8, halfx8>::type;

// The lane's two 16-byte pieces of each of its X rows (32 bytes of k) of one step
template <int PATH, int MR>
__device__ __forceinline__ void load_x(const float* const (&arow)[MR], u32x4 (&x)[MR][2], int k0, int kx) {
#pragma unroll
    for (int r = 0; r < MR; ++r)
#pragma unroll
        for (int i = 0; i < 2; ++i)
            x[r][i] = *reinterpret_cast<const u32x4*>(arow[r] + (PATH ? (k0 >> 5) * 512 + 256 * i : kx + 4 * i));
}

// part += the products of one step, smallest part of X first
template <int PATH, int MR, int NR>
__device__ __forceinline__ void step(const u32x4 (&xa)[MR][2], const u32x4 (&wb)[NR], const float (&xs)[MR],
                                     floatx4 (&part)[MR][NR]) {
    using OpT = operand<PATH>;
    constexpr int NP = PATH == kBf16 ? 3 : 2;
#pragma unroll
    for (int r = 0; r < MR; ++r) {
        OpT aop[NP];
        if constexpr (PATH == kF16Planes) {
            aop[0] = __builtin_bit_cast(OpT, xa[r][0]);
            aop[1] = __builtin_bit_cast(OpT, xa[r][1]);
        } else {
            const float4 x0 = __builtin_bit_cast(float4, xa[r][0]), x1 = __builtin_bit_cast(float4, xa[r][1]);
            uint32_t h[4], m[4], l[4];
            if constexpr (PATH == kF16) {
                const float sc = xs[r];
                split2h_pair(x0.x * sc, x0.y * sc, h[0], l[0]);
                split2h_pair(x0.z * sc, x0.w * sc, h[1], l[1]);
                split2h_pair(x1.x * sc, x1.y * sc, h[2], l[2]);
                split2h_pair(x1.z * sc, x1.w * sc, h[3], l[3]);
            } else {
                split3_pair(x0.x, x0.y, h[0], m[0], l[0]);
                split3_pair(x0.z, x0.w, h[1], m[1], l[1]);
                split3_pair(x1.x, x1.y, h[2], m[2], l[2]);
                split3_pair(x1.z, x1.w, h[3], m[3], l[3]);
                aop[1] = __builtin_bit_cast(OpT, u32x4{m[0], m[1], m[2], m[3]});
            }
            aop[0] = __builtin_bit_cast(OpT, u32x4{h[0], h[1], h[2], h[3]});
            aop[NP - 1] = __builtin_bit_cast(OpT, u32x4{l[0], l[1], l[2], l[3]});
        }
#pragma unroll
        for (int p = NP - 1; p >= 0; --p)
#pragma unroll
            for (int j = 0; j < NR; ++j) {
                const OpT w = __builtin_bit_cast(OpT, wb[j]);
                if constexpr (PATH == kBf16) part[r][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(aop[p], w, part[r][j], 0, 0, 0);
                else part[r][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(aop[p], w, part[r][j], 0, 0, 0);
            }
    }
}

template <int MR, int NR>
__device__ __forceinline__ void zero(floatx4 (&part)[MR][NR]) {
#pragma unroll
    for (int r = 0; r < MR; ++r)
#pragma unroll
        for (int j = 0; j < NR; ++j) part[r][j] = floatx4{0.f, 0.f, 0.f, 0.f};
}

// Partial sum of one whole 512-deep K block of a (16 MR) x (16 NR) tile by one wave.
template <int PATH, int MR, int NR>
__device__ __forceinline__ void block_part(const float* const (&arow)[MR], const float (&xs)[MR],
                                           const uint16_t* const (&wrow)[NR], int kb, floatx4 (&part)[MR][NR]) {
    // Requests go out for two steps (64 k, one 128-byte line of a W row) at a time. Pairs
    // ahead: a compute unit holds about 32 KB of requested lines, 8 KB a wave.
    constexpr int PA = MR == 1 ? 3 : MR == 2 ? 2 : 1;
    constexpr int PB = NR == 1 ? 4 : NR == 2 ? 3 : NR == 3 ? 2 : MR >= 3 ? 1 : 2;
    const int kq = ((threadIdx.x & 63) >> 4) * 8;
    u32x4 xa[PA][2][MR][2], wb[PB][NR][2];
    auto load_w = [&](u32x4 (&w)[NR][2], int q) {
#pragma unroll
        for (int j = 0; j < NR; ++j)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                w[j][h] = *reinterpret_cast<const u32x4*>(wrow[j] + kb + (2 * q + h) * kStep + kq);
    };
    auto load_xp = [&](u32x4 (&x)[2][MR][2], int q) {
#pragma unroll
        for (int h = 0; h < 2; ++h) load_x<PATH>(arow, x[h], kb + (2 * q + h) * kStep, kb + (2 * q + h) * kStep + kq);
    };
#pragma unroll
    for (int q = 0; q < (PA > PB ? PA : PB); ++q) {
        if (q < PB) load_w(wb[q], q);
        if (q < PA) load_xp(xa[q], q);
    }
    zero(part);
#pragma unroll
    for (int q = 0; q < kSteps / 2; ++q) {
        __builtin_amdgcn_sched_barrier(0);  // the requests stay ahead of the products
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            u32x4 w[NR];
#pragma unroll
            for (int j = 0; j < NR; ++j) w[j] = wb[q % PB][j][h];
            step<PATH, MR, NR>(xa[q % PA][h], w, xs, part);
        }
        if (q + PA < kSteps / 2) load_xp(xa[q % PA], q + PA);
        if (q + PB < kSteps / 2) load_w(wb[q % PB], q + PB);
    }
}

// The same for a last block that ends at K: two steps at a time, what lies past K as zeros
// (K % 8 == 0, so a lane's 8 k are wholly inside or wholly past K).
template <int PATH, int MR, int NR>
__device__ __forceinline__ void block_part_tail(const float* const (&arow)[MR], const float (&xs)[MR],
                                                const uint16_t* const (&wrow)[NR], int kb, int K, floatx4 (&part)[MR][NR]) {
    constexpr int U = MR * NR == 1 || MR * NR == 4 ? 4 : 2;
    const int kq = ((threadIdx.x & 63) >> 4) * 8;
    zero(part);
#pragma unroll 1
    for (int k0 = kb; k0 < K; k0 += U * kStep) {
        u32x4 xa[U][MR][2], wb[U][NR];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int ks = min(k0 + u * kStep, (K - 1) & ~(kStep - 1)), kl = min(k0 + u * kStep + kq, K - 8);
            load_x<PATH>(arow, xa[u], ks, kl);
#pragma unroll
            for (int j = 0; j < NR; ++j) wb[u][j] = *reinterpret_cast<const u32x4*>(wrow[j] + kl);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (k0 + u * kStep + kq >= K) {
#pragma unroll
                for (int r = 0; r < MR; ++r) xa[u][r][0] = xa[u][r][1] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
                for (int j = 0; j < NR; ++j) wb[u][j] = u32x4{0u, 0u, 0u, 0u};
            }
            step<PATH, MR, NR>(xa[u], wb[u], xs, part);
        }
    }
}

// start of piece i when n units are cut into `pieces` as evenly as they come
__device__ __forceinline__ int cut(int n, int pieces, int i) { return static_cast<int>(static_cast<int64_t>(n) * i / pieces); }

template <int PATH, int MR, int NR>
__global__ __launch_bounds__(64 * max_waves(MR, NR), max_waves(MR, NR) == 4 ? 2 : 1) void gemm_small_kernel(GemmArgs a,
                                                                                                          SmallPlan p) {
    constexpr int NB = MR * NR;
    extern __shared__ __align__(16) floatx4 slots[];  // [waves][NB][64]
    __shared__ int xe_s[16 * MR];
    __shared__ unsigned ym_s[16 * MR];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nwaves = blockDim.x >> 6;
    const int l16 = lane & 15, g4 = lane >> 4;
    // workgroups go to the 8 XCDs in turn: the row tiles of one column tile get ids of one
    // residue mod 8, next to each other, so its W rows are fetched into one L2 once
    int tx = blockIdx.x, ty = 0;
    if (p.rt > 1) {
        const int i = blockIdx.x / kXcds;
        tx = (i / p.rt) * kXcds + (blockIdx.x & (kXcds - 1));
        ty = i % p.rt;
        if (tx >= p.ct) return;  // uniform
    }
    const int units = (a.N + p.unit - 1) / p.unit, blocks = (a.M + 15) >> 4;
    const int n0 = cut(units, p.ct, tx) * p.unit, n1 = min(cut(units, p.ct, tx + 1) * p.unit, a.N);
    const int m0 = cut(blocks, p.rt, ty) * 16, m1 = min(cut(blocks, p.rt, ty + 1) * 16, a.M);

    const float* arow[MR];
    float xs[MR];
#pragma unroll
    for (int r = 0; r < MR; ++r) {  // rows past the tile: its first block or row again, stored by nobody
        const int row = min(m0 + 16 * r + l16, m1 - 1);
        const int blk = m0 + 16 * r < m1 ? (m0 >> 4) + r : m0 >> 4;
        arow[r] = PATH ? a.X + static_cast<int64_t>(blk) * (a.K >> 5) * 512 + (PATH == kF16Planes ? lane << 2 : (l16 << 4) + (g4 << 2))
                       : a.X + static_cast<int64_t>(row) * a.ldx;
        xs[r] = 1.0f;
        if constexpr (PATH != kBf16) {
            float mx = 0.0f;
            const float* xm = a.xmax + static_cast<int64_t>(row) * a.xmax_n;
            if ((a.xmax_n & 3) == 0 && (reinterpret_cast<uintptr_t>(a.xmax) & 15) == 0) {  // uniform
                for (int j = 4 * g4; j < a.xmax_n; j += 16) {
                    const float4 q = *reinterpret_cast<const float4*>(xm + j);
                    mx = fmaxf(mx, fmaxf(fmaxf(q.x, q.y), fmaxf(q.z, q.w)));
                }
            } else {
                for (int j = g4; j < a.xmax_n; j += 4) mx = fmaxf(mx, xm[j]);
            }
            mx = fmaxf(mx, __shfl_xor(mx, 16));
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            const int xe = split_row_exp(mx);
            xs[r] = ldexpf(1.0f, xe);
            if (wave == 0 && lane < 16) xe_s[16 * r + lane] = xe;
        }
    }
    if (tid < 16 * MR) ym_s[tid] = 0u;
    const uint16_t* wrow[NR];
#pragma unroll
    for (int j = 0; j < NR; ++j) wrow[j] = (PATH ? a.Wh : a.W) + static_cast<int64_t>(min(n0 + 16 * j + l16, n1 - 1)) * a.K;

    // one output block (16 rows x 16 columns; lane: rows 4 g4 .. + 3 of column l16)
    auto epilogue = [&](int b, floatx4 t) {
        const int br = b / NR, bj = b - br * NR;
        const int lrow = 16 * br + 4 * g4, rbase = m0 + lrow, col = n0 + 16 * bj + l16;
        if constexpr (PATH != kBf16) {
#pragma unroll
            for (int v = 0; v < 4; ++v) t[v] *= ldexpf(1.0f, -(xe_s[lrow + v] + a.w_exp));
        }
        if (a.swiglu) {  // columns (2 i, 2 i + 1) are (gate, up): adjacent lanes, n0 even
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const float up = __shfl_xor(t[v], 1);
                const int row = rbase + v;
                const float h = silu_f(t[v]) * up;
                const bool mine = !(lane & 1) && col + 1 < n1;
                if (mine && row < m1)
                    a.Y[a.y_tiled ? xt_off(row, col >> 1, a.N >> 1) : static_cast<int64_t>(row) * a.ldy + (col >> 1)] = h;
                if (a.ymax) {  // uniform; the bits of non-negative floats order as integers do
                    float m = mine ? fmaxf(0.0f, fabsf(h)) : 0.0f;
                    m = fmaxf(m, __shfl_xor(m, 2));
                    m = fmaxf(m, __shfl_xor(m, 4));
                    m = fmaxf(m, __shfl_xor(m, 8));
                    if (l16 == 0) atomicMax(&ym_s[lrow + v], __float_as_uint(m));
                }
            }
        } else if (col < n1) {
            float rv[4] = {0.f, 0.f, 0.f, 0.f};
            if (a.R) {  // uniform; the residual may be Y: all reads before the first write
#pragma unroll
                for (int v = 0; v < 4; ++v) rv[v] = a.R[static_cast<int64_t>(min(rbase + v, m1 - 1)) * a.ldr + col];
            }
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (rbase + v < m1) a.Y[static_cast<int64_t>(rbase + v) * a.ldy + col] = a.R ? rv[v] + t[v] : t[v];
        }
    };

    const int nblk = (a.K + kBlk - 1) / kBlk;
    for (int b0 = 0; b0 < nblk; b0 += nwaves) {
        const int blk = b0 + wave;
        if (blk < nblk) {  // uniform per wave
            floatx4 part[MR][NR];
            if (kBlk * (blk + 1) <= a.K) block_part<PATH, MR, NR>(arow, xs, wrow, kBlk * blk, part);
            else block_part_tail<PATH, MR, NR>(arow, xs, wrow, kBlk * blk, a.K, part);
#pragma unroll
            for (int r = 0; r < MR; ++r)
#pragma unroll
                for (int j = 0; j < NR; ++j) {
                    floatx4& s = slots[(wave * NB + r * NR + j) * 64 + lane];
                    // slot 0 keeps the running total of the rounds before
                    s = (wave == 0 ? (b0 ? s : floatx4{0.f, 0.f, 0.f, 0.f}) + part[r][j] : part[r][j]);
                }
        }
        lds_barrier();
        const int nw = min(nwaves, nblk - b0);
        const bool last = b0 + nwaves >= nblk;
        for (int b = wave; b < NB; b += nwaves) {  // the partial sums in K order
            floatx4 t = slots[b * 64 + lane];
            for (int w = 1; w < nw; ++w) t += slots[(w * NB + b) * 64 + lane];
            if (last) epilogue(b, t);
            else slots[b * 64 + lane] = t;
        }
        if (!last) lds_barrier();
    }
    if (a.swiglu && a.ymax) {  // each row's maximum over this tile's outputs
        lds_barrier();
        if (tid < m1 - m0) a.ymax[static_cast<int64_t>(m0 + tid) * p.ct + tx] = __uint_as_float(ym_s[tid]);
    }
}

template <int PATH, int MR, int NR>
hipError_t launch_tile(const GemmArgs& a, const SmallPlan& p, hipStream_t s) {
    const int nblk = (a.K + kBlk - 1) / kBlk, mw = max_waves(MR, NR);
    const int rounds = (nblk + mw - 1) / mw, waves = (nblk + rounds - 1) / rounds;
    const uint32_t lds = static_cast<uint32_t>(waves) * MR * NR * 64 * 16;  // at most 64 KB, (4, 4); 0.5 KB more are static
    const int grid = p.rt > 1 ? (p.ct + kXcds - 1) / kXcds * kXcds * p.rt : p.ct;
    klaunch(gemm_small_kernel<PATH, MR, NR>, dim3(grid), 64 * waves, lds, s, a, p);
    return hipGetLastError();
}

template <int PATH>
hipError_t launch_path(const GemmArgs& a, const SmallPlan& p, hipStream_t s) {
    switch (p.mr * 10 + p.nr) {
        case 11: return launch_tile<PATH, 1, 1>(a, p, s);
        case 12: return launch_tile<PATH, 1, 2>(a, p, s);
        case 13: return launch_tile<PATH, 1, 3>(a, p, s);
        case 15: return launch_tile<PATH, 1, 5>(a, p, s);
        case 22: return launch_tile<PATH, 2, 2>(a, p, s);
        case 23: return launch_tile<PATH, 2, 3>(a, p, s);
        case 24: return launch_tile<PATH, 2, 4>(a, p, s);
        case 25: return launch_tile<PATH, 2, 5>(a, p, s);
        case 33: return launch_tile<PATH, 3, 3>(a, p, s);
        case 35: return launch_tile<PATH, 3, 5>(a, p, s);
        case 43: return launch_tile<PATH, 4, 3>(a, p, s);
        case 44: return launch_tile<PATH, 4, 4>(a, p, s);
        default: return hipErrorInvalidValue;
    }
}

int path_of(const GemmArgs& a) {  // as launch_gemm's
    return a.Wh && a.xmax && a.xmax_n > 0 && a.x_tiled ? (a.x_planes ? kF16Planes : kF16) : kBf16;
}

bool small_plan(const GemmArgs& a, SmallPlan* best) {
    return gemm_small_plan(a.M, a.N, a.K, a.swiglu != 0, path_of(a), device_cu_count(), best);
}

}  // namespace

bool launch_gemm_small(const GemmArgs& a, hipStream_t s, hipError_t* e) {
    SmallPlan p;
    if (!small_plan(a, &p)) return false;
    switch (path_of(a)) {
        case kF16Planes: *e = launch_path<kF16Planes>(a, p, s); break;
        case kF16: *e = launch_path<kF16>(a, p, s); break;
        default: *e = launch_path<kBf16>(a, p, s);
    }
    return true;
}

int gemm_ymax_parts(const GemmArgs& a) {
    SmallPlan p;
    return small_plan(a, &p) ? p.ct : gemm_col_tiles(a.N);
}

}  // namespace q35k
