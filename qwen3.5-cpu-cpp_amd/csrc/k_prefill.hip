// Whole-prompt mixers (QwenForward::mix_gdn src/qwen_forward.cpp:83-152 and
// QwenForward::mix_attention src/qwen_forward.cpp:20-80), on a block of T tokens that starts
// at position pos0 and continues from the model's state (so prefill and decode hand over).
//
// Gated DeltaNet, chunked (chunk C = 64, the WY form of the gated delta rule):
//   chunk    per (v-head, chunk), from the raw projection rows: conv window + SiLU per
//            channel (the three inputs before the block come from the conv ring), l2norm of
//            q and k per token, q scaled by DK^-1/2, beta = sigmoid(b),
//            g = -exp(A_log) softplus(a + dt_bias); rows past the block (padding to whole
//            chunks) have q = k = v = 0, beta = g = 0 and change nothing. q goes head-major to
//            the workspace for the output pass. gamma = cumsum(g) in double (every decay factor
//            below is e^(a difference of gammas) rounded once: an fp32 running sum would lose
//            ~1e-6 of each exponent to cancellation, gamma reaching -40 within a chunk); the
//            chunk's e^gamma and e^(gamma_last - gamma) go to the workspace for the later passes;
//            Q K^T and K K^T on the fp32 matrix cores (the 10 lower-triangle 16 x 16 blocks);
//              P[i][j] = q_i.k_j e^(gamma_i - gamma_j)      (j <= i)
//              A[i][j] = beta_i k_i.k_j e^(gamma_i - gamma_j)  (j < i)
//              [U | W] = (I + A)^-1 [beta v | beta e^gamma k]  (by 16-row blocks on the
//                                                               matrix cores)
//   state    per (v-head, 8-column slice of the state), sequential over the chunks, on the
//            fp32 matrix cores: store the chunk-start state S_c, v_new = U - W S,
//              S <- e^(gamma_last) S + K^T (e^(gamma_last - gamma) v_new)
//            The delta rule is column-separable, so the 16 slices of a head are independent.
//            Then the last three raw inputs of the block go to their ring slots (the chunk
//            pass has read the old ones).
//   output   per (v-head, chunk), in parallel: o = e^gamma (Q S_c) + P v_new on the matrix
//            cores, then rmsnorm_gated per (token, v-head) (src/forward_pass.cpp:86-93).
// Causal attention, flash form on the bf16 matrix cores:
//   prep     q_norm + RoPE of every query row (head-major), k_norm + RoPE of every key and
//            the values appended to the KV cache at pos0 + t (angles in double; a bf16 cache
//            stores them rounded to nearest even and the flash kernel widens them back).
//   flash    per block of 128 (bf16 cache: 64) rows, a row one (token, head of the group):
//            waves of 16 rows with their q in registers (as three bf16 parts); 32-position
//            K / V tiles in LDS (in bf16 parts); S = Q K^T and O += P V on the bf16 matrix
//            cores from six part products each; running max / sum per row; epilogue
//            O / l * sigmoid(gate). Long key ranges are cut and merged (flash_plan).
#include <math.h>

#include "dev_common.hpp"
#include "launch.hpp"

namespace q35k {
namespace {

constexpr int kD = 128;   // GDN head dim
constexpr int kC = 64;    // chunk length
constexpr int kHD = 256;  // attention head dim

// ring slots of the block's last three raw inputs (blocks of few tokens whose v-heads share
// k-heads: there no workgroup is the only reader of a channel's old slots)
__global__ __launch_bounds__(256) void gdn_ring_kernel(GdnPrefillArgs a) {
    const int KD = a.KH * kD, VD = a.VH * kD, CONV = 2 * KD + VD;
    const int t0 = a.T > 3 ? a.T - 3 : 0;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < (a.T - t0) * CONV; i += gridDim.x * 256) {
        const int t = t0 + i / CONV, ch = i % CONV;
        a.conv_ring[static_cast<int64_t>((a.pos0 + t) & 3) * CONV + ch] = a.qkv[static_cast<int64_t>(t) * a.ld_qkv + ch];
    }
}

// v_mfma_f32_16x16x4_f32, one block: lane l supplies A[l % 16][l / 16] and B[l / 16][l % 16];
// result register v of lane l is D[4 (l / 16) + v][l % 16].
typedef float floatx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ floatx4 mfma4(float a, float b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// ------------------------------------------------------------------ GDN chunk
constexpr int kLdC = kD + 4;
constexpr int kLdA = 20;  // rows of A's 16 x 16 blocks
constexpr int kRun = 8;   // tokens per conv run

// block (r, b) of the lower triangle of 16 x 16 blocks
__device__ __forceinline__ constexpr int tri(int r, int b) { return r * (r + 1) / 2 + b; }

// 4 x 4 transpose over the four lanes of a quad and four registers
__device__ __forceinline__ floatx4 quad_transpose(floatx4 x, int lane) {
    const bool o1 = lane & 1, o2 = lane & 2;
    const float s0 = dpp_f<0xB1>(o1 ? x[0] : x[1]), s1 = dpp_f<0xB1>(o1 ? x[2] : x[3]);  // from lane ^ 1
    x = o1 ? floatx4{s0, x[1], s1, x[3]} : floatx4{x[0], s0, x[2], s1};
    const float t0 = dpp_f<0x4E>(o2 ? x[0] : x[2]), t1 = dpp_f<0x4E>(o2 ? x[1] : x[3]);  // from lane ^ 2
    return o2 ? floatx4{t0, t1, x[2], x[3]} : floatx4{x[0], x[1], t0, t1};
}

// Wave WV's share of the chunk's products: Q K^T of row block WV and K K^T of row block 3 - WV,
// five 16 x 16 blocks of the lower triangle in all. P goes to memory, A to LDS: blocks below
// the diagonal negated, the diagonal one as T = (I + A)^-1 (column lane % 16 by substitution).
template <int WV>
__device__ __forceinline__ void gdn_products(const float (*Qs)[kLdC], const float (*Ks)[kLdC], float (*As)[16][kLdA],
                                             const double* gam, const float* beta, float* P, int lane) {
    constexpr int RK = 3 - WV, NB = (WV > RK ? WV : RK) + 1;
    const int lr = lane & 15, lg = lane >> 4;
    floatx4 sq[WV + 1] = {}, sk[RK + 1] = {};
    // MFMA j of a 16-deep step takes dim 4 lg + j of lane group lg: operands 16 bytes at a time
#pragma unroll 2
    for (int k = 0; k < kD; k += 16) {
        const floatx4 q = *reinterpret_cast<const floatx4*>(&Qs[16 * WV + lr][k + 4 * lg]);
        floatx4 kb[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) kb[b] = *reinterpret_cast<const floatx4*>(&Ks[16 * b + lr][k + 4 * lg]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int b = 0; b <= WV; ++b) sq[b] = mfma4(q[j], kb[b][j], sq[b]);
#pragma unroll
            for (int b = 0; b <= RK; ++b) sk[b] = mfma4(kb[RK][j], kb[b][j], sk[b]);
        }
    }
#pragma unroll
    for (int b = 0; b <= RK; ++b)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int i = 16 * RK + 4 * lg + v, j = 16 * b + lr;
            const float x = j < i ? beta[i] * sk[b][v] * expf(static_cast<float>(gam[i] - gam[j])) : 0.0f;
            As[tri(RK, b)][4 * lg + v][lr] = b < RK ? -x : x;
        }
#pragma unroll
    for (int b = 0; b <= WV; ++b)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int i = 16 * WV + 4 * lg + v, j = 16 * b + lr;
            P[i * kC + j] = j <= i ? sq[b][v] * expf(static_cast<float>(gam[i] - gam[j])) : 0.0f;
        }
    float (*D)[kLdA] = As[tri(RK, RK)];
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        x[i] = i == lr ? 1.0f : 0.0f;
#pragma unroll
        for (int k = 0; k < i; ++k) x[i] = fmaf(-D[i][k], x[k], x[i]);
    }
    if (lg == 0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) D[i][lr] = x[i];
    }
}

// grid (VH, Tp / 64), 256 threads: the whole chunk pass of one (v-head, chunk of 64 tokens).
//   inputs   thread (run, quad) convolves channels 4 quad .. + 3 of the head's q, k and v over
//            tokens 8 run .. + 7 of the chunk (eleven raw rows, 16 bytes per load), and each
//            32-lane half-wave (one run) sums a token's squares for the l2norm (in double);
//            wave 0 forms beta and g and their running sum (a wave scan in double).
//   products P and A on the fp32 matrix cores over the lower triangle of 16 x 16 blocks, five
//            blocks per wave (gdn_products); K and Q rows padded to 132 floats so that the 16
//            rows of an operand read fall in 64 distinct banks.
//   solve    [U | W] in 16 column groups, four per wave, block by block on the matrix cores:
//            X_b = T_bb (R_b - sum of A_bc X_c over c < b). A product's result registers
//            (rows 4 lg + v of column lr) are the next one's operands with its steps in the
//            order 4 lg + j, so X stays in registers.
// beta v takes Q's place once the products are done (80 KB of LDS: two workgroups per CU).
// 4096 tokens of 16 heads: 115 us with the solve as substitution, one column of 64 per thread
// (2016 dependent fused multiply-adds and 20 KB of code), one thread summing gamma and the v
// columns convolved by half the threads; 90 so, and one chunk's passes 58 -> 43 us. Of the 90 the
// exact SiLU divisions take 16 and the products 8; 250 MB of inputs and results take 53 at the
// rate of a large copy.
__global__ __launch_bounds__(256, 2) void gdn_chunk_kernel(GdnPrefillArgs a) {
    const int vh = blockIdx.x, c = blockIdx.y, tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 15, lg = lane >> 4;
    const int rep = a.VH / a.KH, kh = vh / rep;
    const int KD = a.KH * kD, VD = a.VH * kD, CONV = 2 * KD + VD;
    const int t0 = c * kC;
    __shared__ __align__(16) float Ks[kC][kLdC];
    __shared__ __align__(16) float QV[kC][kLdC];  // Q, then beta v
    __shared__ __align__(16) float As[10][16][kLdA];
    __shared__ double gam[kC];
    __shared__ __align__(16) float beta[kC], bex[kC], edl[kC];  // beta, beta e^gamma, e^(gamma_last - gamma)
    // raw input of block token s (s < 0: the conv ring; s >= T: a padding row, zeroed below)
    auto xin4 = [&](int s, int ch) -> float4 {
        if (s >= 0) return *reinterpret_cast<const float4*>(a.qkv + static_cast<int64_t>(min(s, a.T - 1)) * a.ld_qkv + ch);
        return *reinterpret_cast<const float4*>(a.conv_ring + static_cast<int64_t>((a.pos0 + s) & 3) * CONV + ch);
    };
    const int run = tid >> 5, c4 = 4 * (tid & 31);
    const int ts0 = t0 + kRun * run;
    auto load_run = [&](int ch, float4 (&x)[kRun + 3], float4 (&w)[4]) {
#pragma unroll
        for (int j = 0; j < kRun + 3; ++j) x[j] = xin4(ts0 - 3 + j, ch);
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = *reinterpret_cast<const float4*>(a.conv_w + static_cast<int64_t>(ch + e) * 4);
    };
    // causal conv + SiLU of four channels over a run (the reference's 4-tap window,
    // src/qwen_forward.cpp:109-118)
    auto conv_run = [&](const float4 (&x)[kRun + 3], const float4 (&w)[4], float (&y)[kRun][4]) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float xs[kRun + 3];
#pragma unroll
            for (int j = 0; j < kRun + 3; ++j) xs[j] = e == 0 ? x[j].x : e == 1 ? x[j].y : e == 2 ? x[j].z : x[j].w;
#pragma unroll
            for (int j = 0; j < kRun; ++j) {
                float acc = 0.0f;
                acc += w[e].x * xs[j];
                acc += w[e].y * xs[j + 1];
                acc += w[e].z * xs[j + 2];
                acc += w[e].w * xs[j + 3];
                y[j][e] = silu_f(acc);
            }
        }
    };
    // l2norm of each token of a run, in place (a token is one half-wave)
    auto l2norm = [&](float (&y)[kRun][4]) {
#pragma unroll
        for (int j = 0; j < kRun; ++j) {
            double ss = 0.0;
#pragma unroll
            for (int e = 0; e < 4; ++e) ss += static_cast<double>(y[j][e]) * y[j][e];
            ss = half_wave_sum(ss);
            const float inv = 1.0f / sqrtf(static_cast<float>(ss) + 1e-6f);
#pragma unroll
            for (int e = 0; e < 4; ++e) y[j][e] *= inv;
        }
    };
    float4 xq[kRun + 3], xk[kRun + 3], xv[kRun + 3], wq[4], wk[4], wv[4];
    load_run(kh * kD + c4, xq, wq);
    load_run(KD + kh * kD + c4, xk, wk);
    if (wave == 0) {
        const int t = t0 + lane;
        float bb = 0.0f, gg = 0.0f;
        if (t < a.T) {
            bb = sigmoid_f(a.b[static_cast<int64_t>(t) * a.ld_ba + vh]);
            gg = -expf(a.A_log[vh]) * softplus_f(a.a[static_cast<int64_t>(t) * a.ld_ba + vh] + a.dt_bias[vh]);
        }
        double g = gg;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const double p = __shfl_up(g, o);
            if (lane >= o) g += p;
        }
        const float eg = expf(static_cast<float>(g));
        gam[lane] = g;
        beta[lane] = bb;
        bex[lane] = bb * eg;
        edl[lane] = expf(static_cast<float>(__shfl(g, 63) - g));
        a.Eg[static_cast<int64_t>(vh) * a.Tp + t] = eg;
    }
    float y[kRun][4];
    {
        // q: l2norm, scaled by DK^-1/2; to LDS and (once per k-head) to the workspace
        const bool write_q = vh % rep == 0;
        const float qs = 1.0f / sqrtf(static_cast<float>(kD));
        conv_run(xq, wq, y);
        load_run(2 * KD + vh * kD + c4, xv, wv);  // in q's registers, for after k
        l2norm(y);
#pragma unroll
        for (int j = 0; j < kRun; ++j) {
            float4 o = make_float4(y[j][0] * qs, y[j][1] * qs, y[j][2] * qs, y[j][3] * qs);
            if (ts0 + j >= a.T) o = make_float4(0.f, 0.f, 0.f, 0.f);
            *reinterpret_cast<float4*>(&QV[kRun * run + j][c4]) = o;
            if (write_q) *reinterpret_cast<float4*>(a.Qg + (static_cast<int64_t>(kh) * a.Tp + ts0 + j) * kD + c4) = o;
        }
    }
    conv_run(xk, wk, y);
    l2norm(y);
#pragma unroll
    for (int j = 0; j < kRun; ++j) {
        float4 o = make_float4(y[j][0], y[j][1], y[j][2], y[j][3]);
        if (ts0 + j >= a.T) o = make_float4(0.f, 0.f, 0.f, 0.f);
        *reinterpret_cast<float4*>(&Ks[kRun * run + j][c4]) = o;
    }
    conv_run(xv, wv, y);
    lds_barrier();  // Q, K, beta and gamma in LDS
    {
        float* P = a.P + (static_cast<int64_t>(vh) * (a.Tp / kC) + c) * kC * kC;
        // (P blocks above the diagonal are never read and are left unwritten)
        if (wave == 0) gdn_products<0>(QV, Ks, As, gam, beta, P, lane);
        else if (wave == 1) gdn_products<1>(QV, Ks, As, gam, beta, P, lane);
        else if (wave == 2) gdn_products<2>(QV, Ks, As, gam, beta, P, lane);
        else gdn_products<3>(QV, Ks, As, gam, beta, P, lane);
    }
    lds_barrier();  // A in LDS; every read of Q done
#pragma unroll
    for (int j = 0; j < kRun; ++j) {
        const float b = beta[kRun * run + j];
        float4 o = make_float4(b * y[j][0], b * y[j][1], b * y[j][2], b * y[j][3]);
        if (ts0 + j >= a.T) o = make_float4(0.f, 0.f, 0.f, 0.f);
        *reinterpret_cast<float4*>(&QV[kRun * run + j][c4]) = o;
    }
    lds_barrier();
    // [U | W] = (I + A)^-1 [beta v | beta e^gamma k]: waves 0 and 1 the columns of U, 2 and 3 of W
    const int64_t head = (static_cast<int64_t>(vh) * a.Tp + t0) * kD;
    floatx4 at[10];
#pragma unroll
    for (int n = 0; n < 10; ++n) at[n] = *reinterpret_cast<const floatx4*>(&As[n][lr][4 * lg]);
    const bool isw = wave >= 2;
    const int g0 = 4 * (wave & 1);  // first of the wave's four column groups
    const float (*R)[kLdC] = isw ? Ks : QV;
    floatx4 x[4][4];  // [block][column group]
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        const floatx4 f = isw ? *reinterpret_cast<const floatx4*>(&bex[16 * b + 4 * lg]) : floatx4{1.f, 1.f, 1.f, 1.f};
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int v = 0; v < 4; ++v) x[b][g][v] = f[v] * R[16 * b + 4 * lg + v][16 * (g0 + g) + lr];
#pragma unroll
        for (int e = 0; e < b; ++e)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int g = 0; g < 4; ++g) x[b][g] = mfma4(at[tri(b, e)][j], x[e][g][j], x[b][g]);
        floatx4 y4[4] = {};
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) y4[g] = mfma4(at[tri(b, b)][j], x[b][g][j], y4[g]);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            x[b][g] = y4[g];
            if (isw) {
                // operand order of the state pass (its comment): row 16 b + r, dims 16 g + 4 q .. + 3 at
                // 16-byte slot (8 b + g) 64 + 16 q + r
                const int q = lr >> 2, r = 4 * lg + (lr & 3);
                *reinterpret_cast<floatx4*>(a.W + head + ((8 * b + g0 + g) * 64 + 16 * q + r) * 4) = quad_transpose(y4[g], lane);
            } else {
#pragma unroll
                for (int v = 0; v < 4; ++v) a.U[head + (16 * b + 4 * lg + v) * kD + 16 * (g0 + g) + lr] = y4[g][v];
            }
        }
    }
    // the decayed keys K[t][d] e^(gamma_last - gamma_t) in operand order: dim 32 w + l % 32,
    // tokens 16 (g / 2) + 8 (l / 32) + 4 (g % 2) .. + 3 at slot (8 w + g) 64 + l
#pragma unroll
    for (int n = 0; n < kC * kD / 4 / 256; ++n) {
        const int f = tid + 256 * n, g = (f >> 6) & 7, w = f >> 9;
        const int t = 16 * (g >> 1) + 8 * (lane >> 5) + 4 * (g & 1), d = 32 * w + (lane & 31);
        const floatx4 e = *reinterpret_cast<const floatx4*>(&edl[t]);
        *reinterpret_cast<floatx4*>(a.Kd + head + f * 4) =
            floatx4{Ks[t][d] * e[0], Ks[t + 1][d] * e[1], Ks[t + 2][d] * e[2], Ks[t + 3][d] * e[3]};
    }
}

// ------------------------------------------------------------------ GDN state scan
constexpr int kSW = 8;  // state columns per state-scan workgroup

// v_mfma_f32_4x4x1_16b_f32, 16 blocks of D[4][4] += a[4] b[4]: lane l supplies a[l % 4] and
// b[l % 4] of block l / 4; result register v of lane l is D[v][l % 4]. Every 2^CB consecutive
// blocks take their a from one of them, the J-th.
template <int CB, int J>
__device__ __forceinline__ floatx4 mfma1(float a, float b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, CB, J, 0);
}

// four steps for both column quads: s0, s1 the state side, w the operands of steps J .. J + 3
template <int CB, int J>
__device__ __forceinline__ void mfma_quad(float s0, float s1, floatx4 w, floatx4 (&acc)[2]) {
    acc[0] = mfma1<CB, J>(s0, w[0], acc[0]);
    acc[1] = mfma1<CB, J>(s1, w[0], acc[1]);
    acc[0] = mfma1<CB, J + 1>(s0, w[1], acc[0]);
    acc[1] = mfma1<CB, J + 1>(s1, w[1], acc[1]);
    acc[0] = mfma1<CB, J + 2>(s0, w[2], acc[0]);
    acc[1] = mfma1<CB, J + 2>(s1, w[2], acc[1]);
    acc[0] = mfma1<CB, J + 3>(s0, w[3], acc[0]);
    acc[1] = mfma1<CB, J + 3>(s1, w[3], acc[1]);
}

__device__ __forceinline__ void swap32(float& a, float& b) {  // lanes 32-63 of a <-> lanes 0-31 of b
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(int, a), __builtin_bit_cast(int, b), false, false);
    a = __builtin_bit_cast(float, static_cast<int>(r[0]));
    b = __builtin_bit_cast(float, static_cast<int>(r[1]));
}
__device__ __forceinline__ void swap16(float& a, float& b) {  // odd 16-lane rows of a <-> even rows of b
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(int, a), __builtin_bit_cast(int, b), false, false);
    a = __builtin_bit_cast(float, static_cast<int>(r[0]));
    b = __builtin_bit_cast(float, static_cast<int>(r[1]));
}

// grid (VH, 128 / kSW), 256 threads: sequential over the chunks of one state column slice, on
// the fp32 matrix cores. Per chunk: store the chunk-start state, v_new = U - W S (written over
// U), then S <- e^(gamma_last) S + (K e^(gamma_last - gamma))^T v_new.
//   The scan's length is fixed, so its time is that of one chunk step; with 16 v-heads 8-column
//   slices give every compute unit a workgroup. The 4x4x1 instruction runs at the rate of
//   16x16x4 and fills at 8 columns: the state (and v_new) is its a operand, four columns wide
//   and broadcast over blocks, W (and the decayed K) its b operand.
//   W and K go from memory into registers in operand order (the chunk pass lays them out so
//   that a lane's 16 bytes are its operands of four steps and a wave's load is 1 KB in a row),
//   two chunks ahead, each load asked for as soon as the eight products that free its registers
//   are issued (requested together, the 32 loads of a phase made the waves wait to issue them:
//   92 us a scan against 81); each value is used for both column quads. Only v_new and the
//   state, 2 KB and 4 KB, pass through LDS, each with one barrier per chunk:
//   v_new  wave w rows 16 w + lane % 16; lane group q = lane / 16 multiplies dims 16 g + 4 q + j
//          (step g, register j), the four groups' sums are added crosswise, and lane (q, r)
//          ends with columns 2 q, 2 q + 1 of its row
//   state  wave w dims 32 w + lane % 32; half p = lane / 32 multiplies tokens 16 g + 8 p + 0..7,
//          and lane (p, d) ends with columns 4 p .. + 3 of its dim, kept in registers
// 4096 tokens of 16 heads: 134 us as 16-column slices of 16x16x4 products with W, K and U staged
// through LDS (128 workgroups, 64 KB of LDS reads and as much of writes a chunk), 81 so; 66
// without the loads, about 30 of it the products.
__global__ __launch_bounds__(256, 2) void gdn_state_kernel(GdnPrefillArgs a) {
    // More heads than the chip holds at once (2 workgroups per unit): the slices of 8 heads follow
    // each other, each head on one XCD, so that a head's W and K are fetched once and not once per
    // round of workgroups (4096 tokens of 48 heads 758 -> 707 us, of 64 974 -> 932; of 24 heads,
    // which fit, 367 -> 377, and 16 and 32 the same either way).
    int vh = blockIdx.x, slice = blockIdx.y;
    if (gridDim.x > 32 && (gridDim.x & 7) == 0) {  // uniform
        const int id = blockIdx.y * gridDim.x + blockIdx.x;
        vh = (id >> 7) * 8 + (id & 7);
        slice = (id >> 3) & 15;
    }
    const int col0 = slice * kSW, tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int lr = lane & 15, q = lane >> 4;  // v_new: row of the wave's 16, lane group
    const int d = 32 * wave + (lane & 31), p = lane >> 5;  // state: dim, half
    const int nchunk = a.Tp / kC;
    __shared__ __align__(16) float St[2][kD][4];   // the state: column quad, dim, column
    __shared__ __align__(16) float Vn[2][kC][4];   // v_new: column quad, token, column
    float* S = a.state + static_cast<int64_t>(vh) * kD * kD + d * kD + col0 + 4 * p;
    floatx4 s = {S[0], S[1], S[2], S[3]};

    floatx4 rw[2][8], rk[2][8];  // operands of two chunks
    float2 ru[2];                // U of two chunks: this lane's two columns of its row
    // (uniform base + 32-bit lane offset: one scalar addition moves all of a chunk's addresses)
    const int64_t head = static_cast<int64_t>(vh) * a.Tp * kD;
    const uint32_t ow = (wave * 512 + lane) * 4, ou = (16 * wave + lr) * kD + col0 + 2 * q, os = d * kD + col0 + 4 * p;
    float re[2];  // e^gamma of two chunks' rows (only the last is used: a uniform address would
                  // be a scalar load, which the next LDS wait would wait for)
    auto chunk = [&](int c) { return head + static_cast<int64_t>(min(c, nchunk - 1)) * kC * kD; };
    auto load_w = [&](int c, floatx4 (&r)[8], float2& u) {
        const float* W = a.W + chunk(c);
#pragma unroll
        for (int g = 0; g < 8; ++g) r[g] = *reinterpret_cast<const floatx4*>(W + g * 256 + ow);
        u = *reinterpret_cast<const float2*>(a.U + chunk(c) + ou);
    };
    auto load_k = [&](int c, floatx4 (&r)[8], float& e) {
        const float* K = a.Kd + chunk(c);
#pragma unroll
        for (int g = 0; g < 8; ++g) r[g] = *reinterpret_cast<const floatx4*>(K + g * 256 + ow);
        e = a.Eg[static_cast<int64_t>(vh) * a.Tp + min(c, nchunk - 1) * kC + lane];
    };
    load_w(0, rw[0], ru[0]);
    load_k(0, rk[0], re[0]);
    load_w(1, rw[1], ru[1]);
    load_k(1, rk[1], re[1]);
    *reinterpret_cast<floatx4*>(&St[p][d][0]) = s;
    lds_barrier();
    auto step = [&](int c, floatx4 (&w)[8], floatx4 (&k)[8], float2& u, float& eg) {
        *reinterpret_cast<floatx4*>(a.Sc + (static_cast<int64_t>(vh) * nchunk + c) * kD * kD + os) = s;
        floatx4 acc[2] = {};
        float sa[2][8];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int g = 0; g < 8; ++g) sa[h][g] = (&St[h][0][0])[64 * g + lane];
        const float* Wn = a.W + chunk(c + 2);
#pragma unroll
        for (int g = 0; g < 8; ++g) {
            mfma_quad<2, 0>(sa[0][g], sa[1][g], w[g], acc);
            w[g] = *reinterpret_cast<const floatx4*>(Wn + g * 256 + ow);
            __builtin_amdgcn_sched_barrier(0);
        }
        float y[4], x[2];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            float lo = acc[0][v], hi = acc[1][v];
            swap32(lo, hi);
            y[v] = lo + hi;  // lanes below 32 column v, the others column 4 + v
        }
#pragma unroll
        for (int v = 0; v < 2; ++v) {
            swap16(y[v], y[v + 2]);
            x[v] = y[v] + y[v + 2];
        }
        const float2 vn = make_float2(u.x - x[0], u.y - x[1]);
        *reinterpret_cast<float2*>(&Vn[q >> 1][16 * wave + lr][2 * (q & 1)]) = vn;
        *reinterpret_cast<float2*>(a.U + chunk(c) + ou) = vn;
        u = *reinterpret_cast<const float2*>(a.U + chunk(c + 2) + ou);
        lds_barrier();  // v_new in LDS; every read of St done
        float va[2][4];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int g = 0; g < 4; ++g) va[h][g] = (&Vn[h][0][0])[64 * g + lane];
        floatx4 e[2] = {};
        const float elast = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, eg), 63));
        const float* Kn = a.Kd + chunk(c + 2);
#pragma unroll
        for (int g = 0; g < 8; ++g) {
            if (g & 1) mfma_quad<3, 4>(va[0][g >> 1], va[1][g >> 1], k[g], e);
            else mfma_quad<3, 0>(va[0][g >> 1], va[1][g >> 1], k[g], e);
            k[g] = *reinterpret_cast<const floatx4*>(Kn + g * 256 + ow);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            float lo = e[0][v], hi = e[1][v];
            swap32(lo, hi);
            s[v] = s[v] * elast + (lo + hi);
        }
        *reinterpret_cast<floatx4*>(&St[p][d][0]) = s;
        eg = a.Eg[static_cast<int64_t>(vh) * a.Tp + min(c + 2, nchunk - 1) * kC + lane];
        lds_barrier();  // the new state in LDS; every read of Vn done
    };
    for (int c = 0; c + 1 < nchunk; c += 2) {
        step(c, rw[0], rk[0], ru[0], re[0]);
        step(c + 1, rw[1], rk[1], ru[1], re[1]);
    }
    if (nchunk & 1) step(nchunk - 1, rw[0], rk[0], ru[0], re[0]);
#pragma unroll
    for (int v = 0; v < 4; ++v) S[v] = s[v];
    // ring slots of the block's last three raw inputs (the chunk pass has read the old ones)
    const int CONV = (2 * a.KH + a.VH) * kD, t0 = a.T > 3 ? a.T - 3 : 0;
    for (int i = (slice * gridDim.x + vh) * 256 + tid; i < (a.T - t0) * CONV; i += gridDim.x * gridDim.y * 256) {
        const int t = t0 + i / CONV, ch = i % CONV;
        a.conv_ring[static_cast<int64_t>((a.pos0 + t) & 3) * CONV + ch] = a.qkv[static_cast<int64_t>(t) * a.ld_qkv + ch];
    }
}

// ------------------------------------------------------------------ GDN chunk output
constexpr int kLdQ = kD + 4;    // Q rows (A operand)
constexpr int kLdS = kD + 16;   // state / v_new rows (B operand)

// grid (VH, Tp / 64), 256 threads: o = e^gamma (Q S_c) + P v_new for one chunk of one v-head,
// then the gated rmsnorm (src/forward_pass.cpp:86-93, sum of squares in double) or the raw
// readout. Wave w owns output rows [16w, 16w + 16), all 128 columns (8 blocks of 16).
// S_c goes through LDS in two halves of 64 rows (71 KB of LDS, two workgroups per CU); every
// operand is requested into registers at the start, so the later phases' loads (the second
// half of S_c, P and v_new, then the epilogue's gate and norm weight) arrive while the
// earlier phases multiply.
__global__ __launch_bounds__(256, 2) void gdn_out_kernel(GdnPrefillArgs a) {
    const int vh = blockIdx.x, c = blockIdx.y, tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6, lr = lane & 15, lg = lane >> 4;
    const int kh = vh / (a.VH / a.KH);
    const int nchunk = a.Tp / kC;
    const int64_t row0 = static_cast<int64_t>(c) * kC;
    // Operand order: within each 16-deep block of the product, MFMA step j takes from lane
    // group lg the index 4 lg + j, so a lane's four A values of the block are one 16-byte
    // read of its row; B rows are stored with their columns permuted (column 16 b + r at
    // 8 r + b), so a lane's eight column blocks of one B row are two 16-byte reads.
    __shared__ __align__(16) float A_s[kC][kLdQ];   // Q, then P
    __shared__ __align__(16) float B_s[kC][kLdS];   // S_c rows [0, 64), then [64, 128), then v_new
    __shared__ float eg[kC];  // e^gamma of the chunk's rows
    const float* Q = a.Qg + (static_cast<int64_t>(kh) * a.Tp + row0) * kD;
    const float* Sc = a.Sc + (static_cast<int64_t>(vh) * nchunk + c) * kD * kD;
    const float* P = a.P + (static_cast<int64_t>(vh) * nchunk + c) * kC * kC;
    const float* Vn = a.U + (static_cast<int64_t>(vh) * a.Tp + row0) * kD;
    constexpr int NQ4 = kC * kD / 4 / 256;  // float4 per thread of a 64 x 128 tile (8)
    constexpr int NP4 = kC * kC / 4 / 256;  // of the 64 x 64 P tile (4)
    auto put_b = [&](int f, floatx4 v) {  // float4 f of a row-major 64 x 128 tile -> B_s, permuted
        const int r = f >> 5, c0 = (f & 31) * 4;
#pragma unroll
        for (int i = 0; i < 4; ++i) B_s[r][((c0 + i) & 15) * 8 + ((c0 + i) >> 4)] = v[i];
    };
    floatx4 acc[8];
#pragma unroll
    for (int b = 0; b < 8; ++b) acc[b] = floatx4{0.f, 0.f, 0.f, 0.f};
    // acc += A[rows 16 w ..][acol .. acol + 15] . B[brow .. brow + 15][all 128 columns]
    auto mma16 = [&](int acol, int brow) {
        const float4 a4 = *reinterpret_cast<const float4*>(&A_s[16 * wave + lr][acol + 4 * lg]);
        const float av[4] = {a4.x, a4.y, a4.z, a4.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float4* bp = reinterpret_cast<const float4*>(&B_s[brow + 4 * lg + j][lr * 8]);
            const float4 b0 = bp[0], b1 = bp[1];
            acc[0] = mfma4(av[j], b0.x, acc[0]);
            acc[1] = mfma4(av[j], b0.y, acc[1]);
            acc[2] = mfma4(av[j], b0.z, acc[2]);
            acc[3] = mfma4(av[j], b0.w, acc[3]);
            acc[4] = mfma4(av[j], b1.x, acc[4]);
            acc[5] = mfma4(av[j], b1.y, acc[5]);
            acc[6] = mfma4(av[j], b1.z, acc[6]);
            acc[7] = mfma4(av[j], b1.w, acc[7]);
        }
    };
    // every operand is requested up front (Q and S_c[0:64) first: loads complete in order
    // for the wait counter, so the first phase waits for those alone)
    // (vector-typed register arrays: arrays of float4 structs were placed in scratch)
    floatx4 rq[NQ4], rs0[NQ4], rs[NQ4], rp[NP4], rv[NQ4];
#pragma unroll
    for (int i = 0; i < NQ4; ++i) {
        rq[i] = *reinterpret_cast<const floatx4*>(Q + (tid + 256 * i) * 4);
        rs0[i] = *reinterpret_cast<const floatx4*>(Sc + (tid + 256 * i) * 4);
    }
#pragma unroll
    for (int i = 0; i < NQ4; ++i) rs[i] = *reinterpret_cast<const floatx4*>(Sc + kC * kD + (tid + 256 * i) * 4);
#pragma unroll
    for (int i = 0; i < NP4; ++i) rp[i] = *reinterpret_cast<const floatx4*>(P + (tid + 256 * i) * 4);
#pragma unroll
    for (int i = 0; i < NQ4; ++i) rv[i] = *reinterpret_cast<const floatx4*>(Vn + (tid + 256 * i) * 4);
    const float egv = a.Eg[static_cast<int64_t>(vh) * a.Tp + row0 + (tid & (kC - 1))];
#pragma unroll
    for (int i = 0; i < NQ4; ++i) {
        const int f = tid + 256 * i;
        *reinterpret_cast<floatx4*>(&A_s[f >> 5][(f & 31) * 4]) = rq[i];
        put_b(f, rs0[i]);
    }
    if (tid < kC) eg[tid] = egv;
    lds_barrier();  // LDS only: S_c[64:128), P and v_new stay in flight
    // the epilogue's gate z (this lane's 4 rows x 8 columns) and norm weight (8 columns),
    // requested now that the Q and S_c[0:64) registers are free (unconditional loads from a
    // valid address: a raw readout reads the S_c tile and ignores it)
    const bool gated = a.norm_w != nullptr;
    float zr[4][8], nw[8];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int64_t t = row0 + 16 * wave + 4 * lg + v;
        const int64_t tc = t < a.T ? t : a.T - 1;  // padding rows compute but store nothing
        const float* zrow = gated ? a.z + tc * a.ld_z + vh * kD : Sc;
#pragma unroll
        for (int b = 0; b < 8; ++b) zr[v][b] = zrow[16 * b + lr];
    }
    {
        const float* nwp = gated ? a.norm_w : Sc;
#pragma unroll
        for (int b = 0; b < 8; ++b) nw[b] = nwp[16 * b + lr];
    }
#pragma unroll
    for (int blk = 0; blk < kC / 16; ++blk) mma16(16 * blk, 16 * blk);
    lds_barrier();  // done with S_c[0:64)
#pragma unroll
    for (int i = 0; i < NQ4; ++i) put_b(tid + 256 * i, rs[i]);
    lds_barrier();
#pragma unroll
    for (int blk = 0; blk < kC / 16; ++blk) mma16(kC + 16 * blk, 16 * blk);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const float e = eg[16 * wave + 4 * lg + v];
#pragma unroll
        for (int b = 0; b < 8; ++b) acc[b][v] *= e;
    }
    lds_barrier();  // done with Q and S_c
#pragma unroll
    for (int i = 0; i < NP4; ++i) {
        const int f = tid + 256 * i;
        *reinterpret_cast<floatx4*>(&A_s[f >> 4][(f & 15) * 4]) = rp[i];
    }
#pragma unroll
    for (int i = 0; i < NQ4; ++i) put_b(tid + 256 * i, rv[i]);
    lds_barrier();
    // P is lower triangular: the row block of wave w needs columns j < 16 (w + 1)
    for (int blk = 0; blk <= wave; ++blk) mma16(16 * blk, 16 * blk);
    // epilogue: rows 16w + 4 lg + v, columns 16 b + lr
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int64_t t = row0 + 16 * wave + 4 * lg + v;
        double ss = 0.0;
#pragma unroll
        for (int b = 0; b < 8; ++b) ss += static_cast<double>(acc[b][v]) * acc[b][v];
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) ss += __shfl_xor(ss, o);  // the 16 lanes of the row
        const float inv = 1.0f / sqrtf(static_cast<float>(ss / kD) + a.eps);
        float* out = a.out + t * (a.VH * kD) + vh * kD;
        float mx = 0.0f;
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const int col = 16 * b + lr;
            const float y = gated ? nw[b] * (acc[b][v] * inv) * silu_f(zr[v][b]) : acc[b][v];
            mx = fmaxf(mx, fabsf(y));
            if (t < a.T) {
                if (a.out_tiled) a.out[xt_off(t, vh * kD + col, a.VH * kD)] = y;
                else out[col] = y;
            }
        }
        if (a.omax) {  // uniform: the row's maximum over this v-head's 128 columns (16 lanes)
            mx = fmaxf(mx, __shfl_xor(mx, 1));
            mx = fmaxf(mx, __shfl_xor(mx, 2));
            mx = fmaxf(mx, __shfl_xor(mx, 4));
            mx = fmaxf(mx, __shfl_xor(mx, 8));
            if (lr == 0 && t < a.T) a.omax[t * a.VH + vh] = mx;
        }
    }
}

// ------------------------------------------------------------------ GDN over few tokens
// sum over the 8 lanes l, l ^ 8, ..., l ^ 56 (the row groups of one column quad)
__device__ __forceinline__ float rowgroup8_sum(float v) {
    v += dpp_f<0x128>(v);
    auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(int, v), __builtin_bit_cast(int, v), false, false);
    v = __builtin_bit_cast(float, static_cast<int>(r[0])) + __builtin_bit_cast(float, static_cast<int>(r[1]));
    r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(int, v), __builtin_bit_cast(int, v), false, false);
    return __builtin_bit_cast(float, static_cast<int>(r[0])) + __builtin_bit_cast(float, static_cast<int>(r[1]));
}

constexpr int kShortT = 36;      // most tokens
constexpr int kShortRun = 4;     // tokens per conv run
constexpr int kShortThreads = 512;

// grid (VH), 512 threads: a whole block of up to kShortT tokens of one v-head in one launch,
// token by token like the decode step, the state in registers throughout.
//   conv   runs of 4 tokens x 4 channels of the head's q, k and v, SiLU, into LDS; beta and
//          the decay of each token
//   norm   each half-wave l2-normalises q or k rows in place (q also scaled by DK^-1/2)
//   scan   waves 0-3 own 32 state columns each: lane l rows 16 (l / 8) .. + 15 of columns
//          4 (l % 8) .. + 3 (as gdn_wave_kernel); the readout takes v's place in LDS
//   out    each half-wave one token: the gated rmsnorm (or the raw readout), row maximum
// The chunked kernels take the time of one chunk of 64 however few tokens there are, most of
// it serial latency (43 us).
__global__ __launch_bounds__(kShortThreads) void gdn_short_kernel(GdnPrefillArgs a) {
    const int vh = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int rep = a.VH / a.KH, kh = vh / rep;
    const int KD = a.KH * kD, CONV = 2 * KD + a.VH * kD;
    __shared__ __align__(16) float qs[kShortT * kD], ks[kShortT * kD], vs[kShortT * kD];  // vs: v, then the readout
    __shared__ float al[kShortT], be[kShortT];
    float* S = a.state + static_cast<int64_t>(vh) * kD * kD;

    // the state slice of the scan waves, requested first
    constexpr int RR = 16;
    const int rg = lane >> 3, col0 = 32 * wave + 4 * (lane & 7);
    float4 s[RR];
    if (wave < 4) {
#pragma unroll
        for (int i = 0; i < RR; ++i) s[i] = *reinterpret_cast<const float4*>(S + (RR * rg + i) * kD + col0);
    }
    // ---- conv
    const int runs = (a.T + kShortRun - 1) / kShortRun;
    for (int item = tid; item < 96 * runs; item += kShortThreads) {
        const int run = item / 96, quad = item - 96 * run;  // quads 0-31 q, 32-63 k, 64-95 v
        const int part = quad >> 5, c4 = 4 * (quad & 31), t0 = kShortRun * run;
        const int ch = (part == 0 ? kh * kD : part == 1 ? KD + kh * kD : 2 * KD + vh * kD) + c4;
        float4 x[kShortRun + 3], w[4];
#pragma unroll
        for (int j = 0; j < kShortRun + 3; ++j) {
            const int t = t0 - 3 + j;  // t < 0: the conv ring
            const float* p = t >= 0 ? a.qkv + static_cast<int64_t>(min(t, a.T - 1)) * a.ld_qkv + ch
                                    : a.conv_ring + static_cast<int64_t>((a.pos0 + t) & 3) * CONV + ch;
            x[j] = *reinterpret_cast<const float4*>(p);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = *reinterpret_cast<const float4*>(a.conv_w + static_cast<int64_t>(ch + e) * 4);
        float* dst = (part == 0 ? qs : part == 1 ? ks : vs) + t0 * kD + c4;
#pragma unroll
        for (int j = 0; j < kShortRun; ++j) {
            float y[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                auto at = [&](const float4& q) { return e == 0 ? q.x : e == 1 ? q.y : e == 2 ? q.z : q.w; };
                float acc = 0.0f;
                acc += w[e].x * at(x[j]);
                acc += w[e].y * at(x[j + 1]);
                acc += w[e].z * at(x[j + 2]);
                acc += w[e].w * at(x[j + 3]);
                y[e] = silu_f(acc);
            }
            if (t0 + j < a.T) *reinterpret_cast<float4*>(dst + j * kD) = make_float4(y[0], y[1], y[2], y[3]);
        }
    }
    if (tid < a.T) {
        const float g = -expf(a.A_log[vh]) * softplus_f(a.a[static_cast<int64_t>(tid) * a.ld_ba + vh] + a.dt_bias[vh]);
        al[tid] = expf(g);
        be[tid] = sigmoid_f(a.b[static_cast<int64_t>(tid) * a.ld_ba + vh]);
    }
    lds_barrier();
    // ---- l2norm (eps 1e-6, sums of squares in double)
    const int half = tid >> 5, l32 = tid & 31;  // 16 half-waves
    for (int r = half; r < 2 * a.T; r += kShortThreads / 32) {
        float* row = (r < a.T ? qs + r * kD : ks + (r - a.T) * kD) + 4 * l32;
        const float4 x = *reinterpret_cast<const float4*>(row);
        double ss = static_cast<double>(x.x) * x.x + static_cast<double>(x.y) * x.y + static_cast<double>(x.z) * x.z +
                    static_cast<double>(x.w) * x.w;
        ss = half_wave_sum(ss);
        const float inv = 1.0f / sqrtf(static_cast<float>(ss) + 1e-6f);
        const float qsc = r < a.T ? 1.0f / sqrtf(static_cast<float>(kD)) : 1.0f;
        *reinterpret_cast<float4*>(row) =
            make_float4((x.x * inv) * qsc, (x.y * inv) * qsc, (x.z * inv) * qsc, (x.w * inv) * qsc);
    }
    // the block's last three raw inputs into the ring (one v-head per k-head: nobody else
    // reads these channels; else gdn_ring_kernel writes it)
    if (rep == 1 && tid < 3 * 96) {
        const int quad = tid % 96, part = quad >> 5, t = a.T - 1 - tid / 96;
        const int ch = (part == 0 ? kh * kD : part == 1 ? KD + kh * kD : 2 * KD + vh * kD) + 4 * (quad & 31);
        if (t >= 0)
            *reinterpret_cast<float4*>(a.conv_ring + static_cast<int64_t>((a.pos0 + t) & 3) * CONV + ch) =
                *reinterpret_cast<const float4*>(a.qkv + static_cast<int64_t>(t) * a.ld_qkv + ch);
    }
    lds_barrier();
    // ---- scan
    if (wave < 4) {
        float4 q4[RR / 4], k4[RR / 4], v4;
        auto read = [&](int t) {
#pragma unroll
            for (int j = 0; j < RR / 4; ++j) {
                q4[j] = *reinterpret_cast<const float4*>(qs + t * kD + RR * rg + 4 * j);
                k4[j] = *reinterpret_cast<const float4*>(ks + t * kD + RR * rg + 4 * j);
            }
            v4 = *reinterpret_cast<const float4*>(vs + t * kD + col0);
        };
        read(0);
#pragma unroll 1
        for (int t = 0; t < a.T; ++t) {
            const float alpha = al[t], beta = be[t];
            float qn[RR], kn[RR];
#pragma unroll
            for (int j = 0; j < RR / 4; ++j) {
                qn[4 * j] = q4[j].x, qn[4 * j + 1] = q4[j].y, qn[4 * j + 2] = q4[j].z, qn[4 * j + 3] = q4[j].w;
                kn[4 * j] = k4[j].x, kn[4 * j + 1] = k4[j].y, kn[4 * j + 2] = k4[j].z, kn[4 * j + 3] = k4[j].w;
            }
            const float4 v = v4;
            if (t + 1 < a.T) read(t + 1);  // uniform: the next token's rows while this one's are used
            float4 km = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int i = 0; i < RR; ++i) {
                s[i].x *= alpha;
                s[i].y *= alpha;
                s[i].z *= alpha;
                s[i].w *= alpha;
                km.x += s[i].x * kn[i];
                km.y += s[i].y * kn[i];
                km.z += s[i].z * kn[i];
                km.w += s[i].w * kn[i];
            }
            km.x = rowgroup8_sum(km.x);
            km.y = rowgroup8_sum(km.y);
            km.z = rowgroup8_sum(km.z);
            km.w = rowgroup8_sum(km.w);
            const float4 d = make_float4((v.x - km.x) * beta, (v.y - km.y) * beta, (v.z - km.z) * beta, (v.w - km.w) * beta);
            float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int i = 0; i < RR; ++i) {
                s[i].x += kn[i] * d.x;
                s[i].y += kn[i] * d.y;
                s[i].z += kn[i] * d.z;
                s[i].w += kn[i] * d.w;
                o.x += s[i].x * qn[i];
                o.y += s[i].y * qn[i];
                o.z += s[i].z * qn[i];
                o.w += s[i].w * qn[i];
            }
            o.x = rowgroup8_sum(o.x);
            o.y = rowgroup8_sum(o.y);
            o.z = rowgroup8_sum(o.z);
            o.w = rowgroup8_sum(o.w);
            if (rg == 0) *reinterpret_cast<float4*>(vs + t * kD + col0) = o;
        }
#pragma unroll
        for (int i = 0; i < RR; ++i) *reinterpret_cast<float4*>(S + (RR * rg + i) * kD + col0) = s[i];
    }
    lds_barrier();
    // ---- out: half-wave h takes tokens h, h + 16, ..; lane l columns l, l + 32, l + 64, l + 96
    for (int t = half; t < a.T; t += kShortThreads / 32) {
        float o[4], z[4] = {0.f, 0.f, 0.f, 0.f}, nw[4] = {1.f, 1.f, 1.f, 1.f};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            o[e] = vs[t * kD + l32 + 32 * e];
            if (a.norm_w) {  // uniform
                z[e] = a.z[static_cast<int64_t>(t) * a.ld_z + vh * kD + l32 + 32 * e];
                nw[e] = a.norm_w[l32 + 32 * e];
            }
        }
        double ss = 0.0;
#pragma unroll
        for (int e = 0; e < 4; ++e) ss += static_cast<double>(o[e]) * o[e];
        ss = half_wave_sum(ss);
        const float inv = 1.0f / sqrtf(static_cast<float>(ss / kD) + a.eps);
        float mx = 0.0f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int c = vh * kD + l32 + 32 * e;
            const float y = a.norm_w ? nw[e] * (o[e] * inv) * silu_f(z[e]) : o[e];
            mx = fmaxf(mx, fabsf(y));
            a.out[a.out_tiled ? xt_off(t, c, a.VH * kD) : static_cast<int64_t>(t) * (a.VH * kD) + c] = y;
        }
        if (a.omax) {  // uniform
            mx = fmaxf(mx, dpp_f<0xB1>(mx));
            mx = fmaxf(mx, dpp_f<0x4E>(mx));
            mx = fmaxf(mx, dpp_f<0x141>(mx));
            mx = fmaxf(mx, dpp_f<0x140>(mx));
            mx = fmaxf(mx, swz16_f(mx));
            if (l32 == 0) a.omax[static_cast<int64_t>(t) * a.VH + vh] = mx;
        }
    }
}

// ------------------------------------------------------------------ attention prep
// Any even rotary width: grid (T, NQ + NKV), one thread per dim.
__global__ __launch_bounds__(256) void attn_prefill_prep_any_kernel(AttnPrefillArgs a) {
    const int t = blockIdx.x, r = blockIdx.y, d = threadIdx.x;
    const int pos = a.pos0 + t;
    __shared__ float buf[kHD];
    __shared__ float cs[2][kHD / 2];
    __shared__ double red[4];
    const float* row = a.qkv + static_cast<int64_t>(t) * a.ld_qkv;
    const float* src;
    const float* w;
    const bool is_q = r < a.NQ;
    const int kh = r - a.NQ;
    const int64_t coff = (static_cast<int64_t>(kh) * a.max_ctx + pos) * kHD;  // cache row (keys)
    if (is_q) {
        src = row + static_cast<int64_t>(r) * 2 * kHD;
        w = a.q_norm;
    } else {
        src = row + static_cast<int64_t>(a.NQ) * 2 * kHD + kh * kHD;
        w = a.k_norm;
        const float v = row[static_cast<int64_t>(a.NQ) * 2 * kHD + static_cast<int64_t>(a.NKV) * kHD + kh * kHD + d];
        if (a.kv_bf16) reinterpret_cast<uint16_t*>(a.v_cache)[coff + d] = f32_to_bf16(v);
        else a.v_cache[coff + d] = v;
    }
    const int half = a.ROT / 2;
    if (d < half) {
        const double inv_freq = pow(a.theta, -static_cast<double>(2 * d) / a.ROT);
        const double ang = static_cast<double>(pos) * inv_freq;
        cs[0][d] = static_cast<float>(cos(ang));
        cs[1][d] = static_cast<float>(sin(ang));
    }
    const float x = src[d];
    const double ss = block_sum(static_cast<double>(x) * x, red);
    const float inv = 1.0f / sqrtf(static_cast<float>(ss / kHD) + a.eps);
    float y = x * inv * (1.0f + w[d]);
    buf[d] = y;
    __syncthreads();
    if (d < a.ROT) {
        const int i = d < half ? d : d - half;
        const float c = cs[0][i], s = cs[1][i];
        const float x1 = buf[i], x2 = buf[i + half];
        y = d < half ? x1 * c - x2 * s : x2 * c + x1 * s;
    }
    if (is_q) a.Qa[(static_cast<int64_t>(r) * a.T + t) * kHD + d] = y;
    else if (a.kv_bf16) reinterpret_cast<uint16_t*>(a.k_cache)[coff + d] = f32_to_bf16(y);
    else a.k_cache[coff + d] = y;
}

// One workgroup per token, all of its rows: the NQ query rows (rmsnorm (1 + q_norm) + RoPE
// -> Qa), the NKV key rows (k_norm + RoPE -> cache) and the NKV value rows (-> cache). A row
// is 4 dims per lane of one wave (sum of squares in double); the RoPE partner dims d +- ROT/2
// come from lane +- ROT/8; cos / sin from the table or from the double-precision angle.
__global__ __launch_bounds__(256) void attn_prefill_prep_kernel(AttnPrefillArgs a) {
    const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int pos = a.pos0 + t;
    const int half = a.ROT / 2, hq = a.ROT / 8;
    const float* row = a.qkv + static_cast<int64_t>(t) * a.ld_qkv;
    // cos / sin of the 4 dims of this lane (dims d mod half, lanes < ROT / 4)
    float4 cs4 = make_float4(1.f, 1.f, 1.f, 1.f), sn4 = make_float4(0.f, 0.f, 0.f, 0.f);
    const int ci = (lane * 4) % max(half, 4);
    if (a.rope_cs) {
        const float* tb = a.rope_cs + static_cast<int64_t>(pos) * a.ROT;
        const int c0 = min(ci, max(half - 4, 0));
        cs4 = *reinterpret_cast<const float4*>(tb + c0);
        sn4 = *reinterpret_cast<const float4*>(tb + half + c0);
    } else {
        rope_cs4(a.theta, a.ROT, pos, lane, cs4, sn4);  // double-precision angles
    }
    const int nrow = a.NQ + 2 * a.NKV;
    for (int r = wave; r < nrow; r += 4) {  // uniform per wave
        if (r >= a.NQ + a.NKV) {  // value row: copied to the cache
            const int kh = r - a.NQ - a.NKV;
            const float4 v = *reinterpret_cast<const float4*>(row + static_cast<int64_t>(a.NQ) * 2 * kHD +
                                                              static_cast<int64_t>(a.NKV + kh) * kHD + lane * 4);
            const int64_t off = (static_cast<int64_t>(kh) * a.max_ctx + pos) * kHD + lane * 4;
            if (a.kv_bf16) {
                *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(a.v_cache) + off) =
                    make_uint2(f32_to_bf16(v.x) | (static_cast<uint32_t>(f32_to_bf16(v.y)) << 16),
                               f32_to_bf16(v.z) | (static_cast<uint32_t>(f32_to_bf16(v.w)) << 16));
            } else {
                *reinterpret_cast<float4*>(a.v_cache + off) = v;
            }
            continue;
        }
        const bool is_q = r < a.NQ;
        const int kh = r - a.NQ;
        const float* src = is_q ? row + static_cast<int64_t>(r) * 2 * kHD
                                : row + static_cast<int64_t>(a.NQ) * 2 * kHD + static_cast<int64_t>(kh) * kHD;
        const float4 x = *reinterpret_cast<const float4*>(src + lane * 4);
        const float4 w = *reinterpret_cast<const float4*>((is_q ? a.q_norm : a.k_norm) + lane * 4);
        double ss = static_cast<double>(x.x) * x.x + static_cast<double>(x.y) * x.y + static_cast<double>(x.z) * x.z +
                    static_cast<double>(x.w) * x.w;
        ss = wave_sum(ss);
        const float inv = 1.0f / sqrtf(static_cast<float>(ss / kHD) + a.eps);
        float4 y;
        y.x = x.x * inv * (1.0f + w.x);
        y.y = x.y * inv * (1.0f + w.y);
        y.z = x.z * inv * (1.0f + w.z);
        y.w = x.w * inv * (1.0f + w.w);
        const int srcl = lane < hq ? lane + hq : lane - hq;
        float4 o;
        o.x = __shfl(y.x, srcl);
        o.y = __shfl(y.y, srcl);
        o.z = __shfl(y.z, srcl);
        o.w = __shfl(y.w, srcl);
        if (lane < hq) {
            y.x = y.x * cs4.x - o.x * sn4.x;
            y.y = y.y * cs4.y - o.y * sn4.y;
            y.z = y.z * cs4.z - o.z * sn4.z;
            y.w = y.w * cs4.w - o.w * sn4.w;
        } else if (lane < 2 * hq) {
            y.x = y.x * cs4.x + o.x * sn4.x;
            y.y = y.y * cs4.y + o.y * sn4.y;
            y.z = y.z * cs4.z + o.z * sn4.z;
            y.w = y.w * cs4.w + o.w * sn4.w;
        }
        if (is_q) {
            *reinterpret_cast<float4*>(a.Qa + (static_cast<int64_t>(r) * a.T + t) * kHD + lane * 4) = y;
        } else {
            const int64_t off = (static_cast<int64_t>(kh) * a.max_ctx + pos) * kHD + lane * 4;
            if (a.kv_bf16) {
                *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(a.k_cache) + off) =
                    make_uint2(f32_to_bf16(y.x) | (static_cast<uint32_t>(f32_to_bf16(y.y)) << 16),
                               f32_to_bf16(y.z) | (static_cast<uint32_t>(f32_to_bf16(y.w)) << 16));
            } else {
                *reinterpret_cast<float4*>(a.k_cache + off) = y;
            }
        }
    }
}

// ------------------------------------------------------------------ flash attention
constexpr float kLog2e = 1.44269504088896341f;

// 128 query rows per workgroup (16 per wave), causal, keys of earlier blocks from the cache,
// 32-key tiles staged through LDS (the next tile's rows are loaded into registers while the
// current one is multiplied), online softmax. One workgroup per CU (96 KB of LDS with three
// parts; a bf16 cache's 4-wave workgroups hold 32 KB, two per CU). A row is a (token, query head of the kv head's group) pair, row = token * group +
// head: the heads of a group read the same keys, so 32 tokens of a group of 4 are one full
// block and not four quarter ones, and a block's rows end within 128 / group tokens of each
// other. Causal work grows with the block, and workgroups are dispatched in linear order, so
// rank L takes the L-th longest block of all kv heads.
//
// Few blocks over many keys (a chat turn: 300 tokens of 2 x 4 heads are 20 blocks, 38 of a bf16
// cache's 64 rows) would leave most compute units idle, so a block's tiles are then cut into
// pieces of `piece` tiles, one workgroup each (flash_plan), whose unnormalised outputs, maxima
// and sums flash_combine_kernel merges. That turn at 7000 cached bf16 positions: 703 us as 24
// blocks of 128 tokens of single heads, 81 as 494 pieces (traced one by one: query rows 6, flash
// 75, merge of 32 MB of partial outputs 12). Bound as the unsplit kernel: products behind LDS
// reads and two barriers a tile.
// Both products run on the bf16 matrix cores (v_mfma_f32_16x16x32_bf16): every fp32 operand
// is the exact sum of three bf16 parts (hi + mid + lo, as in the bf16 path of the projection GEMM), and a
// product a.b is the sum of the six part products a_i b_j with i + j <= 2 (parts counted
// from 0): the three dropped ones (mid.lo, lo.mid, lo.lo) are below 2^-23 |a||b| together,
// the size of an fp32 rounding, and each bf16 x bf16 part product is exact in fp32. A bf16
// cache holds K and V exactly, so only Q and P are split (three products each).
//   S^T = K Q^T per 16-key half of the tile: keys as rows (K parts from LDS, 8 consecutive
//         dims per lane), the lane's own query row as the column (Q parts in registers, split
//         once); lane (r16, g) ends with keys 4g + v of each half for query r16.
//   O += P V, 32 keys deep: those eight scores are the A operand (query r16) without data
//         movement, taking the k slots 8g .. 8g + 7 of the product as keys 4g .. 4g + 3 of the
//         first half and of the second; the dim-major V rows in LDS store the keys in that
//         order (one 16-byte read per lane and dim block); lane (r16, g) ends with dims
//         16t + r16 of queries 4g + v. (16-key tiles would need the 16-deep bf16 product,
//         which the gfx950 matrix cores run at half the 32-deep one's rate.)
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// the three bf16 parts of four floats, each part as four packed bf16 (element 0 low)
__device__ __forceinline__ void split3_4(const float (&x)[4], uint2 (&part)[3]) {
    uint32_t h[4], m[4], l[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) split3(x[e], h[e], m[e], l[e]);
    part[0] = make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
    part[1] = make_uint2(m[0] | (m[1] << 16), m[2] | (m[3] << 16));
    part[2] = make_uint2(l[0] | (l[1] << 16), l[2] | (l[3] << 16));
}

// eight floats as three 16-byte chunks, the exact bf16 parts of each (elements 0..7 in order)
__device__ __forceinline__ void split3_8(const float (&x)[8], uint4 (&c)[3]) {
    const float lo[4] = {x[0], x[1], x[2], x[3]}, hi[4] = {x[4], x[5], x[6], x[7]};
    uint2 p0[3], p1[3];
    split3_4(lo, p0);
    split3_4(hi, p1);
#pragma unroll
    for (int p = 0; p < 3; ++p) c[p] = make_uint4(p0[p].x, p0[p].y, p1[p].x, p1[p].y);
}

// The flash kernel's LDS image of one 32-key tile of an fp32 cache: K chunks Kc[3][2][32][16]
// then V chunks Vc[3][16][4][16] (the layouts described at that kernel), 16-byte chunks.
static_assert(kImgK == 3 * 2 * (kHD / 8) * 16, "K chunks of a tile");
// key of slot 8 g + j of a V chunk: keys 4 g .. + 3 of the tile's first half, then the same
// four of its second half
__device__ __forceinline__ int vslot_key(int g, int j) { return (j < 4 ? 0 : 12) + 4 * g + j; }

// grid (tiles, NKV), 256 threads: writes the LDS image of every tile of keys [0, pos0 + T) of
// one kv head (rows past the last key are copies of it), so that the flash kernel stages a
// tile by a plain copy instead of splitting it again in every query-block workgroup.
__global__ __launch_bounds__(256) void attn_kv_image_kernel(AttnPrefillArgs a) {
    const int ti = blockIdx.x, kh = blockIdx.y, tid = threadIdx.x;
    const int last = a.pos0 + a.T - 1;
    const int64_t hoff = static_cast<int64_t>(kh) * a.max_ctx * kHD;
    uint4* img = static_cast<uint4*>(a.kv_img) + (static_cast<int64_t>(kh) * gridDim.x + ti) * kImgTile;
    // K chunk (key, dims 8 dc ..): lanes walk the dim chunks of one key
    for (int e = tid; e < kKT * (kHD / 8); e += 256) {
        const int key = e >> 5, dc = e & 31;
        const float* src = a.k_cache + hoff + static_cast<int64_t>(min(ti * kKT + key, last)) * kHD + 8 * dc;
        const float4 u = *reinterpret_cast<const float4*>(src), w = *reinterpret_cast<const float4*>(src + 4);
        const float x[8] = {u.x, u.y, u.z, u.w, w.x, w.y, w.z, w.w};
        uint4 c[3];
        split3_8(x, c);
#pragma unroll
        for (int p = 0; p < 3; ++p) img[((p * 2 + (key >> 4)) * (kHD / 8) + dc) * 16 + (key & 15)] = c[p];
    }
    // V chunk (dim d, slot chunk g): lanes walk the dims of the same eight keys
    for (int e = tid; e < kHD * 4; e += 256) {
        const int d = e & (kHD - 1), g = e >> 8;
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
            x[j] = a.v_cache[hoff + static_cast<int64_t>(min(ti * kKT + vslot_key(g, j), last)) * kHD + d];
        uint4 c[3];
        split3_8(x, c);
#pragma unroll
        for (int p = 0; p < 3; ++p) img[kImgK + ((p * (kHD / 16) + (d >> 4)) * 4 + g) * 16 + ((d & 15) ^ (4 * g))] = c[p];
    }
}

// Online softmax of one 32-key tile for the lane's query: the scores S^T[key 16 hf + 4 g4 + v]
// become weights p[4 hf + v], (m, l) the row's running maximum and sum. Returns the factor of
// the output so far. The reference max moves only when a score exceeds it by more than 8; a
// row with no key yet keeps -inf and weight 0. e^y as the native 2^(y log2 e): y = score -
// max is formed exactly, so the product's rounding moves a weight by |y| 2^-24 relative (1 ulp
// of v_exp_f32 besides), negligible where the weights are large.
__device__ __forceinline__ float flash_softmax(const floatx4 (&St)[2], int kv0, int qpos, int kv_end, float sc, int g4,
                                               float& m, float& l, float (&p)[8]) {
    float sv[8];
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int key = kv0 + 16 * hf + 4 * g4 + v;
            sv[4 * hf + v] = key <= qpos && key < kv_end ? St[hf][v] * sc : -INFINITY;
        }
    float tm = sv[0];
#pragma unroll
    for (int i = 1; i < 8; ++i) tm = fmaxf(tm, sv[i]);
    tm = fmaxf(tm, __shfl_xor(tm, 16));
    tm = fmaxf(tm, __shfl_xor(tm, 32));
    const float m_new = tm > m + 8.0f ? tm : m;
    const bool live = m_new != -INFINITY;
    const float f = live ? __builtin_amdgcn_exp2f((m - m_new) * kLog2e) : 1.0f;
    float ps = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        p[i] = live ? __builtin_amdgcn_exp2f((sv[i] - m_new) * kLog2e) : 0.0f;
        ps += p[i];
    }
    ps += __shfl_xor(ps, 16);
    ps += __shfl_xor(ps, 32);
    l = l * f + ps;
    m = m_new;
    return f;
}
// output rows 4 g4 + r of the wave times the factors f of lanes 4 g4 + r
__device__ __forceinline__ void flash_rescale(float f, int g4, floatx4 (&o)[16]) {
    if (!__any(f != 1.0f)) return;
    float fr[4];
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) fr[rr] = __shfl(f, 4 * g4 + rr);
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        o[t][0] *= fr[0];
        o[t][1] *= fr[1];
        o[t][2] *= fr[2];
        o[t][3] *= fr[3];
    }
}

// Epilogue of 16 rows of a block from `rbase`: o / (row sum) times the gate.
__device__ __forceinline__ void flash_store(const AttnPrefillArgs& a, const floatx4 (&o)[16], const float (&lr)[4], int kh,
                                            int grp, int rows, int rbase, int lane) {
    const int r16 = lane & 15, g4 = lane >> 4;
    // every gate value requested before the first store: the output may alias them as far as
    // the compiler knows, and a load after a store would wait for its own round trip, 64 in a
    // row (35 us a workgroup; 4096 tokens 762 -> 722 us)
    float gt[4][16];
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
        const int rc = min(rbase + 4 * g4 + rr, rows - 1);  // rows past the block store nothing
        const float* gate = a.qkv + static_cast<int64_t>(rc / grp) * a.ld_qkv +
                            static_cast<int64_t>(kh * grp + rc % grp) * 2 * kHD + kHD;
#pragma unroll
        for (int tt = 0; tt < 16; ++tt) gt[rr][tt] = gate[16 * tt + r16];
    }
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
        const int row = rbase + 4 * g4 + rr;
        const int rc = min(row, rows - 1);
        const int t = rc / grp, h = kh * grp + rc % grp;
        const float inv = 1.0f / lr[rr];
        float* out = a.out + static_cast<int64_t>(t) * (a.NQ * kHD) + static_cast<int64_t>(h) * kHD;
        float mx = 0.0f;
#pragma unroll
        for (int tt = 0; tt < 16; ++tt) {
            const int dd = 16 * tt + r16;
            const float y = (o[tt][rr] * inv) * sigmoid_f(gt[rr][tt]);
            mx = fmaxf(mx, fabsf(y));
            if (row < rows) {
                if (a.out_tiled) a.out[xt_off(t, h * kHD + dd, a.NQ * kHD)] = y;
                else out[dd] = y;
            }
        }
        if (a.omax) {  // uniform: the row's maximum over this head's 256 dims (16 lanes)
            mx = fmaxf(mx, __shfl_xor(mx, 1));
            mx = fmaxf(mx, __shfl_xor(mx, 2));
            mx = fmaxf(mx, __shfl_xor(mx, 4));
            mx = fmaxf(mx, __shfl_xor(mx, 8));
            if (r16 == 0 && row < rows) a.omax[static_cast<int64_t>(t) * a.NQ + h] = mx;
        }
    }
}

// SPLIT: grid (pieces, blocks of all kv heads), else grid (blocks).
template <bool KVB, bool SPLIT>
__global__ __launch_bounds__(flash_waves(KVB) * 64, KVB ? 8 / flash_waves(KVB) : 1) void flash_attn_kernel(AttnPrefillArgs a) {
    constexpr int kFW = flash_waves(KVB), kQT = 16 * kFW;
    constexpr int SS = 8 / kFW;  // staging passes (one thread's share of a tile by 512 threads each)
    constexpr int NP = KVB ? 1 : 3;  // parts of K and V
    const int grp = a.NQ / a.NKV, rows = a.T * grp, nblk = (rows + kQT - 1) / kQT;
    const int rank = SPLIT ? blockIdx.y : blockIdx.x;
    const int qt = nblk - 1 - rank / a.NKV, kh = rank % a.NKV;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int row0 = qt * kQT;
    // keys of the block, and this workgroup's piece of them
    const int kv_end = a.pos0 + min(rows - 1, row0 + kQT - 1) / grp + 1;
    const int piece_keys = a.plan.piece * kKT;
    const int kv_lo = SPLIT ? static_cast<int>(blockIdx.x) * piece_keys : 0;
    if (SPLIT && kv_lo >= kv_end) return;  // uniform: the block has fewer pieces
    const int kv_hi = SPLIT ? min(kv_end, kv_lo + piece_keys) : kv_end;
    const bool whole = !SPLIT || kv_end <= piece_keys;  // the block's only piece: final output
    const int r16 = lane & 15, g4 = lane >> 4;
    // LDS in 16-byte chunks (8 bf16) so that the 16 lanes of a lane group read one whole
    // 256-byte row of 16 chunks (any order within the row runs at full rate; rows of padded
    // or scattered chunks at 0.6 of it): K chunk (key, dims 8 dc ..) at Kc[p][key / 16][dc]
    // [key % 16], V chunk (dim, key slots 8 g ..) at Vc[p][dim / 16][g][(dim % 16) ^ 4 g]
    // (the XOR puts the 8 lanes of each staging store on distinct banks).
    __shared__ __align__(16) uint4 Kc[NP][2][kHD / 8][16];
    __shared__ __align__(16) uint4 Vc[NP][kHD / 16][4][16];
    const float sc = 1.0f / sqrtf(static_cast<float>(kHD));

    // this lane's query row, dims 32c + 8 g4 .. + 7, as three bf16 parts (the B operand)
    const int qrow = min(row0 + wave * 16 + r16, rows - 1);
    bf16x8 qp[3][8];
    {
        const float* src = a.Qa + (static_cast<int64_t>(kh * grp + qrow % grp) * a.T + qrow / grp) * kHD + 8 * g4;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const float4 x0 = *reinterpret_cast<const float4*>(src + 32 * c);
            const float4 x1 = *reinterpret_cast<const float4*>(src + 32 * c + 4);
            const float v0[4] = {x0.x, x0.y, x0.z, x0.w}, v1[4] = {x1.x, x1.y, x1.z, x1.w};
            uint2 p0[3], p1[3];
            split3_4(v0, p0);
            split3_4(v1, p1);
#pragma unroll
            for (int p = 0; p < 3; ++p)
                qp[p][c] = __builtin_bit_cast(bf16x8, make_uint4(p0[p].x, p0[p].y, p1[p].x, p1[p].y));
        }
    }
    const int qpos = a.pos0 + qrow / grp;
    // the wave's last query position: tiles starting past it hold no key its rows attend
    const int wlast = a.pos0 + min(row0 + wave * 16 + 15, rows - 1) / grp;
    floatx4 o[16];  // dims 16 t + r16 of query rows 4 g4 + v
#pragma unroll
    for (int t = 0; t < 16; ++t) o[t] = floatx4{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.0f;

    const int64_t hoff = static_cast<int64_t>(kh) * a.max_ctx * kHD;
    // staging of one tile, in registers while the previous tile is multiplied: K key
    // 8 (wave % 4) + lane % 8, dim chunks 8 c + lane / 8 for c = 2 (wave / 4) + i, i < 2 (two
    // float4 each); V dims 2 (tid / 4), + 1 of the eight keys of slot chunk g = tid % 4 (keys
    // 4 g .. + 3 and 16 + 4 g .. + 3, one float2 each); split (or widened) when stored to LDS
    const int ks_row = 8 * (wave & 3) + (lane & 7), ks_c0 = 16 * (wave >> 2) + (lane >> 3);
    const int vs_g = tid & 3, vs_d = (tid >> 2) * 2;
    float4 kst[KVB ? 1 : 4];
    float2 vst[KVB ? 1 : 8];
    // (vector-typed: an array of uint4 structs here was placed in scratch memory)
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    // bf16 cache: the stored bits are the operands, K chunks as they lie, V pairs of dims
    // (8-byte aligned, as the cache rows' other accesses)
    typedef uint32_t u32x4_a8 __attribute__((ext_vector_type(4), aligned(8)));
    u32x4 kbs[KVB ? 2 * SS : 1];
    uint32_t vbs[KVB ? 8 * SS : 1];
    auto vkey = [&](int j) { return vslot_key(vs_g, j); };
    auto load_tile = [&](int kv0) {
        const bool live = kv0 < kv_end;
        if constexpr (KVB) {
            const uint16_t *kc = reinterpret_cast<const uint16_t*>(a.k_cache) + hoff,
                           *vc = reinterpret_cast<const uint16_t*>(a.v_cache) + hoff;
            const int64_t ok = live ? static_cast<int64_t>(min(kv0 + ks_row, kv_end - 1)) * kHD : 0;
#pragma unroll
            for (int j = 0; j < 2 * SS; ++j) kbs[j] = *reinterpret_cast<const u32x4_a8*>(kc + ok + 8 * (ks_c0 + 8 * j));
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int64_t ov = live ? static_cast<int64_t>(min(kv0 + vkey(j), kv_end - 1)) * kHD + vs_d : 0;
#pragma unroll
                for (int e = 0; e < SS; ++e) vbs[8 * e + j] = *reinterpret_cast<const uint32_t*>(vc + ov + e * (kHD / SS));
            }
            return;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int pk = min(kv0 + ks_row, kv_end - 1);
            const int64_t ok = live ? static_cast<int64_t>(pk) * kHD + 8 * (ks_c0 + 8 * (j >> 1)) + 4 * (j & 1) : 0;
            kst[j] = *reinterpret_cast<const float4*>(a.k_cache + hoff + ok);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int pv = min(kv0 + vkey(j), kv_end - 1);
            const int64_t ov = live ? static_cast<int64_t>(pv) * kHD + vs_d : 0;
            vst[j] = *reinterpret_cast<const float2*>(a.v_cache + hoff + ov);
        }
    };
    // Rows past the end of the keys are copies of the last one (finite): their scores are
    // masked to -inf, so their weights are exactly 0 and 0 * V adds nothing.
    auto store_tile = [&]() {
        if constexpr (KVB) {
#pragma unroll
            for (int j = 0; j < 2 * SS; ++j)
                Kc[0][ks_row >> 4][ks_c0 + 8 * j][ks_row & 15] = __builtin_bit_cast(uint4, kbs[j]);
#pragma unroll
            for (int e = 0; e < SS; ++e) {
                const int d = vs_d + e * (kHD / SS);
                uint4 lo, hi;  // dims d and d + 1 of the eight keys
                uint32_t* pl = &lo.x;
                uint32_t* ph = &hi.x;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t x = vbs[8 * e + 2 * j], y = vbs[8 * e + 2 * j + 1];
                    pl[j] = (x & 0xffffu) | (y << 16);
                    ph[j] = (x >> 16) | (y & 0xffff0000u);
                }
                Vc[0][d >> 4][vs_g][(d & 15) ^ (4 * vs_g)] = lo;
                Vc[0][d >> 4][vs_g][((d + 1) & 15) ^ (4 * vs_g)] = hi;
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const float4 u = kst[2 * i], w = kst[2 * i + 1];
            const float x[8] = {u.x, u.y, u.z, u.w, w.x, w.y, w.z, w.w};
            uint4 c[3];
            split3_8(x, c);
#pragma unroll
            for (int p = 0; p < NP; ++p) Kc[p][ks_row >> 4][ks_c0 + 8 * i][ks_row & 15] = c[p];
        }
        // V, dim-major: dims vs_d, vs_d + 1 get the eight keys of slot chunk vs_g
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            float x[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j] = e ? vst[j].y : vst[j].x;
            uint4 c[3];
            split3_8(x, c);
            const int d = vs_d + e;
#pragma unroll
            for (int p = 0; p < NP; ++p) Vc[p][d >> 4][vs_g][(d & 15) ^ (4 * vs_g)] = c[p];
        }
    };
    load_tile(kv_lo);
    store_tile();
    lds_barrier();
    for (int kv0 = kv_lo; kv0 < kv_hi; kv0 += kKT) {
        load_tile(kv0 + kKT);  // in flight during this tile's products
        if (kv0 <= wlast) {    // uniform per wave
            // S^T[key 16 hf + 4 g4 + v][query r16]: the hi.hi products and the smaller part
            // products in separate accumulators, each split over even / odd dim blocks
            floatx4 St[2];
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {
                floatx4 sa[2], sb[2];
#pragma unroll
                for (int e = 0; e < 2; ++e) sa[e] = sb[e] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int c = 0; c < 8; ++c) {
                    bf16x8 kop[NP];
#pragma unroll
                    for (int p = 0; p < NP; ++p)
                        kop[p] = __builtin_bit_cast(bf16x8, Kc[p][hf][4 * c + g4][r16]);
                    floatx4& b = sb[c & 1];
                    if constexpr (KVB) {
                        b = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kop[0], qp[2][c], b, 0, 0, 0);
                        b = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kop[0], qp[1][c], b, 0, 0, 0);
                    } else {
                        b = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kop[2 % NP], qp[0][c], b, 0, 0, 0);
                        b = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kop[1 % NP], qp[1][c], b, 0, 0, 0);
                        b = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kop[0], qp[2][c], b, 0, 0, 0);
                        b = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kop[1 % NP], qp[0][c], b, 0, 0, 0);
                        b = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kop[0], qp[1][c], b, 0, 0, 0);
                    }
                    sa[c & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kop[0], qp[0][c], sa[c & 1], 0, 0, 0);
                }
                St[hf] = (sb[0] + sb[1]) + (sa[0] + sa[1]);
            }
            float p[8];
            const float f = flash_softmax(St, kv0, qpos, kv_end, sc, g4, m_run, l_run, p);
            flash_rescale(f, g4, o);
            // O[query 4 g4 + v][dim 16 t + r16] += P[query][keys] V[keys][dim], k slots
            // 8 g4 .. + 7 = keys 4 g4 .. + 3 of both halves
            bf16x8 pa[3];
            {
                const float p0[4] = {p[0], p[1], p[2], p[3]}, p1[4] = {p[4], p[5], p[6], p[7]};
                uint2 q0[3], q1[3];
                split3_4(p0, q0);
                split3_4(p1, q1);
#pragma unroll
                for (int q = 0; q < 3; ++q) pa[q] = __builtin_bit_cast(bf16x8, make_uint4(q0[q].x, q0[q].y, q1[q].x, q1[q].y));
            }
#pragma unroll
            for (int t = 0; t < 16; ++t) {
                bf16x8 vb[NP];
#pragma unroll
                for (int q = 0; q < NP; ++q) vb[q] = __builtin_bit_cast(bf16x8, Vc[q][t][g4][r16 ^ (4 * g4)]);
                // the part products straight into the running output, smallest first
                if constexpr (KVB) {
                    o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa[2], vb[0], o[t], 0, 0, 0);
                    o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa[1], vb[0], o[t], 0, 0, 0);
                } else {
                    o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa[2], vb[0], o[t], 0, 0, 0);
                    o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa[1], vb[1 % NP], o[t], 0, 0, 0);
                    o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa[0], vb[2 % NP], o[t], 0, 0, 0);
                    o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa[1], vb[0], o[t], 0, 0, 0);
                    o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa[0], vb[1 % NP], o[t], 0, 0, 0);
                }
                o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa[0], vb[0], o[t], 0, 0, 0);
            }
        }
        lds_barrier();  // every wave is done with this tile
        if (kv0 + kKT < kv_hi) {
            store_tile();
            lds_barrier();
        }
    }
    if (!whole) {  // uniform: the piece's output and (max, sum) as they stand, lane by lane
        const int64_t slot = static_cast<int64_t>(blockIdx.y) * gridDim.x + blockIdx.x;
        floatx4* po = reinterpret_cast<floatx4*>(a.part) + (slot * kFW + wave) * 16 * 64 + lane;
#pragma unroll
        for (int t = 0; t < 16; ++t) po[64 * t] = o[t];
        if (g4 == 0) a.part_ml[slot * kQT + wave * 16 + r16] = make_float2(m_run, l_run);
        return;
    }
    float lr[4];
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) lr[rr] = __shfl(l_run, 4 * g4 + rr);
    flash_store(a, o, lr, kh, grp, rows, row0 + wave * 16, lane);
}

// The same block of 128 rows of an fp32 cache from the tile image attn_kv_image_kernel wrote:
// the same products and sums as flash_attn_kernel without an image, bit for bit. The image is
// the LDS contents, so a tile is copied straight into LDS (global_load_lds, 16 bytes a lane)
// with no registers in between: K of the next tile goes into a second buffer while this tile
// is worked on, V of this tile arrives under S = K Q^T (144 KB of LDS). Against staging in 48
// registers a thread the 4096-token attention went from 724.6 to 715.7 us in turn on one
// board; its 825 GFLOP of bf16 part products take 578 us at the rate of a large matrix product
// there, and the clock falls as the matrix cores fill. Ruled out: 4 waves of 32 rows (half the
// LDS reads, but one wave a SIMD overlaps nothing: 28% slower), the next step's operands read
// under this step's products (0.4% slower), one K array with two halves (every read waited
// for the copy in flight: 5% slower).
template <bool SPLIT>
__global__ __launch_bounds__(512, 1) void flash_image_kernel(AttnPrefillArgs a) {
    constexpr int kQT = 128, W = 8;
    const int grp = a.NQ / a.NKV, rows = a.T * grp, nblk = (rows + kQT - 1) / kQT;
    const int rank = SPLIT ? blockIdx.y : blockIdx.x;
    const int qt = nblk - 1 - rank / a.NKV, kh = rank % a.NKV;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row0 = qt * kQT;
    const int kv_end = a.pos0 + min(rows - 1, row0 + kQT - 1) / grp + 1;
    const int piece_keys = a.plan.piece * kKT;
    const int kv_lo = SPLIT ? static_cast<int>(blockIdx.x) * piece_keys : 0;
    if (SPLIT && kv_lo >= kv_end) return;  // uniform: the block has fewer pieces
    const int kv_hi = SPLIT ? min(kv_end, kv_lo + piece_keys) : kv_end;
    const bool whole = !SPLIT || kv_end <= piece_keys;  // the block's only piece: final output
    const int r16 = lane & 15, g4 = lane >> 4;
    // (separate arrays: the compiler then knows that a copy into one need not be waited for
    // before reads of another)
    typedef uint4 KTile[3][2][kHD / 8][16];
    __shared__ __align__(16) KTile K0, K1;
    __shared__ __align__(16) uint4 Vc[3][kHD / 16][4][16];
    const float sc = 1.0f / sqrtf(static_cast<float>(kHD));

    // K (half 0) or V (half 1) of a tile of the image into LDS: each wave 1 KB per instruction
    constexpr int kCopies = kImgK / (64 * W);
    auto copy = [&](int kv0, int half, uint4* dst) {
        const uint4* src = static_cast<const uint4*>(a.kv_img) +
                           (static_cast<int64_t>(kh) * a.img_tiles + min(kv0, kv_end - 1) / kKT) * kImgTile + half * kImgK;
#pragma unroll
        for (int j = 0; j < kCopies; ++j) {
            const int c = 64 * (W * j + wave);
            __builtin_amdgcn_global_load_lds(
                reinterpret_cast<const __attribute__((address_space(1))) void*>(reinterpret_cast<uintptr_t>(src + c + lane)),
                (__attribute__((address_space(3))) void*)(dst + c), 16, 0, 0);
        }
    };
    // s_waitcnt with only the vector-memory counter given: none left, or one copy's loads left
    constexpr int kWaitAll = 0x0f70, kWaitNewestK = 0x0f70 | kCopies;

    copy(kv_lo, 0, &K0[0][0][0][0]);
    // this lane's query row, dims 32c + 8 g4 .. + 7, as three bf16 parts (the B operand)
    const int qrow = min(row0 + wave * 16 + r16, rows - 1);
    const int qpos = a.pos0 + qrow / grp;
    bf16x8 qp[3][8];
    {
        const float* src = a.Qa + (static_cast<int64_t>(kh * grp + qrow % grp) * a.T + qrow / grp) * kHD + 8 * g4;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const float4 x0 = *reinterpret_cast<const float4*>(src + 32 * c);
            const float4 x1 = *reinterpret_cast<const float4*>(src + 32 * c + 4);
            const float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
            uint4 p3[3];
            split3_8(x, p3);
#pragma unroll
            for (int p = 0; p < 3; ++p) qp[p][c] = __builtin_bit_cast(bf16x8, p3[p]);
        }
    }
    // the wave's last query position: tiles starting past it hold no key its rows attend
    const int wlast = a.pos0 + min(row0 + wave * 16 + 15, rows - 1) / grp;
    floatx4 o[16];  // dims 16 t + r16 of query rows 4 g4 + v
#pragma unroll
    for (int t = 0; t < 16; ++t) o[t] = floatx4{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.0f;

    __builtin_amdgcn_s_waitcnt(kWaitAll);
    lds_barrier();
    copy(kv_lo, 1, &Vc[0][0][0][0]);
    auto tile = [&](int kv0, const KTile& Kc, KTile& Kn) {
        copy(kv0 + kKT, 0, &Kn[0][0][0][0]);  // past the last tile: the last one again
        const bool live_wave = kv0 <= wlast;  // uniform per wave
        bf16x8 pa[3];
        // (K or P part, Q or V part) from the smallest product
        constexpr int lo[6] = {2, 1, 0, 1, 0, 0}, ro[6] = {0, 1, 2, 0, 1, 0};
        if (live_wave) {
            // S^T[key 16 hf + 4 g4 + v][query r16]: the hi.hi products and the smaller part
            // products in separate accumulators, each split over even / odd dim blocks
            floatx4 St[2];
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {
                floatx4 sa[2], sb[2];
#pragma unroll
                for (int e = 0; e < 2; ++e) sa[e] = sb[e] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int c2 = 0; c2 < 4; ++c2) {
                    bf16x8 kop[2][3];
#pragma unroll
                    for (int e = 0; e < 2; ++e)
#pragma unroll
                        for (int p = 0; p < 3; ++p)
                            kop[e][p] = __builtin_bit_cast(bf16x8, Kc[p][hf][4 * (2 * c2 + e) + g4][r16]);
#pragma unroll
                    for (int i = 0; i < 6; ++i)
#pragma unroll
                        for (int e = 0; e < 2; ++e) {
                            floatx4& s = i < 5 ? sb[e] : sa[e];
                            s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kop[e][lo[i]], qp[ro[i]][2 * c2 + e], s, 0, 0, 0);
                        }
                }
                St[hf] = (sb[0] + sb[1]) + (sa[0] + sa[1]);
            }
            float p[8];
            const float f = flash_softmax(St, kv0, qpos, kv_end, sc, g4, m_run, l_run, p);
            flash_rescale(f, g4, o);
            uint4 p3[3];
            split3_8(p, p3);
#pragma unroll
            for (int q = 0; q < 3; ++q) pa[q] = __builtin_bit_cast(bf16x8, p3[q]);
        }
        // this wave's share of V is in LDS (the next K's need not be: lds_barrier would wait for
        // it), then every wave's
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(kWaitNewestK);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        if (live_wave) {
            // O[query 4 g4 + v][dim 16 t + r16] += P[query][keys] V[keys][dim], the part products
            // straight into the running output
#pragma unroll
            for (int t2 = 0; t2 < 8; ++t2) {
                bf16x8 vb[2][3];
#pragma unroll
                for (int e = 0; e < 2; ++e)
#pragma unroll
                    for (int q = 0; q < 3; ++q) vb[e][q] = __builtin_bit_cast(bf16x8, Vc[q][2 * t2 + e][g4][r16 ^ (4 * g4)]);
#pragma unroll
                for (int i = 0; i < 6; ++i)
#pragma unroll
                    for (int e = 0; e < 2; ++e)
                        o[2 * t2 + e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa[lo[i]], vb[e][ro[i]], o[2 * t2 + e], 0, 0, 0);
            }
        }
        __builtin_amdgcn_s_waitcnt(kWaitAll);  // this wave's share of the next K (asked for a tile ago)
        lds_barrier();                         // every wave is done with this V, every share of the next K is in
        copy(kv0 + kKT, 1, &Vc[0][0][0][0]);
    };
    for (int kv0 = kv_lo; kv0 < kv_hi; kv0 += 2 * kKT) {
        tile(kv0, K0, K1);
        if (kv0 + kKT < kv_hi) tile(kv0 + kKT, K1, K0);  // uniform
    }
    __builtin_amdgcn_s_waitcnt(kWaitAll);  // nothing is on its way into LDS when the workgroup ends
    if (!whole) {  // uniform: the piece's output and (max, sum) as they stand, lane by lane
        const int64_t slot = static_cast<int64_t>(blockIdx.y) * gridDim.x + blockIdx.x;
        floatx4* po = reinterpret_cast<floatx4*>(a.part) + (slot * W + wave) * 16 * 64 + lane;
#pragma unroll
        for (int t = 0; t < 16; ++t) po[64 * t] = o[t];
        if (g4 == 0) a.part_ml[slot * kQT + wave * 16 + r16] = make_float2(m_run, l_run);
        return;
    }
    float lr[4];
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) lr[rr] = __shfl(l_run, 4 * g4 + rr);
    flash_store(a, o, lr, kh, grp, rows, row0 + wave * 16, lane);
}

// Merges the pieces of one 16-row group of a block (grid: wave groups, blocks of all kv
// heads): every piece's output scaled by e^(its row maximum - the row's), over the sum of the
// row sums scaled alike, then the gate. The scales of all pieces are formed first, in LDS, so
// that the partial outputs stream with nothing between their loads; each of the 16 waves takes
// one output register (dims 16 w + r16 of rows 4 g4 + v, as the flash kernel left them) of
// every piece, in order.
template <int W>
__global__ __launch_bounds__(1024) void flash_combine_kernel(AttnPrefillArgs a, int pieces) {
    constexpr int QT = 16 * W;
    const int grp = a.NQ / a.NKV, rows = a.T * grp, nblk = (rows + QT - 1) / QT;
    const int qt = nblk - 1 - static_cast<int>(blockIdx.y) / a.NKV, kh = blockIdx.y % a.NKV;
    const int group = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r16 = lane & 15, g4 = lane >> 4;
    const int row0 = qt * QT + 16 * group;
    const int kv_end = a.pos0 + min(rows - 1, qt * QT + QT - 1) / grp + 1;
    const int n = (kv_end + a.plan.piece * kKT - 1) / (a.plan.piece * kKT);
    if (n <= 1 || row0 >= rows) return;  // uniform: already final, or no rows
    __shared__ __align__(16) float f_s[kFlashPieces][16];
    __shared__ float red[64][17], mred[16][16];
    const int64_t slot0 = static_cast<int64_t>(blockIdx.y) * pieces;
    // thread (row tid % 16, pieces tid / 16 and 64 + tid / 16): the row's maximum, its scales
    static_assert(kFlashPieces <= 128, "two pieces per thread");
    const float2* ml = a.part_ml + slot0 * QT + group * 16 + (tid & 15);
    const float2 none = make_float2(-INFINITY, 0.0f);
    const int q0 = tid >> 4;
    const float2 x0 = q0 < n ? ml[q0 * QT] : none, x1 = 64 + q0 < n ? ml[(64 + q0) * QT] : none;
    red[q0][tid & 15] = fmaxf(x0.x, x1.x);
    lds_barrier();
    float m = -INFINITY;
    for (int i = 0; i < min(n, 64); ++i) m = fmaxf(m, red[i][tid & 15]);
    const float f0 = __builtin_amdgcn_exp2f((x0.x - m) * kLog2e);  // 0 for a piece without keys of the row
    const float f1 = __builtin_amdgcn_exp2f((x1.x - m) * kLog2e);
    f_s[q0][tid & 15] = f0;
    f_s[64 + q0][tid & 15] = f1;
    lds_barrier();
    red[q0][tid & 15] = x0.y * f0 + x1.y * f1;
    lds_barrier();
    floatx4 o = floatx4{0.f, 0.f, 0.f, 0.f};
    const floatx4* po = reinterpret_cast<const floatx4*>(a.part) + ((slot0 * W + group) * 16 + wave) * 64 + lane;
#pragma unroll 8
    for (int q = 0; q < n; ++q)
        o += po[static_cast<int64_t>(q) * W * 16 * 64] * *reinterpret_cast<const floatx4*>(&f_s[q][4 * g4]);
    const int dd = 16 * wave + r16;
    float gt[4];  // requested before the first store
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int rc = min(row0 + 4 * g4 + v, rows - 1);
        gt[v] = a.qkv[static_cast<int64_t>(rc / grp) * a.ld_qkv + static_cast<int64_t>(kh * grp + rc % grp) * 2 * kHD + kHD + dd];
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        float l = 0.0f;
        for (int i = 0; i < min(n, 64); ++i) l += red[i][4 * g4 + v];
        const int row = row0 + 4 * g4 + v;
        const int rc = min(row, rows - 1), t = rc / grp, h = kh * grp + rc % grp;
        const float y = (o[v] * (1.0f / l)) * sigmoid_f(gt[v]);
        if (row < rows) {
            if (a.out_tiled) a.out[xt_off(t, h * kHD + dd, a.NQ * kHD)] = y;
            else a.out[static_cast<int64_t>(t) * (a.NQ * kHD) + static_cast<int64_t>(h) * kHD + dd] = y;
        }
        float mx = fabsf(y);
        mx = fmaxf(mx, __shfl_xor(mx, 1));
        mx = fmaxf(mx, __shfl_xor(mx, 2));
        mx = fmaxf(mx, __shfl_xor(mx, 4));
        mx = fmaxf(mx, __shfl_xor(mx, 8));
        if (r16 == 0) mred[wave][4 * g4 + v] = mx;
    }
    if (a.omax) {  // uniform: each row's maximum over this head's 256 dims
        lds_barrier();
        const int row = row0 + tid;
        if (tid < 16 && row < rows) {
            float mx = 0.0f;
#pragma unroll
            for (int i = 0; i < 16; ++i) mx = fmaxf(mx, mred[i][tid]);
            a.omax[static_cast<int64_t>(row / grp) * a.NQ + kh * grp + row % grp] = mx;
        }
    }
}

// ------------------------------------------------------------------ small prefill helpers
__global__ __launch_bounds__(256) void embed_rows_kernel(const uint16_t* embed, const int* ids, float* hidden, int T,
                                                         int H) {
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < static_cast<int64_t>(T) * H;
         i += static_cast<int64_t>(gridDim.x) * 256) {
        const int64_t t = i / H, c = i % H;
        hidden[i] = bf16_to_f32(embed[static_cast<int64_t>(ids[t]) * H + c]);
    }
}

int blocks_for(int64_t n) {
    const int64_t b = (n + 255) / 256;
    return static_cast<int>(b < 8192 ? (b > 0 ? b : 1) : 8192);
}

}  // namespace

int64_t gdn_prefill_workspace_floats(int KH, int VH, int T) {
    const int64_t Tp = (T + kC - 1) / kC * kC;
    return (KH + 2 * static_cast<int64_t>(VH)) * Tp * kD  // Qg U W
           + static_cast<int64_t>(VH) * Tp                 // Eg
           + static_cast<int64_t>(VH) * Tp * kD            // Kd
           + static_cast<int64_t>(VH) * Tp * kC            // P
           + static_cast<int64_t>(VH) * (Tp / kC) * kD * kD  // Sc (chunk-start states)
           + 64 * 6;                                       // alignment slack
}

void gdn_prefill_carve(GdnPrefillArgs& a, float* ws) {
    a.Tp = (a.T + kC - 1) / kC * kC;
    auto take = [&](int64_t n) {
        float* p = ws;
        ws += (n + 63) / 64 * 64;
        return p;
    };
    a.Qg = take(static_cast<int64_t>(a.KH) * a.Tp * kD);
    a.U = take(static_cast<int64_t>(a.VH) * a.Tp * kD);
    a.W = take(static_cast<int64_t>(a.VH) * a.Tp * kD);
    a.Eg = take(static_cast<int64_t>(a.VH) * a.Tp);
    a.Kd = take(static_cast<int64_t>(a.VH) * a.Tp * kD);
    a.P = take(static_cast<int64_t>(a.VH) * a.Tp * kC);
    a.Sc = take(static_cast<int64_t>(a.VH) * (a.Tp / kC) * kD * kD);
}

hipError_t launch_gdn_prefill(GdnPrefillArgs& a, hipStream_t s) {
    // Few tokens: token by token in one launch (the state is read 16 bytes at a time). The scan
    // takes about 1 us a token, 330 instructions of one wave per SIMD; the chunked kernels one
    // chunk's 43 us up to 64 tokens: 6.1 us for 1 token, 20.3 for 16, 35.8 for 32, 40.5 for 36,
    // 44.0 for 40, 52.0 for 48 (16 heads; 42.3 for 36 with two v-heads per k-head). Closer to
    // float64, 1.4e-7 against 2.0e-7.
    if (a.T <= kShortT && (reinterpret_cast<uintptr_t>(a.state) & 15) == 0) {
        klaunch(gdn_short_kernel, a.VH, kShortThreads, 0, s, a);
        if (a.VH != a.KH) klaunch(gdn_ring_kernel, blocks_for(3 * (2 * a.KH * kD + a.VH * kD)), 256, 0, s, a);
        return hipGetLastError();
    }
    klaunch(gdn_chunk_kernel, dim3(a.VH, a.Tp / kC), 256, 0, s, a);
    klaunch(gdn_state_kernel, dim3(a.VH, kD / kSW), 256, 0, s, a);
    klaunch(gdn_out_kernel, dim3(a.VH, a.Tp / kC), 256, 0, s, a);
    return hipGetLastError();
}

void attn_prefill_carve(AttnPrefillArgs& a, float* ws, int64_t floats) {
    a.Qa = ws;
    const int64_t used = attn_prefill_workspace_floats(a.NQ, a.T);
    const AttnRoom r = attn_prefill_room(a.T, a.NQ, a.NKV, a.pos0, a.kv_bf16, device_cu_count(), floats - used);
    ws += used;
    if (r.image) {
        a.kv_img = ws;
        ws += attn_prefill_image_floats(a.NKV, a.pos0, a.T);
    }
    a.plan = r.plan;
    if (r.plan.pieces) {
        a.part = ws;
        a.part_ml = reinterpret_cast<float2*>(ws + static_cast<int64_t>(r.plan.slots) * 16 * kHD);
    }
}

hipError_t launch_attn_prefill(const AttnPrefillArgs& in, hipStream_t s) {
    AttnPrefillArgs a = in;
    if (a.ROT % 8 == 0) klaunch(attn_prefill_prep_kernel, a.T, 256, 0, s, a);
    else klaunch(attn_prefill_prep_any_kernel, dim3(a.T, a.NQ + a.NKV), 256, 0, s, a);
    const int waves = flash_waves(a.kv_bf16), kQT = 16 * waves;
    const int blocks = (a.T * (a.NQ / a.NKV) + kQT - 1) / kQT * a.NKV;
    const FlashPlan& p = a.plan;
    const dim3 grid = p.pieces ? dim3(p.pieces, blocks) : dim3(blocks);
    const bool img = !a.kv_bf16 && a.kv_img;
    if (img) {
        a.img_tiles = attn_prefill_image_tiles(a.pos0, a.T);
        klaunch(attn_kv_image_kernel, dim3(a.img_tiles, a.NKV), 256, 0, s, a);
    }
    if (p.pieces) {
        if (a.kv_bf16) klaunch(flash_attn_kernel<true, true>, grid, 64 * waves, 0, s, a);
        else if (img) klaunch(flash_image_kernel<true>, grid, 512, 0, s, a);
        else klaunch(flash_attn_kernel<false, true>, grid, 64 * waves, 0, s, a);
        if (a.kv_bf16) klaunch(flash_combine_kernel<flash_waves(true)>, dim3(waves, blocks), 1024, 0, s, a, p.pieces);
        else klaunch(flash_combine_kernel<flash_waves(false)>, dim3(waves, blocks), 1024, 0, s, a, p.pieces);
    } else if (a.kv_bf16) {
        klaunch(flash_attn_kernel<true, false>, grid, 64 * waves, 0, s, a);
    } else if (img) {
        klaunch(flash_image_kernel<false>, grid, 512, 0, s, a);
    } else {
        klaunch(flash_attn_kernel<false, false>, grid, 64 * waves, 0, s, a);
    }
    return hipGetLastError();
}

hipError_t launch_embed_rows(const uint16_t* embed, const int* ids, float* hidden, int T, int H, hipStream_t s) {
    klaunch(embed_rows_kernel, blocks_for(static_cast<int64_t>(T) * H), 256, 0, s, embed, ids, hidden, T, H);
    return hipGetLastError();
}

}  // namespace q35k
