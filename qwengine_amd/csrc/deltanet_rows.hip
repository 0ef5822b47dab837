// Gated DeltaNet prefill of B tokens (gfx950): the token mixer of deltanet.hip over a chunk of prompt rows.  Entry point
// and state conventions: src/cuda/prefill.cuh:37-44; semantics: src/reference/ref_model.cpp:169-256.
//
// Three launches: k_dn_conv_prep (token-parallel: conv, unit q / k, and every coefficient of the chunked recurrence that
// does not need the state), k_dn_chunk_rows (the sequential chunks of 16 tokens, on fp32 MFMA) and k_dn_gnorm_rows (the
// gated norm to fp16).
#include <type_traits>
#include <utility>

#include "deltanet.hpp"

namespace qwa {

constexpr int DN_CT = 16;      // tokens per chunk of the chunked recurrence
constexpr int DN_RG = 4;               // workgroups (column groups) per head of the recurrence
constexpr int DN_RC = DN_HD / DN_RG;   // 32 value columns per workgroup
constexpr int DN_RN = DN_RC / 16;      // column tiles
constexpr int DN_CW = 4;               // waves per workgroup (32 key dims each)
// coefficient block of one (chunk, value head): T [16][16] | M' [16][16] (row-major) | {c2, gamma} [16] | E [16]
constexpr int DN_CM = 256, DN_CG = 512, DN_CE = 544;
constexpr int DN_NCOEF = 704;  // floats per block in the workspace
constexpr int DN_BLK = DN_CT * DN_HD;  // floats of one head's chunk of q, k or v
// The operands of the recurrence, per chunk and head in the order in which its lanes hold them (lane = 16 g4 + l16), so
// that every load instruction of a wave is 16 bytes per lane of one contiguous 1 KB span.  Tokens past B are zeros.
struct DnRows {
    float* v;     // [nch][48][8 column tiles][64 lanes][4]: beta v[token 4 g4 + e][16 tile + l16] (after conv and SiLU)
    float* q;     // [nch][16][4 waves][2][64][4]: unit q[token l16][32 w + 16 m + 4 g4 + e]
    float* k;     // the same of unit k
    float* kt;    // [nch][16][4][2][64][4]: unit k[token 4 g4 + e][32 w + 16 m + l16]
    float* coef;  // [nch][48][DN_NCOEF]
};

__host__ __device__ inline DnRows dn_rows_split(void* work, int nch) {
    float* f = static_cast<float*>(work);
    DnRows r;
    r.v = f;
    f += (size_t)nch * DN_VH * DN_BLK;
    r.q = f;
    f += (size_t)nch * DN_KH * DN_BLK;
    r.k = f;
    f += (size_t)nch * DN_KH * DN_BLK;
    r.kt = f;
    f += (size_t)nch * DN_KH * DN_BLK;
    r.coef = f;
    return r;
}

// `need`: 14400 floats per token of the padded chunks, 12288 of v, q, k and kt and 2112 of coefficients.  For whole chunks
// the stated size stays the one that this entry point has always stated (`least`: rows in token order, no padding), with
// nothing stored in the difference; short and ragged calls need the padding (1 token: 922 KB).
size_t dn_work_bytes(int B) {
    const size_t nch = (B + DN_CT - 1) / DN_CT;
    const size_t need = nch * (DN_BLK * (DN_VH + 3 * DN_KH) + DN_VH * DN_NCOEF);
    const size_t least = (size_t)B * (DN_CH + 2 * DN_QK + 2 * DN_VH) + nch * DN_VH * DN_NCOEF;
    return (need > least ? need : least) * sizeof(float);
}

// ---- the chunked recurrence.  For a chunk of 16 tokens with S the state before it, decays g, write strengths beta,
// G(s, t) = g_{s+1} ... g_t and gamma_t = g_0 ... g_t, the per-token rule
//     S <- g S;  u = beta (v - S^T k);  S += k u^T;  o = S^T q
// unrolls to
//     a_t = S^T k_t, b_t = S^T q_t
//     (I + L) U = W,  L[t][s] = beta_t G(s, t) k_s.k_t (s < t),  W_t = beta_t v_t - c2_t a_t,  c2_t = beta_t gamma_t
//     o_t = gamma_t b_t + sum_{s<=t} M'[t][s] u_s,  M'[t][s] = G(s, t) k_s.q_t
//     S'  = gamma_15 S + sum_s E_s k_s u_s^T,  E_s = G(s, 15).
// k_dn_conv_prep does everything that does not need the state: the conv, the unit q and k, beta v, and per (chunk,
// value head) T = (I + L)^-1, M' and the token scalars.  k_dn_chunk_rows walks the chunks.  Tokens past B are padded
// with k = q = v = 0, beta = 0, g = 1, which change nothing.
__device__ __forceinline__ f4 mfma4f32(float a, float b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// conv[t][c] = silu(sum_k w[c][k] in(t - 3 + k)), in(i) = qkv[i][c] for i >= 0, else row 3 + i of the old window, for
// the N tokens from t0 on of one channel (inputs read once, sliding in registers); the run that holds token B - 1 also
// writes the window after the chunk (rows k = input B - 3 + k) into the other buffer.
template <int N>
__device__ __forceinline__ void dn_conv_run(const float* __restrict__ qkv, const float* __restrict__ cs_old,
                                            float* __restrict__ cs_new, float4 w, int c, int t0, int B, float* y) {
    float x[N + 3];
#pragma unroll
    for (int k = 0; k < N + 3; k++) {
        const int i = t0 - 3 + k;
        x[k] = i < 0 ? cs_old[(size_t)(3 + i) * DN_CH + c] : i < B ? qkv[(size_t)i * DN_CH + c] : 0.0f;
    }
    if (t0 + N >= B) {
#pragma unroll
        for (int k = 0; k < N + 3; k++) {
            const int kk = t0 - 3 + k - (B - 3);
            if (kk >= 0 && kk < 3) cs_new[(size_t)kk * DN_CH + c] = x[k];
        }
    }
#pragma unroll
    for (int u = 0; u < N; u++) y[u] = dn_silu(w.x * x[u] + w.y * x[u + 1] + w.z * x[u + 2] + w.w * x[u + 3]);
}

__device__ __forceinline__ float dn_sigmoid(float x) { return 1.0f / (1.0f + expf(-x)); }

// One launch, two kinds of blocks of 256 threads (bound by the bytes: for 1024 tokens 42 MB read and 57 MB written, 20 us
// at the card's copy rate).
//  * blocks 0 .. 16 nch - 1: (key head, chunk).  Thread = channel of the key head's q | k; the conv of the chunk's 16
//    tokens, L2 norms through LDS (unit q / k written out and kept in LDS), the Gram products k.k and q.k on fp32
//    MFMA (each wave half of the 128 dims of one of the two), then wave v < 3 forms the coefficient block of value head
//    kh + 16 v: L and M' from the Gram entries and the decay products, T by forward substitution (lane = column).
//    The three value heads of a key head share the conv, the norms and the Gram products.
//  * the rest: (256 v channels, run of 8 tokens): the conv, times the token's beta for the head.
// Measured for 1024 tokens: 24 us, 21 once the clock has settled (a conv kernel and a per-value-head preparation kernel
// before: 21 + 22 us, 18 + 20 settled).
constexpr int DN_CR = 8;                  // tokens per run of the v channels
constexpr int DN_XP = 2 * DN_HD + 4;      // padded row (floats) of the chunk's q | k in LDS
__global__ void __launch_bounds__(256) k_dn_conv_prep(const float* __restrict__ qkv, const float* __restrict__ cs_old,
                                                      const float* __restrict__ conv_w, DnRows r,
                                                      const float* __restrict__ beta_raw,
                                                      const float* __restrict__ alpha_raw,
                                                      const float* __restrict__ dt_bias,
                                                      const float* __restrict__ ssm_a, float eps, int B, int nch,
                                                      float* __restrict__ cs_new) {
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
    __shared__ __attribute__((aligned(16))) float sx[DN_CT][DN_XP];      // q (dims 0 .. 127) | k (128 .. 255)
    __shared__ float sp[4][DN_CT][DN_CT + 1];                            // partial Gram: k.k (waves 0, 1), q.k (2, 3)
    __shared__ __attribute__((aligned(16))) float sL[3][DN_CT][DN_CT + 4];
    __shared__ __attribute__((aligned(16))) float sg[3][DN_CT], sb[3][DN_CT];
    const int qk_blocks = DN_KH * nch;
    if ((int)blockIdx.x >= qk_blocks) {
        constexpr int NX = DN_VD / 256;
        const int b = blockIdx.x - qk_blocks, t0 = b / NX * DN_CR, cv = b % NX * 256, c = 2 * DN_QK + cv + t;
        const int hv = (cv + t) / DN_HD, col = t % DN_HD;
        if (t < 2 * DN_CR) {  // beta of (token t0 + t % 8, head cv / 128 + t / 8)
            const int i = t0 + t % DN_CR;
            sb[0][t] = i < B ? dn_sigmoid(beta_raw[(size_t)i * DN_VH + cv / DN_HD + t / DN_CR]) : 0.0f;
        }
        float y[DN_CR];
        dn_conv_run<DN_CR>(qkv, cs_old, cs_new, *reinterpret_cast<const float4*>(conv_w + (size_t)c * 4), c, t0, B, y);
        __syncthreads();
        float* dst =
            r.v + ((size_t)(t0 / DN_CT) * DN_VH + hv) * DN_BLK + col / 16 * 256 + col % 16 * 4 + t0 % DN_CT * 16;
#pragma unroll
        for (int u = 0; u < DN_CR; u += 4) {
            float x[4];
#pragma unroll
            for (int e = 0; e < 4; e++) x[e] = t0 + u + e < B ? y[u + e] * sb[0][(t >> 7) * DN_CR + u + e] : 0.0f;
            *reinterpret_cast<float4*>(dst + 16 * u) = make_float4(x[0], x[1], x[2], x[3]);
        }
        return;
    }
    const int kh = blockIdx.x % DN_KH, ch = blockIdx.x / DN_KH, t0 = ch * DN_CT;
    const int c = (t >> 7) * DN_QK + kh * DN_HD + (t & (DN_HD - 1));
    if (t < 3 * DN_CT) {  // decay and beta of (value head kh + 16 (t / 16), token t0 + t % 16)
        const int i = t0 + t % DN_CT, hv = t / DN_CT, h = kh + DN_KH * hv;
        float g = 1.0f, be = 0.0f;
        if (i < B) {
            const float a = alpha_raw[(size_t)i * DN_VH + h] + dt_bias[h];
            const float spl = a > 20.0f ? a : logf(1.0f + expf(a));
            g = expf(spl * ssm_a[h]);
            be = dn_sigmoid(beta_raw[(size_t)i * DN_VH + h]);
        }
        sg[hv][t % DN_CT] = g;
        sb[hv][t % DN_CT] = be;
    }
    {
        float y[DN_CT];
        dn_conv_run<DN_CT>(qkv, cs_old, cs_new, *reinterpret_cast<const float4*>(conv_w + (size_t)c * 4), c, t0, B, y);
#pragma unroll
        for (int u = 0; u < DN_CT; u++) sx[u][t] = y[u];
    }
    __syncthreads();
    // the (token, q or k) rows 8 wave .. 8 wave + 7, lane holding dims lane and lane + 64
#pragma unroll
    for (int p = 0; p < 8; p++) {
        const int u = 4 * wave + (p >> 1), hw = p & 1;
        const float v0 = sx[u][DN_HD * hw + lane], v1 = sx[u][DN_HD * hw + lane + 64];
        const float iv = 1.0f / fmaxf(sqrtf(wave_sum(v0 * v0 + v1 * v1)), eps);
        const bool in = t0 + u < B;
        const float n0 = in ? v0 * iv : 0.0f, n1 = in ? v1 * iv : 0.0f;
        sx[u][DN_HD * hw + lane] = n0;
        sx[u][DN_HD * hw + lane + 64] = n1;
    }
    __syncthreads();
    const int g4 = lane >> 4, l16 = lane & 15;
    {
        // the recurrence's operands of wave `wave`, in lane order
        const size_t base = ((size_t)ch * DN_KH + kh) * DN_BLK + 512 * wave + 4 * lane;
#pragma unroll
        for (int m = 0; m < 2; m++) {
            const int d = 32 * wave + 16 * m;
            *reinterpret_cast<float4*>(r.q + base + 256 * m) = *reinterpret_cast<const float4*>(&sx[l16][d + 4 * g4]);
            *reinterpret_cast<float4*>(r.k + base + 256 * m) =
                *reinterpret_cast<const float4*>(&sx[l16][DN_HD + d + 4 * g4]);
            const float* kc = &sx[4 * g4][DN_HD + d + l16];
            *reinterpret_cast<float4*>(r.kt + base + 256 * m) =
                make_float4(kc[0], kc[DN_XP], kc[2 * DN_XP], kc[3 * DN_XP]);
        }
    }
    {
        // Gram: D[row][col] = x_row . k_col over dims 64 (wave & 1) .. + 63, x = k (waves 0, 1) or q (waves 2, 3)
        f4 acc = f4{0.0f, 0.0f, 0.0f, 0.0f};
        const float* xr = &sx[l16][(wave < 2 ? DN_HD : 0) + 64 * (wave & 1) + 4 * g4];
        const float* kr = &sx[l16][DN_HD + 64 * (wave & 1) + 4 * g4];
#pragma unroll
        for (int m = 0; m < 4; m++) {
            const float4 x = *reinterpret_cast<const float4*>(xr + 16 * m);
            const float4 k = *reinterpret_cast<const float4*>(kr + 16 * m);
            acc = mfma4f32(x.x, k.x, acc);
            acc = mfma4f32(x.y, k.y, acc);
            acc = mfma4f32(x.z, k.z, acc);
            acc = mfma4f32(x.w, k.w, acc);
        }
#pragma unroll
        for (int rr = 0; rr < 4; rr++) sp[wave][4 * g4 + rr][l16] = acc[rr];
    }
    __syncthreads();
    if (wave == 3) return;
    const int h = kh + DN_KH * wave;
    float* cf = r.coef + ((size_t)ch * DN_VH + h) * DN_NCOEF;
    float g[DN_CT];
#pragma unroll
    for (int e = 0; e < DN_CT; e++) g[e] = sg[wave][e];
    // lane: column s = l16, rows u = 4 g4 + rr.  G(s, u): the product of the decays s + 1 .. u, in order
    {
        float G = 1.0f, Gu[4] = {1.0f, 1.0f, 1.0f, 1.0f};
#pragma unroll
        for (int e = 0; e < DN_CT; e++) {
            G = e > l16 ? G * g[e] : G;
            if ((e >> 2) == g4) Gu[e & 3] = G;
        }
#pragma unroll
        for (int rr = 0; rr < 4; rr++) {
            const int s = l16, u = 4 * g4 + rr;
            const float kk = sp[0][u][s] + sp[1][u][s], qk = sp[2][u][s] + sp[3][u][s];
            sL[wave][u][s] = s < u ? sb[wave][u] * Gu[rr] * kk : 0.0f;
            cf[DN_CM + u * DN_CT + s] = s <= u ? Gu[rr] * qk : 0.0f;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // sL: written above, read below by other lanes of the wave
    __builtin_amdgcn_wave_barrier();
    if (lane < DN_CT) {
        // column s = lane of T = (I + L)^-1 by forward substitution: T[u][s] = [u == s] - sum_{q<u} L[u][q] T[q][s]
        float x[DN_CT], gam = 1.0f, E = 1.0f;
#pragma unroll
        for (int u = 0; u < DN_CT; u++) {
            float acc = u == lane ? 1.0f : 0.0f;
#pragma unroll
            for (int q = 0; q < u; q++) acc = fmaf(-sL[wave][u][q], x[q], acc);
            x[u] = u < lane ? 0.0f : acc;
            cf[u * DN_CT + lane] = x[u];
        }
#pragma unroll
        for (int e = 0; e < DN_CT; e++) {
            gam = e <= lane ? gam * g[e] : gam;
            E = e > lane ? E * g[e] : E;
        }
        *reinterpret_cast<float2*>(cf + DN_CG + 2 * lane) = make_float2(sb[wave][lane] * gam, gam);
        cf[DN_CE + lane] = E;
    }
}

// The sequential part: one workgroup of 4 waves per (value head, 32 value columns); wave w holds key dims 32 w .. 32 w
// + 31 of its 128 x 32 slice of S (two 16-column tiles) in fp32 MFMA accumulators.  A chunk is matrix products on
// v_mfma_f32_16x16x4_f32, per wave:
//   a = K S (16 MFMAs, partial over the wave's key dims), summed through LDS behind the chunk's one barrier;
//   b = Q S (16, mostly under the latency of that exchange);
//   U = T W (8, in every wave: it is the operand of the wave's own update);  S = gamma_15 S + K^T (E U) (16);
//   O = gamma b + M' U: each wave adds the product over its quarter of the tokens s (s mod 4 = w: 2) to its own partial
//   gamma b (gamma_t scales q_t, and c2_t k_t, before the products) and leaves the sum in LDS, where the next chunk's
//   barrier makes it visible; the threads then add the four waves' partials and store.
// All operands come straight from global memory (L2) into registers in lane order, two chunks ahead; nothing is staged
// through LDS.
// What bounds it: one wave's in-order issue, on 192 of the 256 CUs: 58 MFMAs (33 cycles each: 55 us for 64 chunks at 2.24
// GHz) and about 28 load, store and LDS instructions per chunk, which take some 50 cycles of issue each, as the CU's four
// waves reach them together.  Measured for 1024 tokens, in one session: 93 us (86 once the clock has settled); with
// compiler-ordered groups of loads and 64-bit lane addresses: 96 us.  Before: 16 columns per workgroup (384 workgroups, half
// of the CUs with two), the operands staged and transposed through LDS by all threads and O in every wave: 131 us.  This
// kernel with the operands in row order (26 load instructions per chunk instead of 12): 104 us; with 8 waves of one column
// tile each: 108 us.

// f(0), f(1), ... with each index a compile-time constant
template <class F, int... S>
__device__ __forceinline__ void static_steps(F&& f, std::integer_sequence<int, S...>) {
    (f(std::integral_constant<int, S>{}), ...);
}

// one chunk's operands of one lane
struct DnOps {
    float4 k[2], q[2], kt[2], v[DN_RN];  // (see DnRows)
    float4 T, E, M;                      // T[l16][4 g4 ..], E[4 g4 ..], M'[l16][4 g4 ..]
    float2 cg;                           // {c2, gamma}[l16]
};

__global__ void __launch_bounds__(DN_CW * 64, 1) k_dn_chunk_rows(DnRows r, float* __restrict__ state, int B,
                                                                 float* __restrict__ core_out) {
    const int h = blockIdx.x, grp = blockIdx.y, kh = h % DN_KH, t = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6), l = t & 63, g4 = l >> 4, l16 = l & 15;
    // the waves' partial a and O of one chunk; two buffers: a slow wave may still read chunk c's while others write
    // c + 1's
    __shared__ __attribute__((aligned(16))) float4 s_a[2][DN_CW][DN_RN][64], s_o[2][DN_CW][DN_RN][64];
    const int nch = (B + DN_CT - 1) / DN_CT;
    const int j = grp * DN_RC + l16;
    float* Sj = state + (size_t)h * DN_HD * DN_HD + (size_t)j * DN_HD + 32 * w + 4 * g4;
    f4 st[DN_RN][2];
#pragma unroll
    for (int n = 0; n < DN_RN; n++)
#pragma unroll
        for (int m = 0; m < 2; m++) {
            const float4 v = *reinterpret_cast<const float4*>(Sj + 16 * n * DN_HD + 16 * m);
            st[n][m] = f4{v.x, v.y, v.z, v.w};
        }
    const float oscale = 1.0f / sqrtf((float)DN_HD);
    uint32_t wm[4];  // all ones for e = w
#pragma unroll
    for (int e = 0; e < 4; e++) wm[e] = e == w ? ~0u : 0u;
    // operand addresses: a uniform chunk base and lane offsets that never change
    const uint32_t ol = 16 * l, oT = (l16 * DN_CT + 4 * g4) * 4, oE = 16 * g4, og = 8 * l16;
    const size_t kofs = (size_t)kh * DN_BLK + 512 * w, vofs = (size_t)h * DN_BLK + 512 * grp;
    // (buffer loads: scalar base, 32-bit lane offset; a 64-bit address per lane takes twice as long to issue)
    auto rsrc = [](const float* p, int bytes) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), 0, bytes, 0x00027000);
    };
    typedef uint32_t u4v __attribute__((ext_vector_type(4)));
    typedef uint32_t u2v __attribute__((ext_vector_type(2)));
    auto ld4 = [&](const float* base, uint32_t off) {
        const u4v v = __builtin_amdgcn_raw_buffer_load_b128(rsrc(base, 1024), off, 0, 0);
        return __builtin_bit_cast(float4, v);
    };
    // load i of a chunk's 12
    constexpr int NLOAD = 12;
    auto fetch = [&](DnOps& x, int c, int i) {
        const size_t kc = (size_t)c * (DN_KH * DN_BLK) + kofs;
        const float* cf = r.coef + ((size_t)c * DN_VH + h) * DN_NCOEF;
        if (i < 2) x.k[i] = ld4(r.k + kc + 256 * i, ol);
        else if (i == 2)
            x.cg = __builtin_bit_cast(float2, (u2v)__builtin_amdgcn_raw_buffer_load_b64(rsrc(cf + DN_CG, 128), og, 0, 0));
        else if (i < 5) x.q[i - 3] = ld4(r.q + kc + 256 * (i - 3), ol);
        else if (i < 7) x.v[i - 5] = ld4(r.v + (size_t)c * (DN_VH * DN_BLK) + vofs + 256 * (i - 5), ol);
        else if (i == 7) x.T = ld4(cf, oT);
        else if (i == 8) x.E = ld4(cf + DN_CE, oE);
        else if (i < 11) x.kt[i - 9] = ld4(r.kt + kc + 256 * (i - 9), ol);
        else x.M = ld4(cf + DN_CM, oT);
    };
    // c2_t k_t and gamma_t q_t: quarter i of a loaded chunk's 16 values
    auto scale = [&](DnOps& x, int i) {
        float4& z = i < 2 ? x.k[i & 1] : x.q[i & 1];
        const float f = i < 2 ? x.cg.x : x.cg.y;
        z = make_float4(f * z.x, f * z.y, f * z.z, f * z.w);
    };
    // sums the waves' partial O of chunk c: thread (wave w, lane l) the rows 4 g4 + 2 (w / 2) + {0, 1} of column tile
    // w % 2 (every token of a chunk is below B except in the last one)
    const int en = w & 1, eh = w >> 1;
    float* const cobase = core_out + (size_t)(4 * g4 + 2 * eh) * DN_VD + h * DN_HD + j + 16 * en;
    float2 eo[DN_CW];
    auto emit_read = [&](int c) {
#pragma unroll
        for (int x = 0; x < DN_CW; x++) eo[x] = reinterpret_cast<const float2*>(&s_o[c & 1][x][en][l])[eh];
    };
    auto emit_sum = [&]() {
        eo[0].x = (((eo[0].x + eo[1].x) + eo[2].x) + eo[3].x) * oscale;
        eo[0].y = (((eo[0].y + eo[1].y) + eo[2].y) + eo[3].y) * oscale;
    };
    float* co = cobase;  // rows of the chunk being stored
    f4 o[DN_RN];         // partial O of the last chunk
    // One chunk on x; z: the next chunk's operands (in registers since the chunk before), y: those of chunk cf, fetched.
    // A wave issues in order, and its own VALU instructions cost nothing only in the shadow of an MFMA (32 cycles), so the
    // order is fixed by a scheduling barrier (DN_SB) after every MFMA and the few instructions that go with it.
#define DN_SB __builtin_amdgcn_sched_barrier(0)
    auto chunk = [&](DnOps& x, int c, DnOps& z, DnOps& y, int cf, auto first) {
        constexpr bool FIRST = decltype(first)::value;
        const int p = c & 1;
        f4 pa[DN_RN], pb[DN_RN], U[DN_RN];
#pragma unroll
        for (int n = 0; n < DN_RN; n++) pa[n] = pb[n] = U[n] = f4{0.0f, 0.0f, 0.0f, 0.0f};
        const float kx[2][4] = {{x.k[0].x, x.k[0].y, x.k[0].z, x.k[0].w}, {x.k[1].x, x.k[1].y, x.k[1].z, x.k[1].w}};
        const float qx[2][4] = {{x.q[0].x, x.q[0].y, x.q[0].z, x.q[0].w}, {x.q[1].x, x.q[1].y, x.q[1].z, x.q[1].w}};
        const float Tx[4] = {x.T.x, x.T.y, x.T.z, x.T.w}, Ex[4] = {x.E.x, x.E.y, x.E.z, x.E.w};
        const float Mx[4] = {x.M.x, x.M.y, x.M.z, x.M.w};
        const float ktx[2][4] = {{x.kt[0].x, x.kt[0].y, x.kt[0].z, x.kt[0].w},
                                 {x.kt[1].x, x.kt[1].y, x.kt[1].z, x.kt[1].w}};
        const float vx[2][4] = {{x.v[0].x, x.v[0].y, x.v[0].z, x.v[0].w}, {x.v[1].x, x.v[1].y, x.v[1].z, x.v[1].w}};
        auto b_mfma = [&](int i, int n) { pb[n] = mfma4f32(qx[i >> 2][i & 3], st[n][i >> 2][i & 3], pb[n]); };
        // a, the partial O of the chunk before to LDS
        static_steps([&](auto step) __attribute__((always_inline)) {
            constexpr int s = step.value, n = s >> 3, i = s & 7;
            pa[n] = mfma4f32(kx[i >> 2][i & 3], st[n][i >> 2][i & 3], pa[n]);
            if constexpr (!FIRST && (s == 2 || s == 3))
                s_o[p ^ 1][w][s - 2][l] = make_float4(o[s - 2][0], o[s - 2][1], o[s - 2][2], o[s - 2][3]);
            if constexpr (s == 11) s_a[p][w][0][l] = make_float4(pa[0][0], pa[0][1], pa[0][2], pa[0][3]);
            if constexpr (s == 5 || s == 8 || s == 14) fetch(y, cf, s == 5 ? 0 : s == 8 ? 1 : 2);
            DN_SB;
        }, std::make_integer_sequence<int, 16>{});
        b_mfma(0, 0);
        DN_SB;
        b_mfma(0, 1);
        DN_SB;
        s_a[p][w][1][l] = make_float4(pa[1][0], pa[1][1], pa[1][2], pa[1][3]);
        __syncthreads();
        float4 ap[DN_RN][DN_CW];
#pragma unroll
        for (int n = 0; n < DN_RN; n++)
#pragma unroll
            for (int v = 0; v < DN_CW; v++) ap[n][v] = s_a[p][v][n][l];
        DN_SB;
        float W[DN_RN][4], eu[DN_RN][4];
        uint32_t mw = 0, uw[DN_RN] = {0, 0};  // M'[l16][4 g4 + w], U[n][w]
        const float g15 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x.cg.y), DN_CT - 1));
        f4 sn[DN_RN][2];
        static_steps([&](auto step) __attribute__((always_inline)) {
            constexpr int s = step.value;
            // the rest of b, U, then per column tile the update and O
            if constexpr (s < 14) b_mfma(1 + (s >> 1), s & 1);
            else if constexpr (s < 22) {
                constexpr int n = (s - 14) >> 2, e = (s - 14) & 3;
                U[n] = mfma4f32(Tx[e], W[n][e], U[n]);
            }
            else {
                constexpr int n = (s - 22) / 9, k = (s - 22) % 9;
                if constexpr (k < 8) sn[n][k & 1] = mfma4f32(ktx[k & 1][k >> 1], eu[n][k >> 1], sn[n][k & 1]);
                else o[n] = mfma4f32(__uint_as_float(mw), __uint_as_float(uw[n]), pb[n]);
            }
            if constexpr (!FIRST) {  // the output of the chunk before
                if constexpr (s == 14) emit_read(c - 1);
                if constexpr (s == 25) emit_sum();
                if constexpr (s == 27) co[0] = eo[0].x;
                if constexpr (s == 30) co[DN_VD] = eo[0].y;
            }
            if constexpr (s >= 6 && s < 14) {  // W = beta v - a
                constexpr int n = (s - 6) >> 2, e = (s - 6) & 3;
                auto at = [&](int v) {
                    return e == 0 ? ap[n][v].x : e == 1 ? ap[n][v].y : e == 2 ? ap[n][v].z : ap[n][v].w;
                };
                W[n][e] = vx[n][e] - (((at(0) + at(1)) + at(2)) + at(3));
            }
            if constexpr (s >= 14 && s < 18) sn[(s - 14) >> 1][s & 1] = st[(s - 14) >> 1][s & 1] * g15;
            if constexpr (s == 20 || s == 24) {
#pragma unroll
                for (int e = 0; e < 4; e++) eu[(s - 20) >> 2][e] = Ex[e] * U[(s - 20) >> 2][e];
            }
            if constexpr (s == 2) {
#pragma unroll
                for (int e = 0; e < 4; e++) mw |= __float_as_uint(Mx[e]) & wm[e];
            }
            if constexpr (s == 26 || s == 28) {
#pragma unroll
                for (int e = 0; e < 4; e++) uw[(s - 26) >> 1] |= __float_as_uint(U[(s - 26) >> 1][e]) & wm[e];
            }
            if constexpr (s >= 34 && s < 38) scale(z, s - 34);
            if constexpr (s % 4 == 1 && s / 4 < NLOAD - 3) fetch(y, cf, 3 + s / 4);
            DN_SB;
        }, std::make_integer_sequence<int, 40>{});
        if constexpr (!FIRST) co += DN_CT * DN_VD;
#pragma unroll
        for (int n = 0; n < DN_RN; n++)
#pragma unroll
            for (int m = 0; m < 2; m++) st[n][m] = sn[n][m];
    };
    // two chunks ahead, three register sets; every fetch is unconditional (past the end: the last chunk again) so that
    // the compiler can count the loads in flight and waits for no later ones
    DnOps xa, xb, xc;
#pragma unroll
    for (int i = 0; i < NLOAD; i++) fetch(xa, 0, i);
#pragma unroll
    for (int i = 0; i < NLOAD; i++) fetch(xb, min(1, nch - 1), i);
#pragma unroll
    for (int i = 0; i < 4; i++) scale(xa, i);
    const int last = nch - 1;
    chunk(xa, 0, xb, xc, min(2, last), std::true_type{});
    int c = 1;
    for (; c + 3 <= nch; c += 3) {
        chunk(xb, c, xc, xa, min(c + 2, last), std::false_type{});
        chunk(xc, c + 1, xa, xb, min(c + 3, last), std::false_type{});
        chunk(xa, c + 2, xb, xc, min(c + 4, last), std::false_type{});
    }
    if (c < nch) chunk(xb, c, xc, xa, last, std::false_type{});
    if (c + 1 < nch) chunk(xc, c + 1, xa, xb, last, std::false_type{});
#pragma unroll
    for (int n = 0; n < DN_RN; n++) s_o[last & 1][w][n][l] = make_float4(o[n][0], o[n][1], o[n][2], o[n][3]);
    __syncthreads();
    emit_read(last);
    emit_sum();
    const int tok = last * DN_CT + 4 * g4 + 2 * eh;
    if (tok < B) co[0] = eo[0].x;
    if (tok + 1 < B) co[DN_VD] = eo[0].y;
#pragma unroll
    for (int n = 0; n < DN_RN; n++)
#pragma unroll
        for (int m = 0; m < 2; m++)
            *reinterpret_cast<float4*>(Sj + 16 * n * DN_HD + 16 * m) =
                make_float4(st[n][m][0], st[n][m][1], st[n][m][2], st[n][m][3]);
#undef DN_SB
}

// gated RMSNorm per (token, value head), fp16 out: grid (B), 256 threads; wave w normalises value heads w, w + 4,
// ..., lane holding dims 2 lane, 2 lane + 1 (all loads of the token issued before the first reduction)
__global__ void __launch_bounds__(256) k_dn_gnorm_rows(const float* __restrict__ core, const float* __restrict__ z,
                                                       const float* __restrict__ nw, float eps,
                                                       uint16_t* __restrict__ o16) {
    constexpr int NHW = DN_VH / 4;  // heads per wave
    const int t = blockIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const float2 w = *reinterpret_cast<const float2*>(nw + 2 * lane);
    float2 v[NHW], zz[NHW];
#pragma unroll
    for (int i = 0; i < NHW; i++) {
        const size_t idx = (size_t)t * DN_VD + (wave + 4 * i) * DN_HD + 2 * lane;
        v[i] = *reinterpret_cast<const float2*>(core + idx);
        zz[i] = *reinterpret_cast<const float2*>(z + idx);
    }
#pragma unroll
    for (int i = 0; i < NHW; i++) {
        const float rs = 1.0f / sqrtf(wave_sum(v[i].x * v[i].x + v[i].y * v[i].y) / DN_HD + eps);
        const uint32_t lo = f2h_bits(v[i].x * rs * w.x * dn_silu(zz[i].x));
        const uint32_t hi = f2h_bits(v[i].y * rs * w.y * dn_silu(zz[i].y));
        *reinterpret_cast<uint32_t*>(o16 + (size_t)t * DN_VD + (wave + 4 * i) * DN_HD + 2 * lane) = lo | (hi << 16);
    }
}

hipError_t launch_dn_rows(const qwa_dn_params& p, const float* qkv, const float* z, const float* beta_raw,
                          const float* alpha_raw, int B, int cin, float eps, void* work, float* core_out,
                          uint16_t* o16, hipStream_t st) {
    const int nch = (B + DN_CT - 1) / DN_CT;
    const DnRows r = dn_rows_split(work, nch);
    const float* cs_old = p.conv_state + (size_t)cin * 3 * DN_CH;
    float* cs_new = p.conv_state + (size_t)(cin ^ 1) * 3 * DN_CH;
    const int runs = nch * (DN_CT / DN_CR);
    hipLaunchKernelGGL(k_dn_conv_prep, dim3(DN_KH * nch + DN_VD / 256 * runs), dim3(256), 0, st, qkv, cs_old, p.conv_w,
                       r, beta_raw, alpha_raw, p.dt_bias, p.ssm_a, eps, B, nch, cs_new);
    hipLaunchKernelGGL(k_dn_chunk_rows, dim3(DN_VH, DN_RG), dim3(DN_CW * 64), 0, st, r, p.ssm_state, B, core_out);
    hipLaunchKernelGGL(k_dn_gnorm_rows, dim3(B), dim3(256), 0, st, core_out, z, p.ssm_norm, eps, o16);
    return hipGetLastError();
}

}  // namespace qwa
