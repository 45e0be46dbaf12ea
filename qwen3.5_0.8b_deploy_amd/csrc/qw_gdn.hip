// qw_gdn.hip -- Gated-DeltaNet decode step for gfx950: everything between the
// input projections (QKV, Z, a, b) and the out projection of a linear-
// attention layer, for T consecutive tokens of each of B sequences (T = 1 is
// the decode step; T > 1 is the serial prefill of the reference's
// forward_batch, linear_attention_cuda.cu:529-680, whose contract is
// equality with T single-token steps, verify_linear_attn_batch.cu:68-112).
//
// Math (reference CPU operator, src/backend/cpu/core/attention/
// language_linear_attn.cpp:143-256; CUDA chain conv1d_update_fused /
// l2norm_qk_fused / gated_delta / norm_gate_fused, linear_attention_cuda.cu:
// 47-172):
//   conv:  c[d] = silu(w[d][K-1]*x[d] + sum_j<K-1 w[d][j]*st[d][j]), then
//          st[d][j] = st[d][j-1] (j > 0), st[d][0] = x[d]   (st[d][0] newest)
//   q, k:  per head L2-normalized (eps 1e-6 under the root), q * 1/sqrt(kd)
//   gates: beta = sigmoid(b), g = -exp(A_log) * softplus(a + dt_bias)
//   state: S *= exp(g); kv = S^T k; delta = (v - kv) * beta; S += k delta^T;
//          o = S^T q                                  (S: kd x vd, FP32)
//   out:   o * rsqrt(mean(o^2) + 1e-6) * norm_w * silu(z)   per head
//
// Work decomposition.  One workgroup of 256 threads per (sequence, head).
// The head's 2*kd + vd conv channels are spread over the threads (two at
// most per thread), each keeping its conv taps and state in registers; q, k,
// v land in LDS per token.  The state S[kd][vd] of the head (64 KB) is read
// once before the first token and written once after the last: thread t owns
// column t % vd for rows [64*(t/vd), +64), so every load and store of a row
// is one coalesced 512-byte access, the column sums kv and o need one two-way
// combine in LDS, and the update happens in registers between the two.
// Bound: at T = 1 HBM (state read + write, ~2 x 64 KB per head); at T > 1
// the per-token barrier chain (the recurrence is serial in T).
#include "qw_stream.hpp"

namespace qwk {

constexpr int GDN_T = 256;

__device__ __forceinline__ float gdn_load(const void* p, int dt, int64_t i) {
    return dt == DT_F32 ? reinterpret_cast<const float*>(p)[i] : load_act(p, dt, i);
}

template <int KD, int VD>
__global__ __launch_bounds__(GDN_T) void gdn_kernel(GdnArgs a) {
    static_assert(GDN_T % VD == 0 && KD % (GDN_T / VD) == 0, "state split");
    static_assert(2 * KD + VD <= 2 * GDN_T, "two conv channels per thread at most");
    constexpr int RH = GDN_T / VD;   // row groups
    constexpr int RPT = KD / RH;     // state rows per thread
    constexpr int SLMAX = 7;         // conv taps kept in registers (K <= 8)
    const int h = blockIdx.x, b = blockIdx.y;
    const int t = threadIdx.x;
    const int nh = a.nh;
    const int K = a.K, SL = a.K - 1;
    const int conv_dim = 2 * nh * KD + nh * VD;
    const int wave = t >> 6, lane = t & 63;

    __shared__ float qs[KD], ks[KD], vs[VD];
    __shared__ float red[RH][VD];
    __shared__ float scal[4];  // |q|, |k|, beta, exp(g)
    __shared__ float wsum[GDN_T / 64];

    // ---- per-thread conv channels (up to two) and their state, in registers ----
    int cd[2];
    float* cdst[2];
    float cw[2][SLMAX + 1], cst[2][SLMAX];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int c = t + u * GDN_T;
        cd[u] = -1;
        cdst[u] = nullptr;
        if (c < 2 * KD + VD) {
            if (c < KD) { cd[u] = h * KD + c; cdst[u] = &qs[c]; }
            else if (c < 2 * KD) { cd[u] = nh * KD + h * KD + (c - KD); cdst[u] = &ks[c - KD]; }
            else { cd[u] = 2 * nh * KD + h * VD + (c - 2 * KD); cdst[u] = &vs[c - 2 * KD]; }
        }
#pragma unroll
        for (int j = 0; j <= SLMAX; ++j) cw[u][j] = (cd[u] >= 0 && j < K) ? a.conv_w[(int64_t)cd[u] * K + j] : 0.0f;
#pragma unroll
        for (int j = 0; j < SLMAX; ++j)
            cst[u][j] = (cd[u] >= 0 && j < SL) ? a.conv_state[((int64_t)b * conv_dim + cd[u]) * SL + j] : 0.0f;
    }
    // ---- the head's state rows of this thread, resident for all tokens ----
    float* S = a.rec_state + ((int64_t)b * nh + h) * KD * VD;
    const int col = t % VD, r0 = (t / VD) * RPT;
    float s[RPT];
#pragma unroll
    for (int i = 0; i < RPT; ++i) s[i] = S[(r0 + i) * VD + col];
    const float q_scale = 1.0f / sqrtf((float)KD);
    const float expA = __expf(a.A_log[h]);

    for (int tok = 0; tok < a.T; ++tok) {
        const int64_t in_row = ((int64_t)b * a.T + tok) * a.ld_in;
        // ---- conv1d + SiLU, state shift (st[0] newest) ----
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            if (cd[u] < 0) continue;
            const float xv = gdn_load(a.mixed, a.in_dt, in_row + cd[u]);
            float sum = 0.0f;
#pragma unroll
            for (int j = 0; j <= SLMAX; ++j)
                if (j == K - 1) sum = cw[u][j] * xv;
#pragma unroll
            for (int j = 0; j < SLMAX; ++j)
                if (j < SL) sum += cw[u][j] * cst[u][j];
#pragma unroll
            for (int j = SLMAX - 1; j > 0; --j) cst[u][j] = cst[u][j - 1];
            cst[u][0] = xv;
            *cdst[u] = silu_f(sum);
        }
        __syncthreads();

        // ---- L2 norms of q and k (waves 0 and 1), gates (thread 128) ----
        if (wave < 2) {
            const float* v = wave == 0 ? qs : ks;
            float ss = 0.0f;
            for (int d = lane; d < KD; d += 64) ss += v[d] * v[d];
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
            if (lane == 0) scal[wave] = sqrtf(ss + 1e-6f);
        } else if (t == 128) {
            const float av = gdn_load(a.a, a.in_dt, in_row + h) + a.dt_bias[h];
            const float bv = gdn_load(a.b, a.in_dt, in_row + h);
            const float sp = av > 20.0f ? av : logf(1.0f + __expf(av));
            scal[2] = 1.0f / (1.0f + __expf(-bv));
            scal[3] = __expf(-expA * sp);
        }
        __syncthreads();
        for (int d = t; d < KD; d += GDN_T) {
            qs[d] = qs[d] / scal[0] * q_scale;
            ks[d] = ks[d] / scal[1];
        }
        __syncthreads();

        // ---- delta rule on this thread's column slice ----
        const float beta = scal[2], gt = scal[3];
        float kv = 0.0f;
#pragma unroll
        for (int i = 0; i < RPT; ++i) {
            s[i] *= gt;
            kv += s[i] * ks[r0 + i];
        }
        red[t / VD][col] = kv;
        __syncthreads();
        float kvs = 0.0f;
#pragma unroll
        for (int g = 0; g < RH; ++g) kvs += red[g][col];
        const float delta = (vs[col] - kvs) * beta;
        float o = 0.0f;
#pragma unroll
        for (int i = 0; i < RPT; ++i) {
            s[i] += ks[r0 + i] * delta;
            o += s[i] * qs[r0 + i];
        }
        __syncthreads();  // every thread has read red[] for kv
        red[t / VD][col] = o;
        __syncthreads();

        // ---- per-head RMSNorm x norm_w x SiLU(z): threads 0 .. VD-1 own a
        // column; every wave takes part in the reduction and its barrier ----
        float os = 0.0f;
        if (t < VD) {
#pragma unroll
            for (int g = 0; g < RH; ++g) os += red[g][t];
        }
        float ss = os * os;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
        if (lane == 0) wsum[wave] = ss;
        __syncthreads();
        if (t < VD) {
            float tot = 0.0f;
#pragma unroll
            for (int w = 0; w < GDN_T / 64; ++w) tot += wsum[w];
            const float inv = 1.0f / sqrtf(tot / (float)VD + 1e-6f);
            const float zv = gdn_load(a.z, a.in_dt, in_row + h * VD + t);
            const float y = os * inv * a.norm_w[t] * silu_f(zv);
            const int64_t oi = ((int64_t)b * a.T + tok) * a.ld_out + h * VD + t;
            if (a.out_dt == DT_F32) reinterpret_cast<float*>(a.out)[oi] = y;
            else store_act(a.out, a.out_dt, oi, y);
        }
        // the next token rewrites qs/ks/vs, red and wsum only after this barrier
        __syncthreads();
    }

    // ---- write back the state: recurrent once, conv taps once ----
#pragma unroll
    for (int i = 0; i < RPT; ++i) S[(r0 + i) * VD + col] = s[i];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        if (cd[u] < 0) continue;
#pragma unroll
        for (int j = 0; j < SLMAX; ++j)
            if (j < SL) a.conv_state[((int64_t)b * conv_dim + cd[u]) * SL + j] = cst[u][j];
    }
}

hipError_t launch_gdn(const GdnArgs& a, hipStream_t stream) {
    if (a.kd != 128 || a.vd != 128 || a.K < 1 || a.K > 8 || a.T < 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL((gdn_kernel<128, 128>), dim3(a.nh, a.B), dim3(GDN_T), 0, stream, a);
    return hipGetLastError();
}

// ===========================================================================
// Chunked form for long token runs.  The serial recurrence above costs one
// barrier chain per token; here the tokens of a sequence are cut into chunks
// of C = 64 and the delta rule is rewritten per chunk (the WY form of the
// delta rule, Yang et al. 2024, "Parallelizing Linear Transformers with the
// Delta Rule over Sequence Length", with the per-token decay of Gated
// DeltaNet).  For a chunk with start state S0, per-token decays gamma_i,
// G_i = sum_{m<=i} log gamma_m (so Gamma_i = exp(G_i)), the serial steps
//   S_i = gamma_i S_{i-1} + k_i u_i^T,  u_i = beta_i (v_i - gamma_i S_{i-1}^T k_i),
//   o_i = S_i^T q_i
// unroll to
//   (I + A) U = diag(beta) V - diag(beta Gamma) K S0,
//       A_ij = beta_i exp(G_i - G_j) k_i.k_j  (j < i, else 0)
//   U = Ut - W S0,  Ut = (I+A)^-1 diag(beta) V,  W = (I+A)^-1 diag(beta Gamma) K
//   O = diag(Gamma) Q S0 + Aq U,  Aq_ij = exp(G_i - G_j) q_i.k_j  (j <= i)
//   S_C = Gamma_C S0 + K^T diag(exp(G_C - G_i)) U.
// Every decay ratio is exp of a non-positive number, so nothing overflows.
// Three launches per segment of tokens:
//   gdn_chunk_prep   (chunk, head, sequence): conv + SiLU, L2 norms, gates,
//                    the two Gram matrices, the unit-triangular solve for Ut
//                    and W, and the decayed Q and K, written to a chunk record;
//   gdn_chunk_state  (16-column slice of the state, head, sequence): the only
//                    serial pass, S_{c+1} = Gamma_C S_c + Kd^T (Ut - W S_c);
//                    it records each chunk's start state S_c and U = Ut - W S_c;
//   gdn_chunk_out    (chunk, head, sequence), in parallel over the chunks:
//                    O = Qd S_c + Aq U, then RMSNorm x norm_w x SiLU(z).
// The state update is column-separable (column j of S only needs column j of
// V), which is what lets the state pass split the state over 8 workgroups.
// Every product runs on FP32 MFMA (exact FP32 products, FP32 accumulation).
//
// Bound at one prompt: latency.  16 heads x T/64 chunks are at most a workgroup
// or two per CU, so each stage's time is that of its longest chain, and the
// FP32 matrix cores (64 FLOP per clock and SIMD) set the floor of each stage.
// The chunk record is therefore laid out as the consumers' MFMA operands (K
// and U transposed, the state by columns, W negated): the state and output
// passes load them from L2 straight into registers as float4, with no LDS
// staging and no transposing stores.  T = 1000, 16 heads, one sequence, before
// (256-thread workgroups, row-major records staged and transposed in LDS) and
// now: prep 41.8 -> 25.8, state 52.1 -> 30.4, outputs 28.8 -> 16.3 us (125 -> 70 us per
// layer).
constexpr int GC_C = 64;     // tokens per chunk
constexpr int GC_D = 128;    // key_dim = value_dim
constexpr int GC_P = GC_D + 4;  // LDS row stride (floats) of the [C][D] tiles
constexpr int GC_AP = GC_C + 4; // LDS row stride of [.][C] tiles
constexpr int GC_VS = 16;    // state columns per state-pass workgroup
constexpr int GC_T = 1024;   // threads of the prep kernel
// chunk record (floats): -W[C][D] | Ut^T[D][C] (U^T after the state pass) | Qd[C][D] | Kd^T[D][C] |
// Aq[C][C] (16x16 tiles on and below the diagonal) | Gamma_C, padding |
// S_c^T[D][D] (start state by columns, written by the state pass).
// Each matrix is stored as 16x16 tiles of 1 KB, row tiles outermost, a tile as
// the float4 of its 64 lanes: lane l holds row l%16, columns 4*(l/16) .. +3 --
// one contiguous 1 KB access per wave and MFMA operand.
constexpr int GR_W = 0, GR_U = GC_C * GC_D, GR_Q = 2 * GC_C * GC_D, GR_K = 3 * GC_C * GC_D,
              GR_AQ = 4 * GC_C * GC_D, GR_G = GR_AQ + GC_C * GC_C, GR_S = GR_G + 64, GR_SIZE = GR_S + GC_D * GC_D;

// FP32 MFMA 16x16x4: lane l supplies A[l%16][l/16] and B[l/16][l%16] and holds
// D[4*(l/16) + r][l%16] in element r.  The k index of a product only has to be
// the same permutation on both sides, so a 16-deep k block is fed as four
// steps q with k = 4*(l/16) + q: a float4 along k per lane and operand, and a
// D tile is directly the B operand of a following product.
__device__ __forceinline__ f32x4 mfma16(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma16x4(f32x4 a, f32x4 b, f32x4 c) {
#pragma unroll
    for (int q = 0; q < 4; ++q) c = mfma16(a[q], b[q], c);
    return c;
}

// float4 of this lane in tile (rt, ct) of a record matrix with NC column tiles
template <int NC>
__device__ __forceinline__ int gr_tile(int rt, int ct, int lane) { return ((rt * NC + ct) * 64 + lane) * 4; }
__device__ __forceinline__ f32x4 ld4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ void st4(float* p, f32x4 v) { *reinterpret_cast<f32x4*>(p) = v; }

__device__ __forceinline__ float gdn_x(const GdnArgs& a, int b, int conv_dim, int d, int tau) {
    // conv input of channel d at token tau of sequence b; tau < 0 reads the conv state
    // (state[0] is token -1), tau >= T is padding
    if (tau >= a.T) return 0.0f;
    if (tau >= 0) return gdn_load(a.mixed, a.in_dt, ((int64_t)b * a.T + tau) * a.ld_in + d);
    return a.conv_state[((int64_t)b * conv_dim + d) * (a.K - 1) + (-tau - 1)];
}

// Workgroups are dealt round robin to the 8 XCDs, each with its own L2: the
// n workgroups of a (sequence, head) pair take ids of one residue mod 8, so
// that what one of the three kernels writes for a head, and what its
// workgroups share, stays in one L2.  Grid: 8 * n * ceil(pairs / 8).
__device__ __forceinline__ bool gdn_pair(const GdnArgs& a, int n, int& i, int& h, int& b) {
    const int lin = blockIdx.x, idx = lin >> 3;
    const int pair = (lin & 7) + 8 * (idx / n);
    i = idx % n;
    h = pair % a.nh;
    b = pair / a.nh;
    return pair < a.nh * a.B;
}
static int gdn_grid(const GdnArgs& a, int n) { return 8 * n * ((a.nh * a.B + 7) / 8); }

// One chunk of one head, 16 waves (the workgroup's LDS fills a CU, so four
// waves per SIMD are what hides the latencies).  KT: conv taps, 0 = a.K.
template <int KT>
__global__ __launch_bounds__(GC_T) void gdn_chunk_prep(GdnArgs a, int t0, int nchunk, float* rec) {
    int c, h, b;
    if (!gdn_pair(a, nchunk, c, h, b)) return;
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63, li = lane & 15, lg = lane >> 4;
    const int nh = a.nh, K = KT ? KT : a.K;
    const int conv_dim = 3 * nh * GC_D;
    const int tc = t0 + c * GC_C;  // first token of the chunk

    __shared__ __attribute__((aligned(16))) float qkv_s[3 * GC_C * GC_P];  // q | k | v tiles [C][P]
    float* const qs = qkv_s;
    float* const ks = qkv_s + GC_C * GC_P;
    float* const vs = qkv_s + 2 * GC_C * GC_P;
    __shared__ __attribute__((aligned(16))) float As[GC_C * GC_AP];  // A^T
    __shared__ __attribute__((aligned(16))) float Tl[4 * 256];       // inverses of A's diagonal blocks
    __shared__ double Gs[GC_C];  // decay prefix sums in FP64: their differences stay exact to ~1e-16
    __shared__ float bs[GC_C], gq[GC_C], gk[GC_C];  // beta_i, exp(G_i), exp(G_C - G_i)

    // ---- conv1d + SiLU + L2 norms (waves 0..11): a half wave takes 8
    // consecutive tokens of one of q, k, v, a lane 4 channels, so a token's
    // norm is a sum over the half wave; the inputs and the K-1 before them
    // come straight from the rows (or the conv state) into registers ----
    if (wave < 12) {
        constexpr int R = 8, HK = KT ? KT - 1 : 7;
        const int hw = t >> 5, g3 = hw % 3, i0 = R * (hw / 3), ch = 4 * (t & 31);
        const int d = g3 * nh * GC_D + h * GC_D + ch;
        const int esz = a.in_dt == DT_F32 ? 4 : 2;
        // vector loads when the rows allow, element loads otherwise
        const bool vec = ((uintptr_t)a.mixed % (4 * esz)) == 0 && (a.ld_in % 4) == 0;
        f32x4 x[R + HK];  // x[n]: token tc + i0 + n - HK
        if (vec) {
#pragma unroll
            for (int n = 0; n < R + HK; ++n) {
                if (!KT && n < HK - (K - 1)) continue;
                const int tau = tc + i0 + n - HK;
                const int64_t o = ((int64_t)b * a.T + max(0, min(tau, a.T - 1))) * a.ld_in + d;
                x[n] = a.in_dt == DT_F32 ? *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(a.mixed) + o)
                                         : load_act4(a.mixed, a.in_dt, o);
            }
        } else {
#pragma unroll
            for (int n = 0; n < R + HK; ++n) {
                if (!KT && n < HK - (K - 1)) continue;
                const int tau = tc + i0 + n - HK;
#pragma unroll
                for (int q = 0; q < 4; ++q) x[n][q] = gdn_x(a, b, conv_dim, d + q, max(tau, 0));
            }
        }
        if (tc + i0 < HK) {  // the sequence's first tokens: inputs before it from the conv state
#pragma unroll
            for (int n = 0; n < HK; ++n) {
                const int tau = tc + i0 + n - HK;
                if ((!KT && n < HK - (K - 1)) || tau >= 0) continue;
#pragma unroll
                for (int q = 0; q < 4; ++q) x[n][q] = gdn_x(a, b, conv_dim, d + q, tau);
            }
        }
        float w[4][HK + 1];
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int j = 0; j <= HK; ++j) w[q][j] = (KT || j < K) ? a.conv_w[(int64_t)(d + q) * K + j] : 0.0f;
        const float qsc = g3 == 0 ? 1.0f / sqrtf((float)GC_D) : 1.0f;
#pragma unroll
        for (int i = 0; i < R; ++i) {
            f32x4 y;
            float ss = 0.0f;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float wl = w[q][HK];
                if (!KT) wl = a.conv_w[(int64_t)(d + q) * K + K - 1];
                float sum = wl * x[i + HK][q];
#pragma unroll
                for (int j = 0; j < HK; ++j)
                    if (KT || j < K - 1) sum += w[q][j] * x[i + HK - 1 - j][q];
                y[q] = tc + i0 + i < a.T ? silu_f(sum) : 0.0f;
                ss += y[q] * y[q];
            }
            if (g3 < 2) {
                ss = dpp_add<0xB1, 0xF>(ss);   // quad_perm [1,0,3,2]
                ss = dpp_add<0x4E, 0xF>(ss);   // quad_perm [2,3,0,1]
                ss = dpp_add<0x141, 0xF>(ss);  // row_half_mirror
                ss = dpp_add<0x140, 0xF>(ss);  // row_mirror: every lane holds its row's sum
                ss += __shfl_xor(ss, 16);
                y = y * (1.0f / sqrtf(ss + 1e-6f) * qsc);
            }
            *reinterpret_cast<f32x4*>(&qkv_s[(g3 * GC_C + i0 + i) * GC_P + ch]) = y;
        }
    } else if (wave == 12) {  // ---- gates and the decay prefix sum, one token per lane ----
        const int tau = tc + lane;
        double g = 0.0;
        float beta = 0.0f;
        if (tau < a.T) {
            const int64_t row = ((int64_t)b * a.T + tau) * a.ld_in;
            const float av = gdn_load(a.a, a.in_dt, row + h) + a.dt_bias[h];
            const float bv = gdn_load(a.b, a.in_dt, row + h);
            const float sp = av > 20.0f ? av : logf(1.0f + __expf(av));
            beta = 1.0f / (1.0f + __expf(-bv));
            g = (double)(-__expf(a.A_log[h]) * sp);
        }
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const double o = __shfl_up(g, off);
            if (lane >= off) g += o;
        }
        const double GC = __shfl(g, 63);
        Gs[lane] = g;
        bs[lane] = beta;
        gq[lane] = __expf((float)g);
        gk[lane] = __expf((float)(GC - g));
    }
    __syncthreads();
    // ---- Gram tiles on MFMA: the 10 lower 16x16 tiles (ti >= tj) of K K^T
    // (jobs 0..9) and Q K^T (10..19); A = beta_i exp(G_i - G_j) k_i.k_j (j < i)
    // into LDS transposed (As[j][i]); Aq = exp(G_i - G_j) q_i.k_j (j <= i) to
    // the record (the tiles above the diagonal are never read) ----
    float* R = rec + ((int64_t)(b * nh + h) * nchunk + c) * GR_SIZE;
    for (int job = wave; job < 20; job += 16) {
        const int tile = job % 10;
        const bool isq = job >= 10;
        const int ti = tile < 1 ? 0 : tile < 3 ? 1 : tile < 6 ? 2 : 3;
        const int tj = tile - ti * (ti + 1) / 2;
        // K K^T gives A's tile as D[i][j]; K Q^T gives Aq's transposed, D[j][i]:
        // a lane then holds four consecutive i of A^T's row j, and four j of Aq's row i
        const float* xa = &ks[(16 * (isq ? tj : ti) + li) * GC_P + 4 * lg];
        const float* xb = isq ? &qs[(16 * ti + li) * GC_P + 4 * lg] : &ks[(16 * tj + li) * GC_P + 4 * lg];
        f32x4 g0 = {0.0f, 0.0f, 0.0f, 0.0f}, g1 = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int kb = 0; kb < GC_D; kb += 32) {
            g0 = mfma16x4(ld4(xa + kb), ld4(xb + kb), g0);
            g1 = mfma16x4(ld4(xa + kb + 16), ld4(xb + kb + 16), g1);
        }
        g0 = g0 + g1;
        f32x4 av;
        if (isq) {
            const int i = 16 * ti + li;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int j = 16 * tj + 4 * lg + r;
                av[r] = j <= i ? __expf((float)(Gs[i] - Gs[j])) * g0[r] : 0.0f;
            }
            st4(&R[GR_AQ + gr_tile<4>(ti, tj, lane)], av);
        } else {
            const int j = 16 * tj + li;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = 16 * ti + 4 * lg + r;
                av[r] = j < i ? bs[i] * __expf((float)(Gs[i] - Gs[j])) * g0[r] : 0.0f;
            }
            st4(&As[j * GC_AP + 16 * ti + 4 * lg], av);
        }
    }
    __syncthreads();
    // ---- (I + A) X = [diag(beta Gamma) K | diag(beta) V] by 16-row blocks:
    // the four diagonal blocks are inverted by substitution (wave 0, one lane
    // per column of a block) while the other waves write the decayed Q and K,
    // then each wave runs the block substitution
    //   X_b = T_bb (R_b - sum_{c<b} A_bc X_c)
    // on MFMA for its 16 of the 256 right-hand-side columns, X in registers ----
    if (wave == 0) {
        const int bb = lg, jc = li;
        float x[16];
#pragma unroll
        for (int m = 0; m < 16; ++m) {
            float v = m == jc ? 1.0f : 0.0f;
#pragma unroll
            for (int n = 0; n < m; ++n) v -= As[(16 * bb + n) * GC_AP + 16 * bb + m] * x[n];
            x[m] = v;
        }
#pragma unroll
        for (int m = 0; m < 16; ++m) Tl[bb * 256 + m * 16 + jc] = x[m];
    } else {
        for (int e = wave - 1; e < 32; e += 15) {  // 16x16 tiles (conflict-free LDS reads)
            const int i = 16 * (e >> 3) + li, d = 16 * (e & 7) + 4 * lg;
            st4(&R[GR_Q + (e * 64 + lane) * 4], ld4(&qs[i * GC_P + d]) * gq[i]);
        }
        for (int e = wave - 1; e < 32; e += 15) {
            const int d = 16 * (e >> 2) + li, i = 16 * (e & 3) + 4 * lg;
            f32x4 kv;
#pragma unroll
            for (int q = 0; q < 4; ++q) kv[q] = ks[(i + q) * GC_P + d] * gk[i + q];
            st4(&R[GR_K + (e * 64 + lane) * 4], kv);
        }
    }
    __syncthreads();
    {
        const bool isw = wave < 8;
        const float* src = isw ? ks : vs;
        const int col = (wave & 7) * 16 + li;  // column within K (waves 0..7) or V (8..15)
        f32x4 X[4];
#pragma unroll
        for (int rb = 0; rb < 4; ++rb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = 16 * rb + 4 * lg + r;
                X[rb][r] = bs[i] * (isw ? gq[i] : 1.0f) * src[i * GC_P + col];
            }
#pragma unroll
        for (int rb = 0; rb < 4; ++rb) {
#pragma unroll
            for (int cb = 0; cb < rb; ++cb) {
                f32x4 na;
#pragma unroll
                for (int q = 0; q < 4; ++q) na[q] = -As[(16 * cb + 4 * lg + q) * GC_AP + 16 * rb + li];
                X[rb] = mfma16x4(na, X[cb], X[rb]);
            }
            const f32x4 ta = *reinterpret_cast<const f32x4*>(&Tl[rb * 256 + li * 16 + 4 * lg]);
            X[rb] = mfma16x4(ta, X[rb], f32x4{0.0f, 0.0f, 0.0f, 0.0f});
        }
#pragma unroll
        for (int rb = 0; rb < 4; ++rb) {
            if (isw) {  // through LDS (over q, which no wave reads any more) into row order
#pragma unroll
                for (int r = 0; r < 4; ++r) qs[(16 * rb + 4 * lg + r) * GC_P + col] = -X[rb][r];
            } else {
                st4(&R[GR_U + gr_tile<4>(wave & 7, rb, lane)], X[rb]);
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int e = wave; e < 32; e += 16)
        st4(&R[GR_W + (e * 64 + lane) * 4], ld4(&qs[(16 * (e >> 3) + li) * GC_P + 16 * (e & 7) + 4 * lg]));
    if (t == 0) R[GR_G] = gq[GC_C - 1];
}

// The serial pass over the chunks of one segment for a 16-column slice of
// one head's state, on MFMA.  Per chunk: record S_c, U = Ut - W S_c (wave w:
// rows 16w..16w+15, written over Ut), S_{c+1} = Gamma_C S_c + Kd^T U (wave w:
// state rows 32w..32w+31, kept in registers across the chunks).  Only U and S
// pass through LDS (12 KB); a wave's W and Kd rows are its own MFMA operands,
// loaded two chunks ahead into two register sets, so a chunk costs its two
// chains of 32 dependent-pair MFMAs (~0.9 us) and two barriers.  On the last
// segment the workgroup also moves the conv state of 48 of the head's 384
// channels (the prep kernel of this segment has finished reading it).
__global__ __launch_bounds__(256, 2) void gdn_chunk_state(GdnArgs a, int nchunk, float* rec, int last_segment) {
    int sl, h, b;
    if (!gdn_pair(a, GC_D / GC_VS, sl, h, b)) return;
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63, li = lane & 15, lg = lane >> 4;
    const int nh = a.nh;
    const int c0 = sl * GC_VS;  // first state column of the slice

    __shared__ __attribute__((aligned(16))) float St[GC_VS * GC_P], Ut[GC_VS * GC_AP];

    struct Chunk {
        f32x4 w[8], k[2][4], u;
        float g;
    };
    float* R0 = rec + (int64_t)(b * nh + h) * nchunk * GR_SIZE;
    auto load_w = [&](Chunk& x, const float* Rc) {
#pragma unroll
        for (int kb = 0; kb < 8; ++kb)
            x.w[kb] = ld4(&Rc[GR_W + gr_tile<8>(wave, kb, lane)]);
        x.u = ld4(&Rc[GR_U + gr_tile<4>(sl, wave, lane)]);
    };
    auto load_k = [&](Chunk& x, const float* Rc) {
#pragma unroll
        for (int dt = 0; dt < 2; ++dt)
#pragma unroll
            for (int ib = 0; ib < 4; ++ib)
                x.k[dt][ib] = ld4(&Rc[GR_K + gr_tile<4>(2 * wave + dt, ib, lane)]);
        x.g = Rc[GR_G];
    };
    // The loads are kept in the order of their use (the scheduler would mix
    // the two sets), so that the compiler's wait counts leave the later ones
    // in flight.
    Chunk x0, x1;
    const float* R1 = R0 + (nchunk > 1 ? GR_SIZE : 0);
    float* Sg = a.rec_state + ((int64_t)b * nh + h) * GC_D * GC_D;
    f32x4 S[2];  // this wave's rows of the slice: S[32w + 16dt + 4lg + r][c0 + li]
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[dt][r] = Sg[(32 * wave + 16 * dt + 4 * lg + r) * GC_D + c0 + li];
    __builtin_amdgcn_sched_barrier(0);
    load_w(x0, R0);
    __builtin_amdgcn_sched_barrier(0);
    load_k(x0, R0);
    __builtin_amdgcn_sched_barrier(0);
    load_w(x1, R1);
    __builtin_amdgcn_sched_barrier(0);
    load_k(x1, R1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int dt = 0; dt < 2; ++dt) st4(&St[li * GC_P + 32 * wave + 16 * dt + 4 * lg], S[dt]);
    __syncthreads();
    auto step = [&](Chunk& x, int c) {
        float* R = R0 + (int64_t)c * GR_SIZE;
        const float* Rn = R0 + (int64_t)min(c + 2, nchunk - 1) * GR_SIZE;
        // the start state of this chunk, by columns
#pragma unroll
        for (int dt = 0; dt < 2; ++dt)
            st4(&R[GR_S + gr_tile<8>(sl, 2 * wave + dt, lane)], S[dt]);
        // U = Ut - W S_c   (rows 16w .. 16w+15)
        f32x4 u0 = x.u, u1 = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int kb = 0; kb < 8; kb += 2) {
            u0 = mfma16x4(x.w[kb], ld4(&St[li * GC_P + 16 * kb + 4 * lg]), u0);
            u1 = mfma16x4(x.w[kb + 1], ld4(&St[li * GC_P + 16 * kb + 16 + 4 * lg]), u1);
        }
        u0 = u0 + u1;
        st4(&Ut[li * GC_AP + 16 * wave + 4 * lg], u0);
        st4(&R[GR_U + gr_tile<4>(sl, wave, lane)], u0);
        __builtin_amdgcn_sched_barrier(0);
        load_w(x, Rn);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        // S_{c+1} = Gamma_C S_c + Kd^T U   (state rows 32w .. 32w+31)
        S[0] = S[0] * x.g;
        S[1] = S[1] * x.g;
#pragma unroll
        for (int ib = 0; ib < 4; ++ib) {
            const f32x4 ub = ld4(&Ut[li * GC_AP + 16 * ib + 4 * lg]);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                S[0] = mfma16(x.k[0][ib][q], ub[q], S[0]);
                S[1] = mfma16(x.k[1][ib][q], ub[q], S[1]);
            }
        }
#pragma unroll
        for (int dt = 0; dt < 2; ++dt) st4(&St[li * GC_P + 32 * wave + 16 * dt + 4 * lg], S[dt]);
        __builtin_amdgcn_sched_barrier(0);
        load_k(x, Rn);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
    };
    int c = 0;
    for (; c + 1 < nchunk; c += 2) {
        step(x0, c);
        step(x1, c + 1);
    }
    if (c < nchunk) step(x0, c);
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
        for (int r = 0; r < 4; ++r) Sg[(32 * wave + 16 * dt + 4 * lg + r) * GC_D + c0 + li] = S[dt][r];

    constexpr int CPS = 3 * GC_D / (GC_D / GC_VS);  // conv channels per slice: 48
    if (last_segment && a.K > 1 && t < CPS) {
        const int conv_dim = 3 * nh * GC_D;
        const int cl = sl * CPS + t;  // 0 .. 383 within the head
        const int d = (cl / GC_D) * nh * GC_D + h * GC_D + cl % GC_D;
        float nv[7];
#pragma unroll
        for (int j = 0; j < 7; ++j) nv[j] = j < a.K - 1 ? gdn_x(a, b, conv_dim, d, a.T - 1 - j) : 0.0f;
#pragma unroll
        for (int j = 0; j < 7; ++j)
            if (j < a.K - 1) a.conv_state[((int64_t)b * conv_dim + d) * (a.K - 1) + j] = nv[j];
    }
}

// Outputs of one chunk of one head on MFMA, transposed (O^T = S^T Qd^T +
// U^T Aq^T), so that a lane holds four consecutive output columns of a token.
// 8 waves: wave (cg, rg) computes columns 32cg .. 32cg+31 of the token tiles rg
// and 3 - rg (together 5 of the 10 tiles of Aq on or below the diagonal), a
// 2 x 2 block of tiles that reads each operand tile once for two products;
// all of a wave's S and Q tiles are in flight before its first product.
// Then per token RMSNorm x norm_w x SiLU(z), the sums of squares combined
// across the waves in LDS.
__global__ __launch_bounds__(512, 2) void gdn_chunk_out(GdnArgs a, int t0, int nchunk, const float* rec) {
    int c, h, b;
    if (!gdn_pair(a, nchunk, c, h, b)) return;
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63, li = lane & 15, lg = lane >> 4;
    const int cg = wave & 3, rg = wave >> 2;
    const int rt[2] = {rg, 3 - rg};
    __shared__ float red[4][GC_C];
    const float* R = rec + ((int64_t)(b * a.nh + h) * nchunk + c) * GR_SIZE;
    f32x4 sa[8][2], qv[8][2];
#pragma unroll
    for (int kb = 0; kb < 8; ++kb)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            sa[kb][u] = ld4(&R[GR_S + gr_tile<8>(2 * cg + u, kb, lane)]);
            qv[kb][u] = ld4(&R[GR_Q + gr_tile<8>(rt[u], kb, lane)]);
        }
    __builtin_amdgcn_sched_barrier(0);
    f32x4 o[2][2];  // [column tile][token tile]
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int v = 0; v < 2; ++v) o[u][v] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int kb = 0; kb < 8; ++kb)
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int v = 0; v < 2; ++v) o[u][v] = mfma16(sa[kb][u][q], qv[kb][v][q], o[u][v]);
#pragma unroll
    for (int ib = 0; ib < 4; ++ib) {
        if (ib > rt[1]) continue;  // uniform over the wave
        const f32x4 u0 = ld4(&R[GR_U + gr_tile<4>(2 * cg, ib, lane)]), u1 = ld4(&R[GR_U + gr_tile<4>(2 * cg + 1, ib, lane)]);
        const f32x4 a1 = ld4(&R[GR_AQ + gr_tile<4>(rt[1], ib, lane)]);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            o[0][1] = mfma16(u0[q], a1[q], o[0][1]);
            o[1][1] = mfma16(u1[q], a1[q], o[1][1]);
        }
        if (ib > rt[0]) continue;
        const f32x4 a0 = ld4(&R[GR_AQ + gr_tile<4>(rt[0], ib, lane)]);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            o[0][0] = mfma16(u0[q], a0[q], o[0][0]);
            o[1][0] = mfma16(u1[q], a0[q], o[1][0]);
        }
    }
    // ---- RMSNorm x norm_w x SiLU(z): lane (lg, li) holds columns
    // 32cg + 16u + 4lg + r of token 16rt[v] + li in o[u][v][r] ----
#pragma unroll
    for (int v = 0; v < 2; ++v) {
        float ss = 0.0f;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int r = 0; r < 4; ++r) ss += o[u][v][r] * o[u][v][r];
        ss += __shfl_xor(ss, 16);
        ss += __shfl_xor(ss, 32);
        if (lg == 0) red[cg][16 * rt[v] + li] = ss;
    }
    const int esz = a.in_dt == DT_F32 ? 4 : 2, osz = a.out_dt == DT_F32 ? 4 : 2;
    const bool zvec = ((uintptr_t)a.z % (4 * esz)) == 0 && (a.ld_in % 4) == 0;
    const bool ovec = ((uintptr_t)a.out % (4 * osz)) == 0 && (a.ld_out % 4) == 0;
    __syncthreads();
#pragma unroll
    for (int v = 0; v < 2; ++v) {
        const int i = 16 * rt[v] + li, tau = t0 + c * GC_C + i;
        if (tau >= a.T) continue;
        const float tot = red[0][i] + red[1][i] + red[2][i] + red[3][i];
        const float inv = 1.0f / sqrtf(tot / (float)GC_D + 1e-6f);
        const int64_t row = (int64_t)b * a.T + tau;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int cl = 32 * cg + 16 * u + 4 * lg;
            const int64_t zi = row * a.ld_in + h * GC_D + cl, oi = row * a.ld_out + h * GC_D + cl;
            f32x4 z, y;
            if (zvec) {
                z = load_act4(a.z, a.in_dt, zi);
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) z[r] = gdn_load(a.z, a.in_dt, zi + r);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) y[r] = o[u][v][r] * inv * a.norm_w[cl + r] * silu_f(z[r]);
            if (ovec) {
                store_act4(a.out, a.out_dt, oi, y);
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) store_act(a.out, a.out_dt, oi + r, y[r]);
            }
        }
    }
}

size_t gdn_chunked_bytes_per_token(int nh) { return (size_t)nh * GR_SIZE * 4 / GC_C; }

hipError_t launch_gdn_chunked(const GdnArgs& a, void* ws, size_t ws_bytes, hipStream_t stream) {
    if (a.kd != GC_D || a.vd != GC_D || a.K < 1 || a.K > 8 || a.T < 1) return hipErrorInvalidValue;
    // tokens per segment: whole chunks whose records fit the workspace
    const size_t per_tok = (size_t)a.B * gdn_chunked_bytes_per_token(a.nh);
    int64_t seg = (int64_t)(ws_bytes / per_tok) / GC_C * GC_C;
    if (seg < GC_C) return hipErrorInvalidValue;
    seg = std::min<int64_t>(seg, ((int64_t)a.T + GC_C - 1) / GC_C * GC_C);
    float* rec = reinterpret_cast<float*>(ws);
    for (int t0 = 0; t0 < a.T; t0 += (int)seg) {
        const int len = (int)std::min<int64_t>(seg, a.T - t0);
        const int nchunk = (len + GC_C - 1) / GC_C;
        const bool last = t0 + len >= a.T;
        if (a.K == 4)
            hipLaunchKernelGGL(gdn_chunk_prep<4>, dim3(gdn_grid(a, nchunk)), dim3(GC_T), 0, stream, a, t0, nchunk, rec);
        else
            hipLaunchKernelGGL(gdn_chunk_prep<0>, dim3(gdn_grid(a, nchunk)), dim3(GC_T), 0, stream, a, t0, nchunk, rec);
        hipLaunchKernelGGL(gdn_chunk_state, dim3(gdn_grid(a, GC_D / GC_VS)), dim3(256), 0, stream, a, nchunk, rec,
                           last ? 1 : 0);
        hipLaunchKernelGGL(gdn_chunk_out, dim3(gdn_grid(a, nchunk)), dim3(512), 0, stream, a, t0, nchunk,
                           (const float*)rec);
    }
    return hipGetLastError();
}

}  // namespace qwk
