// qw_attn.hip -- gated full attention between the projections for gfx950:
// per-head RMSNorm (1 + w) of q and k, partial RoPE, the KV-cache write
// (INT8 with one scale per token and KV head, or FP32), causal GQA attention
// over the cache, and the sigmoid gate.  B sequences of T new tokens each.
//
// Math (reference CPU operator, src/backend/cpu/core/attention/
// language_full_attn.cpp:77-108,156-207; INT8 cache recipe of
// fused_kv_cache_int8_kernel, full_attention_cuda.cu:75-155):
//   q_h = rmsnorm(q_h) * (1 + q_norm_w), k_g likewise, eps 1e-6
//   RoPE on dims d < rot, pairs (d, d+1): angle = pos / theta^(d / rot)
//   K/V INT8: scale = max|x| / 127 (1 when <= 1e-8), round half away, clamp 127
//   o_h = softmax(q_h . K_g^T / sqrt(hd)) V_g over positions 0 .. pos (causal),
//   g = h / (nh / nkv); out = o * sigmoid(gate)
//
// Launches per segment of rows:
//   decode and short runs: attn_prep (norms, RoPE, cache write, normalized q to
//     the workspace), one workgroup per (key split, KV head, row)
//     (attn_decode_i8h on f16 MFMA, attn_split for an FP32 cache), attn_combine
//     (merges the splits, gate, output); a small INT8 decode step is the one
//     launch attn_decode_i8h<., true>;
//   INT8 prefill: attn_prep_rows, attn_expand (the cached codes and scales to
//     f16 MFMA operands), attn_pf (64-token query blocks, keys cut into runs of
//     equal work), attn_pf_merge; calls that do not pay for these four launches
//     (pf_pays) or whose expanded keys the workspace does not hold: attn_prep,
//     attn_prefill_i8h (16-token blocks), attn_combine;
//   FP32 prefill: attn_prep, attn_prefill (16-token blocks, keys cut into shares
//     where the blocks leave the chip idle), attn_combine.
// A token whose position lies outside the
// cache (or beyond the max_len the launch was sized for) writes nothing,
// outputs zeros and raises the context's device error flag.
#include "qw_stream.hpp"

namespace qwk {

constexpr int AT_KT = 32;  // keys per LDS tile

// FP32 MFMA 16x16x4: lane l supplies A[l%16][l/16] and B[l/16][l%16] and holds
// D[4*(l/16) + r][l%16] in element r.
__device__ __forceinline__ f32x4 at_mfma16(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ float at_load(const void* p, int dt, int64_t i) {
    return dt == DT_F32 ? reinterpret_cast<const float*>(p)[i] : load_act(p, dt, i);
}

// E consecutive elements from i; vec: the address is a multiple of E elements
template <int E>
__device__ __forceinline__ void at_load_row(const void* p, int dt, int64_t i, bool vec, float (&x)[E]) {
    if (E == 4 && vec) {
        const f32x4 v = load_act4(p, dt, i);
#pragma unroll
        for (int e = 0; e < E; ++e) x[e] = v[e];
        return;
    }
#pragma unroll
    for (int e = 0; e < E; ++e) x[e] = at_load(p, dt, i + e);
}

// v of lane l ^ OFF, for a value that the lanes l ^ 2 OFF, l ^ 4 OFF, .. already
// share (a butterfly from 32 down): register moves instead of LDS round trips
template <int OFF>
__device__ __forceinline__ float butterfly(float v) {
    const int x = __builtin_bit_cast(int, v);
    if constexpr (OFF == 32 || OFF == 16) {
        const auto s = OFF == 32 ? __builtin_amdgcn_permlane32_swap(x, x, false, false)
                                 : __builtin_amdgcn_permlane16_swap(x, x, false, false);
        // the two results hold both halves' values; the one that is not this lane's
        const bool upper = threadIdx.x & OFF;
        return __builtin_bit_cast(float, upper ? s[0] : s[1]);
    } else {
        // row_ror:8, row_ror:4 (= xor 4 where xor 8 agrees), quad_perm [2,3,0,1], [1,0,3,2]
        constexpr int CTRL = OFF == 8 ? 0x128 : OFF == 4 ? 0x124 : OFF == 2 ? 0x4E : 0xB1;
        return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, x, CTRL, 0xF, 0xF, false));
    }
}

__device__ __forceinline__ float wave_sum(float v) {
    v += butterfly<32>(v);
    v += butterfly<16>(v);
    v += butterfly<8>(v);
    v += butterfly<4>(v);
    v += butterfly<2>(v);
    return v + butterfly<1>(v);
}

__device__ __forceinline__ float wave_max(float v) {
    v = fmaxf(v, butterfly<32>(v));
    v = fmaxf(v, butterfly<16>(v));
    v = fmaxf(v, butterfly<8>(v));
    v = fmaxf(v, butterfly<4>(v));
    v = fmaxf(v, butterfly<2>(v));
    return fmaxf(v, butterfly<1>(v));
}

// Sum of squares of a lane's elements and rotation of a pair, the roundings
// spelled out: every kernel that writes cache codes has to round them alike.
template <int E>
__device__ __forceinline__ float sum_squares(const float (&x)[E]) {
    float ss = __builtin_fmaf(x[0], x[0], x[1] * x[1]);
#pragma unroll
    for (int e = 2; e < E; ++e) ss = __builtin_fmaf(x[e], x[e], ss);
    return ss;
}
__device__ __forceinline__ float rope0(float x0, float x1, float c, float s) { return __builtin_fmaf(x0, c, -(x1 * s)); }
__device__ __forceinline__ float rope1(float x0, float x1, float c, float s) { return __builtin_fmaf(x1, c, x0 * s); }

// ---------------------------------------------------------------------------
// prep: one workgroup per row with one wave per work item (nh q heads, nkv k
// heads, nkv v heads; 64 x items threads); lane l holds dims [l*E, l*E + E).
template <int HD>
__global__ __launch_bounds__(1024) void attn_prep(AttnArgs a) {
    constexpr int E = HD / 64;
    const int rl = blockIdx.x, r = a.row0 + rl;
    const int b = r / a.T, t = r % a.T;
    const int P = a.pos[b] + t;
    // a position outside the cache, or past the keys the launch was sized for
    const bool ok = P >= 0 && P < a.cap && P < a.lim;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (!ok && threadIdx.x == 0) *a.err = 1u;
    // the rotation of this position, shared by every q and k head
    __shared__ float rc[HD / 2], rs[HD / 2];
    if ((int)threadIdx.x < a.rot / 2) {
        const float freq = 1.0f / powf(a.theta, (float)(2 * threadIdx.x) / (float)a.rot);
        const float ang = (float)P * freq;
        rc[threadIdx.x] = cosf(ang);
        rs[threadIdx.x] = sinf(ang);
    }
    __syncthreads();
    const int items = a.nh + 2 * a.nkv;
    const int64_t row = (int64_t)r * a.ld_in;
    for (int it = wave; it < items; it += blockDim.x >> 6) {
        const bool isq = it < a.nh, isk = !isq && it < a.nh + a.nkv;
        const int h = isq ? it : (isk ? it - a.nh : it - a.nh - a.nkv);
        const void* src = isq ? a.q : (isk ? a.k : a.v);
        const int64_t base = row + (isq ? (int64_t)h * a.q_hs : (int64_t)h * HD) + lane * E;
        float x[E];
#pragma unroll
        for (int e = 0; e < E; ++e) x[e] = at_load(src, a.in_dt, base + e);
        if (isq || isk) {
            const float ss = wave_sum(sum_squares(x));
            const float rms = sqrtf(ss / (float)HD + 1e-6f);
            const float* w = isq ? a.qn_w : a.kn_w;
#pragma unroll
            for (int e = 0; e < E; ++e) x[e] = x[e] / rms * (1.0f + w[lane * E + e]);
#pragma unroll
            for (int e = 0; e < E; e += 2) {
                const int d = lane * E + e;
                if (d < a.rot) {
                    const float c = rc[d / 2], s = rs[d / 2];
                    const float x0 = x[e], x1 = x[e + 1];
                    x[e] = rope0(x0, x1, c, s);
                    x[e + 1] = rope1(x0, x1, c, s);
                }
            }
        }
        if (isq) {
            float* dst = a.qn + ((int64_t)rl * a.nh + h) * HD + lane * E;
#pragma unroll
            for (int e = 0; e < E; ++e) dst[e] = x[e];
            continue;
        }
        if (!ok) continue;
        const int64_t slot = ((int64_t)b * a.cap + P) * a.nkv + h;
        if (a.kv_dt == DT_I8) {
            float m = 0.0f;
#pragma unroll
            for (int e = 0; e < E; ++e) m = fmaxf(m, fabsf(x[e]));
            m = wave_max(m);
            float sc = m / 127.0f;
            sc = sc > 1e-8f ? sc : 1.0f;
            int8_t* dst = reinterpret_cast<int8_t*>(isk ? a.kc : a.vc) + slot * HD + lane * E;
#pragma unroll
            for (int e = 0; e < E; ++e) dst[e] = (int8_t)fmaxf(-127.0f, fminf(127.0f, roundf(x[e] / sc)));
            if (lane == 0) (isk ? a.ks : a.vs)[slot] = sc;
        } else {
            float* dst = reinterpret_cast<float*>(isk ? a.kc : a.vc) + slot * HD + lane * E;
#pragma unroll
            for (int e = 0; e < E; ++e) dst[e] = x[e];
        }
    }
}

// The same for attn_pf's segments, R rows per workgroup (the same values bit
// for bit; q as f16).
// The rotation's powf / cosf / sinf chain is paid once for R rows, whose loads
// are in flight under it, and rows are read and written 16 bytes per lane: 4096
// rows 33.6 -> 27.6 us.
template <int HD, int R>
__global__ __launch_bounds__(1024) void attn_prep_rows(AttnArgs a) {
    constexpr int E = HD / 64;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    __shared__ float rc[R][HD / 2], rs[R][HD / 2];
    const int items = a.nh + 2 * a.nkv, nr = min(R, a.rows - (int)blockIdx.x * R);
    const int esz = a.in_dt == DT_F32 ? 4 : 2;
    const bool vec = (((uintptr_t)a.q | (uintptr_t)a.k | (uintptr_t)a.v) % (4 * esz)) == 0 && a.ld_in % 4 == 0 && a.q_hs % 4 == 0;
    auto position = [&](int rl, int& b) {
        const int r = a.row0 + rl;
        b = r / a.T;
        return a.pos[b] + r % a.T;
    };
    // a position outside the cache, or past the keys the launch was sized for
    auto valid = [&](int P) { return P >= 0 && P < a.cap && P < a.lim; };
    for (int it0 = 0; it0 < items; it0 += blockDim.x >> 6) {
        const int it = it0 + wave;
        const bool isq = it < a.nh, isk = !isq && it < a.nh + a.nkv;
        const int h = isq ? it : (isk ? it - a.nh : it - a.nh - a.nkv);
        const void* src = isq ? a.q : (isk ? a.k : a.v);
        float x[R][E];
        if (it < items) {
#pragma unroll
            for (int i = 0; i < R; ++i) {
                const int64_t row = (int64_t)(a.row0 + (int)blockIdx.x * R + min(i, nr - 1)) * a.ld_in;
                const int64_t base = row + (isq ? (int64_t)h * a.q_hs : (int64_t)h * HD) + lane * E;
                at_load_row(src, a.in_dt, base, vec, x[i]);
            }
        }
        if (it0 == 0) {
            // the rotations of these positions, shared by every q and k head
            for (int j = threadIdx.x; j < nr * (a.rot / 2); j += blockDim.x) {
                const int i = j / (a.rot / 2), d2 = j % (a.rot / 2);
                int b;
                const int P = position(blockIdx.x * R + i, b);
                const float freq = 1.0f / powf(a.theta, (float)(2 * d2) / (float)a.rot);
                const float ang = (float)P * freq;
                rc[i][d2] = cosf(ang);
                rs[i][d2] = sinf(ang);
                if (d2 == 0 && !valid(P)) *a.err = 1u;
            }
            if (a.rot == 0 && (int)threadIdx.x < nr) {
                int b;
                if (!valid(position(blockIdx.x * R + threadIdx.x, b))) *a.err = 1u;
            }
            __syncthreads();
        }
        if (it >= items) continue;
#pragma unroll
        for (int i = 0; i < R; ++i) {
            if (i >= nr) break;
            const int rl = blockIdx.x * R + i;
            if (isq || isk) {
                const float ss = wave_sum(sum_squares(x[i]));
                const float rms = sqrtf(ss / (float)HD + 1e-6f);
                const float* w = isq ? a.qn_w : a.kn_w;
#pragma unroll
                for (int e = 0; e < E; ++e) x[i][e] = x[i][e] / rms * (1.0f + w[lane * E + e]);
#pragma unroll
                for (int e = 0; e < E; e += 2) {
                    const int d = lane * E + e;
                    if (d < a.rot) {
                        const float c = rc[i][d / 2], s = rs[i][d / 2];
                        const float x0 = x[i][e], x1 = x[i][e + 1];
                        x[i][e] = rope0(x0, x1, c, s);
                        x[i][e + 1] = rope1(x0, x1, c, s);
                    }
                }
            }
            if (isq) {
                const int64_t qo = ((int64_t)rl * a.nh + h) * HD + lane * E;
                typedef _Float16 f16e __attribute__((ext_vector_type(E)));
                f16e y;
#pragma unroll
                for (int e = 0; e < E; ++e) y[e] = (_Float16)x[i][e];
                *reinterpret_cast<f16e*>(reinterpret_cast<_Float16*>(a.qn) + qo) = y;
                continue;
            }
            int b;
            const int P = position(rl, b);
            if (!valid(P)) continue;
            const int64_t slot = ((int64_t)b * a.cap + P) * a.nkv + h;
            float m = 0.0f;
#pragma unroll
            for (int e = 0; e < E; ++e) m = fmaxf(m, fabsf(x[i][e]));
            m = wave_max(m);
            float sc = m / 127.0f;
            sc = sc > 1e-8f ? sc : 1.0f;
            typedef int8_t i8e __attribute__((ext_vector_type(E)));
            i8e y;
#pragma unroll
            for (int e = 0; e < E; ++e) y[e] = (int8_t)fmaxf(-127.0f, fminf(127.0f, roundf(x[i][e] / sc)));
            int8_t* dst = reinterpret_cast<int8_t*>(isk ? a.kc : a.vc) + slot * HD + lane * E;
            if (((uintptr_t)(isk ? a.kc : a.vc)) % E == 0) {
                *reinterpret_cast<i8e*>(dst) = y;
            } else {
#pragma unroll
                for (int e = 0; e < E; ++e) dst[e] = y[e];
            }
            if (lane == 0) (isk ? a.ks : a.vs)[slot] = sc;
        }
    }
}

template <int HD>
static void launch_prep(const AttnArgs& a, hipStream_t stream) {
    const dim3 t(64 * std::min(16, a.nh + 2 * a.nkv));
    if (a.pf_units) hipLaunchKernelGGL((attn_prep_rows<HD, 4>), dim3((a.rows + 3) / 4), t, 0, stream, a);
    else hipLaunchKernelGGL(attn_prep<HD>, dim3(a.rows), t, 0, stream, a);
}

// ---------------------------------------------------------------------------
// split: (key split s, KV head g, row rl); wave w < G handles query head g*G + w.
// The K and V tiles of 32 keys are staged in LDS once for the whole KV group:
// INT8 codes as they are (the scales multiply the score and the probability),
// FP32 values as they are; every thread issues its share of the next tile's
// loads before the current tile is computed.
template <int HD, bool I8>
struct AtTile {
    static constexpr int KROW = I8 ? HD + 4 : (HD + 4) * 4;   // K row stride, bytes (bank spread)
    static constexpr int VROW = I8 ? HD : HD * 4;             // V row stride, bytes
    static constexpr int CH = AT_KT * (I8 ? HD : HD * 4) / 16; // 16-byte chunks per K (or V) tile
    static constexpr int PER = 2 * CH / 256;                   // chunks per thread (K and V)
};

template <int HD, bool I8>
__global__ __launch_bounds__(256) void attn_split(AttnArgs a) {
    using Tl = AtTile<HD, I8>;
    constexpr int E = HD / 64, ESZ = I8 ? 1 : 4, CPR = HD * ESZ / 16;  // chunks per row
    const int s = blockIdx.x, g = blockIdx.y, rl = blockIdx.z, r = a.row0 + rl;
    const int b = r / a.T, t = r % a.T;
    const int P = a.pos[b] + t;
    const int L = (P >= 0 && P < a.cap && P < a.lim) ? P + 1 : 0;  // causal: keys 0 .. P
    const int k0 = s * a.split, k1 = min(k0 + a.split, L);
    const int G = a.nh / a.nkv;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int h = g * G + wave;
    if (k0 >= k1) {  // uniform over the workgroup
        if (L == 0 && a.nsplit == 1 && wave < G) {  // a flagged token without a combine step: zeros
            const int64_t oi = (int64_t)r * a.ld_out + (int64_t)h * HD + lane * E;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                if (a.out_dt == DT_F32) reinterpret_cast<float*>(a.out)[oi + e] = 0.0f;
                else store_act(a.out, a.out_dt, oi + e, 0.0f);
            }
        }
        return;
    }

    __shared__ __attribute__((aligned(16))) float qs[4][HD];
    __shared__ __attribute__((aligned(16))) uint8_t Kt[AT_KT * Tl::KROW];
    __shared__ __attribute__((aligned(16))) uint8_t Vt[AT_KT * Tl::VROW];
    __shared__ float ksc[AT_KT], vsc[AT_KT];

    const uint8_t* kbase = reinterpret_cast<const uint8_t*>(a.kc);
    const uint8_t* vbase = reinterpret_cast<const uint8_t*>(a.vc);
    const int64_t slot0 = (int64_t)b * a.cap * a.nkv + g;  // slot of key j: slot0 + j * nkv
    u32x4 pre[Tl::PER];
    float psc = 0.0f;
    auto issue = [&](int kt) {  // the loads of the tile starting at key kt
        const int n = min(AT_KT, k1 - kt);
#pragma unroll
        for (int i = 0; i < Tl::PER; ++i) {
            const int c = threadIdx.x + 256 * i, isv = c >= Tl::CH, cc = c - isv * Tl::CH;
            const int j = cc / CPR, part = cc % CPR;
            const int64_t slot = slot0 + (int64_t)(kt + j) * a.nkv;
            if (j < n) pre[i] = *reinterpret_cast<const u32x4*>((isv ? vbase : kbase) + slot * (HD * ESZ) + part * 16);
            else pre[i] = u32x4{0u, 0u, 0u, 0u};
        }
        if (I8 && threadIdx.x < 2 * AT_KT) {
            const int j = threadIdx.x & (AT_KT - 1);
            psc = j < n ? (threadIdx.x < AT_KT ? a.ks : a.vs)[slot0 + (int64_t)(kt + j) * a.nkv] : 0.0f;
        }
    };
    issue(k0);
    for (int e = threadIdx.x; e < G * HD; e += 256) qs[e / HD][e % HD] = a.qn[((int64_t)rl * a.nh + g * G) * HD + e];
    const float scale = 1.0f / sqrtf((float)HD);
    float m = -INFINITY, l = 0.0f, o[E];
#pragma unroll
    for (int e = 0; e < E; ++e) o[e] = 0.0f;
    const int kj = lane >> 1, half = lane & 1;  // score lane: key kj of the tile, half of the dims

    for (int kt = k0; kt < k1; kt += AT_KT) {
        const int n = min(AT_KT, k1 - kt);
        __syncthreads();  // the previous tile is consumed; qs is in place
#pragma unroll
        for (int i = 0; i < Tl::PER; ++i) {
            const int c = threadIdx.x + 256 * i, isv = c >= Tl::CH, cc = c - isv * Tl::CH;
            const int j = cc / CPR, part = cc % CPR;
            if (isv) {
                *reinterpret_cast<u32x4*>(&Vt[j * Tl::VROW + part * 16]) = pre[i];
            } else {
                uint32_t* d32 = reinterpret_cast<uint32_t*>(&Kt[j * Tl::KROW + part * 16]);
                d32[0] = pre[i][0]; d32[1] = pre[i][1]; d32[2] = pre[i][2]; d32[3] = pre[i][3];
            }
        }
        if (I8 && threadIdx.x < 2 * AT_KT) (threadIdx.x < AT_KT ? ksc : vsc)[threadIdx.x & (AT_KT - 1)] = psc;
        if (kt + AT_KT < k1) issue(kt + AT_KT);
        __syncthreads();
        if (wave < G) {
            float dot = 0.0f;
            if (kj < n) {
                const float* qr = &qs[wave][half * (HD / 2)];
                if (I8) {
                    const uint32_t* kr = reinterpret_cast<const uint32_t*>(&Kt[kj * Tl::KROW + half * (HD / 2)]);
#pragma unroll 8
                    for (int w = 0; w < HD / 8; ++w) {
                        const uint32_t c4 = kr[w];
                        const float4 qv = *reinterpret_cast<const float4*>(qr + 4 * w);
                        dot += qv.x * (float)(int8_t)(c4 & 0xff) + qv.y * (float)(int8_t)((c4 >> 8) & 0xff) +
                               qv.z * (float)(int8_t)((c4 >> 16) & 0xff) + qv.w * (float)(int8_t)(c4 >> 24);
                    }
                    dot *= ksc[kj];
                } else {
                    const float* kr = reinterpret_cast<const float*>(&Kt[kj * Tl::KROW]) + half * (HD / 2);
#pragma unroll 8
                    for (int d = 0; d < HD / 2; d += 4) {
                        const float4 kv = *reinterpret_cast<const float4*>(kr + d);
                        const float4 qv = *reinterpret_cast<const float4*>(qr + d);
                        dot += qv.x * kv.x + qv.y * kv.y + qv.z * kv.z + qv.w * kv.w;
                    }
                }
            }
            dot += __shfl_xor(dot, 1);
            const float sc = kj < n ? dot * scale : -INFINITY;
            const float mt = wave_max(sc);
            const float mn = fmaxf(m, mt);
            const float corr = __expf(m - mn);  // m = -inf on the first tile: 0
            const float p = kj < n ? __expf(sc - mn) : 0.0f;
            l = l * corr + wave_sum(half == 0 ? p : 0.0f);
            const float pv = I8 ? p * vsc[kj < n ? kj : 0] : p;  // probability times the V row's scale
#pragma unroll
            for (int e = 0; e < E; ++e) o[e] *= corr;
            for (int j = 0; j < n; ++j) {
                const float pj = __shfl(pv, 2 * j);
                if (I8 && E == 4) {
                    const uint32_t c4 = reinterpret_cast<const uint32_t*>(&Vt[j * Tl::VROW])[lane];
#pragma unroll
                    for (int e = 0; e < E; ++e) o[e] += pj * (float)(int8_t)((c4 >> (8 * e)) & 0xff);
                } else if (I8) {
#pragma unroll
                    for (int e = 0; e < E; ++e) o[e] += pj * (float)(int8_t)Vt[j * Tl::VROW + lane * E + e];
                } else {
                    const float* vr = reinterpret_cast<const float*>(&Vt[j * Tl::VROW]) + lane * E;
#pragma unroll
                    for (int e = 0; e < E; ++e) o[e] += pj * vr[e];
                }
            }
            m = mn;
        }
    }
    if (wave >= G) return;
    if (a.nsplit == 1) {  // the only split: finish the row here
        const float inv = 1.0f / l;
        const int64_t gi = (int64_t)r * a.ld_in + (int64_t)h * a.q_hs + lane * E;
        const int64_t oi = (int64_t)r * a.ld_out + (int64_t)h * HD + lane * E;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const float y = o[e] * inv * (1.0f / (1.0f + __expf(-at_load(a.gate, a.in_dt, gi + e))));
            if (a.out_dt == DT_F32) reinterpret_cast<float*>(a.out)[oi + e] = y;
            else store_act(a.out, a.out_dt, oi + e, y);
        }
        return;
    }
    float* dst = a.part + (((int64_t)rl * a.nh + h) * a.nsplit + s) * (HD + 2);
#pragma unroll
    for (int e = 0; e < E; ++e) dst[lane * E + e] = o[e];
    if (lane == 0) {
        dst[HD] = m;
        dst[HD + 1] = l;
    }
}

// ---------------------------------------------------------------------------
// combine: one workgroup of NW waves per (row, head) (NW = 1 for up to 16
// splits, else 4).  The split maxima are reduced over all threads; each wave
// then sums the partial outputs of every NW-th split, eight splits' loads in
// flight; the wave sums are merged in LDS.
// Merge of ns split partials (o, max, sum) of one (row, head) by one wave,
// in a fixed order; COH: device-coherent loads (partials written by other
// workgroups of the same launch).  Returns the unnormalized o and the sum.
template <bool COH>
__device__ __forceinline__ float part_ld(const float* p) {
    if constexpr (COH) return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else return *p;
}

template <int HD, bool COH>
__device__ __forceinline__ void merge_splits_wave(const float* pp, int ns, int lane, float (&o)[HD / 64], float& l) {
    constexpr int E = HD / 64;
    float M = -INFINITY;
    for (int s = lane; s < ns; s += 64) M = fmaxf(M, part_ld<COH>(pp + s * (HD + 2) + HD));
    M = wave_max(M);
    l = 0.0f;
    for (int s = lane; s < ns; s += 64)
        l += __expf(part_ld<COH>(pp + s * (HD + 2) + HD) - M) * part_ld<COH>(pp + s * (HD + 2) + HD + 1);
    l = wave_sum(l);
#pragma unroll
    for (int e = 0; e < E; ++e) o[e] = 0.0f;
    int s = 0;
    for (; s + 7 < ns; s += 8) {  // splits s .. s+7
        float w[8], v[8][E];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            w[u] = part_ld<COH>(pp + (s + u) * (HD + 2) + HD);
#pragma unroll
            for (int e = 0; e < E; ++e) v[u][e] = part_ld<COH>(pp + (s + u) * (HD + 2) + lane * E + e);
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const float wu = __expf(w[u] - M);
#pragma unroll
            for (int e = 0; e < E; ++e) o[e] += wu * v[u][e];
        }
    }
    for (; s < ns; ++s) {
        const float wu = __expf(part_ld<COH>(pp + s * (HD + 2) + HD) - M);
#pragma unroll
        for (int e = 0; e < E; ++e) o[e] += wu * part_ld<COH>(pp + s * (HD + 2) + lane * E + e);
    }
}

// out = o / l * sigmoid(gate) for the E dims of this lane
template <int HD>
__device__ __forceinline__ void gate_store(const AttnArgs& a, int r, int h, int lane, const float (&o)[HD / 64], float inv) {
    constexpr int E = HD / 64;
    const int64_t gi = (int64_t)r * a.ld_in + (int64_t)h * a.q_hs + lane * E;
    const int64_t oi = (int64_t)r * a.ld_out + (int64_t)h * HD + lane * E;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const float y = o[e] * inv * (1.0f / (1.0f + __expf(-at_load(a.gate, a.in_dt, gi + e))));
        if (a.out_dt == DT_F32) reinterpret_cast<float*>(a.out)[oi + e] = y;
        else store_act(a.out, a.out_dt, oi + e, y);
    }
}

// Keys per share of a query block with L keys (the FP32 query-block kernel).
__device__ __forceinline__ int block_share(const AttnArgs& a, int L) {
    return max(128, ((L + a.nsplit - 1) / a.nsplit + AT_KT - 1) / AT_KT * AT_KT);
}

// DC > 1 (many splits): blockIdx.z takes HD/DC of the head's dims, so more
// workgroups share the split partials' reads (each recomputes M and l from
// the splits' two floats).
template <int HD, int NW, int DC = 1>
__global__ __launch_bounds__(64 * NW) void attn_combine(AttnArgs a) {
    static_assert(DC == 1 || NW > 1, "dim chunks with the multi-wave merge");
    constexpr int E = HD / 64 / DC;  // dims per lane
    const int d0 = (int)blockIdx.z * (HD / DC);
    const int rl = blockIdx.x, h = blockIdx.y, r = a.row0 + rl;
    const int b = r / a.T, t = r % a.T;
    const int P = a.pos[b] + t;
    const int L = (P >= 0 && P < a.cap && P < a.lim) ? P + 1 : 0;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    int split = a.split;
    if (a.blk) {  // cut by blocks: the keys of this row's block
        const int last = min(a.tb + (t - a.tb) / a.blk * a.blk + a.blk, a.tb + a.ntok) - 1;
        const int Lb = P - t >= 0 ? min(P - t + last, min(a.cap, a.lim) - 1) + 1 : 0;
        split = block_share(a, Lb);
        if (Lb <= split) return;  // one share: the row is written
    }
    const int ns = (L + split - 1) / split;
    const float* pp = a.part + ((int64_t)rl * a.nh + h) * a.nsplit * (HD + 2);
    __shared__ float red[2][NW];
    __shared__ __attribute__((aligned(16))) float osum[NW][HD / DC];
    if constexpr (NW == 1) {
        float o[E], l;
        merge_splits_wave<HD, false>(pp, ns, lane, o, l);
        gate_store<HD>(a, r, h, lane, o, L > 0 ? 1.0f / l : 0.0f);
        return;
    }
    float M = -INFINITY;
    for (int s = threadIdx.x; s < ns; s += 64 * NW) M = fmaxf(M, pp[s * (HD + 2) + HD]);
    M = wave_max(M);
    if (NW > 1) {
        if (lane == 0) red[0][wave] = M;
        __syncthreads();
        M = red[0][0];
#pragma unroll
        for (int w = 1; w < NW; ++w) M = fmaxf(M, red[0][w]);
    }
    float l = 0.0f;
    for (int s = threadIdx.x; s < ns; s += 64 * NW) l += __expf(pp[s * (HD + 2) + HD] - M) * pp[s * (HD + 2) + HD + 1];
    l = wave_sum(l);
    if (NW > 1 && lane == 0) red[1][wave] = l;
    float o[E];
#pragma unroll
    for (int e = 0; e < E; ++e) o[e] = 0.0f;
    int s = wave;
    for (; s + 7 * NW < ns; s += 8 * NW) {  // splits s, s+NW, ..., s+7NW
        float w[8], v[8][E];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            w[u] = pp[(s + NW * u) * (HD + 2) + HD];
#pragma unroll
            for (int e = 0; e < E; ++e) v[u][e] = pp[(s + NW * u) * (HD + 2) + d0 + lane * E + e];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const float wu = __expf(w[u] - M);
#pragma unroll
            for (int e = 0; e < E; ++e) o[e] += wu * v[u][e];
        }
    }
    for (; s < ns; s += NW) {
        const float wu = __expf(pp[s * (HD + 2) + HD] - M);
#pragma unroll
        for (int e = 0; e < E; ++e) o[e] += wu * pp[s * (HD + 2) + d0 + lane * E + e];
    }
    if (NW > 1) {
#pragma unroll
        for (int e = 0; e < E; ++e) osum[wave][lane * E + e] = o[e];
        __syncthreads();
        if (wave != 0) return;
        l = red[1][0];
#pragma unroll
        for (int w = 1; w < NW; ++w) l += red[1][w];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            float t = 0.0f;
#pragma unroll
            for (int w = 0; w < NW; ++w) t += osum[w][lane * E + e];
            o[e] = t;
        }
    }
    const float inv = L > 0 ? 1.0f / l : 0.0f;
    const int64_t gi = (int64_t)r * a.ld_in + (int64_t)h * a.q_hs + d0 + lane * E;
    const int64_t oi = (int64_t)r * a.ld_out + (int64_t)h * HD + d0 + lane * E;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int d = lane * E + e;
        const float y = o[e] * inv * (1.0f / (1.0f + __expf(-at_load(a.gate, a.in_dt, gi + e))));
        if (a.out_dt == DT_F32) reinterpret_cast<float*>(a.out)[oi + e] = y;
        else store_act(a.out, a.out_dt, oi + e, y);
    }
}

// Gate and output of one query's row of a 16-token block: acc[dt] element rr is
// dim 16 dt + 4 lg + rr of row r, head h.  Four dims per access where the
// alignment allows: by elements, the unrolled type tests made the INT8 kernel 29 KB,
// and a call of a few workgroups waited for its instructions (INT8, BF16 out, one
// split: 61 tokens 30.2 -> 19.0 us, 16 x 100 49.9 -> 36.6).
template <int HD>
__device__ __forceinline__ void tile_gate_store(const AttnArgs& a, const f32x4 (&acc)[HD / 16], float inv, int64_t r, int h,
                                                int lg) {
    constexpr int DT = HD / 16;
    const int esz = a.in_dt == DT_F32 ? 4 : 2, osz = a.out_dt == DT_F32 ? 4 : 2;
    const bool vec = ((uintptr_t)a.gate % (4 * esz)) == 0 && a.ld_in % 4 == 0 && a.q_hs % 4 == 0 &&
                     ((uintptr_t)a.out % (4 * osz)) == 0 && a.ld_out % 4 == 0;
    const int64_t gi = r * a.ld_in + (int64_t)h * a.q_hs + 4 * lg, oi = r * a.ld_out + (int64_t)h * HD + 4 * lg;
    if (vec) {
#pragma unroll
        for (int d0 = 0; d0 < DT; d0 += 4) {
            f32x4 gt[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) gt[e] = load_act4(a.gate, a.in_dt, gi + 16 * (d0 + e));
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                f32x4 y;
#pragma unroll
                for (int rr = 0; rr < 4; ++rr) y[rr] = acc[d0 + e][rr] * inv * (1.0f / (1.0f + __expf(-gt[e][rr])));
                store_act4(a.out, a.out_dt, oi + 16 * (d0 + e), y);
            }
        }
        return;
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr)
            store_act(a.out, a.out_dt, oi + 16 * dt + rr,
                      acc[dt][rr] * inv * (1.0f / (1.0f + __expf(-at_load(a.gate, a.in_dt, gi + 16 * dt + rr)))));
}

// ---------------------------------------------------------------------------
// prefill: (16-token query block, KV head g, sequence b); wave w handles query
// head g*G + w for the 16 tokens of the block, all on FP32 MFMA (16x16x4):
//   S^T = K Q^T (32 keys x 16 queries per tile; Q in registers as the B
//   operand), causal mask, online softmax per query column, O^T += V^T P^T
//   (P^T is the score tile's own D layout: the B operand needs no shuffle).
// K and V tiles of 32 keys of the FP32 cache are staged in LDS once for the KV
// group, each under the other's product.
// Bound: the FP32 matrix cores (256 MFMAs of 32 cycles per wave and tile).  A
// block's keys are cut into up to a.nsplit equal shares (at least 128 keys; the
// number is chosen for about 2.5 workgroups per CU, two of which are resident),
// merged by attn_combine: without, 2 x 600 tokens make 152 workgroups, one per CU and
// the longest alone at the end (317 -> 138 us, and 15 for the merge; without the cut 25.6 -> 15.7 us
// at 8 x 21 tokens, from the V rows spread over the LDS banks and 16-byte gates).
template <int HD>
__global__ __launch_bounds__(256, 2) void attn_prefill(AttnArgs a) {
    constexpr int ROW = HD + 4;                // LDS row stride, floats (bank spread)
    constexpr int PER = AT_KT * HD / 4 / 256;  // 16-byte chunks of a K (or V) tile per thread
    constexpr int KB = HD / 16, DT = HD / 16;
    // shares outermost: those that short sequences do not have come last, and the
    // first ones spread over all XCDs (workgroup ids mod 8)
    const int qb = blockIdx.x, sp = blockIdx.z / a.nb, g = blockIdx.y, b = a.b0 + blockIdx.z % a.nb;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
    const int G = a.nh / a.nkv;
    const int h = g * G + min(wave, G - 1);
    const int tok0 = a.tb + qb * 16;
    const int P0 = a.pos[b];
    const int nq = min(16, a.tb + a.ntok - tok0);          // valid queries of the block
    const int plast = P0 + tok0 + nq - 1;                  // last query position
    const int pend = min(a.cap, a.lim);       // positions must stay below this
    const int L = P0 >= 0 ? min(plast, pend - 1) + 1 : 0;  // keys 0 .. last valid query position
    const int qpos = P0 + tok0 + li;                       // this lane's query position
    const bool qvalid = li < nq && P0 >= 0 && qpos < pend; // an invalid query outputs zeros
    // this workgroup's share of the keys: [k0, k1)
    const int share = block_share(a, L), k0 = sp * share, k1 = min(k0 + share, L);
    if (k0 >= k1 && sp > 0) return;  // uniform; the first share of a flagged block still writes zeros
    const bool lone = L <= share;

    __shared__ __attribute__((aligned(16))) float Kt[AT_KT * ROW], Vt[AT_KT * ROW];

    const int64_t slot0 = (int64_t)b * a.cap * a.nkv + g;
    // one register set for both: K of the next tile is on its way under the
    // V product, V under the scores
    f32x4 pre[PER];
    auto issue = [&](const void* base, int kt) {
        const int n = min(AT_KT, k1 - kt);
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int c = threadIdx.x + 256 * i, j = c / (HD / 4), part = c % (HD / 4);
            pre[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            if (j < n) pre[i] = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(base) + (slot0 + (int64_t)(kt + j) * a.nkv) * HD + part * 4);
        }
    };
    auto stage = [&](float* tile) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int c = threadIdx.x + 256 * i, j = c / (HD / 4), part = c % (HD / 4);
            *reinterpret_cast<f32x4*>(&tile[j * ROW + part * 4]) = pre[i];
        }
    };
    if (k0 < k1) issue(a.kc, k0);

    // Q block of this wave's head in registers: lane (lg, li) holds Q[li][16kb + 4lg + q]
    f32x4 qr[KB];
    {
        const int64_t row = (int64_t)b * a.T + tok0 + li - a.row0;  // segment-local row
        const float* qp = a.qn + (row * a.nh + h) * HD + 4 * lg;
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) qr[kb] = li < nq ? *reinterpret_cast<const f32x4*>(qp + 16 * kb) : f32x4{0, 0, 0, 0};
    }
    const float scale = 1.0f / sqrtf((float)HD);
    f32x4 acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) acc[dt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    float m = -INFINITY, l = 0.0f;

    for (int kt = k0; kt < k1; kt += AT_KT) {
        stage(Kt);  // (the waves are past the previous scores)
        issue(a.vc, kt);
        __syncthreads();
        // S^T for keys kt + 16*sub + (4lg + r), queries li
        f32x4 pb[2];
        float corr = 1.0f;
        if (wave < G) {
            f32x4 sc[2];
#pragma unroll
            for (int sub = 0; sub < 2; ++sub) {
                f32x4 sacc = {0.0f, 0.0f, 0.0f, 0.0f};
                const float* kr = &Kt[(16 * sub + li) * ROW + 4 * lg];  // A operand row: key, k = dim
#pragma unroll
                for (int kb = 0; kb < KB; ++kb) {
                    const f32x4 k4 = *reinterpret_cast<const f32x4*>(kr + 16 * kb);
#pragma unroll
                    for (int q = 0; q < 4; ++q) sacc = at_mfma16(k4[q], qr[kb][q], sacc);
                }
                sc[sub] = sacc;
            }
            // scale, mask, running max per query column li
            float mt = -INFINITY;
#pragma unroll
            for (int sub = 0; sub < 2; ++sub)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int kp = kt + 16 * sub + 4 * lg + r;
                    const float v = qvalid && kp <= qpos && kp < k1 ? sc[sub][r] * scale : -INFINITY;
                    sc[sub][r] = v;
                    mt = fmaxf(mt, v);
                }
            mt = fmaxf(mt, __shfl_xor(mt, 16));
            mt = fmaxf(mt, __shfl_xor(mt, 32));
            const float mn = fmaxf(m, mt);
            corr = mn == -INFINITY ? 1.0f : __expf(m - mn);
            float ps = 0.0f;
#pragma unroll
            for (int sub = 0; sub < 2; ++sub)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float p = mn == -INFINITY ? 0.0f : __expf(sc[sub][r] - mn);
                    ps += p;
                    pb[sub][r] = p;  // B operand of P V: (key 4lg+r, query li)
                }
            ps += __shfl_xor(ps, 16);
            ps += __shfl_xor(ps, 32);
            l = l * corr + ps;
            m = mn;
        }
        stage(Vt);  // (the waves are past the previous V product)
        if (kt + AT_KT < k1) issue(a.kc, kt + AT_KT);
        __syncthreads();
        if (wave < G) {
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) acc[dt] = acc[dt] * corr;
            // O^T[d][query] += V^T[d][key] P^T[key][query]
#pragma unroll
            for (int sub = 0; sub < 2; ++sub)
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        acc[dt] = at_mfma16(Vt[(16 * sub + 4 * lg + q) * ROW + 16 * dt + li], pb[sub][q], acc[dt]);
        }
    }
    if (wave >= G || li >= nq) return;
    // acc[dt] lane (lg, li) element r: O^T[16dt + 4lg + r][query li]
    const int64_t r = (int64_t)b * a.T + tok0 + li;
    if (!lone) {  // a partial (o, max, sum) for the combine kernel
        if (!qvalid || qpos < k0) return;  // never read for this query
        float* dst = a.part + (((r - a.row0) * a.nh + h) * a.nsplit + sp) * (HD + 2);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) dst[16 * dt + 4 * lg + rr] = acc[dt][rr];
        if (lg == 0) {
            dst[HD] = m;
            dst[HD + 1] = l;
        }
        return;
    }
    tile_gate_store<HD>(a, acc, L > 0 && l > 0.0f ? 1.0f / l : 0.0f, r, h, lg);
}

// ---------------------------------------------------------------------------
// prefill over an INT8 cache on f16 MFMA (16x16x16): the cached codes are
// integers of at most 127 in magnitude, exact in f16, and their scales are
// applied in FP32 (to the scores, and to the probabilities before P V), so
// only q and p are rounded to f16 (relative 2^-11).  Same work decomposition
// as attn_prefill; each tile is converted to f16 once as it is staged (K by
// rows, V transposed, VhT[d][key], built from 4-key x 4-dim blocks), so the
// MFMA operands are single 64-bit LDS reads.
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));

// Four signed INT8 codes to f16 without conversions: each byte u = c + 128
// is placed under the f16 exponent of 1024 (bits 0x6400 | u = 1024 + u) by a
// byte permute, then one packed f16 subtraction of 1152 leaves c (exact).
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f16x4 i8x4_to_h4(uint32_t c4) {
    const uint32_t u = c4 ^ 0x80808080u;
    const uint32_t lo = __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u);
    const uint32_t hi = __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u);
    const f16x2 off = {(_Float16)1152.0f, (_Float16)1152.0f};
    const f16x2 x = __builtin_bit_cast(f16x2, lo) - off, y = __builtin_bit_cast(f16x2, hi) - off;
    return f16x4{x[0], x[1], y[0], y[1]};
}

// 4x4 byte transpose: byte q of o[e] = byte e of w[q] (four keys' codes of one
// dim from four keys' rows of four dims)
__device__ __forceinline__ void transpose4x4(const uint32_t w[4], uint32_t o[4]) {
    const uint32_t t0 = __builtin_amdgcn_perm(w[1], w[0], 0x05010400u);
    const uint32_t t1 = __builtin_amdgcn_perm(w[3], w[2], 0x05010400u);
    const uint32_t t2 = __builtin_amdgcn_perm(w[1], w[0], 0x07030602u);
    const uint32_t t3 = __builtin_amdgcn_perm(w[3], w[2], 0x07030602u);
    o[0] = __builtin_amdgcn_perm(t1, t0, 0x05040100u);
    o[1] = __builtin_amdgcn_perm(t1, t0, 0x07060302u);
    o[2] = __builtin_amdgcn_perm(t3, t2, 0x05040100u);
    o[3] = __builtin_amdgcn_perm(t3, t2, 0x07060302u);
}

template <int HD>
__global__ __launch_bounds__(256) void attn_prefill_i8h(AttnArgs a) {
    constexpr int KB = HD / 16, DT = HD / 16;
    constexpr int KHP = HD + 8;           // f16 K row stride (elements)
    constexpr int VHP = AT_KT + 4;        // f16 V^T row stride (elements)
    constexpr int KCH = AT_KT * HD / 16;  // 16-code chunks of the K tile
    constexpr int KPER = KCH / 256;       // per thread
    constexpr int VBL = AT_KT * HD / 16;  // 4-key x 4-dim blocks of the V tile
    constexpr int VPER = VBL / 256;
    constexpr int KT4 = AT_KT / 4;        // lanes take consecutive 4-key groups: conflict-free V^T stores
    const int qb = blockIdx.x / a.nsplit, sp = blockIdx.x % a.nsplit, g = blockIdx.y, b = a.b0 + blockIdx.z;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
    const int G = a.nh / a.nkv;
    const int h = g * G + min(wave, G - 1);
    const int tok0 = a.tb + qb * 16;
    const int P0 = a.pos[b];
    const int nq = min(16, a.tb + a.ntok - tok0);
    const int plast = P0 + tok0 + nq - 1;
    const int pend = min(a.cap, a.lim);
    const int L = P0 >= 0 ? min(plast, pend - 1) + 1 : 0;
    const int qpos = P0 + tok0 + li;
    const bool qvalid = li < nq && P0 >= 0 && qpos < pend;
    // this workgroup's keys: [k0, k1) of the block's causal range
    const int k0 = sp * a.split, k1 = min(k0 + a.split, L);
    if (k0 >= k1 && !(k0 == 0 && a.nsplit == 1)) return;  // uniform; a lone split still writes zeros

    __shared__ __attribute__((aligned(16))) _Float16 Kh[AT_KT * KHP];
    __shared__ __attribute__((aligned(16))) _Float16 VhT[HD * VHP];
    __shared__ float ksc[AT_KT], vsc[AT_KT];

    const uint8_t* kbase = reinterpret_cast<const uint8_t*>(a.kc);
    const uint8_t* vbase = reinterpret_cast<const uint8_t*>(a.vc);
    const int64_t slot0 = (int64_t)b * a.cap * a.nkv + g;
    u32x4 kpre[KPER];
    uint32_t vpre[VPER][4];
    float psc = 0.0f;
    auto issue = [&](int kt) {
        const int n = min(AT_KT, k1 - kt);
#pragma unroll
        for (int i = 0; i < KPER; ++i) {  // K: 16 consecutive codes of one key
            const int c = threadIdx.x + 256 * i, j = c / (HD / 16), part = c % (HD / 16);
            // keys past the range read the range's last key: finite, masked out later
            kpre[i] = *reinterpret_cast<const u32x4*>(kbase + (slot0 + (int64_t)(kt + min(j, n - 1)) * a.nkv) * HD + part * 16);
        }
#pragma unroll
        for (int i = 0; i < VPER; ++i) {  // V: 4 dims of 4 consecutive keys
            const int blk = threadIdx.x + 256 * i, k4 = blk % (KT4), d4 = blk / (KT4);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int j = 4 * k4 + q;
                vpre[i][q] = *reinterpret_cast<const uint32_t*>(vbase + (slot0 + (int64_t)(kt + min(j, n - 1)) * a.nkv) * HD + 4 * d4);
            }
        }
        if (threadIdx.x < 2 * AT_KT) {
            const int j = threadIdx.x & (AT_KT - 1);
            psc = (threadIdx.x < AT_KT ? a.ks : a.vs)[slot0 + (int64_t)(kt + min(j, n - 1)) * a.nkv];
        }
    };

    f16x4 qh[KB];
    {
        const int64_t row = (int64_t)b * a.T + tok0 + li - a.row0;
        const float* qp = a.qn + (row * a.nh + h) * HD + 4 * lg;
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
            const f32x4 v = li < nq ? *reinterpret_cast<const f32x4*>(qp + 16 * kb) : f32x4{0, 0, 0, 0};
#pragma unroll
            for (int q = 0; q < 4; ++q) qh[kb][q] = (_Float16)v[q];
        }
    }
    if (k0 < k1) issue(k0);  // after the q loads, so that waiting for q does not wait for the tile
    const float scale = 1.0f / sqrtf((float)HD);
    f32x4 acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) acc[dt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    float m = -INFINITY, l = 0.0f;

    for (int kt = k0; kt < k1; kt += AT_KT) {
        __syncthreads();
        // stage the tile as f16, converting every code once
#pragma unroll
        for (int i = 0; i < KPER; ++i) {
            const int c = threadIdx.x + 256 * i, j = c / (HD / 16), part = c % (HD / 16);
            f16x4 hv[4];
#pragma unroll
            for (int w = 0; w < 4; ++w) hv[w] = i8x4_to_h4(kpre[i][w]);
            u32x4* dst = reinterpret_cast<u32x4*>(&Kh[j * KHP + part * 16]);
            dst[0] = __builtin_bit_cast(u32x4, __builtin_shufflevector(hv[0], hv[1], 0, 1, 2, 3, 4, 5, 6, 7));
            dst[1] = __builtin_bit_cast(u32x4, __builtin_shufflevector(hv[2], hv[3], 0, 1, 2, 3, 4, 5, 6, 7));
        }
#pragma unroll
        for (int i = 0; i < VPER; ++i) {
            const int blk = threadIdx.x + 256 * i, k4 = blk % (KT4), d4 = blk / (KT4);
            uint32_t tw[4];
            transpose4x4(vpre[i], tw);  // tw[e]: dim 4*d4 + e of keys 4*k4 .. 4*k4+3
#pragma unroll
            for (int e = 0; e < 4; ++e) *reinterpret_cast<f16x4*>(&VhT[(4 * d4 + e) * VHP + 4 * k4]) = i8x4_to_h4(tw[e]);
        }
        if (threadIdx.x < 2 * AT_KT) (threadIdx.x < AT_KT ? ksc : vsc)[threadIdx.x & (AT_KT - 1)] = psc;
        if (kt + AT_KT < k1) issue(kt + AT_KT);
        __syncthreads();
        if (wave >= G) continue;
        f32x4 sc[2];
#pragma unroll
        for (int sub = 0; sub < 2; ++sub) {
            f32x4 sacc = {0.0f, 0.0f, 0.0f, 0.0f};
            const _Float16* kr = &Kh[(16 * sub + li) * KHP + 4 * lg];
#pragma unroll
            for (int kb = 0; kb < KB; ++kb)
                sacc = __builtin_amdgcn_mfma_f32_16x16x16f16(*reinterpret_cast<const f16x4*>(kr + 16 * kb), qh[kb], sacc, 0, 0, 0);
            sc[sub] = sacc;
        }
        float mt = -INFINITY;
#pragma unroll
        for (int sub = 0; sub < 2; ++sub)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int kl = 16 * sub + 4 * lg + r, kp = kt + kl;
                float v = sc[sub][r] * scale * ksc[kl];
                v = (qvalid && kp <= qpos && kp < k1) ? v : -INFINITY;
                sc[sub][r] = v;
                mt = fmaxf(mt, v);
            }
        mt = fmaxf(mt, __shfl_xor(mt, 16));
        mt = fmaxf(mt, __shfl_xor(mt, 32));
        const float mn = fmaxf(m, mt);
        const float corr = mn == -INFINITY ? 1.0f : __expf(m - mn);
        float ps = 0.0f;
        f16x4 pb[2];
#pragma unroll
        for (int sub = 0; sub < 2; ++sub)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int kl = 16 * sub + 4 * lg + r;
                const float p = mn == -INFINITY ? 0.0f : __expf(sc[sub][r] - mn);
                ps += p;
                pb[sub][r] = (_Float16)(p * vsc[kl]);
            }
        ps += __shfl_xor(ps, 16);
        ps += __shfl_xor(ps, 32);
        l = l * corr + ps;
        m = mn;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) acc[dt] = acc[dt] * corr;
#pragma unroll
        for (int sub = 0; sub < 2; ++sub)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
                acc[dt] = __builtin_amdgcn_mfma_f32_16x16x16f16(
                    *reinterpret_cast<const f16x4*>(&VhT[(16 * dt + li) * VHP + 16 * sub + 4 * lg]), pb[sub], acc[dt],
                    0, 0, 0);
    }
    if (wave >= G || li >= nq) return;
    const int64_t r = (int64_t)b * a.T + tok0 + li;
    if (a.nsplit > 1) {  // a partial (o, max, sum) for the combine kernel
        if (!qvalid || qpos < k0) return;  // never read for this query
        float* dst = a.part + (((r - a.row0) * a.nh + h) * a.nsplit + sp) * (HD + 2);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int rr = 0; rr < 4; ++rr) dst[16 * dt + 4 * lg + rr] = acc[dt][rr];
        if (lg == 0) {
            dst[HD] = m;
            dst[HD + 1] = l;
        }
        return;
    }
    tile_gate_store<HD>(a, acc, L > 0 && l > 0.0f ? 1.0f / l : 0.0f, r, h, lg);
}

// ---------------------------------------------------------------------------
// prefill over an INT8 cache, long token runs: three launches after the
// segment's attn_prep.
//
//   attn_expand   (32-key tile, KV head, sequence): the cached codes as f16
//                 MFMA operands, once per call instead of once per query
//                 block: K as the A tiles of S^T = K Q^T, V^T as the A tiles of
//                 O^T = V^T P^T, 1 KB units in the order the consumer's waves
//                 read them, and per tile the 32 K scales (times log2(e) /
//                 sqrt(head dim)) and the 32 V scales;
//   attn_pf       (unit): a 64-token query block of a KV group, all its keys or,
//                 for long blocks, a share of them;
//   attn_pf_merge (block, 16 tokens of a head, sequence): merges the shares,
//                 gate, output.
//
// Units.  A triangle of blocks has no balanced split by blocks: a block is cut
// into n = ceil(tiles / ut) units, ut = 1.3 times the tiles per CU -- about one
// unit per CU at 4096 tokens, no cut where the blocks alone far outnumber the
// CUs -- and the units are dealt longest block first (1.1 times: 363 units, a
// second round for some CUs, 142 against 118 us).  Where the blocks are
// fewer than the CUs (pf_lone 0), uncut blocks leave a partial too: their gate
// reads miss every cache and take 20 us in one workgroup, but are hidden by the
// many of the merge (777 tokens: 24 instead of 42 us).  Only the device knows the
// positions, so the plan is made there; the grid is an upper bound whose
// superfluous workgroups come last (empty ones between the others hold up the
// in-order dispatch: with up to 4 key splits per block in the grid, half the
// CUs idled on average at 4096 tokens, 184 us).
//
// attn_pf: 2 G waves, wave (tg, w) handles the 32 tokens tg of the block for
// query head w of the group.  Per 32-key tile: S^T (32 keys x 32 queries,
// 32x32x16 f16 MFMA, Q in registers), online softmax per query column in FP32,
// O^T += V^T P^T, where P^T is the score tile's own register layout (V's keys
// are stored in that order).  Tiles reach LDS by direct loads two tiles ahead
// (four stages), one barrier per tile.  The two waves of a SIMD belong to the
// two token groups; group 1 runs half a tile late, so that one wave's softmax
// runs under the other's MFMAs -- in step they take turns to idle both units.
//
// Bound: the f16 matrix cores (4 HD flop per key and query), closely followed
// by the softmax's VALU work and the LDS reads of the operands (32 KB per wave
// and tile against 1024 MFMA cycles; 16-query tiles would read twice that);
// 64-token blocks keep the tile traffic from L2 at 256 flop per byte.
// The running maximum is only raised when a tile exceeds it by more than a
// factor of 2^4 (the exponentials stay below 2^4, far inside f16's range while
// V's scales are below 1024; above, every increase counts), which leaves the
// 128-register accumulator unscaled for nearly all tiles.  It is kept a whole
// number (log2), so that neither it nor the cut into units changes the f16
// rounding of the probabilities (down to f16's subnormals).
// Measured, INT8 cache, one sequence, 4096 tokens from position 0: the call 809 ->
// 159 us; in a kernel trace, which adds up to ~1 us to a launch, attn_pf 104, prep 28,
// merge 26, expand 6 us (the 16-token kernels: 759, 40, 43, -).  777 tokens: 24 + 11 +
// 13 + 5 us.
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ uint32_t pf_uni(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

__device__ __forceinline__ PfSeq pf_seq(const AttnArgs& a, int P0) { return PfSeq(min(a.cap, a.lim), a.tb, a.ntok, P0); }

__device__ __forceinline__ uint32_t pf_sum(uint32_t v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return pf_uni(v);
}

// Longest unit, in tiles, of the segment's plan.  All lanes take part.
__device__ __forceinline__ uint32_t pf_longest(const AttnArgs& a) {
    uint32_t v = 0;
    for (int i = threadIdx.x & 63; i < a.nb; i += 64) v += pf_seq(a, a.pos[a.b0 + i]).all();
    return pf_unit_tiles(pf_sum(v) * a.nkv, a.pf_units);
}

// Whether a block's units leave partials
__device__ __forceinline__ bool pf_cut(const AttnArgs& a, uint32_t n) { return n > 1 || !a.pf_lone; }

// Units, and units that leave partials, of the blocks before block `end` of a
// sequence: summed over the lanes of the wave, or by each lane for itself.
template <bool WAVE>
__device__ __forceinline__ void pf_count(const AttnArgs& a, const PfSeq& q, uint32_t ut, uint32_t end, uint32_t& units,
                                         uint32_t& cut) {
    uint32_t u = 0, k = 0;
    for (uint32_t j = WAVE ? threadIdx.x & 63 : 0; j < end; j += WAVE ? 64 : 1) {
        const uint32_t n = pf_shares(q, ut, j);
        u += n;
        k += pf_cut(a, n) ? n : 0u;
    }
    units = WAVE ? pf_sum(u) : u;
    cut = WAVE ? pf_sum(k) : k;
}

// Inclusive prefix sums over the lanes of a wave.
__device__ __forceinline__ void pf_scan(uint32_t& x, uint32_t& y) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t o = __shfl_up(x, off), k = __shfl_up(y, off);
        if (lane >= off) {
            x += o;
            y += k;
        }
    }
}

// The sequence of unit u (of one KV head), u then relative to it, and the
// shares of cut blocks before it; a.nb if there is none.  The lanes take
// sequences where they outnumber the blocks, else the blocks of one after another.
__device__ __forceinline__ int pf_seq_of(const AttnArgs& a, uint32_t ut, uint32_t& u, uint32_t& slot) {
    const int lane = threadIdx.x & 63;
    uint32_t units = 0, cut = 0;
    if (a.nb == 1) return 0;
    if (a.nb > (a.ntok + PF_Q - 1) / PF_Q) {
        for (int i0 = 0; i0 < a.nb; i0 += 64) {
            units = cut = 0;
            if (i0 + lane < a.nb) {
                const PfSeq q = pf_seq(a, a.pos[a.b0 + i0 + lane]);
                pf_count<false>(a, q, ut, q.nblk, units, cut);
            }
            uint32_t iu = units, ic = cut;
            pf_scan(iu, ic);
            const uint64_t hit = __ballot(iu > u);
            if (hit) {
                const int first = __ffsll((unsigned long long)hit) - 1;
                u -= pf_uni(__shfl(iu - units, first));
                slot += pf_uni(__shfl(ic - cut, first));
                return i0 + first;
            }
            u -= pf_uni(__shfl(iu, 63));
            slot += pf_uni(__shfl(ic, 63));
        }
        return a.nb;
    }
    int bl = 0;
    for (; bl < a.nb; ++bl) {
        const PfSeq q = pf_seq(a, __builtin_amdgcn_readfirstlane(a.pos[a.b0 + bl]));
        pf_count<true>(a, q, ut, q.nblk, units, cut);
        if (u < units) break;
        u -= units;
        slot += cut;
    }
    return bl;
}

// floats of a share's partial: 64 rows of HD per head of the group, then (max, sum) per row
__device__ __forceinline__ int64_t pf_piece(int G, int HD) { return (int64_t)G * PF_Q * (HD + 2); }

template <int HD>
__global__ __launch_bounds__(256) void attn_expand(AttnArgs a) {
    constexpr int KS = HD / 16, DT = HD / 32;
    const int tile = blockIdx.x, g = blockIdx.y, b = a.b0 + blockIdx.z;
    const int P0 = a.pos[b];
    const int total = min(P0 + a.tb + a.ntok, min(a.cap, a.lim));  // keys in the cache after attn_prep
    const int k0 = tile * PF_KT;
    if (P0 < 0 || k0 >= total) return;
    const int nk = min(PF_KT, total - k0);
    __shared__ __attribute__((aligned(16))) uint8_t Vt[PF_KT * HD];
    const int64_t pair = (int64_t)blockIdx.z * a.nkv + g;
    const int64_t slot0 = ((int64_t)b * a.cap + k0) * a.nkv + g;
    const uint8_t* kbase = reinterpret_cast<const uint8_t*>(a.kc);
    const uint8_t* vbase = reinterpret_cast<const uint8_t*>(a.vc);
    uint8_t* kx = a.kx + (pair * a.pf_keys + k0) * (HD * 2);
    uint8_t* vx = a.vx + (pair * a.pf_keys + k0) * (HD * 2);
    for (int c = threadIdx.x; c < PF_KT * HD / 16; c += 256) {
        const int key = c / (HD / 16), part = c % (HD / 16);
        u32x4 v = {0u, 0u, 0u, 0u};
        if (key < nk) v = *reinterpret_cast<const u32x4*>(vbase + (slot0 + (int64_t)key * a.nkv) * HD + part * 16);
        *reinterpret_cast<u32x4*>(&Vt[key * HD + part * 16]) = v;
    }
    // K: unit ks, lane l: dims 16 ks + 8 (l / 32) .. +7 of key l % 32
    for (int c = threadIdx.x; c < KS * 64; c += 256) {
        const int ks = c >> 6, key = c & 31, hi = (c >> 5) & 1;
        u32x2 w = {0u, 0u};
        if (key < nk) w = *reinterpret_cast<const u32x2*>(kbase + (slot0 + (int64_t)key * a.nkv) * HD + ks * 16 + hi * 8);
        const f16x4 x = i8x4_to_h4(w[0]), y = i8x4_to_h4(w[1]);
        *reinterpret_cast<f16x8*>(kx + c * 16) = __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7);
    }
    if (threadIdx.x < 64) {
        const int key = threadIdx.x & 31;
        const bool isv = threadIdx.x >= 32;
        float v = key < nk ? (isv ? a.vs : a.ks)[slot0 + (int64_t)key * a.nkv] : 0.0f;
        // the V scales' maximum decides how far the running maximum may lag
        float big = isv ? v : 0.0f;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) big = fmaxf(big, __shfl_xor(big, off));
        if (!isv) v *= 1.44269504f / sqrtf((float)HD);
        float* sx = a.sx + (pair * (a.pf_keys / PF_KT) + tile) * PF_SC;
        sx[threadIdx.x] = v;
        if (threadIdx.x == 0) sx[64] = big < 1024.0f ? 4.0f : 0.0f;
    }
    __syncthreads();
    // V: unit (m, dt), lane l: dim 32 dt + l % 32 of the keys that lane half
    // l / 32 holds of a score tile's rows 16 m .. 16 m + 15
    for (int c = threadIdx.x; c < 2 * DT * 64; c += 256) {
        const int m = c / (DT * 64), d = (c >> 6) % DT * 32 + (c & 31), hi = (c >> 5) & 1;
        f16x8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int key = 16 * m + 4 * hi + (j & 3) + 8 * (j >> 2);
            o[j] = (_Float16)(short)(int8_t)Vt[key * HD + d];
        }
        *reinterpret_cast<f16x8*>(vx + c * 16) = o;
    }
}

template <int HD>
__global__ __launch_bounds__(512, 2) void attn_pf(AttnArgs a) {
    constexpr int KS = HD / 16, DT = HD / 32, LA = 3;
    constexpr int KB = PF_KT * HD * 2;      // bytes of a K (or V) tile: 16 KB
    constexpr int ST = 2 * KB + 512, NS = 4;  // a stage: K | V | scales
    static_assert(8 * 16 * HD * 4 <= NS * ST, "output rows over the stages");
    __shared__ __attribute__((aligned(16))) uint8_t lds[NS * ST];

    const int G = a.nh / a.nkv;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, li = lane & 31, hi = lane >> 5;
    const int tg = wave >= G, w = wave - tg * G;
    // unit -> (sequence, KV head, block, share); the KV heads take turns, so that
    // with two of them an XCD (workgroup ids mod 8) reads the keys of one
    const uint32_t ut = pf_longest(a);
    uint32_t u = blockIdx.x / a.nkv, slot = 0;
    const int g = blockIdx.x % a.nkv;
    const int bl = pf_seq_of(a, ut, u, slot);
    if (bl >= a.nb) return;  // uniform
    const int P0 = __builtin_amdgcn_readfirstlane(a.pos[a.b0 + bl]);
    const PfSeq sq = pf_seq(a, P0);
    uint32_t jb = 0, n = 0;  // block in unit order, its units; u: the share
    for (uint32_t j0 = 0; j0 < sq.nblk; j0 += 64) {
        const uint32_t v = j0 + lane < sq.nblk ? pf_shares(sq, ut, j0 + lane) : 0u, k = pf_cut(a, v) ? v : 0u;
        uint32_t iu = v, ic = k;
        pf_scan(iu, ic);
        const uint64_t hit = __ballot(iu > u);
        if (hit) {
            const int first = __ffsll((unsigned long long)hit) - 1;
            n = pf_uni(__shfl(v, first));
            jb = j0 + first;
            u -= pf_uni(__shfl(iu - v, first));
            slot += pf_uni(__shfl(ic - k, first)) + u;
            break;
        }
        u -= pf_uni(__shfl(iu, 63));
        slot += pf_uni(__shfl(ic, 63));
    }
    if (n == 0) return;  // past the last unit; uniform
    // The grid's last workgroup of a head lies past every plan, and the partials
    // hold every plan's (pf_most_units, pf_most_shares): flagged if that were not so
    if ((int)blockIdx.x >= a.pf_room || (pf_cut(a, n) && (int)slot * a.nkv + g >= a.pf_pieces)) {
        if (threadIdx.x == 0) *a.err = 1u;
        return;
    }
    const int qb = (int)(sq.nblk - 1 - jb);
    const int pend = min(a.cap, a.lim);
    const int b = a.b0 + bl, h = g * G + w, tok0 = a.tb + qb * PF_Q + 32 * tg;
    const int nq = max(0, min(32, a.tb + a.ntok - tok0));  // of this wave's 32 tokens
    // shares are cut at whole multiples of ut: workgroups with the same share
    // index sweep the same keys at the same time, out of L2 (128 workgroups read
    // a head's 4 MB of K and V at 4096 tokens)
    const int t0 = (int)(u * ut), t1 = (int)min((u + 1) * ut, sq.tiles(jb));
    // keys 0 .. last valid query position of the wave's tokens
    const int L = P0 >= 0 && nq > 0 ? min(P0 + tok0 + nq - 1, pend - 1) + 1 : 0;
    const int tlast = min(t1, (L + PF_KT - 1) / PF_KT);
    const int qpos = P0 + tok0 + li;
    const int qlim = li < nq && P0 >= 0 && qpos < pend ? qpos : -1;  // last key this lane's query attends to
    // tiles that need no mask: below every query of 32 valid ones
    const int tfull = nq == 32 && P0 >= 0 && P0 + tok0 + 31 < pend ? (P0 + tok0 + 1) / PF_KT : 0;

    const uint32_t kvbytes = (uint32_t)a.pf_keys * (HD * 2), scbytes = (uint32_t)(a.pf_keys / PF_KT) * (PF_SC * 4);
    const int64_t pair = (int64_t)bl * a.nkv + g;
    const __amdgpu_buffer_rsrc_t rk = make_rsrc(a.kx + pair * kvbytes, kvbytes);
    const __amdgpu_buffer_rsrc_t rv = make_rsrc(a.vx + pair * kvbytes, kvbytes);
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(reinterpret_cast<uint8_t*>(a.sx) + pair * scbytes, scbytes);
    const uint32_t lane16 = lane * 16;
    const int waves = 2 * G, per = (2 * KS + waves - 1) / waves;
    // tile t -> its stage: 1 KB units dealt to the waves (`per` each, the last one
    // repeated where they do not divide), the scales by every wave, so that all
    // waves have the same number of loads in flight
    auto issue = [&](int t) {
        uint8_t* st = lds + (t & (NS - 1)) * ST;
        for (int i = 0; i < per; ++i) {
            const int x = min(wave + i * waves, 2 * KS - 1);
            lds_dma16s(x < KS ? rk : rv, st + x * 1024, lane16, (uint32_t)t * KB + (x & (KS - 1)) * 1024);
        }
        if (lane < 32) lds_dma16s(rs, st + 2 * KB, lane16, (uint32_t)t * (PF_SC * 4));
    };
    if (t0 < t1) issue(t0);
    if (t0 + 1 < t1) issue(t0 + 1);
    f16x8 q[KS];
    {
        const int64_t row = (int64_t)b * a.T + min(tok0 + min(li, max(nq - 1, 0)), a.tb + a.ntok - 1) - a.row0;
        const _Float16* qp = reinterpret_cast<const _Float16*>(a.qn) + (row * a.nh + h) * HD + 8 * hi;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) q[ks] = *reinterpret_cast<const f16x8*>(qp + 16 * ks);
        // waited for here, so that no later wait of the compiler's counts the tile loads
        __builtin_amdgcn_s_waitcnt(vm_wait(0));
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(q[ks]));
    }
    f32x16 acc[DT], s;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[dt][r] = 0.0f;
    float m = -INFINITY, l = 0.0f;  // l: this lane's keys only

    // S^T of a tile: element r of a lane is key 8 (r / 4) + 4 hi + r % 4 of
    // query li.  Operands are read LA MFMAs ahead through a ring of
    // registers, in this order: the LDS latency hides behind the matrix cores.
    auto scores = [&](const uint8_t* kt) {
        f16x8 f[LA + 1];
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = 0.0f;
#pragma unroll
        for (int u = 0; u < LA; ++u) f[u] = *reinterpret_cast<const f16x8*>(kt + u * 1024);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < KS; ++u) {
            if (u + LA < KS) f[(u + LA) % (LA + 1)] = *reinterpret_cast<const f16x8*>(kt + (u + LA) * 1024);
            __builtin_amdgcn_sched_barrier(0);
            s = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[u % (LA + 1)], q[u], s, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // softmax and V product of tile t, whose scores are in s
    auto update = [&](const uint8_t* vt, const float* sc, int t) {
        const float thr = sc[64], m0 = m == -INFINITY ? 0.0f : m;
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
            const f32x4 k4 = *reinterpret_cast<const f32x4*>(sc + 8 * r4 + 4 * hi);
#pragma unroll
            for (int r = 0; r < 4; ++r) s[4 * r4 + r] = __builtin_fmaf(s[4 * r4 + r], k4[r], -m0);
        }
        // the first V units on their way under the softmax
        f16x8 f[LA + 1];
#pragma unroll
        for (int u = 0; u < LA; ++u) f[u] = *reinterpret_cast<const f16x8*>(vt + u * 1024);
        __builtin_amdgcn_sched_barrier(0);
        if (t >= tfull) {
#pragma unroll
            for (int r = 0; r < 16; ++r)
                s[r] = PF_KT * t + 8 * (r >> 2) + 4 * hi + (r & 3) <= qlim ? s[r] : -INFINITY;
        }
        float mt = s[0];
#pragma unroll
        for (int r = 1; r < 16; ++r) mt = fmaxf(mt, s[r]);
        mt = fmaxf(mt, __shfl_xor(mt, 32));
        if (__any(mt > thr || m == -INFINITY)) {  // raise the running maximum (s is relative to m0)
            const float up = m == -INFINITY ? ceilf(mt) : fmaxf(ceilf(mt), 0.0f);
            const float corr = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(-up);
            m = m0 + up;
            l *= corr;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) acc[dt] = acc[dt] * corr;
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = up == -INFINITY ? -INFINITY : s[r] - up;  // no key of this query yet
        }
        f16x8 pb[2];
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
            const f32x4 v4 = *reinterpret_cast<const f32x4*>(sc + 32 + 8 * r4 + 4 * hi);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float e = __builtin_amdgcn_exp2f(s[4 * r4 + r]);
                l += e;
                pb[r4 >> 1][4 * (r4 & 1) + r] = (_Float16)(e * v4[r]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < KS; ++u) {
            if (u + LA < KS) f[(u + LA) % (LA + 1)] = *reinterpret_cast<const f16x8*>(vt + (u + LA) * 1024);
            __builtin_amdgcn_sched_barrier(0);
            acc[u % DT] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[u % (LA + 1)], pb[u / DT], acc[u % DT], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // Tile t is complete behind barrier t, and the stage that is filled behind
    // it (t + 2's) is no longer read.  Group 0 passes barrier t before its scores
    // of tile t, group 1 between its scores of tile t - 1 and the update with
    // them; every wave passes t1 - t0 + 1 barriers.
    auto pass = [&](int t) {
        if (G == 4 && t + 1 < t1) __builtin_amdgcn_s_waitcnt(vm_wait(2 * KS / 8 + 1));  // all but tile t + 1's
        else __builtin_amdgcn_s_waitcnt(vm_wait(0));
        __syncthreads();
        if (t + 2 < t1) issue(t + 2);
    };
    if (tg) pass(t0);
    for (int t = t0; t < t1; ++t) {
        if (!tg) pass(t);
        const uint8_t* st = lds + (t & (NS - 1)) * ST;
        if (t < tlast) scores(st + lane16);
        if (tg) pass(t + 1);
        if (t < tlast) update(st + KB + lane16, reinterpret_cast<const float*>(st + 2 * KB), t);
    }
    if (!tg) pass(t1);
    l += __shfl_xor(l, 32);
    __syncthreads();  // the stages are no longer read

    // ---- rows: 16 at a time through the wave's own 16 KB, 16-byte chunks
    // XOR-swizzled by row.  Rolled loops: this code runs once per workgroup, and
    // unrolled (3400 instructions) its instruction fetches alone took 28 us ----
    const bool lone = !pf_cut(a, n);
    const float inv = lone ? (l > 0.0f ? 1.0f / l : 0.0f) : 1.0f;
    float* piece = a.part + ((int64_t)slot * a.nkv + g) * pf_piece(G, HD);
    if (!lone && hi == 0) {
        float* ml = piece + G * PF_Q * HD + (w * PF_Q + 32 * tg + li) * 2;
        ml[0] = m;
        ml[1] = l;
    }
    piece += (w * PF_Q + 32 * tg) * HD;
    constexpr int RL = HD / 4, RI = 64 / RL;  // lanes per row, rows per access
    float* stg = reinterpret_cast<float*>(lds + wave * (16 * HD * 4));
    const int esz = a.in_dt == DT_F32 ? 4 : 2, osz = a.out_dt == DT_F32 ? 4 : 2;
    const bool gvec = ((uintptr_t)a.gate % (4 * esz)) == 0 && a.ld_in % 4 == 0 && a.q_hs % 4 == 0;
    const bool ovec = ((uintptr_t)a.out % (4 * osz)) == 0 && a.ld_out % 4 == 0;
#pragma unroll 1
    for (int p = 0; p < 2; ++p) {
        if ((li >> 4) == p) {
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4) {
                    f32x4 y;
#pragma unroll
                    for (int r = 0; r < 4; ++r) y[r] = acc[dt][4 * r4 + r] * inv;
                    *reinterpret_cast<f32x4*>(&stg[(li & 15) * HD + 4 * ((8 * dt + 2 * r4 + hi) ^ (li & 15))]) = y;
                }
        }
        __builtin_amdgcn_wave_barrier();
        constexpr int U = 4;  // accesses in flight
#pragma unroll 1
        for (int j0 = 0; j0 < 16; j0 += U * RI) {
            const int d = 4 * (lane % RL);
            f32x4 gt[U], y[U];
#pragma unroll
            for (int e = 0; e < U; ++e) {
                const int rr = j0 + e * RI + lane / RL;  // row of the 16
                y[e] = *reinterpret_cast<const f32x4*>(&stg[rr * HD + 4 * ((lane % RL) ^ rr)]);
                gt[e] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                if (!lone || 16 * p + rr >= nq) continue;
                const int64_t gi = ((int64_t)b * a.T + tok0 + 16 * p + rr) * a.ld_in + (int64_t)h * a.q_hs + d;
                if (gvec) {
                    gt[e] = load_act4(a.gate, a.in_dt, gi);
                } else {
#pragma unroll
                    for (int c = 0; c < 4; ++c) gt[e][c] = at_load(a.gate, a.in_dt, gi + c);
                }
            }
#pragma unroll
            for (int e = 0; e < U; ++e) {
                const int qr = 16 * p + j0 + e * RI + lane / RL;
                if (!lone) {
                    *reinterpret_cast<f32x4*>(piece + qr * HD + d) = y[e];
                    continue;
                }
                if (qr >= nq) continue;
#pragma unroll
                for (int c = 0; c < 4; ++c) y[e][c] *= 1.0f / (1.0f + __expf(-gt[e][c]));
                const int64_t oi = ((int64_t)b * a.T + tok0 + qr) * a.ld_out + (int64_t)h * HD + d;
                if (ovec) {
                    store_act4(a.out, a.out_dt, oi, y[e]);
                } else {
#pragma unroll
                    for (int c = 0; c < 4; ++c) store_act(a.out, a.out_dt, oi + c, y[e][c]);
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// Merges the shares of the blocks that were cut: one workgroup per (block, 16
// of its tokens of a head, sequence), four rows per wave in flight together.
template <int HD>
__global__ __launch_bounds__(256) void attn_pf_merge(AttnArgs a) {
    constexpr int E = HD / 64;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int h = blockIdx.y / (PF_Q / 16), bl = blockIdx.z, G = a.nh / a.nkv, g = h / G, w = h % G;
    const uint32_t jb = blockIdx.x, ut = pf_longest(a);
    const PfSeq sq = pf_seq(a, __builtin_amdgcn_readfirstlane(a.pos[a.b0 + bl]));
    const int n = (int)pf_shares(sq, ut, jb);
    if (!pf_cut(a, n)) return;
    uint32_t slot = 0, units, cut;
    for (int i = threadIdx.x & 63; i < bl && (uint32_t)bl > sq.nblk; i += 64) {  // lanes take sequences
        const PfSeq o = pf_seq(a, a.pos[a.b0 + i]);
        pf_count<false>(a, o, ut, o.nblk, units, cut);
        slot += cut;
    }
    slot = pf_sum(slot);
    for (int i = 0; i < bl && (uint32_t)bl <= sq.nblk; ++i) {  // lanes take blocks
        const PfSeq o = pf_seq(a, __builtin_amdgcn_readfirstlane(a.pos[a.b0 + i]));
        pf_count<true>(a, o, ut, o.nblk, units, cut);
        slot += cut;
    }
    pf_count<true>(a, sq, ut, jb, units, cut);
    slot += cut;
    if ((int)(slot + n - 1) * a.nkv + g >= a.pf_pieces) {  // never (as in attn_pf)
        if (threadIdx.x == 0) *a.err = 1u;
        return;
    }
    const int qb = (int)(sq.nblk - 1 - jb), nq = min(PF_Q, a.ntok - qb * PF_Q);
    const int64_t ps = pf_piece(G, HD), next = ps * a.nkv;
    const float* p0 = a.part + ((int64_t)slot * a.nkv + g) * ps;
    const int qr = blockIdx.y % (PF_Q / 16) * 16 + wave * 4;
    const float* ml = p0 + G * PF_Q * HD + (w * PF_Q + qr) * 2;
    const float* src = p0 + (int64_t)(w * PF_Q + qr) * HD + lane * E;
    float M[4], l[4], o[4][E];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        M[r] = -INFINITY;
        l[r] = 0.0f;
#pragma unroll
        for (int e = 0; e < E; ++e) o[r][e] = 0.0f;
    }
    for (int i = 0; i < n; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) M[r] = fmaxf(M[r], ml[i * next + 2 * r]);
    for (int i = 0; i < n; ++i) {
        float x[4][E];
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int e = 0; e < E; ++e) x[r][e] = src[i * next + r * HD + e];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float mi = ml[i * next + 2 * r];
            const float wi = mi == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mi - M[r]);  // no key of this query in the share
            l[r] += wi * ml[i * next + 2 * r + 1];
#pragma unroll
            for (int e = 0; e < E; ++e) o[r][e] += wi * x[r][e];
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
        if (qr + r < nq)
            gate_store<HD>(a, (a.b0 + bl) * a.T + a.tb + qb * PF_Q + qr + r, h, lane, o[r], l[r] > 0.0f ? 1.0f / l[r] : 0.0f);
}

// ---------------------------------------------------------------------------
// decode over an INT8 cache on f16 MFMA: (key split, KV head g, row).  The
// group's query heads are the MFMA columns (B = Q^T, 16 columns of which G
// are used); a 64-key tile is staged as f16 once (K rows, V transposed) and
// wave w takes its 16-key quarter: S^T = K Q^T, an online softmax of its own
// per column, O^T += V^T P^T.  The four waves' (max, sum, O) are merged in LDS
// at the end; a lone split writes the output, otherwise a partial.
constexpr int AD_KT = 64;  // keys per tile

// FUSED (one new token per sequence): the kernel also does the work of
// attn_prep and attn_combine, saving two launches per decode step:
//   * every workgroup normalizes and rotates its G query heads itself (one
//     wave each) from the projection output;
//   * the workgroup whose key range holds the new position P computes the
//     new token's K and V of its KV head (norm, RoPE, INT8 codes and scale,
//     as attn_prep), writes them to the cache for later steps, and puts the
//     same codes and scales into its LDS tile in place of the cache's (so
//     nothing in this launch reads the slot it writes);
//   * the splits of a (row, KV head) hand their partials over with
//     agent-scope stores and an arrival count; the last one to arrive merges
//     them (merge_splits_wave, as attn_combine) and writes the gated output.
// No workgroup waits for another, so the launch cannot stall.
template <int HD, bool FUSED, bool VCOAL>
__global__ __launch_bounds__(256) void attn_decode_i8h(AttnArgs a) {
    constexpr int KB = HD / 16, DT = HD / 16, E = HD / 64;
    constexpr int KHP = HD + 8, VHP = AD_KT + 4;
    constexpr int KPER = AD_KT * HD / 16 / 256;  // 16-code K chunks per thread
    // V tile loads, two patterns (VCOAL chosen per launch):
    //   VCOAL: 16 codes of each of 4 consecutive keys per thread, consecutive
    //     threads on consecutive 16-byte chunks of a key row (coalesced rows);
    //   else: 4 codes of each of 4 consecutive keys per thread, consecutive
    //     threads on consecutive key groups (conflict-free V^T stores).
    // Measured: the coalesced rows win once the launch fills the chip (B=32,
    // context 4096: 84 vs 97 us; B=1, context 32768: 42 vs 43 us) and lose
    // with few workgroups (B=1, context 4096, 64 workgroups: 33 vs 24 us).
    constexpr int VNG = AD_KT / 4 * (HD / 16);  // 4-key x 16-dim groups of the V tile
    constexpr int VPG = (VNG + 255) / 256;      // per thread
    constexpr int VPER = AD_KT * HD / 16 / 256;  // 4x4 V blocks per thread (scattered pattern)
    constexpr int KT4 = AD_KT / 4;
    const int s = blockIdx.x, g = blockIdx.y, rl = blockIdx.z, r = a.row0 + rl;
    const int b = r / a.T, t = r % a.T;
    const int P = a.pos[b] + t;
    const int L = (P >= 0 && P < a.cap && P < a.lim) ? P + 1 : 0;
    const int k0 = s * a.split, k1 = min(k0 + a.split, L);
    const int G = a.nh / a.nkv;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
    if (k0 >= k1) {  // uniform over the workgroup
        if (FUSED && L == 0 && s == 0 && g == 0 && threadIdx.x == 0) *a.err = 1u;
        if (L == 0 && (a.nsplit == 1 || (FUSED && s == 0)) && wave < G) {
            const int64_t oi = (int64_t)r * a.ld_out + (int64_t)(g * G + wave) * HD + lane * E;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                if (a.out_dt == DT_F32) reinterpret_cast<float*>(a.out)[oi + e] = 0.0f;
                else store_act(a.out, a.out_dt, oi + e, 0.0f);
            }
        }
        return;
    }

    __shared__ __attribute__((aligned(16))) _Float16 Kh[AD_KT * KHP];
    __shared__ __attribute__((aligned(16))) _Float16 VhT[HD * VHP];
    __shared__ float ksc[AD_KT], vsc[AD_KT];
    __shared__ float wm[4][16], wl[4][16];

    const uint8_t* kbase = reinterpret_cast<const uint8_t*>(a.kc);
    const uint8_t* vbase = reinterpret_cast<const uint8_t*>(a.vc);
    const int64_t slot0 = (int64_t)b * a.cap * a.nkv + g;
    u32x4 kpre[KPER];
    u32x4 vpre[VCOAL ? VPG : 1][4];
    uint32_t vpre4[VCOAL ? 1 : VPER][4];
    float psc = 0.0f;
    auto issue = [&](int kt) {
        const int n = min(AD_KT, k1 - kt);
#pragma unroll
        for (int i = 0; i < KPER; ++i) {
            const int c = threadIdx.x + 256 * i, j = c / (HD / 16), part = c % (HD / 16);
            // keys past the range read the range's last key: finite, masked out later
            kpre[i] = *reinterpret_cast<const u32x4*>(kbase + (slot0 + (int64_t)(kt + min(j, n - 1)) * a.nkv) * HD + part * 16);
        }
        if constexpr (VCOAL) {
            for (int i = 0; i < VPG; ++i) {  // V: 16 codes of each of 4 consecutive keys
                const int grp = threadIdx.x + 256 * i, c = grp % (HD / 16), k4 = grp / (HD / 16);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int j = 4 * k4 + q;
                    if (VNG % 256 == 0 || grp < VNG)
                        vpre[i][q] = *reinterpret_cast<const u32x4*>(vbase + (slot0 + (int64_t)(kt + min(j, n - 1)) * a.nkv) * HD + 16 * c);
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < VPER; ++i) {  // V: 4 codes of each of 4 consecutive keys
                const int blk = threadIdx.x + 256 * i, k4 = blk % (KT4), d4 = blk / (KT4);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int j = 4 * k4 + q;
                    vpre4[i][q] = *reinterpret_cast<const uint32_t*>(vbase + (slot0 + (int64_t)(kt + min(j, n - 1)) * a.nkv) * HD + 4 * d4);
                }
            }
        }
        if (threadIdx.x < 2 * AD_KT) {
            const int j = threadIdx.x & (AD_KT - 1);
            psc = (threadIdx.x < AD_KT ? a.ks : a.vs)[slot0 + (int64_t)(kt + min(j, n - 1)) * a.nkv];
        }
    };
    // fused: q of the G heads (wave w: head g*G + w), and -- in the workgroup
    // that holds position P -- the new K and V of head g, as attn_prep
    const bool owner = FUSED && k1 == L;  // this split's range ends at P
    __shared__ __attribute__((aligned(16))) float qs[FUSED ? 4 : 1][FUSED ? HD : 1];
    __shared__ float rc[FUSED ? HD / 2 : 1], rs[FUSED ? HD / 2 : 1];
    __shared__ int8_t newkv[FUSED ? 2 : 1][FUSED ? HD : 1];
    __shared__ float newsc[2];
    if constexpr (FUSED) {
        // the first tile's loads go out before the q work: they do not depend
        // on it (a stale slot P is replaced in LDS below), and the q loads
        // then wait for the tile instead of the tile waiting for the q work
        issue(k0);
        if ((int)threadIdx.x < a.rot / 2) {
            const float freq = 1.0f / powf(a.theta, (float)(2 * threadIdx.x) / (float)a.rot);
            const float ang = (float)P * freq;
            rc[threadIdx.x] = cosf(ang);
            rs[threadIdx.x] = sinf(ang);
        }
        __syncthreads();
        const int64_t row = (int64_t)r * a.ld_in;
        // items: q head g*G + it for it < G; then (owner) it = G: k, G+1: v of head g
        for (int it = wave; it < G + (owner ? 2 : 0); it += 4) {
            const bool isq = it < G, isk = it == G;
            const void* src = isq ? a.q : (isk ? a.k : a.v);
            const int64_t base = row + (isq ? (int64_t)(g * G + it) * a.q_hs : (int64_t)g * HD) + lane * E;
            float x[E];
#pragma unroll
            for (int e = 0; e < E; ++e) x[e] = at_load(src, a.in_dt, base + e);
            if (it <= G) {  // q or k: RMSNorm (1 + w), then RoPE on d < rot
                const float ss = wave_sum(sum_squares(x));
                const float rms = sqrtf(ss / (float)HD + 1e-6f);
                const float* w = isq ? a.qn_w : a.kn_w;
#pragma unroll
                for (int e = 0; e < E; ++e) x[e] = x[e] / rms * (1.0f + w[lane * E + e]);
#pragma unroll
                for (int e = 0; e < E; e += 2) {
                    const int d = lane * E + e;
                    if (d < a.rot) {
                        const float c = rc[d / 2], sn = rs[d / 2];
                        const float x0 = x[e], x1 = x[e + 1];
                        x[e] = rope0(x0, x1, c, sn);
                        x[e + 1] = rope1(x0, x1, c, sn);
                    }
                }
            }
            if (isq) {
#pragma unroll
                for (int e = 0; e < E; ++e) qs[it][lane * E + e] = x[e];
                continue;
            }
            // the new token's INT8 codes and scale (kv 0: K, 1: V)
            const int kv = isk ? 0 : 1;
            float m = 0.0f;
#pragma unroll
            for (int e = 0; e < E; ++e) m = fmaxf(m, fabsf(x[e]));
            m = wave_max(m);
            float sc = m / 127.0f;
            sc = sc > 1e-8f ? sc : 1.0f;
            const int64_t slot = ((int64_t)b * a.cap + P) * a.nkv + g;
            int8_t* cdst = reinterpret_cast<int8_t*>(isk ? a.kc : a.vc) + slot * HD + lane * E;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int8_t c = (int8_t)fmaxf(-127.0f, fminf(127.0f, roundf(x[e] / sc)));
                cdst[e] = c;
                newkv[kv][lane * E + e] = c;
            }
            if (lane == 0) {
                (isk ? a.ks : a.vs)[slot] = sc;
                newsc[kv] = sc;
            }
        }
        __syncthreads();
    }
    // B operand: column li = query head g*G + li of this row (zero for li >= G)
    f16x4 qh[KB];
    {
        const float* qp = FUSED ? &qs[min(li, G - 1)][4 * lg]
                                : a.qn + ((int64_t)rl * a.nh + g * G + min(li, G - 1)) * HD + 4 * lg;
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
            const f32x4 v = li < G ? *reinterpret_cast<const f32x4*>(qp + 16 * kb) : f32x4{0, 0, 0, 0};
#pragma unroll
            for (int q = 0; q < 4; ++q) qh[kb][q] = (_Float16)v[q];
        }
    }
    if constexpr (!FUSED) issue(k0);  // after the q loads, so that waiting for q does not wait for the tile
    const float scale = 1.0f / sqrtf((float)HD);
    f32x4 acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) acc[dt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    float m = -INFINITY, l = 0.0f;

    for (int kt = k0; kt < k1; kt += AD_KT) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < KPER; ++i) {
            const int c = threadIdx.x + 256 * i, j = c / (HD / 16), part = c % (HD / 16);
            f16x4 hv[4];
#pragma unroll
            for (int w = 0; w < 4; ++w) hv[w] = i8x4_to_h4(kpre[i][w]);
            u32x4* dst = reinterpret_cast<u32x4*>(&Kh[j * KHP + part * 16]);
            dst[0] = __builtin_bit_cast(u32x4, __builtin_shufflevector(hv[0], hv[1], 0, 1, 2, 3, 4, 5, 6, 7));
            dst[1] = __builtin_bit_cast(u32x4, __builtin_shufflevector(hv[2], hv[3], 0, 1, 2, 3, 4, 5, 6, 7));
        }
        if constexpr (VCOAL) {
            for (int i = 0; i < VPG; ++i) {
                const int grp = threadIdx.x + 256 * i, c = grp % (HD / 16), k4 = grp / (HD / 16);
                if (VNG % 256 == 0 || grp < VNG) {
#pragma unroll
                    for (int blk = 0; blk < 4; ++blk) {
                        const uint32_t w4[4] = {vpre[i][0][blk], vpre[i][1][blk], vpre[i][2][blk], vpre[i][3][blk]};
                        uint32_t tw[4];
                        transpose4x4(w4, tw);  // tw[e]: dim 16*c + 4*blk + e of keys 4*k4 .. 4*k4+3
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            *reinterpret_cast<f16x4*>(&VhT[(16 * c + 4 * blk + e) * VHP + 4 * k4]) = i8x4_to_h4(tw[e]);
                    }
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < VPER; ++i) {
                const int blk = threadIdx.x + 256 * i, k4 = blk % (KT4), d4 = blk / (KT4);
                uint32_t tw[4];
                transpose4x4(vpre4[i], tw);  // tw[e]: dim 4*d4 + e of keys 4*k4 .. 4*k4+3
#pragma unroll
                for (int e = 0; e < 4; ++e) *reinterpret_cast<f16x4*>(&VhT[(4 * d4 + e) * VHP + 4 * k4]) = i8x4_to_h4(tw[e]);
            }
        }
        if (threadIdx.x < 2 * AD_KT) (threadIdx.x < AD_KT ? ksc : vsc)[threadIdx.x & (AD_KT - 1)] = psc;
        if (kt + AD_KT < k1) issue(kt + AD_KT);
        __syncthreads();
        if (owner && P < kt + AD_KT) {  // the tile of position P: its K/V from this launch, not the cache
            const int jp = P - kt;
            for (int d = threadIdx.x; d < HD; d += 256) {
                Kh[jp * KHP + d] = (_Float16)newkv[0][d];
                VhT[d * VHP + jp] = (_Float16)newkv[1][d];
            }
            if (threadIdx.x < 2) (threadIdx.x == 0 ? ksc : vsc)[jp] = newsc[threadIdx.x];
            __syncthreads();
        }
        const int kw = 16 * wave;  // this wave's quarter of the tile
        if (kt + kw >= k1) continue;
        f32x4 sacc = {0.0f, 0.0f, 0.0f, 0.0f};
        const _Float16* kr = &Kh[(kw + li) * KHP + 4 * lg];
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
            sacc = __builtin_amdgcn_mfma_f32_16x16x16f16(*reinterpret_cast<const f16x4*>(kr + 16 * kb), qh[kb], sacc, 0, 0, 0);
        float mt = -INFINITY;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int kl = kw + 4 * lg + q;
            const float v = kt + kl < k1 ? sacc[q] * scale * ksc[kl] : -INFINITY;
            sacc[q] = v;
            mt = fmaxf(mt, v);
        }
        mt = fmaxf(mt, __shfl_xor(mt, 16));
        mt = fmaxf(mt, __shfl_xor(mt, 32));
        const float mn = fmaxf(m, mt);  // finite: the quarter has at least one key
        const float corr = __expf(m - mn);
        float ps = 0.0f;
        f16x4 pb;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float p = __expf(sacc[q] - mn);
            ps += p;
            pb[q] = (_Float16)(p * vsc[kw + 4 * lg + q]);
        }
        ps += __shfl_xor(ps, 16);
        ps += __shfl_xor(ps, 32);
        l = l * corr + ps;
        m = mn;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            acc[dt] = acc[dt] * corr;
            acc[dt] = __builtin_amdgcn_mfma_f32_16x16x16f16(
                *reinterpret_cast<const f16x4*>(&VhT[(16 * dt + li) * VHP + kw + 4 * lg]), pb, acc[dt], 0, 0, 0);
        }
    }
    // merge the four waves: column li of each wave's (m, l, O^T)
    __syncthreads();  // the tiles are no longer read; reuse VhT for the wave outputs
    float* ow = reinterpret_cast<float*>(VhT);  // [4 waves][G cols][HD]
    if (lg == 0) {
        wm[wave][li] = m;
        wl[wave][li] = l;
    }
    if (li < G) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<f32x4*>(&ow[(wave * 4 + li) * HD + 16 * dt + 4 * lg]) = acc[dt];
    }
    __syncthreads();
    // wave w < G finishes query head g*G + w: merge the four waves' columns
    auto wave_merge = [&](float (&o)[E], float& M, float& lt) {
        const int col = wave;
        M = -INFINITY;
#pragma unroll
        for (int w = 0; w < 4; ++w) M = fmaxf(M, wm[w][col]);
        float wsc[4];
        lt = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            wsc[w] = wm[w][col] == -INFINITY ? 0.0f : __expf(wm[w][col] - M);
            lt += wsc[w] * wl[w][col];
        }
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int d = lane * E + e;
            float v = 0.0f;
#pragma unroll
            for (int w = 0; w < 4; ++w) v += wsc[w] * ow[(w * 4 + col) * HD + d];
            o[e] = v;
        }
    };
    const int h = g * G + wave;
    if constexpr (!FUSED) {
        if (wave >= G) return;
        float o[E], M, lt;
        wave_merge(o, M, lt);
        if (a.nsplit == 1) {
            gate_store<HD>(a, r, h, lane, o, 1.0f / lt);
            return;
        }
        float* dst = a.part + (((int64_t)rl * a.nh + h) * a.nsplit + s) * (HD + 2);
#pragma unroll
        for (int e = 0; e < E; ++e) dst[lane * E + e] = o[e];
        if (lane == 0) {
            dst[HD] = M;
            dst[HD + 1] = lt;
        }
    } else {
        const int ns = (L + a.split - 1) / a.split;  // splits holding keys of this row
        __shared__ unsigned last_s;
        if (wave < G) {
            float o[E], M, lt;
            wave_merge(o, M, lt);
            if (ns == 1) {
                gate_store<HD>(a, r, h, lane, o, 1.0f / lt);
            } else {
                // hand-off: agent-scope stores of the partial
                float* dst = a.part + (((int64_t)rl * a.nh + h) * a.nsplit + s) * (HD + 2);
#pragma unroll
                for (int e = 0; e < E; ++e)
                    __hip_atomic_store(dst + lane * E + e, o[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (lane == 0) {
                    __hip_atomic_store(dst + HD, M, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    __hip_atomic_store(dst + HD + 1, lt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
        }
        if (ns > 1) {  // uniform over the workgroup
            // every wave waits for its stores' completion, then one arrival
            // count per workgroup; the last split of (row, g) merges them all
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            if (threadIdx.x == 0) {
                unsigned* cnt = a.cnt + (int64_t)rl * a.nkv + g;
                const unsigned old = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                last_s = old == (unsigned)(ns - 1) ? 1u : 0u;
                if (old == (unsigned)(ns - 1)) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            __syncthreads();
            if (last_s && wave < G) {
                const float* pp = a.part + ((int64_t)rl * a.nh + h) * a.nsplit * (HD + 2);
                float om[E], l;
                merge_splits_wave<HD, true>(pp, ns, lane, om, l);
                gate_store<HD>(a, r, h, lane, om, 1.0f / l);
            }
        }
    }
}

size_t attn_bytes_per_row(int nh, int hd, int nsplit) {
    return (size_t)nh * hd * 4 + (size_t)nh * nsplit * (hd + 2) * 4;
}

template <int HD>
static void launch_combine(const AttnArgs& a, hipStream_t stream) {
    if (a.nsplit <= 1) return;
    if (a.nsplit <= 16) hipLaunchKernelGGL((attn_combine<HD, 1>), dim3(a.rows, a.nh), dim3(64), 0, stream, a);
    else hipLaunchKernelGGL((attn_combine<HD, 4, HD / 64>), dim3(a.rows, a.nh, HD / 64), dim3(256), 0, stream, a);
}

template <int HD>
static hipError_t launch_attn_hd(const AttnArgs& a, hipStream_t stream) {
    if (a.prefill) {
        launch_prep<HD>(a, stream);
        if (a.pf_units) {
            hipLaunchKernelGGL(attn_expand<HD>, dim3(a.pf_keys / PF_KT, a.nkv, a.nb), dim3(256), 0, stream, a);
            hipLaunchKernelGGL(attn_pf<HD>, dim3(a.pf_grid), dim3(128 * (a.nh / a.nkv)), 0, stream, a);
            hipLaunchKernelGGL(attn_pf_merge<HD>, dim3((a.ntok + PF_Q - 1) / PF_Q, a.nh * (PF_Q / 16), a.nb), dim3(256), 0, stream, a);
            return hipGetLastError();
        }
        // INT8: query blocks x key splits (f16 MFMA), merged by attn_combine;
        // FP32: the same on FP32 MFMA, the keys cut by blocks
        if (a.kv_dt == DT_I8) {
            hipLaunchKernelGGL(attn_prefill_i8h<HD>, dim3((a.ntok + 15) / 16 * a.nsplit, a.nkv, a.nb), dim3(256), 0,
                               stream, a);
            launch_combine<HD>(a, stream);
        } else {
            // (nsplit > 1 only where blocks are few, so nb * nsplit stays a valid grid)
            hipLaunchKernelGGL((attn_prefill<HD>), dim3((a.ntok + 15) / 16, a.nkv, a.nb * a.nsplit), dim3(256), 0,
                               stream, a);
            launch_combine<HD>(a, stream);
        }
        return hipGetLastError();
    }
    if (a.kv_dt == DT_I8 && a.T == 1 && a.cnt) {  // one launch: prep and combine inside
        if (a.vcoal) hipLaunchKernelGGL((attn_decode_i8h<HD, true, true>), dim3(a.nsplit, a.nkv, a.rows), dim3(256), 0, stream, a);
        else hipLaunchKernelGGL((attn_decode_i8h<HD, true, false>), dim3(a.nsplit, a.nkv, a.rows), dim3(256), 0, stream, a);
        return hipGetLastError();
    }
    launch_prep<HD>(a, stream);
    if (a.kv_dt == DT_I8 && a.vcoal) hipLaunchKernelGGL((attn_decode_i8h<HD, false, true>), dim3(a.nsplit, a.nkv, a.rows), dim3(256), 0, stream, a);
    else if (a.kv_dt == DT_I8) hipLaunchKernelGGL((attn_decode_i8h<HD, false, false>), dim3(a.nsplit, a.nkv, a.rows), dim3(256), 0, stream, a);
    else hipLaunchKernelGGL((attn_split<HD, false>), dim3(a.nsplit, a.nkv, a.rows), dim3(256), 0, stream, a);
    launch_combine<HD>(a, stream);
    return hipGetLastError();
}

hipError_t launch_attn(const AttnArgs& a, hipStream_t stream) {
    if (a.nkv < 1 || a.nh % a.nkv || a.nh / a.nkv > 4 || a.rot % 2 || a.rot > a.hd) return hipErrorInvalidValue;
    if (a.hd == 256) return launch_attn_hd<256>(a, stream);
    if (a.hd == 128) return launch_attn_hd<128>(a, stream);
    return hipErrorInvalidValue;
}

}  // namespace qwk
