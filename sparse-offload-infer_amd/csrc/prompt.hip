// A whole prompt through one decoder layer at a time (gfx950): the decode step's operators over T tokens.
//
// The decode step (gemv_int4.hip, decode_attention.hip, decoder.hip) takes one token through every layer, so a
// prompt fed through it reads every weight once per token and pays every launch once per token. Here each weight
// row is read once for a tile of tokens, and a layer is a handful of launches whatever the prompt's length.
//
// Values: these kernels evaluate, for every (token, row) and (token, head), the expressions of the decode step in
// the decode step's order (the lane partition and reduction tree of gemv_int4_tile, the norm's partition, the
// split plan and combine of the attention), so hidden states, caches and selections are bit for bit those of
// the same tokens fed one at a time. The linears of dense prompts of 9 tokens up are the exception: they run in
// prompt_mfma.hip, whose sums take another order (here are their norms, attention and, for group sizes or widths that
// kernel does not take, their linears too). Reference: the prompt loop of generate_streaming / generate_dip
// (python/soinfer/runtime/generate.py:429-520), one token per step.
//
// Measured (Qwen3-1.7B shape, dense): 8 tokens through 4 layers 289 us against 732 with one layers-graph replay per
// token. With the linears on the matrix cores, 28 layers, a 256-token prompt and its first token 3.8 ms against 146 (13.2
// with these linears); 48 tokens and 4 new ones with 8 layers streamed from host memory 19.7 against 197 (the weights
// cross PCIe once for the prompt instead of once per token).
#include "soi_device.h"
#include "soi_host.h"
#include "soi_attn.h"
#include "soi_int4_tile.h"
#include "soi_prompt.h"

namespace soi {

// ---------------------------------------------------------------------------
// embedding rows
// ---------------------------------------------------------------------------
// out[t] = table[tokens[t]] (zeros for a token outside the table, as embed_kernel); one workgroup per token.
__global__ __launch_bounds__(256) void embed_tokens_kernel(const uint16_t* __restrict__ table, int64_t rows,
                                                           int hidden, const int32_t* __restrict__ tokens,
                                                           uint16_t* __restrict__ out) {
    const int t = ldg(tokens + blockIdx.x);
    const bool ok = t >= 0 && t < rows;
    const uint16_t* src = table + (ok ? static_cast<int64_t>(t) : 0) * hidden;
    uint16_t* dst = out + static_cast<int64_t>(blockIdx.x) * hidden;
    for (int i = threadIdx.x; i < hidden; i += 256) stg(dst + i, ok ? ldg(src + i) : uint16_t(0));
}

// ---------------------------------------------------------------------------
// RMSNorm rows
// ---------------------------------------------------------------------------
// h[t] = rmsnorm(x[t], w), one wave per token, with the partition of the norm-fused GEMVs: REG, the one-pass form
// (hidden 2048: lane l sums its 32 elements), else NormX's (lane l sums 16-byte chunks l, l + 64, ...). frag: h in
// fragment layout.
constexpr int kNormTokens = 4;  // waves (tokens) per workgroup

template <bool REG>
__global__ __launch_bounds__(kNormTokens * kWave) void norm_tokens_kernel(const uint16_t* __restrict__ x,
                                                                          const uint16_t* __restrict__ w, float eps,
                                                                          uint16_t* __restrict__ h, int T, int K, int frag) {
    const int lane = threadIdx.x & 63;
    const int t = static_cast<int>(blockIdx.x) * kNormTokens + static_cast<int>(threadIdx.x >> 6);
    if (t >= T) return;  // wave-uniform
    const u32x4* a4 = reinterpret_cast<const u32x4*>(x + static_cast<int64_t>(t) * K);
    const u32x4* w4 = reinterpret_cast<const u32x4*>(w);
    u32x4* h4 = reinterpret_cast<u32x4*>(h + static_cast<int64_t>(t) * K);
    const int n8 = K >> 3;
    float ss = 0.0f;
    if (REG) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const u32x4 s = ldg(a4 + 4 * lane + i);
            ss += sumsq_f16x2(s.x) + sumsq_f16x2(s.y) + sumsq_f16x2(s.z) + sumsq_f16x2(s.w);
        }
    } else {
        for (int c = lane; c < n8; c += kWave) {
            const u32x4 s = ldg(a4 + c);
            ss += sumsq_f16x2(s.x) + sumsq_f16x2(s.y) + sumsq_f16x2(s.z) + sumsq_f16x2(s.w);
        }
    }
    const float inv = rsqrtf(wave_sum_bcast(ss) / static_cast<float>(K) + eps);
    for (int c = lane; c < n8; c += kWave) {
        const u32x4 s = ldg(a4 + c), g = ldg(w4 + c);
        u32x4 r;
        r.x = norm_f16x2(s.x, g.x, inv);
        r.y = norm_f16x2(s.y, g.y, inv);
        r.z = norm_f16x2(s.z, g.z, inv);
        r.w = norm_f16x2(s.w, g.w, inv);
        stg(frag ? reinterpret_cast<u32x4*>(h + frag_offset(t, 8 * c, K)) : h4 + c, r);
    }
}

// ---------------------------------------------------------------------------
// INT4 rows x tokens, the GEMV's arithmetic
// ---------------------------------------------------------------------------
// Epilogues: total (token t, row) -> y[t, row], or (ADD) x[t, row] = x[t, row] + y as one binary16 addition.
struct TokenStore {
    uint16_t* y;
    __device__ __forceinline__ void store(int64_t i, float total) const { stg(y + i, f32_to_f16_bits(total)); }
};
struct TokenAdd {
    uint16_t* x;
    __device__ __forceinline__ void store(int64_t i, float total) const {
        stg(x + i, static_cast<uint16_t>(add_f16x2(ldg(x + i), f32_to_f16_bits(total))));
    }
};

// The value of lane (l ^ 4) in lane l: each 4-lane bank takes the bank 4 lanes up or down (DPP row_shl:4 into
// banks 0 and 2, row_shr:4 into banks 1 and 3).
__device__ __forceinline__ float xor4(float v) {
    const int u = __builtin_bit_cast(int, v);
    const int a = __builtin_amdgcn_update_dpp(u, u, 0x104, 0xf, 0x5, false);
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(a, u, 0x114, 0xf, 0xa, false));
}

// Transposed reduction of V (a power of two, 8 to 64) per-lane partials over the 64 lanes: lane pairs 32, 16, 8, 1,
// 2, 4 apart are added in that order (reduce_rows' tree: addition commutes, so which lane of a pair keeps a value
// does not matter), and each exchange halves the values a lane still holds. Lane l ends with the total of value
// reduce_tile_index<V>(l).
template <int V>
__device__ __forceinline__ float reduce_tile(float (&a)[V], int lane) {
    static_assert(V >= 8 && V <= 64, "8 to 64 values");
#pragma unroll
    for (int j = 0; j < V / 2; ++j) {
        float hi = a[j + V / 2], lo = a[j];
        swap32(hi, lo);
        a[j] = hi + lo;
    }
#pragma unroll
    for (int j = 0; j < V / 4; ++j) {
        float hi = a[j + V / 4], lo = a[j];
        swap16(hi, lo);
        a[j] = hi + lo;
    }
#pragma unroll
    for (int j = 0; j < V / 8; ++j) {
        const bool e = lane & 8;
        const float keep = e ? a[j] : a[j + V / 8], send = e ? a[j + V / 8] : a[j];
        a[j] = keep + dpp_f<0x128>(send);
    }
#pragma unroll
    for (int j = 0; j < (V >= 16 ? V / 16 : 1); ++j) {
        const bool e = lane & 1;
        const float keep = (V < 16 || e) ? a[j] : a[j + V / 16], send = (V < 16 || !e) ? a[j] : a[j + V / 16];
        a[j] = V < 16 ? a[j] + dpp_f<0xb1>(a[j]) : keep + dpp_f<0xb1>(send);
    }
#pragma unroll
    for (int j = 0; j < (V >= 32 ? V / 32 : 1); ++j) {
        const bool e = lane & 2;
        const float keep = (V < 32 || e) ? a[j] : a[j + V / 32], send = (V < 32 || !e) ? a[j] : a[j + V / 32];
        a[j] = V < 32 ? a[j] + dpp_f<0x4e>(a[j]) : keep + dpp_f<0x4e>(send);
    }
    if (V >= 64) {
        const bool e = lane & 4;
        const float keep = e ? a[0] : a[V >= 64 ? 1 : 0], send = e ? a[V >= 64 ? 1 : 0] : a[0];
        return keep + xor4(send);
    }
    return a[0] + xor4(a[0]);
}

// the upper half of a pair stays where the lane bit is 0 (bits 5, 4, 3, 0, 1, 2 from the top index bit down)
template <int V>
__device__ __forceinline__ int reduce_tile_index(int lane) {
    const int order[6] = {5, 4, 3, 0, 1, 2};
    int v = 0;
#pragma unroll
    for (int b = 0, n = V; n > 1; ++b, n >>= 1) v = 2 * v + (((lane >> order[b]) & 1) ^ 1);
    return v;
}

// One wave: R rows x TT tokens per tile, `tiles` row tiles one after another. Lane l owns chunk l (32 elements) of
// every 64-chunk pass, as in gemv_int4_tile; per (row, token) the lane's chain is the GEMV's (two 8-step v_dot2
// chains, -8 sum(x), one fma with the scale per chunk) and the wave's sum is its tree, so each y is the GEMV's.
//
// Bound by v_dot2 issue: a row's chunk costs 20 instructions to unpack, shared by TT tokens of 16 dot products + 3
// fmas each. The tokens' x chunks stay in registers (16 VGPRs a token) over the row tiles when a row is one pass.
template <int R, int TT, bool FULL, class EP>
__global__ __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(2, 3))) void gemm_int4_tokens_kernel(
    const uint8_t* __restrict__ W, const float* __restrict__ S, int64_t row_bytes, int G,
    const uint16_t* __restrict__ X, int64_t N, int K, int gs, int T, int tiles, EP ep) {
    const int lane = threadIdx.x;
    const int chunks = K >> 5;
    const int t0 = static_cast<int>(blockIdx.y) * TT;
    const bool one_pass = chunks <= kWave;
    const u32x4* z = reinterpret_cast<const u32x4*>(g_zero16);
    const float* zf = reinterpret_cast<const float*>(g_zero16);
    f16x2 xv[TT][16];
    float xs[TT];
    const int vi = reduce_tile_index<R * TT>(lane);  // value index = token * R + row
    const int vt = vi / R, vr = vi % R;
    const bool writer = (lane & 63 & ~(R * TT >= 64 ? 63 : R * TT == 32 ? 59 : R * TT == 16 ? 57 : 56)) == 0;

    for (int tile = 0; tile < tiles; ++tile) {
        const int64_t row0 = (static_cast<int64_t>(blockIdx.x) * tiles + tile) * R;
        if (row0 >= N) return;
        const uint8_t* wr[R];
        const float* sr[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int64_t row = row0 + r < N ? row0 + r : N - 1;
            wr[r] = W + row * row_bytes;
            sr[r] = S + row * G;
        }
        float acc[R * TT];
#pragma unroll
        for (int i = 0; i < R * TT; ++i) acc[i] = 0.0f;
        for (int c0 = 0; c0 < chunks; c0 += kWave) {
            const int c = c0 + lane;
            const bool cv = FULL || c < chunks;
            u32x4 wv[R];
            float sc[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                wv[r] = ldg(cv ? reinterpret_cast<const u32x4*>(wr[r]) + c : z);
                sc[r] = ldg(cv ? sr[r] + (32 * c) / gs : zf);
            }
            if (!one_pass || tile == 0) {
#pragma unroll
                for (int t = 0; t < TT; ++t) {
                    const int tk = t0 + t < T ? t0 + t : T - 1;
                    const u32x4* xp = reinterpret_cast<const u32x4*>(X + static_cast<int64_t>(tk) * K) + 4 * c;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const u32x4 q = ldg(cv ? xp + i : z);
                        xv[t][4 * i + 0] = as_f16x2(q.x);
                        xv[t][4 * i + 1] = as_f16x2(q.y);
                        xv[t][4 * i + 2] = as_f16x2(q.z);
                        xv[t][4 * i + 3] = as_f16x2(q.w);
                    }
                }
                const f16x2 ones = {(f16)1.0f, (f16)1.0f};
#pragma unroll
                for (int t = 0; t < TT; ++t) {
                    float s = 0.0f;
#pragma unroll
                    for (int e = 0; e < 16; ++e) s = dot2(xv[t][e], ones, s);
                    xs[t] = -8.0f * s;
                }
            }
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const uint32_t wd[4] = {wv[r].x, wv[r].y, wv[r].z, wv[r].w};
                f16x2 lo[4][2], hi[4][2];
#pragma unroll
                for (int i = 0; i < 4; ++i) int4x8_subnormal_bitfield(wd[i], lo[i], hi[i]);
#pragma unroll
                for (int t = 0; t < TT; ++t) {
                    float ta = 0.0f, tb = 0.0f;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        ta = dot2(lo[i][0], xv[t][4 * i + 0], ta);
                        tb = dot2(hi[i][0], xv[t][4 * i + 1], tb);
                        ta = dot2(lo[i][1], xv[t][4 * i + 2], ta);
                        tb = dot2(hi[i][1], xv[t][4 * i + 3], tb);
                    }
                    const float v = fmaf(ta, kTwo24, fmaf(tb, kTwo20, xs[t]));
                    acc[t * R + r] = fmaf(sc[r], v, acc[t * R + r]);
                }
            }
        }
        const float total = reduce_tile<R * TT>(acc, lane);
        if (writer && t0 + vt < T && row0 + vr < N) ep.store(static_cast<int64_t>(t0 + vt) * N + row0 + vr, total);
    }
}

// h[t, i] = fp16(silu(gate) * up) of the [gate | up] rows of gu [T, 2 I] (INTERLEAVED: rows in 8-row tiles of 4 gate
// and the 4 matching up rows).
template <bool INTERLEAVED>
__global__ __launch_bounds__(256) void silu_tokens_kernel(const uint16_t* __restrict__ gu, uint16_t* __restrict__ h,
                                                          int64_t n, int I) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n) return;
    const int64_t t = i / I;
    const int c = static_cast<int>(i - t * I);
    const uint16_t* row = gu + t * 2 * I;
    const int gi = INTERLEAVED ? 8 * (c >> 2) + (c & 3) : c;
    const float g = f16_bits_to_f32(ldg(row + gi)), u = f16_bits_to_f32(ldg(row + gi + (INTERLEAVED ? 4 : I)));
    stg(h + i, f32_to_f16_bits(silu_f32(g) * u));
}

// ---------------------------------------------------------------------------
// q/k norm, RoPE and KV append
// ---------------------------------------------------------------------------
// Token t is at position p = pos[0] + t. One wave per (head, token), the arithmetic of the decode step's prologue:
// q rows go to q_out [T, NQ, hd], k rows normed and rotated and v rows as they are to the caches at p. Past the
// cache (p >= max_seq) q takes the last table row and nothing is appended, as in the step.
constexpr int kRopeWaves = 4;

__global__ __launch_bounds__(kRopeWaves * kWave) void qk_norm_rope_tokens_kernel(
    const uint16_t* __restrict__ qkv, const uint16_t* __restrict__ q_norm, const uint16_t* __restrict__ k_norm,
    const float* __restrict__ cos_t, const float* __restrict__ sin_t, const int32_t* __restrict__ pos_ptr,
    uint16_t* __restrict__ q_out, uint16_t* __restrict__ kc, uint16_t* __restrict__ vc, int NQ, int NKV, int S, int hd,
    float eps) {
    const int lane = threadIdx.x & 63;
    const int heads = NQ + 2 * NKV;
    const int h = static_cast<int>(blockIdx.x) * kRopeWaves + static_cast<int>(threadIdx.x >> 6);
    if (h >= heads) return;  // wave-uniform
    const int t = blockIdx.y;
    const int p = ldg(pos_ptr) + t;
    const bool pvalid = p >= 0 && p < S;
    const int prow = pvalid ? p : (p < 0 ? 0 : S - 1);
    const int half = hd >> 1;
    const uint16_t* src = qkv + (static_cast<int64_t>(t) * heads + h) * hd;
    if (h >= NQ + NKV) {
        if (!pvalid) return;
        uint16_t* vd = vc + (static_cast<int64_t>(h - NQ - NKV) * S + p) * hd;
        for (int i = lane; i < hd; i += kWave) stg(vd + i, ldg(src + i));
        return;
    }
    if (h >= NQ && !pvalid) return;
    const uint16_t* wn = h < NQ ? q_norm : k_norm;
    float ss = 0.0f;
    for (int i = lane; i < hd; i += kWave) {
        const float v = f16_bits_to_f32(ldg(src + i));
        ss = fmaf(v, v, ss);
    }
    const float inv = rsqrtf(wave_sum_bcast(ss) / static_cast<float>(hd) + eps);
    uint16_t* dst = h < NQ ? q_out + (static_cast<int64_t>(t) * NQ + h) * hd
                           : kc + (static_cast<int64_t>(h - NQ) * S + p) * hd;
    for (int i = lane; i < half; i += kWave) {
        const float a = f16_bits_to_f32(
            f32_to_f16_bits(f16_bits_to_f32(ldg(src + i)) * inv * f16_bits_to_f32(ldg(wn + i))));
        const float b = f16_bits_to_f32(f32_to_f16_bits(f16_bits_to_f32(ldg(src + i + half)) * inv *
                                                        f16_bits_to_f32(ldg(wn + i + half))));
        float o1, o2;
        rope_pair(a, b, ldg(cos_t + static_cast<int64_t>(prow) * half + i),
                  ldg(sin_t + static_cast<int64_t>(prow) * half + i), o1, o2);
        stg(dst + i, f32_to_f16_bits(o1));
        stg(dst + i + half, f32_to_f16_bits(o2));
    }
}

// ---------------------------------------------------------------------------
// attention of every prompt token
// ---------------------------------------------------------------------------
// Workgroup (query head h, token t): attention over pos[0] + t + 1 timesteps with the decode attention's passes,
// split plan and combine. The splits of a longer context run one after another in the workgroup and leave their
// states in LDS, so there is no workspace, arrival or second launch: the T x NQ workgroups fill the chip without
// splitting a token over several.
template <int LPR>
__global__ __launch_bounds__(kAttnThreads) void attn_tokens_kernel(const uint16_t* __restrict__ q,
                                                                   const uint16_t* __restrict__ kc,
                                                                   const uint16_t* __restrict__ vc,
                                                                   uint16_t* __restrict__ out,
                                                                   const int32_t* __restrict__ pos_ptr, int NQ, int NKV,
                                                                   int S, float scale_log2, int frag) {
    constexpr int HD = LPR * 8;
    constexpr int RPI = kWave / LPR;
    constexpr int STEP = RPI * kAttnWaves;
    __shared__ float s_state[kAttnWaves][1][HD + 2];
    extern __shared__ float s_split[];  // [splits][HD + 2], a split context only
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int u = lane % LPR;
    const int h = blockIdx.x, t_q = blockIdx.y;
    const int kvh = h / (NQ / NKV);
    const int p = ldg(pos_ptr) + t_q;
    const int L = p < 0 ? 1 : (p >= S ? S : p + 1);
    int tps, ns;
    split_plan(L, NKV, STEP, tps, ns);
    const uint16_t* kbase = kc + static_cast<int64_t>(kvh) * S * HD;
    const uint16_t* vbase = vc + static_cast<int64_t>(kvh) * S * HD;
    const int64_t qo = (static_cast<int64_t>(t_q) * NQ + h) * HD;
    // element d of the head's output: fragment layout (the o projection's x on the matrix cores) or [T, NQ * HD]
    auto out_at = [&](int d) { return out + (frag ? frag_offset(t_q, h * HD + d, static_cast<int64_t>(NQ) * HD) : qo + d); };
    f16x2 qv[1][4];
    {
        const u32x4 r = ldg(reinterpret_cast<const u32x4*>(q + qo) + u);
        qv[0][0] = as_f16x2(r.x);
        qv[0][1] = as_f16x2(r.y);
        qv[0][2] = as_f16x2(r.z);
        qv[0][3] = as_f16x2(r.w);
    }
    for (int split = 0; split < ns; ++split) {
        const int t0 = split * tps, t1 = min(L, t0 + tps);
        const int tb0 = t0 + wave * RPI;
        const int npass = (t1 - t0 + STEP - 1) / STEP;
        AttnState<LPR, 1> st;
        attn_range<LPR, 1>(st, qv, kbase, vbase, tb0, t1, npass, scale_log2);
        attn_wave_state<LPR, 1, HD>(st, s_state[wave], lane);
        __syncthreads();
        for (int e = tid; e < HD + 2; e += kAttnThreads) {
            float w[kAttnWaves];
            const float M = wave_weights<1, HD>(s_state, 0, w);
            const float v = e == 0 ? M : wave_sum<1, HD>(s_state, 0, e, w);
            if (ns > 1) {
                s_split[split * (HD + 2) + e] = v;
            } else if (e >= 2) {
                const float lsum = wave_sum<1, HD>(s_state, 0, 1, w);
                stg(out_at(e - 2), f32_to_f16_bits(v / lsum));
            }
        }
        __syncthreads();  // the split's state is read before the next split's waves overwrite s_state
    }
    if (ns == 1) return;
    for (int d = tid; d < HD; d += kAttnThreads) {
        float M = kNegBig;
        for (int s = 0; s < ns; ++s) M = fmaxf(M, s_split[s * (HD + 2)]);
        float lsum = 0.0f, acc = 0.0f;
        for (int s = 0; s < ns; ++s) {
            const float w = fast_exp2(s_split[s * (HD + 2)] - M);
            lsum = fmaf(s_split[s * (HD + 2) + 1], w, lsum);
            acc = fmaf(s_split[s * (HD + 2) + 2 + d], w, acc);
        }
        stg(out_at(d), f32_to_f16_bits(acc / lsum));
    }
}

// ---------------------------------------------------------------------------
// host
// ---------------------------------------------------------------------------

// LDS of the split states of a context of up to max_seq timesteps; 0: head_dim outside the fast attention kernels,
// or more states than one workgroup's LDS takes.
static size_t attn_tokens_lds(int64_t NQ, int64_t NKV, int64_t hd, int64_t max_seq) {
    const int64_t lpr = hd / 8;
    if (NKV < 1 || NQ % NKV || hd % 8 || lpr < 1 || lpr > 32 || (lpr & (lpr - 1)) || NQ / NKV > 8 ||
        max_seq * NKV >= (int64_t(1) << 31))
        return 0;
    const int64_t step = (kWave / lpr) * kAttnWaves;
    const int64_t by_len = ceil_div64(max_seq, step), by_heads = ceil_div64(kAttnTargetGroups, NKV);
    const int64_t cap = by_len < by_heads ? by_len : by_heads;
    const size_t bytes = static_cast<size_t>(cap < 1 ? 1 : cap) * static_cast<size_t>(hd + 2) * sizeof(float);
    return bytes <= 48 * 1024 ? bytes : 0;
}

static int check_tokens(int64_t T, const char* what) {
    SOI_REQUIRE(T >= 1 && T <= 65535, "%s: the token count must be in [1, 65535], got %lld", what, (long long)T);
    return SOI_OK;
}

// R rows x 8 tokens per tile for 5 tokens up, x 4 below; row tiles per wave so that about 2048 waves (8 per CU) are
// left: fewer would leave SIMDs idle, more would load the tokens' x again for each.
template <class EP>
static int launch_gemm_tokens(const uint8_t* W, const float* S, const uint16_t* X, int64_t N, int64_t K, int64_t gs,
                              int64_t T, const EP& ep, hipStream_t st, const char* what) {
    const int64_t row_bytes = K / 2, G = ceil_div64(K, gs);
    const bool full = (K / 32) % kWave == 0;
    constexpr int R = 4;
    const int TT = T > 4 ? 8 : 4;
    const int64_t tt = ceil_div64(T, TT), rt = ceil_div64(N, R);
    int64_t tiles = rt * tt / 2048;
    tiles = tiles < 1 ? 1 : tiles > 16 ? 16 : tiles;
    const dim3 grid(static_cast<unsigned>(ceil_div64(rt, tiles)), static_cast<unsigned>(tt));
#define SOI_T(TTT, FL)                                                                                              \
    hipLaunchKernelGGL((gemm_int4_tokens_kernel<R, TTT, FL, EP>), grid, dim3(kWave), 0, st, W, S, row_bytes,       \
                       static_cast<int>(G), X, N, static_cast<int>(K), static_cast<int>(gs), static_cast<int>(T),  \
                       static_cast<int>(tiles), ep)
    if (TT == 8) {
        if (full) SOI_T(8, true); else SOI_T(8, false);
    } else {
        if (full) SOI_T(4, true); else SOI_T(4, false);
    }
#undef SOI_T
    return launch_status(what);
}

}  // namespace soi

using namespace soi;

extern "C" int soi_embed_tokens(const uint16_t* table, int64_t rows, int64_t hidden, const int32_t* tokens, int64_t T,
                                uint16_t* out, void* stream) {
    const char* what = "soi_embed_tokens";
    int s = check_tokens(T, what);
    if (s) return s;
    SOI_REQUIRE(rows >= 1 && hidden >= 1 && hidden <= (int64_t(1) << 24), "%s: size out of range", what);
    SOI_REQUIRE(table && tokens && out, "%s: null pointer", what);
    hipLaunchKernelGGL(embed_tokens_kernel, dim3(static_cast<unsigned>(T)), dim3(256), 0, as_stream(stream), table,
                       rows, static_cast<int>(hidden), tokens, out);
    return launch_status(what);
}

extern "C" int soi_norm_tokens(const uint16_t* x, const uint16_t* weight, float eps, uint16_t* h, int64_t T,
                               int64_t hidden, int one_pass, int frag, void* stream) {
    const char* what = "soi_norm_tokens";
    int s = check_tokens(T, what);
    if (s) return s;
    SOI_REQUIRE(hidden >= 8 && hidden % 8 == 0 && hidden <= (int64_t(1) << 24),
                "%s: hidden must be a multiple of 8 in [8, 2^24]", what);
    SOI_REQUIRE(!frag || hidden % 128 == 0, "%s: the fragment layout needs hidden %% 128 == 0", what);
    SOI_REQUIRE(!one_pass || hidden == 2048, "%s: the one-pass partition is for hidden = 2048", what);
    SOI_REQUIRE(x && weight && h && h != x, "%s: null pointer or h = x", what);
    SOI_REQUIRE(aligned16(x) && aligned16(weight) && aligned16(h), "%s: vectors must be 16-byte aligned", what);
    const dim3 grid(static_cast<unsigned>(ceil_div64(T, kNormTokens)));
    if (one_pass)
        hipLaunchKernelGGL(norm_tokens_kernel<true>, grid, dim3(kNormTokens * kWave), 0, as_stream(stream), x, weight,
                           eps, h, static_cast<int>(T), static_cast<int>(hidden), frag);
    else
        hipLaunchKernelGGL(norm_tokens_kernel<false>, grid, dim3(kNormTokens * kWave), 0, as_stream(stream), x, weight,
                           eps, h, static_cast<int>(T), static_cast<int>(hidden), frag);
    return launch_status(what);
}

extern "C" int soi_gemm_w4a16_tokens(const uint8_t* Wq, const float* scale, const uint16_t* x, uint16_t* y, int64_t N,
                                     int64_t K, int64_t group_size, int64_t T, int add, void* stream) {
    const char* what = "soi_gemm_w4a16_tokens";
    int s = check_tokens(T, what);
    if (s) return s;
    SOI_REQUIRE(N >= 1 && N <= (int64_t(1) << 31) - 1, "%s: N out of range", what);
    SOI_REQUIRE(K >= 32 && K % 32 == 0 && K <= (int64_t(1) << 30), "%s: K must be a multiple of 32", what);
    SOI_REQUIRE(group_size >= 32 && group_size % 32 == 0, "%s: group_size must be a multiple of 32", what);
    SOI_REQUIRE(Wq && scale && x && y && y != x, "%s: null pointer or y = x", what);
    SOI_REQUIRE(aligned16(Wq) && aligned16(x), "%s: weights and x must be 16-byte aligned", what);
    hipStream_t st = as_stream(stream);
    if (add) return launch_gemm_tokens(Wq, scale, x, N, K, group_size, T, TokenAdd{y}, st, what);
    return launch_gemm_tokens(Wq, scale, x, N, K, group_size, T, TokenStore{y}, st, what);
}

extern "C" int soi_silu_mul_tokens(const uint16_t* gate_up, uint16_t* h, int64_t T, int64_t I, int interleaved,
                                   void* stream) {
    const char* what = "soi_silu_mul_tokens";
    int s = check_tokens(T, what);
    if (s) return s;
    SOI_REQUIRE(I >= 1 && I <= (int64_t(1) << 30) && (!interleaved || I % 4 == 0), "%s: I out of range", what);
    SOI_REQUIRE(gate_up && h, "%s: null pointer", what);
    const int64_t n = T * I;
    SOI_REQUIRE(ceil_div64(n, 256) <= (int64_t(1) << 31) - 1, "%s: T * I out of range", what);
    const dim3 grid(static_cast<unsigned>(ceil_div64(n, 256)));
    if (interleaved)
        hipLaunchKernelGGL(silu_tokens_kernel<true>, grid, dim3(256), 0, as_stream(stream), gate_up, h, n,
                           static_cast<int>(I));
    else
        hipLaunchKernelGGL(silu_tokens_kernel<false>, grid, dim3(256), 0, as_stream(stream), gate_up, h, n,
                           static_cast<int>(I));
    return launch_status(what);
}

extern "C" int soi_qk_norm_rope_tokens(const uint16_t* qkv, const uint16_t* q_norm, const uint16_t* k_norm,
                                       const float* cos_table, const float* sin_table, const int32_t* pos,
                                       uint16_t* q_out, uint16_t* k_cache, uint16_t* v_cache, int64_t T,
                                       int64_t num_q_heads, int64_t num_kv_heads, int64_t max_seq, int64_t head_dim,
                                       float eps, void* stream) {
    const char* what = "soi_qk_norm_rope_tokens";
    int s = check_tokens(T, what);
    if (s) return s;
    SOI_REQUIRE(num_q_heads >= 1 && num_kv_heads >= 1 && num_q_heads + 2 * num_kv_heads <= 65535,
                "%s: head counts out of range", what);
    SOI_REQUIRE(head_dim >= 2 && head_dim % 2 == 0 && head_dim <= 4096, "%s: head_dim must be even, in [2, 4096]",
                what);
    SOI_REQUIRE(max_seq >= 1 && max_seq <= (int64_t(1) << 30), "%s: max_seq_len out of range", what);
    SOI_REQUIRE(qkv && q_norm && k_norm && cos_table && sin_table && pos && q_out && k_cache && v_cache,
                "%s: null pointer", what);
    const dim3 grid(static_cast<unsigned>(ceil_div64(num_q_heads + 2 * num_kv_heads, kRopeWaves)),
                    static_cast<unsigned>(T));
    hipLaunchKernelGGL(qk_norm_rope_tokens_kernel, grid, dim3(kRopeWaves * kWave), 0, as_stream(stream), qkv, q_norm,
                       k_norm, cos_table, sin_table, pos, q_out, k_cache, v_cache, static_cast<int>(num_q_heads),
                       static_cast<int>(num_kv_heads), static_cast<int>(max_seq), static_cast<int>(head_dim), eps);
    return launch_status(what);
}

extern "C" int soi_attention_tokens_supported(int64_t NQ, int64_t NKV, int64_t head_dim, int64_t max_seq) {
    return attn_tokens_lds(NQ, NKV, head_dim, max_seq) > 0 ? 1 : 0;
}

extern "C" int soi_attention_tokens(const uint16_t* q, const uint16_t* k_cache, const uint16_t* v_cache, uint16_t* out,
                                    const int32_t* pos, int64_t T, int64_t NQ, int64_t NKV, int64_t max_seq,
                                    int64_t head_dim, float scale, int frag, void* stream) {
    const char* what = "soi_attention_tokens";
    int s = check_tokens(T, what);
    if (s) return s;
    SOI_REQUIRE(NQ >= 1 && NKV >= 1 && NQ % NKV == 0 && max_seq >= 1, "%s: bad head counts or max_seq_len", what);
    SOI_REQUIRE(q && k_cache && v_cache && out && pos, "%s: null pointer", what);
    SOI_REQUIRE(!frag || NQ * head_dim % 128 == 0, "%s: the fragment layout needs NQ * head_dim %% 128 == 0", what);
    const size_t lds = attn_tokens_lds(NQ, NKV, head_dim, max_seq);
    if (!lds) {
        set_last_error("%s: head_dim must be a power of two in [8, 256], at most 8 query heads per KV head and a "
                       "context whose split states fit in 48 KB",
                       what);
        return SOI_ERR_UNSUPPORTED;
    }
    SOI_REQUIRE(aligned16(q) && aligned16(k_cache) && aligned16(v_cache), "%s: operands must be 16-byte aligned", what);
    const dim3 grid(static_cast<unsigned>(NQ), static_cast<unsigned>(T));
    const float scale_log2 = scale * kLog2e;
    hipStream_t st = as_stream(stream);
#define SOI_A(LL)                                                                                                     \
    hipLaunchKernelGGL(attn_tokens_kernel<LL>, grid, dim3(kAttnThreads), lds, st, q, k_cache, v_cache, out, pos,      \
                       static_cast<int>(NQ), static_cast<int>(NKV), static_cast<int>(max_seq), scale_log2, frag)
    switch (head_dim / 8) {
        case 1: SOI_A(1); break;
        case 2: SOI_A(2); break;
        case 4: SOI_A(4); break;
        case 8: SOI_A(8); break;
        case 16: SOI_A(16); break;
        default: SOI_A(32); break;
    }
#undef SOI_A
    return launch_status(what);
}
