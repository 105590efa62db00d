// Building blocks of the batch-1 attention kernels (decode_attention.hip: one query token; prompt.hip: every token of a
// prompt): row requests, scores, the online-softmax chunk, the wave and workgroup states. See decode_attention.hip
// for the layout. Kernels built on them give the same bytes for the same query, rows and split plan.
#pragma once

#include "soi_attn_plan.h"
#include "soi_device.h"

namespace soi {

constexpr int kAttnWaves = 8;
constexpr int kAttnThreads = kAttnWaves * kWave;
constexpr float kNegBig = -1e30f;
constexpr float kLog2e = 1.4426950408889634f;

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Context length: the host value, or (device form) pos[0] + 1 clamped to [1, S].
__device__ __forceinline__ int cur_len_of(int L_arg, const int32_t* pos, int S) {
    if (!pos) return L_arg;
    const int p = ldg(pos);
    return p < 0 ? 1 : (p >= S ? S : p + 1);
}


// Sum over the LPR lanes of a row group, every lane of the group gets it. Up to
// 16 lanes this is DPP inside a 16-lane row (a few cycles per step, against
// ~100 for an LDS-crossbar shuffle): rotations by 8 and 4 (or the 8-lane
// mirror), then the two quad exchanges; each step doubles the lanes summed.
template <int LPR>
__device__ __forceinline__ float group_sum(float v) {
    if (LPR >= 16) {
        v += dpp_f<0x128>(v);  // row_ror:8
        v += dpp_f<0x124>(v);  // row_ror:4
    } else if (LPR == 8) {
        v += dpp_f<0x141>(v);  // row_half_mirror: lane i <-> 7-i
    }
    if (LPR >= 4) v += dpp_f<0x4e>(v);  // quad_perm [2,3,0,1]
    if (LPR >= 2) v += dpp_f<0xb1>(v);  // quad_perm [1,0,3,2]
    if (LPR == 32) v += xor_lanes<16>(v);
    return v;
}

template <int LPR, int REP>
struct AttnState {
    float m[REP], l[REP], acc[REP][8];
};

// Score of the lane's row (K kk) for every query head, pre-multiplied by scale * log2(e): v_dot2 over the
// lane's 8 dims, then a sum over the row's lanes (every lane of the group takes part); -inf for a row past the
// range. Heads past rep (rep not a power of two) are computed on head 0's q and never written.
template <int LPR, int REP>
__device__ __forceinline__ void attn_scores(float (&sc)[REP], const f16x2 (&qv)[REP][4], bool valid, const u32x4& kk,
                                            float scale_log2) {
    const f16x2 k0 = as_f16x2(kk.x), k1 = as_f16x2(kk.y), k2 = as_f16x2(kk.z), k3 = as_f16x2(kk.w);
#pragma unroll
    for (int hh = 0; hh < REP; ++hh) {
        float part_s = dot2(qv[hh][0], k0, 0.0f);
        part_s = dot2(qv[hh][1], k1, part_s);
        part_s = dot2(qv[hh][2], k2, part_s);
        part_s = dot2(qv[hh][3], k3, part_s);
        const float sc_h = group_sum<LPR>(part_s) * scale_log2;
        sc[hh] = valid ? sc_h : -__builtin_inff();
    }
}

// The lane's row (V vv) with weight 2^(sc - m) enters every query head's sum (m already covers sc).
template <int LPR, int REP>
__device__ __forceinline__ void attn_accumulate(AttnState<LPR, REP>& st, const float (&sc)[REP], const u32x4& vv) {
    const uint32_t vw[4] = {vv.x, vv.y, vv.z, vv.w};
    float v[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const f16x2 v2 = as_f16x2(vw[e]);
        v[2 * e] = static_cast<float>(v2.x);
        v[2 * e + 1] = static_cast<float>(v2.y);
    }
#pragma unroll
    for (int hh = 0; hh < REP; ++hh) {
        const float p = fast_exp2(sc[hh] - st.m[hh]);
        st.l[hh] += p;
#pragma unroll
        for (int d = 0; d < 8; ++d) st.acc[hh][d] = fmaf(p, v[d], st.acc[hh][d]);
    }
}

// a + b of lane pairs swapped across 16-lane rows (ROWS = 16) or wave halves (ROWS = 32) by
// v_permlane16_swap / v_permlane32_swap on two values (swap16 / swap32: the upper row of each pair of VDST
// trades places with the lower row of VSRC0): with vdst = x, vsrc = y, lanes of the lower row of each pair end
// with x of both rows, lanes of the upper row with y of both, summed in row order.
template <int ROWS>
__device__ __forceinline__ float swap_sum(float x, float y) {
    float a = x, b = y;
    if constexpr (ROWS == 16) {
        swap16(a, b);
    } else {
        swap32(a, b);
    }
    return a + b;
}

// Max over the lane groups of a wave (lane exchanges across masks LPR .. 32; the lanes of a group hold the
// same value): every lane gets it.
template <int LPR>
__device__ __forceinline__ float groups_max(float v) {
    if constexpr (LPR <= 1) v = fmaxf(v, xor_lanes<1>(v));
    if constexpr (LPR <= 2) v = fmaxf(v, xor_lanes<2>(v));
    if constexpr (LPR <= 4) v = fmaxf(v, xor_lanes<4>(v));
    if constexpr (LPR <= 8) v = fmaxf(v, xor_lanes<8>(v));
    if constexpr (LPR <= 16) {
        float a = v, b = v;
        swap16(a, b);
        v = fmaxf(a, b);
    }
    float a = v, b = v;
    swap32(a, b);
    return fmaxf(a, b);
}

// The wave's state into s_row (= s_state[wave]): its lane groups share the running max, so l and acc are plain
// sums over the groups. Groups inside a 16-lane row are summed by lane exchanges first (LPR < 16); the rows
// are then summed by a reduce-scatter of swap_sum: level 16 leaves row r with dims (2i + (r & 1)) of its 8,
// level 32 with dims r and 4 + r, each summed over the 4 rows in a fixed order (wave halves: dims 2i + half).
template <int LPR, int REP, int HD>
__device__ __forceinline__ void attn_wave_state(AttnState<LPR, REP>& st, float (*s_row)[HD + 2], int lane) {
    if constexpr (LPR < 16) {
#pragma unroll
        for (int mask = LPR; mask < 16; mask *= 2) {
#pragma unroll
            for (int hh = 0; hh < REP; ++hh) {
                if (mask == 1) st.l[hh] += xor_lanes<1>(st.l[hh]);
                if (mask == 2) st.l[hh] += xor_lanes<2>(st.l[hh]);
                if (mask == 4) st.l[hh] += xor_lanes<4>(st.l[hh]);
                if (mask == 8) st.l[hh] += xor_lanes<8>(st.l[hh]);
#pragma unroll
                for (int d = 0; d < 8; ++d) {
                    if (mask == 1) st.acc[hh][d] += xor_lanes<1>(st.acc[hh][d]);
                    if (mask == 2) st.acc[hh][d] += xor_lanes<2>(st.acc[hh][d]);
                    if (mask == 4) st.acc[hh][d] += xor_lanes<4>(st.acc[hh][d]);
                    if (mask == 8) st.acc[hh][d] += xor_lanes<8>(st.acc[hh][d]);
                }
            }
        }
    }
    const int u = lane % LPR;
#pragma unroll
    for (int hh = 0; hh < REP; ++hh) {
        if constexpr (LPR <= 16) {
            const float l2 = swap_sum<16>(st.l[hh], st.l[hh]);
            const float l4 = swap_sum<32>(l2, l2);
            float b[4], c[2];
#pragma unroll
            for (int i = 0; i < 4; ++i) b[i] = swap_sum<16>(st.acc[hh][2 * i], st.acc[hh][2 * i + 1]);
#pragma unroll
            for (int i = 0; i < 2; ++i) c[i] = swap_sum<32>(b[2 * i], b[2 * i + 1]);
            const int r = lane >> 4;
            if ((lane & 15) < LPR) {
                s_row[hh][2 + 8 * u + r] = c[0];
                s_row[hh][2 + 8 * u + 4 + r] = c[1];
            }
            if (lane == 0) {
                s_row[hh][0] = st.m[hh];
                s_row[hh][1] = l4;
            }
        } else {  // LPR == 32: two groups, the wave halves
            const float l2 = swap_sum<32>(st.l[hh], st.l[hh]);
            const int half = lane >> 5;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                s_row[hh][2 + 8 * u + 2 * i + half] = swap_sum<32>(st.acc[hh][2 * i], st.acc[hh][2 * i + 1]);
            if (lane == 0) {
                s_row[hh][0] = st.m[hh];
                s_row[hh][1] = l2;
            }
        }
    }
}

// The K/V rows of a chunk of up to kAttnPassMax passes, requested together.
// Pass i of wave w reads timestep tb0 + i*kAttnWaves*RPI + (lane / LPR) with
// tb0 = t0 + w*RPI; rows at or past t1 are clamped to t1 - 1 (a legal
// address) and masked out of the softmax.
template <int LPR>
struct AttnRows {
    u32x4 k[kAttnPassMax], v[kAttnPassMax];
    __device__ __forceinline__ void load(const uint16_t* kbase, const uint16_t* vbase, int tb0, int t1, int npass) {
        constexpr int HD = LPR * 8;
        constexpr int RPI = kWave / LPR;
        const int lane = threadIdx.x & 63;
        const int g = lane / LPR, u = lane % LPR;
        // pairs of passes past npass are not requested (one wave-uniform branch per pair, as the pass loop
        // takes them): a clamped request would repeat row t1 - 1, and repeated loads of one address queue
        // behind each other
#pragma unroll
        for (int i = 0; i < kAttnPassMax; i += 2) {
            if (i < npass) {
#pragma unroll
                for (int j = i; j < i + 2; ++j) {
                    const int t = tb0 + j * kAttnWaves * RPI + g;
                    const int tl = (j < npass && t < t1) ? t : t1 - 1;
                    k[j] = ldg(reinterpret_cast<const u32x4*>(kbase + static_cast<int64_t>(tl) * HD) + u);
                    v[j] = ldg(reinterpret_cast<const u32x4*>(vbase + static_cast<int64_t>(tl) * HD) + u);
                }
            }
        }
    }
};

// The waves' states of query head hh combined: M = the largest m, w[s] = 2^(m_s - M) (wave order).
template <int REP, int HD>
__device__ __forceinline__ float wave_weights(const float (*s_state)[REP][HD + 2], int hh, float (&w)[kAttnWaves]) {
    float M = kNegBig;
#pragma unroll
    for (int s = 0; s < kAttnWaves; ++s) M = fmaxf(M, s_state[s][hh][0]);
#pragma unroll
    for (int s = 0; s < kAttnWaves; ++s) w[s] = fast_exp2(s_state[s][hh][0] - M);
    return M;
}

// sum_s w[s] * (state element e of wave s), e = 1: l, e = 2 + d: acc[d]; in wave order.
template <int REP, int HD>
__device__ __forceinline__ float wave_sum(const float (*s_state)[REP][HD + 2], int hh, int e,
                                          const float (&w)[kAttnWaves]) {
    float v = 0.0f;
#pragma unroll
    for (int s = 0; s < kAttnWaves; ++s) v = fmaf(s_state[s][hh][e], w[s], v);
    return v;
}

// One chunk of up to kAttnPassMax passes whose rows are requested (pass j of the wave starts at timestep
// tb + j * kAttnWaves * RPI): the scores of every pass first (independent of each other), then the running max moves
// once to cover them all (acc, l rescaled once), then the rows enter the sums. The online-softmax recurrence of the
// reference with the chunk's rows as one step. Passes go in pairs: one uniform branch per pair; the second pass of
// a pair past the chunk scores -inf. PATCH: timestep tnew's row is knew / vnew instead.
template <int LPR, int REP, bool PATCH>
__device__ __forceinline__ void attn_chunk(AttnState<LPR, REP>& st, const f16x2 (&qv)[REP][4], const AttnRows<LPR>& rows,
                                           int tb, int t1, int np, int tnew, const u32x4& knew, const u32x4& vnew,
                                           float scale_log2) {
    constexpr int STEP = kWave / LPR * kAttnWaves;
    const int g = (threadIdx.x & 63) / LPR;
    float sc[kAttnPassMax][REP];
#pragma unroll
    for (int i = 0; i < kAttnPassMax; i += 2) {
        if (i < np) {
#pragma unroll
            for (int j = i; j < i + 2; ++j) {
                const int t = tb + j * STEP + g;
                const u32x4 kk = (PATCH && t == tnew) ? knew : rows.k[j];
                attn_scores<LPR, REP>(sc[j], qv, j < np && t < t1, kk, scale_log2);
            }
        } else {
#pragma unroll
            for (int j = i; j < i + 2; ++j)
#pragma unroll
                for (int hh = 0; hh < REP; ++hh) sc[j][hh] = -__builtin_inff();
        }
    }
#pragma unroll
    for (int hh = 0; hh < REP; ++hh) {
        float mn = st.m[hh];
#pragma unroll
        for (int j = 0; j < kAttnPassMax; ++j) mn = fmaxf(mn, sc[j][hh]);
        mn = groups_max<LPR>(mn);  // one running max for all the wave's lane groups
        const float corr = fast_exp2(st.m[hh] - mn);
        st.l[hh] *= corr;
#pragma unroll
        for (int d = 0; d < 8; ++d) st.acc[hh][d] *= corr;
        st.m[hh] = mn;
    }
#pragma unroll
    for (int i = 0; i < kAttnPassMax; i += 2) {
        if (i < np) {
#pragma unroll
            for (int j = i; j < i + 2; ++j) {
                const int t = tb + j * STEP + g;
                const u32x4 vv = (PATCH && t == tnew) ? vnew : rows.v[j];
                attn_accumulate<LPR, REP>(st, sc[j], vv);
            }
        }
    }
}

template <int LPR, int REP>
__device__ __forceinline__ void attn_state_zero(AttnState<LPR, REP>& st) {
#pragma unroll
    for (int hh = 0; hh < REP; ++hh) {
        st.m[hh] = kNegBig;
        st.l[hh] = 0.0f;
#pragma unroll
        for (int d = 0; d < 8; ++d) st.acc[hh][d] = 0.0f;
    }
}

// The wave's state over the npass passes of timesteps [tb0.., t1) of one KV head's cache.
template <int LPR, int REP>
__device__ __forceinline__ void attn_range(AttnState<LPR, REP>& st, const f16x2 (&qv)[REP][4], const uint16_t* kbase,
                                           const uint16_t* vbase, int tb0, int t1, int npass, float scale_log2) {
    constexpr int STEP = kWave / LPR * kAttnWaves;
    attn_state_zero(st);
    AttnRows<LPR> rows;
    for (int c0 = 0; c0 < npass; c0 += kAttnPassMax) {
        const int np = npass - c0 < kAttnPassMax ? npass - c0 : kAttnPassMax;
        rows.load(kbase, vbase, tb0 + c0 * STEP, t1, np);
        attn_chunk<LPR, REP, false>(st, qv, rows, tb0 + c0 * STEP, t1, np, -1, u32x4{0u, 0u, 0u, 0u},
                                    u32x4{0u, 0u, 0u, 0u}, scale_log2);
    }
}

}  // namespace soi
