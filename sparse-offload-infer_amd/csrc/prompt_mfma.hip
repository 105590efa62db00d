// INT4 rows x prompt tokens on the matrix cores (gfx950): y[t, n] = sum_k s[n, k/gs] q[n, k] x[t, k] for T tokens.
//
// A prompt's linears are contractions over many tokens, which v_dot2 (prompt.hip, the decode step's order) runs at a
// tenth of the matrix cores' rate. Here a wave holds 16-row x 16-token tiles of v_mfma_f32_16x16x32_f16:
//   * operands are exact: the nibbles become binary16 integers in registers (dequant_int4x8_bitfield), x is binary16,
//     products and sums are binary32. The sum over a 128-element step starts from zero and enters the total as
//     total = fma(scale, sum, total), so the fp32 scale multiplies a binary32 sum, as in the GEMV;
//   * lane (m = lane & 15, g = lane >> 4) loads 16 bytes of row m: the 32 elements 128 s + 32 g .. + 31 of step s,
//     one packed word per MFMA. The MFMA's k slots (g, j) of instruction i are elements 128 s + 32 g + 8 i + j for
//     both operands (a contraction may take its terms in any order), so the weights need no rearranging;
//   * x comes in fragment layout (soi_prompt.h): each operand load is 1 KB contiguous. Read from [T, K] rows, whose
//     16 tokens lie 2 K bytes apart and so share L1 sets and an L2 channel, x arrived at 11 bytes per clock and CU
//     (2048 x 6144, 64 tokens: 28 us);
//   * the KW waves of a workgroup take every KW-th step of the same tile and meet in LDS (fixed order), so a short
//     launch (2048 rows x 64 tokens) still has waves on every SIMD and each wave's loads are a fraction of a row.
// Sums run in another order than the GEMV's, with the same operands, products and accumulator width (error against
// binary64 over 9 to 1000 tokens and the Qwen3-1.7B linears: 2.07e-4 rms, the GEMV's order 2.08e-4).
//
// Measured, 256 tokens: 12288 x 2048 28.6 us (450 TFLOP/s) against 182 us on v_dot2, 2048 x 6144 16.4 against 118,
// 4096 x 2048 12.8 against 70, 2048 x 2048 8.6 against 39. Bound by the operands' way into the registers: every
// workgroup reads its own x tiles from L2.
#include "soi_device.h"
#include "soi_host.h"
#include "soi_prompt.h"

namespace soi {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// Epilogues: lane (n, g) holds the totals of rows row .. row + 3 of one token.
struct MfmaStore {  // y[t, row] = fp16(total)
    uint16_t* y;
    __device__ __forceinline__ void store(int64_t t, int64_t row, int64_t N, const f32x4& v, int) const {
        if (row >= N) return;  // N % 4 == 0
        u32x2 o = {pack_f16x2(v.x, v.y), pack_f16x2(v.z, v.w)};
        stg(reinterpret_cast<u32x2*>(y + t * N + row), o);
    }
};
struct MfmaAdd {  // x[t, row] = x[t, row] + fp16(total), one binary16 addition
    uint16_t* x;
    __device__ __forceinline__ void store(int64_t t, int64_t row, int64_t N, const f32x4& v, int) const {
        if (row >= N) return;
        u32x2* p = reinterpret_cast<u32x2*>(x + t * N + row);
        const u32x2 a = ldg(p);
        u32x2 o = {add_f16x2(a.x, pack_f16x2(v.x, v.y)), add_f16x2(a.y, pack_f16x2(v.z, v.w))};
        stg(p, o);
    }
};
struct MfmaSwiglu {  // rows in 8-row tiles, 4 gate then 4 up: h[t, row / 2 ..] = fp16(silu(fp16 gate) * fp16 up)
    uint16_t* h;  // [T, N / 2] in fragment layout: the next product's x
    __device__ __forceinline__ void store(int64_t t, int64_t row, int64_t N, const f32x4& v, int g) const {
        float u[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) u[i] = __shfl_xor(v[i], 16, kWave);  // a gate row's up row is 16 lanes on
        if (row >= N || (g & 1)) return;
        float o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            o[i] = silu_f32(f16_bits_to_f32(f32_to_f16_bits(v[i]))) * f16_bits_to_f32(f32_to_f16_bits(u[i]));
        u32x2 w = {pack_f16x2(o[0], o[1]), pack_f16x2(o[2], o[3])};
        stg(reinterpret_cast<u32x2*>(h + frag_offset(t, row >> 1, N >> 1)), w);
    }
};

template <int MF, int NF>
struct MfmaStep {  // the operands of one 128-element step
    u32x4 a[MF], b[NF][4];
    float s[MF][4];
};

template <int MF, int NF, int KW, class EP>
__global__ __launch_bounds__(KW * kWave) __attribute__((amdgpu_waves_per_eu(1, KW / 4 * 2))) void gemm_int4_mfma_kernel(const uint8_t* __restrict__ W,
                                                                    const float* __restrict__ S, int64_t row_bytes,
                                                                    int G, const uint16_t* __restrict__ X, int64_t N,
                                                                    int K, int spg, int T, EP ep) {
    __shared__ f32x4 red[KW][MF * NF][kWave];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m = lane & 15, g = lane >> 4;
    const int64_t row0 = static_cast<int64_t>(blockIdx.x) * (16 * MF);
    const int t0 = static_cast<int>(blockIdx.y) * (16 * NF);
    const int steps = K >> 7;
    const uint8_t* wa[MF];
    const float* ws[MF];
#pragma unroll
    for (int f = 0; f < MF; ++f) {
        const int64_t ra = row0 + 16 * f + m, rs = row0 + 16 * f + 4 * g;  // rows past N read the last ones
        wa[f] = W + (ra < N ? ra : N - 1) * row_bytes + 16 * g;
        ws[f] = S + (rs < N ? rs : N - 4) * G;
    }
    const uint16_t* xb[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) {
        const int tt = (t0 >> 4) + f, last = (T - 1) >> 4;  // tiles past the last one read the last one
        xb[f] = X + static_cast<int64_t>(tt < last ? tt : last) * 16 * K + 8 * lane;
    }
    auto load = [&](MfmaStep<MF, NF>& o, int s) {
#pragma unroll
        for (int f = 0; f < MF; ++f) {
            o.a[f] = ldg(reinterpret_cast<const u32x4*>(wa[f] + 64 * s));
#pragma unroll
            for (int i = 0; i < 4; ++i) o.s[f][i] = ldg(ws[f] + static_cast<int64_t>(i) * G + s / spg);
        }
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int i = 0; i < 4; ++i) o.b[f][i] = ldg(reinterpret_cast<const u32x4*>(xb[f] + static_cast<int64_t>(s) * 2048 + 512 * i));
    };
    f32x4 acc[MF][NF];
#pragma unroll
    for (int f = 0; f < MF; ++f)
#pragma unroll
        for (int n = 0; n < NF; ++n) acc[f][n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    MfmaStep<MF, NF> cur;
    if (wave < steps) load(cur, wave);
    for (int s = wave; s < steps; s += KW) {
        MfmaStep<MF, NF> nxt;
        load(nxt, s + KW < steps ? s + KW : s);  // the next step's operands are in flight during this one's MFMAs
        __builtin_amdgcn_sched_barrier(0);       // (without the barrier the scheduler sinks these loads to their use)
#pragma unroll
        for (int f = 0; f < MF; ++f) {
            f16x8 a[4];
            const uint32_t wd[4] = {cur.a[f].x, cur.a[f].y, cur.a[f].z, cur.a[f].w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                f16x2 q[4];
                dequant_int4x8_bitfield(wd[i], q);
                a[i] = f16x8{q[0].x, q[0].y, q[1].x, q[1].y, q[2].x, q[2].y, q[3].x, q[3].y};
            }
            f32x4 sum[NF];
#pragma unroll
            for (int n = 0; n < NF; ++n) sum[n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int n = 0; n < NF; ++n)
                    sum[n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], __builtin_bit_cast(f16x8, cur.b[n][i]),
                                                                    sum[n], 0, 0, 0);
#pragma unroll
            for (int n = 0; n < NF; ++n)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[f][n][i] = fmaf(cur.s[f][i], sum[n][i], acc[f][n][i]);
        }
        cur = nxt;
    }
#pragma unroll
    for (int f = 0; f < MF; ++f)
#pragma unroll
        for (int n = 0; n < NF; ++n) red[wave][f * NF + n][lane] = acc[f][n];
    __syncthreads();
#pragma unroll
    for (int f0 = 0; f0 < MF * NF; f0 += KW) {
        const int f = f0 + wave;
        if (f < MF * NF) {  // wave-uniform
            f32x4 v = red[0][f][lane];
#pragma unroll
            for (int w = 1; w < KW; ++w) v += red[w][f][lane];
            const int t = t0 + 16 * (f % NF) + m;
            if (16 * (f % NF) + t0 < T) {  // wave-uniform: the swiglu epilogue exchanges lanes
                const int64_t row = row0 + 16 * (f / NF) + 4 * g;
                if (t < T)
                    ep.store(t, row, N, v, g);
                // lanes of tokens past T take no part: their exchange partners (same token) are past T too
            }
        }
    }
}

template <class EP>
static int launch_gemm_mfma(const uint8_t* W, const float* S, const uint16_t* X, int64_t N, int64_t K, int64_t gs,
                            int64_t T, const EP& ep, hipStream_t st, const char* what) {
    const int64_t G = ceil_div64(K, gs);
    const int NF = T <= 16 ? 1 : T <= 32 ? 2 : 4;
    const int64_t tt = ceil_div64(T, 16 * NF);
    // taller tiles read x less often, shorter ones leave more workgroups: 4 x 16 rows from 512 workgroups on, 2 x 16
    // from 256; a launch that still has at most one workgroup per CU splits its steps over 8 waves instead of 4
    const int64_t r16 = ceil_div64(N, 16) * tt;  // 16-row tiles in all
    const int MF = r16 >= 4 * 512 ? 4 : r16 >= 2 * 256 ? 2 : 1;
    const int64_t wgs = ceil_div64(N, 16 * MF) * tt;
    const bool wide = MF <= 2 && wgs <= 256 && K >= 8 * 128;
    const dim3 grid(static_cast<unsigned>(ceil_div64(N, 16 * MF)), static_cast<unsigned>(tt));
#define SOI_M(MM, NN, KK)                                                                                           \
    hipLaunchKernelGGL((gemm_int4_mfma_kernel<MM, NN, KK, EP>), grid, dim3(KK * kWave), 0, st, W, S, K / 2,          \
                       static_cast<int>(G), X, N, static_cast<int>(K), static_cast<int>(gs / 128),                  \
                       static_cast<int>(T), ep)
#define SOI_MN(MM, KK)                                                                  \
    do {                                                                                \
        if (NF == 1) SOI_M(MM, 1, KK); else if (NF == 2) SOI_M(MM, 2, KK); else SOI_M(MM, 4, KK); \
    } while (0)
    if (MF == 4) SOI_MN(4, 4);
    else if (MF == 2 && wide) SOI_MN(2, 8);
    else if (MF == 2) SOI_MN(2, 4);
    else if (wide) SOI_MN(1, 8);
    else SOI_MN(1, 4);
#undef SOI_MN
#undef SOI_M
    return launch_status(what);
}

}  // namespace soi

using namespace soi;

extern "C" int soi_gemm_w4a16_mfma_supported(int64_t N, int64_t K, int64_t group_size) {
    return N >= 4 && N % 4 == 0 && K >= 128 && K % 128 == 0 && group_size >= 128 && group_size % 128 == 0 ? 1 : 0;
}

extern "C" int soi_gemm_w4a16_mfma(const uint8_t* Wq, const float* scale, const uint16_t* x, uint16_t* y, int64_t N,
                                   int64_t K, int64_t group_size, int64_t T, int epilogue, void* stream) {
    const char* what = "soi_gemm_w4a16_mfma";
    SOI_REQUIRE(T >= 1 && T <= 65535, "%s: the token count must be in [1, 65535], got %lld", what, (long long)T);
    SOI_REQUIRE(N <= (int64_t(1) << 31) - 1 && K <= (int64_t(1) << 30) && soi_gemm_w4a16_mfma_supported(N, K, group_size),
                "%s: N must be a multiple of 4, K and group_size multiples of 128", what);
    SOI_REQUIRE(epilogue >= 0 && epilogue <= 2 && (epilogue != 2 || N % 256 == 0), "%s: unknown epilogue, or SwiGLU with "
                "N not a multiple of 256", what);
    SOI_REQUIRE(Wq && scale && x && y && y != x, "%s: null pointer or y = x", what);
    SOI_REQUIRE(aligned16(Wq) && aligned16(x) && (reinterpret_cast<uintptr_t>(y) & 7u) == 0,
                "%s: weights and x must be 16-byte aligned, y 8-byte", what);
    hipStream_t st = as_stream(stream);
    if (epilogue == 0) return launch_gemm_mfma(Wq, scale, x, N, K, group_size, T, MfmaStore{y}, st, what);
    if (epilogue == 1) return launch_gemm_mfma(Wq, scale, x, N, K, group_size, T, MfmaAdd{y}, st, what);
    return launch_gemm_mfma(Wq, scale, x, N, K, group_size, T, MfmaSwiglu{y}, st, what);
}
