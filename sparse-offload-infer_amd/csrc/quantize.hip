// Symmetric group quantization and INT4 packing on the device (gfx950): the producers of every INT4 kernel's bytes.
//
// Same values as the tensor expressions of soinfer/quant/formats.py and pack.py (reference python/soinfer/quant/
// formats.py:24-123, pack.py:14-69): scale = max(|w|) / qmax by IEEE division, floored at the smallest normal
// binary32; q = clamp(round_half_even(w / scale), -qmax, qmax), again by IEEE division; NaN and infinities as there.
//
// Bound by HBM: one pass over the weights, each element read once and each code written once. A 6144 x 2048 binary32
// matrix takes 15.3 us to quantize from HBM (63 MB, 4.1 TB/s; 12.2 us once the last-level cache holds it) and 5.0 us to
// pack (19 MB, 3.8 TB/s; 3.2); 4 elements per lane instead of 8 took 2 us longer. As tensor operations the two were 25
// passes, 338 us.
#include "soi_device.h"
#include "soi_host.h"

namespace soi {

constexpr int kQuantThreads = 256;

// 4 consecutive elements of one row from element k0 on (zeros past K).
template <bool VEC>
__device__ __forceinline__ f32x4 load4(const float* row, int64_t k0, int64_t K) {
    if (VEC) {
        const f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f};
        return k0 < K ? ldg(reinterpret_cast<const f32x4*>(row + k0)) : z;
    }
    f32x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = k0 + i < K ? ldg(row + k0 + i) : 0.0f;
    return v;
}

// LPG lanes per group of 8 LPG elements; lane `sub` takes elements 4 sub .. + 3 of each half, so both loads of a wave are
// contiguous and in flight together. The group's largest magnitude is taken on the bit patterns (non-negative
// binary32 order like unsigned integers, NaN above infinity: torch.amax's order).
template <int LPG, bool VEC>
__global__ __launch_bounds__(kQuantThreads) void quantize_group_kernel(const float* __restrict__ w,
                                                                       int8_t* __restrict__ q, float* __restrict__ scale,
                                                                       int64_t groups, int G, int64_t K, float qmax) {
    const int64_t id = static_cast<int64_t>(blockIdx.x) * kQuantThreads + threadIdx.x;
    const int64_t grp = id / LPG;
    if (grp >= groups) return;  // whole groups: LPG divides the block
    const int sub = static_cast<int>(id % LPG);
    const int64_t row = grp / G;
    const int64_t k0 = (grp - row * G) * (8 * LPG) + 4 * sub;
    f32x4 v[2];
#pragma unroll
    for (int half = 0; half < 2; ++half) v[half] = load4<VEC>(w + row * K, k0 + half * 4 * LPG, K);
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float e = v[i >> 2][i & 3];  // (a bit cast of the vector element itself reads element 0)
        const uint32_t b = __builtin_bit_cast(uint32_t, e) & 0x7fffffffu;
        m = b > m ? b : m;
    }
#pragma unroll
    for (int d = 1; d < LPG; d <<= 1) {
        const uint32_t o = static_cast<uint32_t>(__shfl_xor(static_cast<int>(m), d, kWave));
        m = o > m ? o : m;
    }
    float s = __fdiv_rn(__builtin_bit_cast(float, m), qmax);
    s = s < 1.17549435e-38f ? 1.17549435e-38f : s;  // NaN stays
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        uint32_t out = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float c = rintf(__fdiv_rn(v[half][i], s));
            c = c < -qmax ? -qmax : c > qmax ? qmax : c;
            out |= (static_cast<uint32_t>(static_cast<int>(c)) & 0xffu) << (8 * i);
        }
        stg(reinterpret_cast<uint32_t*>(q) + grp * (2 * LPG) + half * LPG + sub, out);
    }
    if (sub == 0) stg(scale + grp, s);
}

// The low nibbles of 8 signed bytes (b0..b3 in lo, b4..b7 in hi) as one AWQ-order word: nibbles 0..3 hold elements 0, 2,
// 4, 6, nibbles 4..7 elements 1, 3, 5, 7.
__device__ __forceinline__ uint32_t pack8(uint32_t lo, uint32_t hi) {
    const uint32_t a = (lo & 0x000f000fu) | ((hi & 0x000f000fu) << 8);            // 0 . 4 . 2 . 6 (nibbles 0, 2, 4, 6)
    const uint32_t b = ((lo >> 8) & 0x000f000fu) | ((hi & 0x0f000f00u));          // 1 . 5 . 3 . 7
    const uint32_t e = (a & 0x0f0fu) | ((a >> 12) & 0xf0f0u), o = (b & 0x0f0fu) | ((b >> 12) & 0xf0f0u);
    return e | (o << 16);
}

// VEC (rows of a multiple of 32 codes, 16-byte aligned): 4 words per thread; else one word per thread, zeros past K.
template <bool VEC>
__global__ __launch_bounds__(kQuantThreads) void pack_int4_kernel(const int8_t* __restrict__ q, uint32_t* __restrict__ out,
                                                                  int64_t n, int64_t words, int64_t K) {
    const int64_t id = static_cast<int64_t>(blockIdx.x) * kQuantThreads + threadIdx.x;
    if (id >= n) return;
    if (VEC) {
        const u32x4* s = reinterpret_cast<const u32x4*>(q) + 2 * id;
        const u32x4 a = ldg(s), b = ldg(s + 1);
        stg(reinterpret_cast<u32x4*>(out) + id, u32x4{pack8(a.x, a.y), pack8(a.z, a.w), pack8(b.x, b.y), pack8(b.z, b.w)});
        return;
    }
    const int64_t row = id / words, k0 = (id - row * words) * 8;
    const int8_t* s = q + row * K;
    uint32_t v[2] = {0u, 0u};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint32_t b = k0 + i < K ? static_cast<uint8_t>(ldg(s + k0 + i)) : 0u;
        v[i >> 2] |= b << (8 * (i & 3));
    }
    stg(out + id, pack8(v[0], v[1]));
}

// out [H, n/8] words = the transpose of the n x H codes of in [n, words] (both AWQ order, no rounding): a workgroup turns a
// 64 x 64 tile in LDS, so both sides move 32-byte row segments. (As tensor
// operations the 28 copies of a Qwen3-1.7B-shaped DIP engine took 7 ms of its construction.)
constexpr int kTile = 64;

__global__ __launch_bounds__(kQuantThreads) void transpose_int4_kernel(const uint32_t* __restrict__ in,
                                                                       uint32_t* __restrict__ out, int n, int H,
                                                                       int words) {
    __shared__ uint8_t s[kTile][kTile + 4];  // [column][channel]
    const int c0 = static_cast<int>(blockIdx.y) * kTile, w0 = static_cast<int>(blockIdx.x) * (kTile / 8);
    const int tid = threadIdx.x;
#pragma unroll
    for (int it = 0; it < 2; ++it) {
        const int id = tid + it * kQuantThreads, ch = id >> 3, w = id & 7;  // 8 words of each of 64 channels
        const uint32_t v = c0 + ch < n && w0 + w < words ? ldg(in + static_cast<int64_t>(c0 + ch) * words + w0 + w) : 0u;
#pragma unroll
        for (int j = 0; j < 8; ++j)  // element j of a word: nibble j / 2 (even j) or 4 + j / 2
            s[8 * w + j][ch] = static_cast<uint8_t>((v >> (4 * ((j >> 1) + ((j & 1) << 2)))) & 15u);
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < 2; ++it) {
        const int id = tid + it * kQuantThreads, col = id >> 3, w = id & 7;
        const int64_t row = static_cast<int64_t>(w0) * 8 + col;
        if (row >= H || c0 + 8 * w >= n) continue;
        const uint32_t* p = reinterpret_cast<const uint32_t*>(&s[col][8 * w]);
        stg(out + row * (n >> 3) + (c0 >> 3) + w, pack8(p[0], p[1]));
    }
}

}  // namespace soi

using namespace soi;

extern "C" int soi_transpose_int4(const uint8_t* Wq, uint8_t* out, int64_t n, int64_t H, void* stream) {
    const char* what = "soi_transpose_int4";
    SOI_REQUIRE(n >= 8 && n % 8 == 0 && n <= 65535 * int64_t(kTile) && H >= 1 && H <= (int64_t(1) << 30),
                "%s: n must be a multiple of 8", what);
    SOI_REQUIRE(Wq && out && ((reinterpret_cast<uintptr_t>(Wq) | reinterpret_cast<uintptr_t>(out)) & 3u) == 0,
                "%s: null pointer or rows not 4-byte aligned", what);
    const int64_t words = ceil_div64(H, 8);
    hipLaunchKernelGGL(transpose_int4_kernel,
                       dim3(static_cast<unsigned>(ceil_div64(words, kTile / 8)),
                            static_cast<unsigned>(ceil_div64(n, kTile))),
                       dim3(kQuantThreads), 0, as_stream(stream), reinterpret_cast<const uint32_t*>(Wq),
                       reinterpret_cast<uint32_t*>(out), static_cast<int>(n), static_cast<int>(H),
                       static_cast<int>(words));
    return launch_status(what);
}

extern "C" int soi_quantize_group_supported(int64_t group_size) {
    return group_size == 32 || group_size == 64 || group_size == 128 || group_size == 256 ? 1 : 0;
}

extern "C" int soi_quantize_group(const float* w, int8_t* q, float* scale, int64_t N, int64_t K, int64_t group_size,
                                  int64_t qmax, void* stream) {
    const char* what = "soi_quantize_group";
    SOI_REQUIRE(soi_quantize_group_supported(group_size), "%s: group_size must be 32, 64, 128 or 256, got %lld", what,
                (long long)group_size);
    SOI_REQUIRE(N >= 0 && K >= 1 && K <= (int64_t(1) << 30) && qmax >= 1 && qmax <= 127, "%s: size out of range", what);
    if (N == 0) return SOI_OK;
    SOI_REQUIRE(w && q && scale, "%s: null pointer", what);
    SOI_REQUIRE((reinterpret_cast<uintptr_t>(q) & 3u) == 0, "%s: q must be 4-byte aligned", what);
    const int64_t G = ceil_div64(K, group_size), groups = N * G, lpg = group_size / 8;
    const int64_t blocks = ceil_div64(groups * lpg, kQuantThreads);
    SOI_REQUIRE(blocks <= (int64_t(1) << 31) - 1, "%s: too many groups", what);
    const bool vec = K % 4 == 0 && aligned16(w);
    hipStream_t st = as_stream(stream);
#define SOI_Q(LL, V)                                                                                                  \
    hipLaunchKernelGGL((quantize_group_kernel<LL, V>), dim3(static_cast<unsigned>(blocks)), dim3(kQuantThreads), 0, \
                       st, w, q, scale, groups, static_cast<int>(G), K, static_cast<float>(qmax))
#define SOI_QV(LL) \
    if (vec) SOI_Q(LL, true); else SOI_Q(LL, false)
    if (lpg == 4) { SOI_QV(4); } else if (lpg == 8) { SOI_QV(8); } else if (lpg == 16) { SOI_QV(16); } else { SOI_QV(32); }
#undef SOI_QV
#undef SOI_Q
    return launch_status(what);
}

extern "C" int soi_pack_int4(const int8_t* q, uint8_t* out, int64_t N, int64_t K, void* stream) {
    const char* what = "soi_pack_int4";
    SOI_REQUIRE(N >= 0 && K >= 1 && K <= (int64_t(1) << 31) - 8, "%s: size out of range", what);
    if (N == 0) return SOI_OK;
    SOI_REQUIRE(q && out && (reinterpret_cast<uintptr_t>(out) & 3u) == 0, "%s: null pointer or out not 4-byte aligned",
                what);
    const int64_t words = ceil_div64(K, 8);
    const bool vec = K % 32 == 0 && aligned16(q) && aligned16(out);
    const int64_t n = vec ? N * words / 4 : N * words;
    const int64_t blocks = ceil_div64(n, kQuantThreads);
    SOI_REQUIRE(blocks <= (int64_t(1) << 31) - 1, "%s: too many words", what);
    const dim3 grid(static_cast<unsigned>(blocks));
    uint32_t* o = reinterpret_cast<uint32_t*>(out);
    if (vec)
        hipLaunchKernelGGL(pack_int4_kernel<true>, grid, dim3(kQuantThreads), 0, as_stream(stream), q, o, n, words, K);
    else
        hipLaunchKernelGGL(pack_int4_kernel<false>, grid, dim3(kQuantThreads), 0, as_stream(stream), q, o, n, words, K);
    return launch_status(what);
}
