// Dynamic Input Pruning over the tokens of a prompt (gfx950): selection, gating, the miss rows and the sparse down
// projection of T tokens in one launch each. Every token's selection, h and y are bit for bit those of the decode
// step's operators (topk_select.hip, the SiLU epilogue, sparse_down.hip): a DIP decoder's later layers hang on the last
// bit of a gate, so nothing here may round differently.
// Reference: the DIP MLP of generate_dip / generate_cached_dip (python/soinfer/runtime/generate.py:276-310, 367-404),
// one token per step.
//
// Measured (28-layer Qwen3-1.7B shape, k/I = 0.5): a 64-token prompt 4.5 ms against 53.6 ms one token at a time (the
// indexed schedule), 256 tokens 13.5 against 218 ms; one layer of 64 tokens takes about 160 us, 90 of them the linears.
#include "soi_device.h"
#include "soi_down.h"
#include "soi_host.h"
#include "soi_prompt.h"
#include "soi_select.h"

namespace soi {

constexpr int kSelThreads = 512;
constexpr int kSelWaves = kSelThreads / kWave;
constexpr int kSelMax = kSelThreads * 32;  // channels one workgroup holds in registers

// Workgroup t: the rule-A selection over |gate[t]| (topk_radix_kernel's partition), ascending, to idx[t, k]. mark: every
// selected channel's word is set to `stamp`, so the union of the tokens' selections needs no clearing between calls.
// last_idx, last_count: the last token's selection as the top-k kernel leaves it (nothing past the count is written).
template <int E>
__global__ __launch_bounds__(kSelThreads) void dip_select_tokens_kernel(const uint16_t* __restrict__ gate, int64_t ld,
                                                                        int n, int k, int32_t* __restrict__ idx,
                                                                        int32_t* __restrict__ mark, int32_t stamp,
                                                                        int32_t* __restrict__ last_idx,
                                                                        int32_t* __restrict__ last_count) {
    __shared__ uint32_t s_hist[radix_hist_offset<F16AbsValues>(F16AbsValues::kPasses)];
    __shared__ float s_max[kSelWaves];
    __shared__ uint32_t s_tot[kSelWaves];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int base_i = wave * kWave * E + lane;
    const F16AbsValues v{gate + static_cast<int64_t>(blockIdx.x) * ld};
    int32_t* out = idx + static_cast<int64_t>(blockIdx.x) * k;
    const bool last = last_idx != nullptr && blockIdx.x + 1 == gridDim.x;
    float val[E];
    uint32_t key[E];
    float local_max = 0.0f;
#pragma unroll
    for (int j = 0; j < E; ++j) {
        const int i = base_i + j * kWave;
        val[j] = v.load(i < n ? i : n - 1);
    }
    rule_a_zero_hist<kSelWaves, F16AbsValues>(s_hist, tid);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < E; ++j) {
        const int i = base_i + j * kWave;
        val[j] = (i < n) ? val[j] : __builtin_nanf("");
        key[j] = F16AbsValues::key_of(val[j]);
        local_max = fmaxf(local_max, val[j]);
    }
    const float tau = rule_a_tau<E, kSelWaves, F16AbsValues, true, NoMid, true>(key, local_max, s_hist, s_max, k, tid);
    const uint32_t total = rule_a_compact<E, kSelWaves>(val, tau, s_tot, tid, [&](uint32_t pos, int j) {
        if (pos >= static_cast<uint32_t>(k)) return;
        const int c = base_i + j * kWave;
        stg(out + pos, c);
        if (mark) stg(mark + c, stamp);
        if (last) stg(last_idx + pos, c);
    });
    if (last && tid == 0) stg(last_count, static_cast<int32_t>(total < static_cast<uint32_t>(k) ? total : k));
    // fewer than k gates that are numbers: the rest of the list names no channel
    for (uint32_t i = total + static_cast<uint32_t>(tid); i < static_cast<uint32_t>(k); i += kSelThreads)
        stg(out + i, -1);
}

// h[t, j] = fp16(silu(gate[t, c]) * up[t, c]), c = idx[t, j] (NaN where it names no channel).
__global__ __launch_bounds__(256) void dip_gate_tokens_kernel(const uint16_t* __restrict__ gate,
                                                              const uint16_t* __restrict__ up, int64_t ld, int n,
                                                              const int32_t* __restrict__ idx,
                                                              uint16_t* __restrict__ h, int k) {
    const int j = static_cast<int>(blockIdx.x) * 256 + static_cast<int>(threadIdx.x);
    if (j >= k) return;
    const int64_t t = blockIdx.y;
    const int c = ldg(idx + t * k + j);
    const bool ok = c >= 0 && c < n;
    const int64_t o = t * ld + (ok ? c : 0);
    const float g = f16_bits_to_f32(ldg(gate + o)), u = f16_bits_to_f32(ldg(up + o));
    stg(h + t * k + j, ok ? f32_to_f16_bits(silu_f32(g) * u) : uint16_t(0x7e00u));
}

// Rows c of up (y = 0) and down^T (y = 1) whose mark is `stamp` into the device images: from the hot cache when
// resident, else from the host arena's device mapping (16 lanes per row, 64 contiguous bytes a lane: the wide PCIe
// reads of gather_rows_vec_kernel). So a row that any token selects crosses PCIe once for the prompt.
struct FetchSide {
    const uint8_t* cache;
    const uint8_t* host;
    uint8_t* image;
    int64_t row_bytes;
};

__global__ __launch_bounds__(64) void dip_fetch_rows_kernel(FetchSide up, FetchSide down, int n, int64_t cache_rows,
                                                            const int32_t* __restrict__ slot_of,
                                                            const int32_t* __restrict__ mark, int32_t stamp) {
    const int lane = threadIdx.x, sub = lane & 15;
    const int c = static_cast<int>(blockIdx.x) * 4 + (lane >> 4);
    if (c >= n || ldg(mark + c) != stamp) return;
    const FetchSide f = blockIdx.y ? down : up;
    const int32_t s = ldg(slot_of + c);
    const bool hit = s >= 0 && s < cache_rows;
    const u32x4* src = reinterpret_cast<const u32x4*>(hit ? f.cache + s * f.row_bytes : f.host + c * f.row_bytes);
    u32x4* dst = reinterpret_cast<u32x4*>(f.image + c * f.row_bytes);
    const int64_t n16 = f.row_bytes / 16;
    const u32x4* z = reinterpret_cast<const u32x4*>(g_zero16);
    for (int64_t base = 4 * sub; base < n16; base += 64) {
        u32x4 v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = ldg(base + i < n16 ? src + base + i : z);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (base + i < n16) stg(dst + base + i, v[i]);
    }
}

// x[t, :] += sum_j h[t, j] * row idx[t, j] of down_proj^T, as one binary16 addition. Workgroup (slice, t) takes the
// 256-column slice of one token and walks the sparse down's row chunks (soi_down.h: rpc rows, R chunks) in order, so
// each chunk's sum, and the sum over the chunks, are those of sparse_down_kernel's workgroups and of its combine, with
// no partial rows in memory and no arrival. The chunks' loads are pipelined: while chunk r is summed, chunk r + 1's
// rows and chunk r + 2's indices are in flight.
//
// Bound by instruction issue: 32 columns of a row take 40 instructions to unpack and 32 mixed fmas. A workgroup id is
// slice + slices * token, so with 8 slices every XCD reads one 128-byte column of each row: the layer's selected
// columns stay in its L2 for all tokens.
struct DownKeys {
    int32_t c[kDownU];
    uint16_t h[kDownU];
};
struct DownRows {
    u32x4 w[kDownU];
    float s[kDownU], h[kDownU];
};

__global__ __launch_bounds__(kDownThreads) void sparse_down_tokens_kernel(
    const uint8_t* __restrict__ W, const float* __restrict__ S, int64_t row_bytes, int G, int nrows,
    const int32_t* __restrict__ idx, const uint16_t* __restrict__ h, uint16_t* __restrict__ x, int k, int H, int gs,
    int rpc, int R) {
    __shared__ float red[kRedFloats];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int rs = lane >> 3, cc = lane & (kSliceChunks - 1);
    const int slice = blockIdx.x;
    const int64_t t = blockIdx.y;
    const int c = slice * kSliceChunks + cc;
    const bool cvalid = c < (H >> 5);
    const int sg = cvalid ? 32 * c / gs : 0;
    const int32_t* ti = idx + t * k;
    const uint16_t* th = h + t * k;
    const u32x4* z = reinterpret_cast<const u32x4*>(g_zero16);

    auto keys = [&](DownKeys& o, int r) {
        const int j0 = r * rpc, j1 = min(j0 + rpc, k);
#pragma unroll
        for (int u = 0; u < kDownU; ++u) {
            const int j = j0 + (u * kDownWaves + wave) * kGroupRows + rs;
            const int jc = j < j1 ? j : j0;
            const int32_t ch = ldg(ti + jc);
            o.h[u] = ldg(th + jc);
            o.c[u] = j < j1 ? ch : nrows;  // nrows: nothing (a channel outside [0, nrows] is unresolvable)
        }
    };
    auto rows = [&](DownRows& o, const DownKeys& q) {
#pragma unroll
        for (int u = 0; u < kDownU; ++u) {
            const bool in = q.c[u] != nrows, ok = q.c[u] >= 0 && q.c[u] < nrows;
            const int64_t row = ok ? q.c[u] : 0;
            o.w[u] = ldg(ok && cvalid ? reinterpret_cast<const u32x4*>(W + row * row_bytes) + c : z);
            o.s[u] = ldg(ok && cvalid ? S + row * G + sg : reinterpret_cast<const float*>(g_zero16));
            o.h[u] = !in ? 0.0f : ok ? f16_bits_to_f32(q.h[u]) : __builtin_nanf("");
        }
    };
    DownKeys kn;
    DownRows cur;
    {
        DownKeys k0;
        keys(k0, 0);
        rows(cur, k0);
        keys(kn, R > 1 ? 1 : 0);
    }
    float sum = 0.0f;
    const int tc = tid >> 5, tl = tid & 31;
    for (int r = 0; r < R; ++r) {
        DownRows nxt;
        rows(nxt, kn);
        keys(kn, r + 2 < R ? r + 2 : R - 1);
        __builtin_amdgcn_sched_barrier(0);
        float acc[32];
#pragma unroll
        for (int i = 0; i < 32; ++i) acc[i] = 0.0f;
#pragma unroll
        for (int u = 0; u < kDownU; ++u) {
            const float cf = cur.h[u] * cur.s[u];
            const uint32_t wd[4] = {cur.w[u].x, cur.w[u].y, cur.w[u].z, cur.w[u].w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                f16x2 q[4];
                dequant_int4x8_bitfield(wd[i], q);
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    acc[8 * i + 2 * p] = fmaf(cf, static_cast<float>(q[p].x), acc[8 * i + 2 * p]);
                    acc[8 * i + 2 * p + 1] = fmaf(cf, static_cast<float>(q[p].y), acc[8 * i + 2 * p + 1]);
                }
            }
        }
        float* red_lane = red + ((wave * kGroupRows + rs) * kSliceChunks + cc) * kRedPitch;
#pragma unroll
        for (int i = 0; i < 32; ++i) red_lane[i] = acc[i];
        __syncthreads();
        float part = 0.0f;
#pragma unroll
        for (int g = 0; g < kDownWaves * kGroupRows; ++g) part += red[(g * kSliceChunks + tc) * kRedPitch + tl];
        sum += part;
        __syncthreads();  // every column of this chunk is read before the next chunk's sums overwrite it
        cur = nxt;
    }
    const int64_t col = static_cast<int64_t>(slice) * kSliceCols + tid;
    if (col < H) {
        uint16_t* p = x + t * H + col;
        stg(p, static_cast<uint16_t>(add_f16x2(ldg(p), f32_to_f16_bits(sum))));
    }
}

}  // namespace soi

using namespace soi;

extern "C" int64_t soi_dip_tokens_max_channels(void) { return kSelMax; }

extern "C" int soi_dip_select_tokens(const uint16_t* gate, int64_t ld, int64_t n, int64_t k, int64_t T, int32_t* idx,
                                     int32_t* mark, int32_t stamp, int32_t* last_idx, int32_t* last_count,
                                     void* stream) {
    const char* what = "soi_dip_select_tokens";
    SOI_REQUIRE(T >= 1 && T <= 65535, "%s: the token count must be in [1, 65535]", what);
    SOI_REQUIRE(n >= 1 && n <= kSelMax && ld >= n, "%s: n must be in [1, %d] and ld >= n", what, kSelMax);
    SOI_REQUIRE(k >= 1 && k <= n, "%s: k must be in [1, n]", what);
    SOI_REQUIRE(gate && idx && !last_idx == !last_count, "%s: null pointer, or one of last_idx and last_count", what);
    const int64_t e = ceil_div64(n, kSelThreads);
#define SOI_S(EE)                                                                                                     \
    hipLaunchKernelGGL(dip_select_tokens_kernel<EE>, dim3(static_cast<unsigned>(T)), dim3(kSelThreads), 0,            \
                       as_stream(stream), gate, ld, static_cast<int>(n), static_cast<int>(k), idx, mark, stamp,  \
                       last_idx, last_count)
    if (e <= 1) SOI_S(1);
    else if (e <= 2) SOI_S(2);
    else if (e <= 4) SOI_S(4);
    else if (e <= 8) SOI_S(8);
    else if (e <= 12) SOI_S(12);
    else if (e <= 16) SOI_S(16);
    else if (e <= 24) SOI_S(24);
    else SOI_S(32);
#undef SOI_S
    return launch_status(what);
}

extern "C" int soi_dip_gate_tokens(const uint16_t* gate, const uint16_t* up, int64_t ld, int64_t n, const int32_t* idx,
                                   uint16_t* h, int64_t k, int64_t T, void* stream) {
    const char* what = "soi_dip_gate_tokens";
    SOI_REQUIRE(T >= 1 && T <= 65535, "%s: the token count must be in [1, 65535]", what);
    SOI_REQUIRE(n >= 1 && n <= (int64_t(1) << 30) && ld >= n && k >= 1 && k <= n, "%s: size out of range", what);
    SOI_REQUIRE(gate && up && idx && h, "%s: null pointer", what);
    hipLaunchKernelGGL(dip_gate_tokens_kernel, dim3(static_cast<unsigned>(ceil_div64(k, 256)), static_cast<unsigned>(T)),
                       dim3(256), 0, as_stream(stream), gate, up, ld, static_cast<int>(n), idx, h, static_cast<int>(k));
    return launch_status(what);
}

extern "C" int soi_dip_fetch_rows(const uint8_t* cache_up, const uint8_t* host_up, uint8_t* image_up,
                                  int64_t up_row_bytes, const uint8_t* cache_down, const uint8_t* host_down,
                                  uint8_t* image_down, int64_t down_row_bytes, int64_t num_channels, int64_t cache_rows,
                                  const int32_t* slot_of, const int32_t* mark, int32_t stamp, void* stream) {
    const char* what = "soi_dip_fetch_rows";
    SOI_REQUIRE(num_channels >= 1 && num_channels <= (int64_t(1) << 30) && cache_rows >= 0, "%s: size out of range",
                what);
    SOI_REQUIRE(host_up && image_up && host_down && image_down && slot_of && mark, "%s: null pointer", what);
    SOI_REQUIRE(cache_rows == 0 || (cache_up && cache_down), "%s: null cache", what);
    SOI_REQUIRE(up_row_bytes > 0 && up_row_bytes % 16 == 0 && down_row_bytes > 0 && down_row_bytes % 16 == 0,
                "%s: rows must be multiples of 16 bytes", what);
    for (const void* p : {static_cast<const void*>(cache_up), static_cast<const void*>(host_up),
                          static_cast<const void*>(image_up), static_cast<const void*>(cache_down),
                          static_cast<const void*>(host_down), static_cast<const void*>(image_down)})
        SOI_REQUIRE(aligned16(p), "%s: rows must be 16-byte aligned", what);
    const FetchSide up{cache_up, host_up, image_up, up_row_bytes}, down{cache_down, host_down, image_down, down_row_bytes};
    hipLaunchKernelGGL(dip_fetch_rows_kernel, dim3(static_cast<unsigned>(ceil_div64(num_channels, 4)), 2), dim3(64), 0,
                       as_stream(stream), up, down, static_cast<int>(num_channels), cache_rows, slot_of, mark, stamp);
    return launch_status(what);
}

extern "C" int soi_sparse_down_tokens(const uint8_t* Wq_T, const float* scale_T, int64_t num_rows, const int32_t* idx,
                                      const uint16_t* h, uint16_t* x, int64_t H, int64_t k, int64_t group_size,
                                      int64_t T, void* stream) {
    const char* what = "soi_sparse_down_tokens";
    SOI_REQUIRE(T >= 1 && T <= 65535, "%s: the token count must be in [1, 65535]", what);
    SOI_REQUIRE(H >= 32 && H % 32 == 0 && H <= (int64_t(1) << 24), "%s: H must be a multiple of 32", what);
    SOI_REQUIRE(group_size >= 32 && group_size % 32 == 0, "%s: group_size must be a multiple of 32", what);
    SOI_REQUIRE(num_rows >= 1 && num_rows <= (int64_t(1) << 30) && k >= 1 && k <= (int64_t(1) << 30),
                "%s: size out of range", what);
    SOI_REQUIRE(Wq_T && scale_T && idx && h && x && aligned16(Wq_T), "%s: null pointer or Wq_T not 16-byte aligned",
                what);
    const DownPlan p = down_plan(H, k);
    SOI_REQUIRE(p.rpc <= static_cast<int64_t>(kDownWaves) * kGroupRows * kDownU, "%s: partition out of range", what);
    hipLaunchKernelGGL(sparse_down_tokens_kernel, dim3(static_cast<unsigned>(p.S), static_cast<unsigned>(T)),
                       dim3(kDownThreads), 0, as_stream(stream), Wq_T, scale_T, H / 2,
                       static_cast<int>(ceil_div64(H, group_size)), static_cast<int>(num_rows), idx, h, x,
                       static_cast<int>(k), static_cast<int>(H), static_cast<int>(group_size), static_cast<int>(p.rpc),
                       static_cast<int>(p.R));
    return launch_status(what);
}
