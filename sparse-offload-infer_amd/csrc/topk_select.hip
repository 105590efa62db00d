// Deterministic threshold top-k (Dynamic Input Pruning channel selection).
//
// Semantics are exactly the reference's topk_threshold_select
// (csrc/kernels/topk_select.cu:10-96):
//   total_max = max(0, max_i v_i);  lo = 0;  hi = fl(total_max + 1e-3f)
//   24 times: mid = fl(0.5f * fl(lo + hi));
//             if count(v_i >= mid) >= k  lo = mid  else  hi = mid
//   out = the first k indices, ascending, with v_i >= lo;  count = #written.
// Counts are integers, so the decisions (and hence tau = lo) do not depend on
// how the counting is parallelised.
//
// gfx950 design: ONE workgroup of 8 waves (16 above 16384 values) holds all values in registers, up to 32768 of them,
// and finds v_(k) by a radix select (topk_radix_kernel); longer inputs are streamed (topk_rule_a_stream_kernel). The
// final compaction is an ordered ballot prefix scan: position = (elements of earlier waves) + (earlier rows of this wave)
// + (earlier lanes in this row), so the output is in ascending index order by construction and identical on every call.
#include "soi_device.h"
#include "soi_host.h"
#include "soi_select.h"

namespace soi {

constexpr int kTopkThreads = 1024;
constexpr int kTopkWaves = kTopkThreads / kWave;

// Block-wide fp32 max of per-thread values (initial value 0.0f, as the reference).
__device__ __forceinline__ float block_max_from(float local, float* s_max, int wave, int lane) {
    const float wm = wave_max_bcast(local);
    if (lane == 0) s_max[wave] = wm;
    __syncthreads();
    float m = 0.0f;
#pragma unroll
    for (int w = 0; w < kTopkWaves; ++w) m = fmaxf(m, s_max[w]);
    return m;
}

// Radix form (n <= 1024*32): rule A depends on the values only through v_(k),
// the k-th largest value: count(v >= mid) >= k exactly when v_(k) >= mid. So
// the kernel finds v_(k) exactly by a radix select on order-preserving keys
// (NaN and padding map to key 0 and never count; see the value sources),
// replays the 24 bisection steps on it in fp32 (the reference's op
// sequence), and compacts.
//
// One workgroup of NW waves, E values per lane in registers, element
// (j, lane) of wave w = w*64E + 64j + lane. Every pass: candidates (keys that
// match the digits found so far) add 1 to an LDS histogram of their next
// digit, one barrier, then EVERY wave scans the histogram itself (lane l
// reads the contiguous bins l*B..l*B+B-1 counted from the top, a DPP prefix
// over lanes finds the lane holding the rank, then B lanes re-read that
// lane's bins and a second prefix finds the bin), so the passes need no
// further barrier. Histograms are zeroed up front and padded by one word per
// 32 bins (conflict-free lane reads); a lane whose element is not a
// candidate adds to a private dummy word instead of branching. fp32 keys take
// digits of 11, 10 and 10 bits; a binary16 magnitude's key is its 15-bit
// pattern, two digits of 9 and 6 bits (16 bins per octave in the first pass,
// so gate magnitudes spread over many bins: few same-address LDS atomics).
// Four (binary16) or five (fp32) barriers in all, against nine for the
// bisection-histogram form. Every global load is issued unconditionally
// (clamped index): a branch per load serialises them.
constexpr int kRadixThreads = 512;

template <int E, int NW, class Values>
__global__ __launch_bounds__(NW * kWave) void topk_radix_kernel(const Values v, int n, int k,
                                                                int32_t* __restrict__ out_idx,
                                                                int32_t* __restrict__ out_count) {
    __shared__ uint32_t s_hist[radix_hist_offset<Values>(Values::kPasses)];
    __shared__ float s_max[NW];
    __shared__ uint32_t s_tot[NW];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int base_i = wave * kWave * E + lane;

    float val[E];
    uint32_t key[E];
    float local_max = 0.0f;
#pragma unroll
    for (int j = 0; j < E; ++j) {  // clamped index: every load is issued unconditionally, no branch per load
        const int i = base_i + j * kWave;
        val[j] = v.load(i < n ? i : n - 1);
    }
    // the histograms are zeroed and published while the values are in flight (rule A's SYNCED form)
    rule_a_zero_hist<NW, Values>(s_hist, tid);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < E; ++j) {
        const int i = base_i + j * kWave;
        val[j] = (i < n) ? val[j] : __builtin_nanf("");
        key[j] = Values::key_of(val[j]);
        local_max = fmaxf(local_max, val[j]);
    }
    const float tau = rule_a_tau<E, NW, Values, true, NoMid, true>(key, local_max, s_hist, s_max, k, tid);
    const uint32_t total = rule_a_compact<E, NW>(val, tau, s_tot, tid, [&](uint32_t pos, int j) {
        if (pos < static_cast<uint32_t>(k)) out_idx[pos] = base_i + j * kWave;
    });
    if (tid == 0) *out_count = static_cast<int32_t>(total < static_cast<uint32_t>(k) ? total : k);
}

// Any n: values streamed from global memory (L2-resident after the first
// pass) in blocks of 1024, same arithmetic and same output order.
template <class Values>
__global__ __launch_bounds__(kTopkThreads) void topk_rule_a_stream_kernel(const Values v, int n, int k,
                                                                           int32_t* __restrict__ out_idx,
                                                                           int32_t* __restrict__ out_count) {
    __shared__ float s_max[kTopkWaves];
    __shared__ uint32_t s_cnt[2][kTopkWaves];
    __shared__ uint32_t s_blk[2][kTopkWaves];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    float local_max = 0.0f;
    for (int i = tid; i < n; i += kTopkThreads) local_max = fmaxf(local_max, v[i]);
    const float total_max = block_max_from(local_max, s_max, wave, lane);

    float lo = 0.0f;
    float hi = total_max + 1e-3f;
    for (int it = 0; it < kBisectionSteps; ++it) {
        const float mid = 0.5f * (lo + hi);
        uint32_t cnt = 0;
        for (int b = 0; b < n; b += kTopkThreads) {
            const int i = b + tid;
            cnt += popc64(ballot(i < n && v[i] >= mid));
        }
        if (lane == 0) s_cnt[it & 1][wave] = cnt;
        __syncthreads();
        uint32_t total = 0;
        for (int w = 0; w < kTopkWaves; ++w) total += s_cnt[it & 1][w];
        if (total >= static_cast<uint32_t>(k))
            lo = mid;
        else
            hi = mid;
    }
    const float tau = lo;
    uint32_t running = 0;
    int parity = 0;
    for (int b = 0; b < n && running < static_cast<uint32_t>(k); b += kTopkThreads, parity ^= 1) {
        const int i = b + tid;
        const bool flag = i < n && v[i] >= tau;
        const uint64_t mk = ballot(flag);
        if (lane == 0) s_blk[parity][wave] = popc64(mk);
        __syncthreads();
        uint32_t before = 0, blk = 0;
        for (int w = 0; w < kTopkWaves; ++w) {
            const uint32_t c = s_blk[parity][w];
            before += (w < wave) ? c : 0u;
            blk += c;
        }
        const uint32_t pos = running + before + mask_prefix(mk);
        if (flag && pos < static_cast<uint32_t>(k)) out_idx[pos] = i;
        running += blk;
    }
    if (tid == 0) *out_count = static_cast<int32_t>(running < static_cast<uint32_t>(k) ? running : k);
}

template <class Values>
static int launch_topk(const Values v, int64_t n, int64_t k, int32_t* out_indices, int32_t* out_count, void* stream,
                       const char* what) {
    SOI_REQUIRE(n >= 1 && n <= (int64_t(1) << 30), "%s: n must be in [1, 2^30]", what);
    SOI_REQUIRE(k >= 1 && k <= n, "%s: k must be in [1, n]", what);
    SOI_REQUIRE(v.p && out_indices && out_count, "%s: null pointer", what);
    hipStream_t st = as_stream(stream);
    const int ni = static_cast<int>(n), ki = static_cast<int>(k);
    const int64_t er = ceil_div64(n, kRadixThreads), e = ceil_div64(n, 2 * kRadixThreads);
#define SOI_R(EE, NW)                                                                                              \
    hipLaunchKernelGGL((topk_radix_kernel<EE, NW, Values>), dim3(1), dim3(NW * kWave), 0, st, v, ni, ki, out_indices, \
                       out_count)
    if (er <= 32) {
        if (er <= 1) SOI_R(1, 8);
        else if (er <= 2) SOI_R(2, 8);
        else if (er <= 4) SOI_R(4, 8);
        else if (er <= 8) SOI_R(8, 8);
        else if (er <= 12) SOI_R(12, 8);
        else if (er <= 16) SOI_R(16, 8);
        else if (er <= 24) SOI_R(24, 8);
        else SOI_R(32, 8);
    } else if (e <= 32) {
        // more than 512 x 32 values: twice the waves (fp32, back to back: 17408 values 13.9 us, 27648 17.4; replaying the
        // bisection from node histograms took 24.1 and 36.9). Below, 16 waves are no faster than 8 (16384: 11.3, 11.6).
        if (e <= 24) SOI_R(24, 16);
        else SOI_R(32, 16);
    } else {
        hipLaunchKernelGGL((topk_rule_a_stream_kernel<Values>), dim3(1), dim3(kTopkThreads), 0, st, v, ni, ki,
                           out_indices, out_count);
    }
#undef SOI_R
    return launch_status(what);
}

}  // namespace soi

using namespace soi;

extern "C" int soi_topk_threshold_select(const float* abs_g, int64_t n, int64_t k, int32_t* out_indices,
                                         int32_t* out_count, void* stream) {
    return launch_topk(F32Values{abs_g}, n, k, out_indices, out_count, stream, "soi_topk_threshold_select");
}

extern "C" int soi_topk_threshold_select_f16abs(const uint16_t* gate, int64_t n, int64_t k, int32_t* out_indices,
                                                int32_t* out_count, void* stream) {
    return launch_topk(F16AbsValues{gate}, n, k, out_indices, out_count, stream, "soi_topk_threshold_select_f16abs");
}
