// Temperature / nucleus sampling of one logits vector on the GPU: sample_logits
// (sampler.cpp:15-52) with the reference's arithmetic, so that the same uniform draw picks
// the same token.
//
//   1. the indices sorted by descending logit (an LSD radix sort of 8-bit digits, stable:
//      equal logits keep ascending indices; std::sort leaves their order unspecified);
//   2. p_i = exp((l_i - max) / T) for every i, with the reference libm's expf (expf_libm.hpp);
//   3. s = p_0 + p_1 + ... in that order, p_i /= s;
//   4. nucleus (top_p < 1): the running sum until it reaches top_p gives the kept count
//      `last` and z (the same sum, so the same float), p_i /= z for i < last;
//   5. the first i whose running sum reaches the draw r, else the last kept index.
//
// The running sums (3-5) are sequential float additions in the reference, so one wave performs
// them in order from registers (64 values per load, eight loads ahead), one lane-broadcast
// addition per element. A sum stops early once the next value is at most a quarter of an ulp
// of the sum: the values do not increase, so none of the rest can change it (sharp
// distributions stop after a handful of elements; a nearly flat one over a 128K vocabulary
// takes the whole pass).
//
// Two ways to the same token:
//   launch_sample_top   only the logits with (l_i - max) / T >= -20 are picked out and sorted
//                       (in LDS, at most kTopCap of them). The others have p_i < 2^-28, below a
//                       quarter ulp of every sum they would be added to (s >= 1, and the sums
//                       of p_i / s end within 2^-11 of 1), so they change nothing; only the
//                       very last index of the order is needed besides (a draw above a sum that
//                       stays below it takes it). Bound by its three launches and one
//                       workgroup's sort: 38 us of kernels for a 128,256-entry vocabulary with
//                       about 300 logits that count, where sorting everything took 530 us.
//   launch_sample       the whole order, where more than kTopCap logits count (flat
//                       distributions), where a logit is NaN or the maximum infinite, or where
//                       the caller asks for the order or the probabilities.
// A call that needs the second after the first pays for both and for the wait between them (about
// 50 us). With 128,256 logits of deviation 10, by temperature (the logits that count; a whole call by
// the whole order alone, before k_rs_scan read whole lines, and now): 0.8 (610) 492 -> 54 us, 2 (54,000)
// 1,140 -> 900, 3 (123,000) 2,940 -> 2,730 to 3,270 -> 3,050 by top_p, 5 (all) 6,170 -> 6,020 to 8,440
// -> 8,290, 10 (all) 9,080 -> 9,010 to 14,060 -> 13,990: there the sums in order take nearly all of it.
#include <algorithm>

#include "dev_common.hpp"
#include "expf_libm.hpp"
#include "tf_internal.hpp"

namespace tfk {
namespace {

constexpr int kSampleThreads = 1024;

// expf_libm's table in constant memory
__constant__ uint64_t kExp2Tab[32] = TF_EXP2_TABLE;

// ---- radix sort of (key, index) pairs
// Keys: the logits mapped to unsigned integers whose ascending order is the logits'
// descending order (-0 taken as +0, as `>` compares them equal). Each wave owns a tile
// of kRsTile consecutive elements; a pass counts the tile's digits, an exclusive scan over
// [digit][tile] turns the counts into offsets, and the wave scatters its tile in index
// order (lanes of a 64-element step that share a digit are ranked by lane), so the sort
// is stable.
constexpr int kRsTile = 1024;
constexpr int kRsWaves = kBlock / kWave;

__device__ __forceinline__ uint32_t desc_key(float f) {
    uint32_t u = __float_as_uint(f == 0.0f ? 0.0f : f);
    u = (u & 0x80000000u) ? ~u : (u | 0x80000000u);  // ascending float order
    return ~u;
}

__global__ __launch_bounds__(kBlock) void k_rs_init(const float* logits, uint32_t* key, int32_t* val, int n) {
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        key[i] = desc_key(logits[i]);
        val[i] = i;
    }
}

__global__ __launch_bounds__(kBlock) void k_rs_hist(const uint32_t* key, int n, int shift, uint32_t* hist,
                                                    int tiles) {
    __shared__ uint32_t cnt[kRsWaves][256];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int tile = blockIdx.x * kRsWaves + wv;
    for (int d = lane; d < 256; d += kWave) cnt[wv][d] = 0;
    __syncthreads();
    if (tile < tiles) {
        const int end = min(n, (tile + 1) * kRsTile);
        for (int i = tile * kRsTile + lane; i < end; i += kWave) atomicAdd(&cnt[wv][(key[i] >> shift) & 255u], 1u);
    }
    __syncthreads();
    if (tile < tiles)
        for (int d = lane; d < 256; d += kWave) hist[(size_t)d * tiles + tile] = cnt[wv][d];
}

// Exclusive prefix sum of m counts (a multiple of 4) in place, one workgroup: segments of 4096
// counts, a uint4 per thread (coalesced; a contiguous run per thread instead, read one word
// at a time, took 57 us for 32,256 counts), the next segment loading while this one is summed.
__global__ __launch_bounds__(1024) void k_rs_scan(uint32_t* hist, int m) {
    __shared__ uint32_t wsum[2][16];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    uint4* h4 = (uint4*)hist;
    const int n4 = m / 4;
    const uint4 zero = make_uint4(0, 0, 0, 0);
    uint32_t base = 0;
    uint4 cur = t < n4 ? h4[t] : zero;
    for (int i0 = 0, it = 0; i0 < n4; i0 += 1024, it ^= 1) {
        const int i = i0 + t;
        const uint4 nxt = i + 1024 < n4 ? h4[i + 1024] : zero;
        const uint32_t sum = cur.x + cur.y + cur.z + cur.w;
        uint32_t inc = sum;  // inclusive scan over the wave
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t v = (uint32_t)__shfl_up((int)inc, o);
            inc += lane >= o ? v : 0u;
        }
        if (lane == 63) wsum[it][wave] = inc;
        __syncthreads();
        uint32_t before = 0, all = 0;
#pragma unroll
        for (int w = 0; w < 16; ++w) {
            before += w < wave ? wsum[it][w] : 0u;
            all += wsum[it][w];
        }
        const uint32_t r = base + before + inc - sum;
        if (i < n4) h4[i] = make_uint4(r, r + cur.x, r + cur.x + cur.y, r + cur.x + cur.y + cur.z);
        base += all;
        cur = nxt;
    }
}

__global__ __launch_bounds__(kBlock) void k_rs_scatter(const uint32_t* kin, const int32_t* vin, uint32_t* kout,
                                                       int32_t* vout, int n, int shift, const uint32_t* hist,
                                                       int tiles) {
    __shared__ uint32_t off[kRsWaves][256];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int tile = blockIdx.x * kRsWaves + wv;
    if (tile >= tiles) return;  // whole waves: no barrier below
    for (int d = lane; d < 256; d += kWave) off[wv][d] = hist[(size_t)d * tiles + tile];
    const uint64_t below = (1ull << lane) - 1ull;
    const int end = min(n, (tile + 1) * kRsTile);
    for (int i0 = tile * kRsTile; i0 < end; i0 += kWave) {
        const int i = i0 + lane;
        const bool valid = i < end;
        const uint32_t k = valid ? kin[i] : 0u;
        const uint32_t d = (k >> shift) & 255u;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int bit = 0; bit < 8; ++bit) {
            const uint64_t set = __ballot((d >> bit) & 1u);
            peers &= ((d >> bit) & 1u) ? set : ~set;
        }
        const uint32_t base = valid ? off[wv][d] : 0u;
        if (valid) {
            const uint32_t dst = base + (uint32_t)__popcll(peers & below);
            kout[dst] = k;
            vout[dst] = vin[i];
            if ((peers >> lane) == 1ull) off[wv][d] = base + (uint32_t)__popcll(peers);  // the group's last lane
        }
    }
}

// The next float above s minus s (s >= 0 finite), a quarter of it: values at or below
// this cannot change s when added.
__device__ __forceinline__ float quarter_ulp(float s) {
    return (__uint_as_float(__float_as_uint(s) + 1u) - s) * 0.25f;
}

__device__ __forceinline__ float lane_value(float v, int j) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), j));
}

// Calls f(i, value) for i = 0, 1, ... over val(0), val(1), ... val(n - 1) in order, one wave:
// 64 values per register, eight registers per refill, the next eight loading while these
// are consumed. `stuck(first)` ends it before a group of 64 whose first (largest) value
// can no longer change the sum; f ends it by returning true.
template <class Val, class Stuck, class F>
__device__ __forceinline__ void in_order(int n, Val val, Stuck stuck, F f) {
    const int lane = threadIdx.x & 63;
    float cur[8], nxt[8];
    auto load = [&](int base, float (&b)[8]) {
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const int i = base + 64 * c + lane;
            b[c] = i < n ? val(i) : 0.0f;
        }
    };
    load(0, cur);
    for (int base = 0; base < n; base += 512) {
        load(base + 512, nxt);
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const int cb = base + 64 * c;
            if (cb < n) {
                if (stuck(lane_value(cur[c], 0))) return;
                const int cnt = min(64, n - cb);
                for (int j = 0; j < cnt; ++j)
                    if (f(cb + j, lane_value(cur[c], j))) return;
            }
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) cur[c] = nxt[c];
    }
}

// Steps 3-5 on one wave over val(0) .. val(n - 1) in descending order: s; the nucleus (z, and how
// many values it keeps of `total`, all where the sum stays below top_p); the place of the draw, or -1
// for the last kept one.
template <class Val>
__device__ __forceinline__ float sum_in_order(int n, Val val) {
    float s = 0.0f;
    in_order(n, val, [&](float v) { return v <= quarter_ulp(s); },
             [&](int, float v) {
                 s += v;
                 return false;
             });
    return s;
}
template <class Val>
__device__ __forceinline__ float nucleus(int n, int total, float top_p, int& last, Val val) {
    float acc = 0.0f;
    last = total;
    in_order(n, val, [&](float v) { return v <= quarter_ulp(acc); },
             [&](int i, float v) {
                 acc += v;
                 if (acc >= top_p) {
                     last = i + 1;
                     return true;
                 }
                 return false;
             });
    return acc;
}
template <class Val>
__device__ __forceinline__ int draw(int n, float r, Val val) {
    float acc = 0.0f;
    int place = -1;
    in_order(n, val, [&](float v) { return v <= quarter_ulp(acc); },
             [&](int i, float v) {
                 acc += v;
                 if (r <= acc) {
                     place = i;
                     return true;
                 }
                 return false;
             });
    return place;
}

// Step 2 for the whole order.
__global__ __launch_bounds__(kBlock) void k_sample_exp(const float* logits, const int32_t* idx, float* p, int n,
                                                       float temperature) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    const float m = logits[idx[0]];
    if (i < n) p[i] = expf_libm((logits[idx[i]] - m) / temperature, kExp2Tab);
}

// Steps 3-5 for the whole order (one workgroup): the token, and the final probabilities in place of
// p. The divisions run on every wave between the sums (on the one wave that adds they took 1.5 % of a
// nearly flat 128K vocabulary's 14 ms).
__global__ __launch_bounds__(kSampleThreads) void k_sample(const int32_t* idx, float* p, int n, float top_p, float r,
                                                           int32_t* out) {
    __shared__ float sh_s, sh_z;
    __shared__ int sh_last;
    const int tid = threadIdx.x;
    const bool w0 = tid < 64;
    auto val = [&](int i) { return p[i]; };
    if (w0) {
        const float s = sum_in_order(n, val);
        if (tid == 0) sh_s = s;
    }
    __syncthreads();
    const float s = sh_s;
    for (int i = tid; i < n; i += kSampleThreads) p[i] = p[i] / s;
    __syncthreads();
    int last = n;
    if (top_p < 1.0f) {
        if (w0) {
            const float z = nucleus(n, n, top_p, last, val);
            if (tid == 0) {
                sh_z = z;
                sh_last = last;
            }
        }
        __syncthreads();
        const float z = sh_z;
        last = sh_last;
        for (int i = tid; i < last; i += kSampleThreads) p[i] = p[i] / z;
        __syncthreads();
    }
    if (w0) {
        const int place = draw(last, r, val);
        if (tid == 0) *out = idx[place >= 0 ? place : last - 1];
    }
}

// ---- the logits that count only (launch_sample_top)

constexpr int kTopCap = 4096;      // entries the LDS sort holds
constexpr int kTopBlocks = 64;     // workgroups of the two passes over the logits
constexpr float kTopCut = -20.0f;  // e^-20 < 2^-28

// Scratch: the passes' results, then the picked (key, index) entries.
struct TopWork {
    unsigned long long hi[kTopBlocks];  // per workgroup: least (key, index), the largest logit
    unsigned long long lo[kTopBlocks];  // greatest (key, index), the last of the order
    int32_t nan[kTopBlocks];            // a NaN among its logits
    int32_t count;                      // entries picked (may exceed kTopCap)
    unsigned long long list[kTopCap];
};

__device__ __forceinline__ unsigned long long top_entry(float l, int i) {
    return ((unsigned long long)desc_key(l) << 32) | (uint32_t)i;
}

// Pass 1: each workgroup's first and last entry of the order.
__global__ __launch_bounds__(kBlock) void k_top_range(const float* logits, int n, TopWork* w) {
    __shared__ unsigned long long sh_hi[kWavesPerBlock], sh_lo[kWavesPerBlock];
    __shared__ int sh_nan[kWavesPerBlock];
    unsigned long long hi = ~0ull, lo = 0ull;
    int nan = 0;
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += kTopBlocks * kBlock) {
        const float l = logits[i];
        const unsigned long long e = top_entry(l, i);
        hi = e < hi ? e : hi;
        lo = e > lo ? e : lo;
        nan |= l != l;
    }
    hi = ~wave_max_u64(~hi);
    lo = wave_max_u64(lo);
    nan = __ballot(nan) != 0ull;
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        sh_hi[wave] = hi;
        sh_lo[wave] = lo;
        sh_nan[wave] = nan;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < kWavesPerBlock; ++k) {
            hi = sh_hi[k] < hi ? sh_hi[k] : hi;
            lo = sh_lo[k] > lo ? sh_lo[k] : lo;
            nan |= sh_nan[k];
        }
        w->hi[blockIdx.x] = hi;
        w->lo[blockIdx.x] = lo;
        w->nan[blockIdx.x] = nan;
        if (blockIdx.x == 0) w->count = 0;
    }
}

// The largest logit: lane b of every wave reads workgroup b's entry (kTopBlocks is a wave).
__device__ __forceinline__ float top_max(const float* logits, const TopWork* w) {
    static_assert(kTopBlocks == kWave, "a lane per workgroup of the first pass");
    return logits[(uint32_t)~wave_max_u64(~w->hi[threadIdx.x & 63])];
}

// Pass 2: the entries that count, in any order (the sort makes it one), a place per wave and
// round from one atomic.
__global__ __launch_bounds__(kBlock) void k_top_pick(const float* logits, int n, float temperature, TopWork* w) {
    const float m = top_max(logits, w);
    const int lane = threadIdx.x & 63;
    for (int i0 = blockIdx.x * kBlock + (threadIdx.x & ~63); i0 < n; i0 += kTopBlocks * kBlock) {
        const int i = i0 + lane;
        const float l = i < n ? logits[i] : 0.0f;
        const bool in = i < n && (l - m) / temperature >= kTopCut;
        const uint64_t mask = __ballot(in);
        if (!mask) continue;
        int base = 0;
        if (lane == 0) base = atomicAdd(&w->count, __popcll(mask));
        base = __builtin_amdgcn_readfirstlane(base) + __popcll(mask & ((1ull << lane) - 1ull));
        if (in && base < kTopCap) w->list[base] = top_entry(l, i);
    }
}

// Sort, probabilities and the pick, one workgroup. *out < 0: the whole order is needed.
__global__ __launch_bounds__(kSampleThreads) void k_top_sample(const float* logits, int n, float temperature,
                                                               float top_p, float r, const TopWork* w, int32_t* out) {
    __shared__ unsigned long long e[kTopCap];
    __shared__ float p[kTopCap];
    const int tid = threadIdx.x, count = w->count;
    const float m = top_max(logits, w);
    const bool nan = __ballot(w->nan[tid & 63] != 0) != 0ull;
    if (nan || !(fabsf(m) < INFINITY) || count > kTopCap || count < 1) {
        if (tid == 0) *out = -1;
        return;
    }
    int size = 64;  // the power of two that holds the entries
    while (size < count) size *= 2;
    for (int i = tid; i < size; i += kSampleThreads) e[i] = i < count ? w->list[i] : ~0ull;
    __syncthreads();
    // bitonic sort, thread t taking pair t (entries 2 t - (t mod j) and + j). A step with
    // j <= 64 stays inside the 128 entries of each wave's pairs, so between two such steps the
    // wave's own LDS order is enough (36 of the 55 steps for 1024 entries)
    for (int k = 2; k <= size; k *= 2)
        for (int j = k / 2; j > 0; j /= 2) {
            for (int t = tid; t < size / 2; t += kSampleThreads) {
                const int a = 2 * t - (t & (j - 1)), b = a + j;
                const unsigned long long x = e[a], y = e[b];
                if ((x > y) == ((a & k) == 0)) {
                    e[a] = y;
                    e[b] = x;
                }
            }
            if (j > 64 || (j == 1 && k > 64)) {  // the next step's distance is j / 2, or k after j = 1
                __syncthreads();
            } else {
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
        }
    __syncthreads();
    for (int i = tid; i < count; i += kSampleThreads)
        p[i] = expf_libm((logits[(uint32_t)e[i]] - m) / temperature, kExp2Tab);
    __syncthreads();
    if (tid < 64) {
        // a division by s or z is the same float wherever it happens: few values, divided as they are read
        const float s = sum_in_order(count, [&](int i) { return p[i]; });
        int last = n;
        float z = 0.0f;
        if (top_p < 1.0f) z = nucleus(count, n, top_p, last, [&](int i) { return p[i] / s; });
        const int place = draw(min(count, last), r, [&](int i) { return top_p < 1.0f ? p[i] / s / z : p[i] / s; });
        const int at = place >= 0 ? place : last - 1;
        // a draw past every sum: the last kept index, the whole order's last one if all are kept
        const unsigned long long lo = wave_max_u64(w->lo[tid]);
        if (tid == 0) *out = (int32_t)(uint32_t)(at < count ? e[at] : lo);
    }
}

}  // namespace

size_t sample_work_bytes(int n) {
    const size_t a = ((size_t)n * 4 + 255) / 256 * 256;
    const size_t tiles = ((size_t)n + kRsTile - 1) / kRsTile;
    return std::max(5 * a + (256 * tiles * 4 + 255) / 256 * 256, sizeof(TopWork));
}

hipError_t launch_sample_top(const float* logits, int n, float temperature, float top_p, float r, void* work,
                             size_t work_bytes, int32_t* d_token, hipStream_t st) {
    if (work_bytes < sizeof(TopWork)) return hipErrorInvalidValue;
    TopWork* w = (TopWork*)work;
    hipLaunchKernelGGL(k_top_range, dim3(kTopBlocks), dim3(kBlock), 0, st, logits, n, w);
    hipLaunchKernelGGL(k_top_pick, dim3(kTopBlocks), dim3(kBlock), 0, st, logits, n, temperature, w);
    hipLaunchKernelGGL(k_top_sample, dim3(1), dim3(kSampleThreads), 0, st, logits, n, temperature, top_p, r, w, d_token);
    return hipGetLastError();
}

hipError_t launch_sample(const float* logits, int n, float temperature, float top_p, float r, void* work,
                         size_t work_bytes, int32_t* d_token, int32_t* d_sorted_idx, float* d_probs, hipStream_t st) {
    const size_t a = ((size_t)n * 4 + 255) / 256 * 256;
    if (work_bytes < sample_work_bytes(n)) return hipErrorInvalidValue;
    uint8_t* w = (uint8_t*)work;
    uint32_t* key[2] = {(uint32_t*)w, (uint32_t*)(w + a)};
    int32_t* val[2] = {(int32_t*)(w + 2 * a), (int32_t*)(w + 3 * a)};
    float* p = d_probs ? d_probs : (float*)(w + 4 * a);
    uint32_t* hist = (uint32_t*)(w + 5 * a);
    const int tiles = (n + kRsTile - 1) / kRsTile;
    const int blocks = (tiles + kRsWaves - 1) / kRsWaves;
    hipLaunchKernelGGL(k_rs_init, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, st, logits, key[0], val[0], n);
    for (int pass = 0; pass < 4; ++pass) {
        const int src = pass & 1;
        hipLaunchKernelGGL(k_rs_hist, dim3(blocks), dim3(kBlock), 0, st, key[src], n, 8 * pass, hist, tiles);
        hipLaunchKernelGGL(k_rs_scan, dim3(1), dim3(1024), 0, st, hist, 256 * tiles);
        hipLaunchKernelGGL(k_rs_scatter, dim3(blocks), dim3(kBlock), 0, st, key[src], val[src], key[src ^ 1],
                           val[src ^ 1], n, 8 * pass, hist, tiles);
    }
    // four passes: the sorted indices are back in val[0]
    const int32_t* idx = val[0];
    if (d_sorted_idx) {
        hipError_t e = hipMemcpyAsync(d_sorted_idx, idx, (size_t)n * 4, hipMemcpyDeviceToDevice, st);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(k_sample_exp, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, st, logits, idx, p, n,
                       temperature);
    hipLaunchKernelGGL(k_sample, dim3(1), dim3(kSampleThreads), 0, st, idx, p, n, top_p, r, d_token);
    return hipGetLastError();
}

}  // namespace tfk
