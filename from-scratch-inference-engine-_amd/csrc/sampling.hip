// Next-token choice on the device, one block per row of float32 logits.
//
//   temperature <= 0 : argmax, ties to the smallest index.
//   temperature  > 0 : temperature -> top-k -> top-p -> inverse CDF against a uniform number u
//                      that the host supplies per row.
// The kept set is the one a sort by logit would give (all tokens tied with the last kept one are
// kept); the draw walks the kept tokens in vocabulary order: first i with u * mass < cumulative.
// Thresholds: the row's range below its maximum (at most 32, in logits) is cut into 2,048 equal bins; a pass over
// the row adds up every bin's count and weight in LDS, a scan finds the bin in which the threshold lies, a second pass
// lays that bin's few hundred tokens side by side, and comparing those with each other gives the token at which the
// kept set ends.  The bins' weights are integers (two limbs of the float's own bits), so the order in which the threads
// add them changes nothing.  Rows that do not fit this (a maximum that is not finite, a NaN, a temperature whose inverse
// is zero or infinite, so that a weight may be a NaN, more than 2,048 tokens in the threshold's bin) are bisected over the order-preserving integer image of the logits, a pass a probe.
// What bounds it is how often a compute unit reads a row of 600 KB from the caches: one pass for greedy, two at a plain
// temperature, 4 with a threshold and 5 with two whose bins differ, where the bisection alone took 32 a threshold (64 rows of
// 152,064, a fifth of them each greedy, at a temperature, top k, top p and both: 152 us, 1,504 with the bisection alone).
// Long rows are shared by several workgroups where the call has few of them (below): 89 us for the same call.
#include "common.h"
#include "api.h"

#include <math.h>
#include <stddef.h>

namespace {

constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / FSIE_WAVE;

__device__ __forceinline__ uint32_t order_key(float v) {
    const uint32_t u = __float_as_uint(v);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ double wave_sum_f64(double v) {
#pragma unroll
    for (int off = FSIE_WAVE / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, FSIE_WAVE);
    return v;
}

__device__ double block_sum_f64(double v, double* scratch) {
    const int lane = threadIdx.x & (FSIE_WAVE - 1), wave = threadIdx.x / FSIE_WAVE;
    v = wave_sum_f64(v);
    __syncthreads();
    if (lane == 0) scratch[wave] = v;
    __syncthreads();
    double total = 0.0;
    for (int w = 0; w < kWaves; ++w) total += scratch[w];
    return total;
}

struct Best {
    float value;
    int index;
};

__device__ __forceinline__ Best better(Best a, Best b) {
    if (b.value > a.value || (b.value == a.value && b.index < a.index)) return b;
    return a;
}

// `low`, `nan`: this thread's smallest value above -inf, and whether it met a NaN.
template <bool RANGE>
__device__ Best block_argmax(const float* row, int vocab, float* sval, int* sidx, float* low, bool* nan) {
    Best best{-INFINITY, 0x7fffffff};
    *low = INFINITY;
    *nan = false;
    auto take = [&](float v, int i) {
        if (RANGE) {
            *nan |= v != v;
            if (v > -INFINITY) *low = fminf(*low, v);
        }
        if (best.index == 0x7fffffff || v > best.value) best = Best{v, i};  // strict: lowest index of a stripe wins
    };
    int done = 0;
    if (reinterpret_cast<uintptr_t>(row) % 16 == 0) {
        // 16-byte loads, four of them in flight per thread
        const int quads = vocab / 4;
        constexpr int U = 4;
        for (int q0 = threadIdx.x; q0 < quads; q0 += blockDim.x * U) {
            float4 v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int q = min(q0 + u * static_cast<int>(blockDim.x), quads - 1);
                v[u] = *reinterpret_cast<const float4*>(row + 4 * q);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int q = q0 + u * blockDim.x;
                if (q < quads) {
                    take(v[u].x, 4 * q);
                    take(v[u].y, 4 * q + 1);
                    take(v[u].z, 4 * q + 2);
                    take(v[u].w, 4 * q + 3);
                }
            }
        }
        done = quads * 4;
    }
    for (int i = done + threadIdx.x; i < vocab; i += blockDim.x) take(row[i], i);
#pragma unroll
    for (int off = FSIE_WAVE / 2; off > 0; off >>= 1) {
        Best other{__shfl_xor(best.value, off, FSIE_WAVE), __shfl_xor(best.index, off, FSIE_WAVE)};
        best = better(best, other);
    }
    const int lane = threadIdx.x & (FSIE_WAVE - 1), wave = threadIdx.x / FSIE_WAVE;
    __syncthreads();
    if (lane == 0) {
        sval[wave] = best.value;
        sidx[wave] = best.index;
    }
    __syncthreads();
    Best total{sval[0], sidx[0]};
    for (int w = 1; w < kWaves; ++w) total = better(total, Best{sval[w], sidx[w]});
    return total;
}

// weight of token i under the row's temperature; mx is the row maximum
__device__ __forceinline__ double token_weight(float logit, float mx, float inv_temp) {
    return static_cast<double>(expf((logit - mx) * inv_temp));
}

// whether every token of a row without NaN and with a finite maximum has a weight that is a number
__device__ __forceinline__ bool weighs(float inv_temp) { return inv_temp > 0.f && inv_temp < INFINITY; }

constexpr int kBins = 2048;        // two a thread
constexpr int kListed = 2048;      // tokens of one bin that are compared with each other
constexpr float kRange = 32.f;     // logits below the maximum that the bins cover; the last one takes the rest
constexpr int kMaxBinned = 1 << 23;  // a vocabulary beyond this leaves the limbs no room for its sum
constexpr int kRuns = 256;         // runs of the vocabulary whose weights the draw adds up first
constexpr int kUnroll = 8;         // loads of a thread in flight

// A weight (a float in [0, 1]) as an integer of 2^-hi_bits units and, for what that leaves, one of 2^-(hi_bits + 40):
// its 24 bits shifted, none rounded away above 2^-(hi_bits + 17).
struct Limbs {
    unsigned long long hi, lo;
};
__device__ __forceinline__ Limbs limbs_of(float w, int hi_bits) {
    const uint32_t u = __float_as_uint(w);
    const int e = static_cast<int>(u >> 23);
    if (e == 0) return Limbs{0, 0};
    const unsigned long long m = (u & 0x7fffffu) | 0x800000u;
    const int up = e - 150 + hi_bits;  // m * 2^(e - 150) in units of 2^-hi_bits
    if (up >= 0) return Limbs{m << up, 0};
    const int down = -up;
    if (down <= 40) return Limbs{down < 24 ? m >> down : 0ull, (m & ((1ull << down) - 1)) << (40 - down)};
    return Limbs{0, down - 40 < 24 ? m >> (down - 40) : 0ull};
}
__device__ __forceinline__ double value_of(Limbs v, int hi_bits) {
    return ldexp(static_cast<double>(v.hi), -hi_bits) + ldexp(static_cast<double>(v.lo), -(hi_bits + 40));
}

// Every element of the row once, kUnroll loads of a thread under way: body(value, index).
template <typename F>
__device__ __forceinline__ void for_row(const float* __restrict__ row, int vocab, F body) {
    for (int i0 = threadIdx.x; i0 < vocab; i0 += kThreads * kUnroll) {
        float v[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) v[u] = row[min(i0 + u * kThreads, vocab - 1)];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            const int i = i0 + u * kThreads;
            if (i < vocab) body(v[u], i);
        }
    }
}

struct Binned {
    unsigned int count[kBins];
    unsigned long long hi[kBins], lo[kBins];
    float listed[kListed], weight[kListed];
    double wave_base[kWaves + 1];
    double above;      // what lies above the chosen bin
    int bin;           // the chosen bin, -1: none found
    unsigned int n_listed;
    uint32_t cut;      // key of the token at which the kept set ends; 0: not found
};
static_assert(sizeof(Binned) <= 60 * 1024, "the bins and the list must fit the LDS a kernel may declare");

__device__ __forceinline__ int bin_of(float v, float mx, float scale) {
    return static_cast<int>(fminf((mx - v) * scale, static_cast<float>(kBins - 1)));  // -inf and all below the range: the last
}

// The bin in which the running sum of the bins' values (from the maximum down) first reaches `target`, and the sum above
// it, left in `s`; returns the sum of all.  Fixed order of additions.
template <typename F>
__device__ double find_bin(Binned& s, double target, F value) {
    const int lane = threadIdx.x & (FSIE_WAVE - 1), wave = threadIdx.x / FSIE_WAVE;
    const double v0 = value(2 * threadIdx.x), v1 = value(2 * threadIdx.x + 1);
    double run = v0 + v1;
#pragma unroll
    for (int off = 1; off < FSIE_WAVE; off <<= 1) {
        const double other = __shfl_up(run, off, FSIE_WAVE);
        if (lane >= off) run += other;
    }
    __syncthreads();
    if (lane == FSIE_WAVE - 1) s.wave_base[wave + 1] = run;
    if (threadIdx.x == 0) {
        s.wave_base[0] = 0.0;
        s.bin = -1;
    }
    __syncthreads();
    double base = 0.0, total = 0.0;
    for (int w = 0; w < kWaves; ++w) {
        if (w == wave) base = total;
        total += s.wave_base[w + 1];
    }
    const double left = __shfl_up(run, 1, FSIE_WAVE);  // (all lanes together: a shuffle reads active lanes only)
    const double before = base + (lane ? left : 0.0);
    const double upto = base + run;
    if (before < target && target <= upto) {
        const bool first = target <= before + v0;
        s.bin = 2 * threadIdx.x + (first ? 0 : 1);
        s.above = first ? before : before + v0;
    }
    __syncthreads();
    return total;
}

// The tokens of bin `bin`, side by side in LDS (their order is left to chance: only sums of integers are taken of them).
// False if they are too many.
__device__ bool list_bin(Binned& s, const float* row, int vocab, float mx, float scale, int bin) {
    if (threadIdx.x == 0) s.n_listed = 0;
    __syncthreads();
    for_row(row, vocab, [&](float v, int) {
        if (bin_of(v, mx, scale) == bin) {
            const unsigned int at = atomicAdd(&s.n_listed, 1u);
            if (at < kListed) s.listed[at] = v;
        }
    });
    __syncthreads();
    return s.n_listed <= kListed;
}

// Sets `cut` to the key at which the kept set ends, by bins; false where the row has to be bisected.
__device__ bool cut_by_bins(Binned& s, const float* row, int vocab, float mx, float low, bool nan, float inv_temp, int k,
                            float p, uint32_t* cut_out) {
    __shared__ float lowest[kWaves];
    __shared__ int odd;
    if (threadIdx.x == 0) odd = 0;
    for (int b = threadIdx.x; b < kBins; b += kThreads) {
        s.count[b] = 0;
        s.hi[b] = s.lo[b] = 0;
    }
    low = -wave_max(-low);
    __syncthreads();
    if ((threadIdx.x & (FSIE_WAVE - 1)) == 0) lowest[threadIdx.x / FSIE_WAVE] = low;
    if (nan) odd = 1;
    __syncthreads();
    for (int w = 0; w < kWaves; ++w) low = fminf(low, lowest[w]);
    const float range = fminf(mx - low, kRange);
    if (odd || !(range > 1e-30f) || !weighs(inv_temp)) return false;
    const float scale = static_cast<float>(kBins - 1) / range;
    const int hi_bits = 63 - (32 - __clz(vocab));  // vocab < 2^(32 - clz): the sum of all weights stays below 2^63
    for_row(row, vocab, [&](float v, int) {
        const int b = bin_of(v, mx, scale);
        if (k > 0) atomicAdd(&s.count[b], 1u);
        if (p < 1.f) {
            const Limbs w = limbs_of(expf((v - mx) * inv_temp), hi_bits);
            if (w.hi) atomicAdd(&s.hi[b], w.hi);
            if (w.lo) atomicAdd(&s.lo[b], w.lo);
        }
    });
    __syncthreads();
    const auto bin_weight = [&](int b) { return value_of(Limbs{s.hi[b], s.lo[b]}, hi_bits); };
    uint32_t cut = 0;
    int k_bin = -1;
    Limbs k_kept{0, 0};  // weight of the listed tokens that top k keeps
    if (k > 0) {
        find_bin(s, static_cast<double>(k), [&](int b) { return static_cast<double>(s.count[b]); });
        k_bin = s.bin;
        if (k_bin < 0 || !list_bin(s, row, vocab, mx, scale, k_bin)) return false;
        const int n = static_cast<int>(s.n_listed), want = k - static_cast<int>(s.above);
        for (int i = threadIdx.x; i < n; i += kThreads) {
            const uint32_t mine = order_key(s.listed[i]);
            int above = 0, upto = 0;
            for (int j = 0; j < n; ++j) {
                const uint32_t other = order_key(s.listed[j]);
                above += other > mine;
                upto += other >= mine;
            }
            if (above < want && want <= upto) s.cut = mine;  // (equal keys write the same)
        }
        __syncthreads();
        cut = s.cut;
        __syncthreads();
    }
    if (p < 1.f) {
        double kept;
        if (k_bin >= 0) {
            // the bins above that of top k, and the kept part of that one
            const int n = static_cast<int>(s.n_listed);
            if (threadIdx.x == 0) s.hi[k_bin] = s.lo[k_bin] = 0;
            __syncthreads();
            for (int i = threadIdx.x; i < n; i += kThreads) {
                if (order_key(s.listed[i]) < cut) continue;
                const Limbs w = limbs_of(expf((s.listed[i] - mx) * inv_temp), hi_bits);
                if (w.hi) atomicAdd(&s.hi[k_bin], w.hi);
                if (w.lo) atomicAdd(&s.lo[k_bin], w.lo);
            }
            for (int b = threadIdx.x; b < kBins; b += kThreads)
                if (b > k_bin) s.hi[b] = s.lo[b] = 0;
            __syncthreads();
        }
        kept = find_bin(s, INFINITY, bin_weight);
        const double target = static_cast<double>(p) * kept;
        if (!(target > 0.0)) {
            *cut_out = order_key(mx);
            return true;
        }
        find_bin(s, target, bin_weight);
        const int bin = s.bin;
        if (bin < 0) return false;  // (a target that rounding puts between two bins)
        const double above = s.above;
        if (bin != k_bin && !list_bin(s, row, vocab, mx, scale, bin)) return false;
        const int n = static_cast<int>(s.n_listed);
        for (int i = threadIdx.x; i < n; i += kThreads) s.weight[i] = expf((s.listed[i] - mx) * inv_temp);
        if (threadIdx.x == 0) s.cut = 0;
        __syncthreads();
        for (int i = threadIdx.x; i < n; i += kThreads) {
            const uint32_t mine = order_key(s.listed[i]);
            if (mine < cut) continue;
            Limbs over{0, 0}, upto{0, 0};
            for (int j = 0; j < n; ++j) {
                const uint32_t other = order_key(s.listed[j]);
                if (other < mine) continue;
                const Limbs w = limbs_of(s.weight[j], hi_bits);
                upto.hi += w.hi;
                upto.lo += w.lo;
                if (other > mine) {
                    over.hi += w.hi;
                    over.lo += w.lo;
                }
            }
            if (above + value_of(over, hi_bits) < target && target <= above + value_of(upto, hi_bits)) s.cut = mine;
        }
        __syncthreads();
        const uint32_t found = s.cut;
        if (found == 0) return false;
        cut = found;
    }
    *cut_out = cut;
    return true;
}

// The same by bisection over the keys, a pass over the row a probe.
__device__ uint32_t cut_by_bisection(const float* row, int vocab, float mx, float inv_temp, int k, float p, double* scratch) {
    const uint32_t key_max = order_key(mx);
    uint32_t cut = 0;
    if (k > 0) {
        // largest key t with count(key >= t) >= k
        uint32_t lo = 0, hi = key_max;
        while (lo < hi) {
            const uint32_t mid = lo + (hi - lo) / 2 + ((hi - lo) & 1);
            double cnt = 0.0;
            for (int i = threadIdx.x; i < vocab; i += blockDim.x) cnt += order_key(row[i]) >= mid ? 1.0 : 0.0;
            cnt = block_sum_f64(cnt, scratch);
            if (cnt >= static_cast<double>(k)) lo = mid; else hi = mid - 1;
        }
        cut = lo;
    }
    if (p < 1.f) {
        double kept = 0.0;
        for (int i = threadIdx.x; i < vocab; i += blockDim.x) {
            const float v = row[i];
            if (order_key(v) >= cut) kept += token_weight(v, mx, inv_temp);
        }
        kept = block_sum_f64(kept, scratch);
        const double target = static_cast<double>(p) * kept;
        // largest key t >= cut with mass(key >= t) >= target
        uint32_t lo = cut, hi = key_max;
        while (lo < hi) {
            const uint32_t mid = lo + (hi - lo) / 2 + ((hi - lo) & 1);
            double mass = 0.0;
            for (int i = threadIdx.x; i < vocab; i += blockDim.x) {
                const float v = row[i];
                if (order_key(v) >= mid) mass += token_weight(v, mx, inv_temp);
            }
            mass = block_sum_f64(mass, scratch);
            if (mass >= target) lo = mid; else hi = mid - 1;
        }
        cut = lo;
    }
    return cut;
}

// The first token, in vocabulary order, at which the running sum of the kept weights passes uniform * their sum, from the
// sums of the runs: every wave finds the run, and the wave that owns it (`own_runs` runs a wave; -1: there is one wave)
// walks it.
__device__ void draw_from_runs(const float* __restrict__ row, int vocab, Best top, float inv_temp, uint32_t cut, double uniform,
                               const double* run_sum, int own_runs, int32_t* out) {
    const int lane = threadIdx.x & (FSIE_WAVE - 1), wave = threadIdx.x / FSIE_WAVE;
    const int rows = ((vocab + FSIE_WAVE - 1) / FSIE_WAVE + kRuns - 1) / kRuns;  // 64 tokens each
    const float mx = top.value;
    // four neighbouring runs a lane
    double part[kRuns / FSIE_WAVE], upto = 0.0;
#pragma unroll
    for (int q = 0; q < kRuns / FSIE_WAVE; ++q) {
        part[q] = run_sum[lane * (kRuns / FSIE_WAVE) + q];
        upto += part[q];
    }
#pragma unroll
    for (int off = 1; off < FSIE_WAVE; off <<= 1) {
        const double other = __shfl_up(upto, off, FSIE_WAVE);
        if (lane >= off) upto += other;
    }
    const double total = __shfl(upto, FSIE_WAVE - 1, FSIE_WAVE);
    const double threshold = uniform * total;
    double before = __shfl_up(upto, 1, FSIE_WAVE);
    if (lane == 0) before = 0.0;
    // the first lane whose running sum passes the threshold, then the first of its runs
    const unsigned long long past = __ballot(threshold < upto);
    if (past == 0) {  // a NaN or no weight at all
        if (threadIdx.x == 0) *out = top.index;
        return;
    }
    const int owner = __ffsll(past) - 1;
    int run = lane * (kRuns / FSIE_WAVE);
    double cum = before;
#pragma unroll
    for (int q = 0; q < kRuns / FSIE_WAVE - 1; ++q) {
        if (run == lane * (kRuns / FSIE_WAVE) + q && threshold >= cum + part[q]) {
            cum += part[q];
            ++run;
        }
    }
    run = __shfl(run, owner, FSIE_WAVE);
    cum = __shfl(cum, owner, FSIE_WAVE);
    if (own_runs > 0 && wave != run / own_runs) return;
    int last_kept = -1;
    for (int j = 0; j < rows; ++j) {
        const int64_t i = (static_cast<int64_t>(run) * rows + j) * FSIE_WAVE + lane;
        const float v = row[i < vocab ? i : vocab - 1];
        const bool kept = i < vocab && order_key(v) >= cut;
        double w = kept ? token_weight(v, mx, inv_temp) : 0.0;
#pragma unroll
        for (int off = 1; off < FSIE_WAVE; off <<= 1) {
            const double other = __shfl_up(w, off, FSIE_WAVE);
            if (lane >= off) w += other;
        }
        const unsigned long long hit = __ballot(kept && threshold < cum + w), any = __ballot(kept);
        if (hit) {
            if (lane == __ffsll(hit) - 1) *out = static_cast<int>(i);
            return;
        }
        if (any) last_kept = static_cast<int>((static_cast<int64_t>(run) * rows + j) * FSIE_WAVE) + 63 - __clzll(any);
        cum += __shfl(w, FSIE_WAVE - 1, FSIE_WAVE);
    }
    if (lane == 0) *out = last_kept >= 0 ? last_kept : top.index;  // rounding at the run's end
}

// Without temperatures: the maximum alone.  A kernel of its own, since the other one's extremes and registers cost this pass
// twice its time (1 row of 151,936: 9.5 us, 18 in the other; 64 rows: 14 and 21).
__global__ __launch_bounds__(kThreads) void sample_greedy_kernel(const float* __restrict__ logits, int vocab, int32_t* __restrict__ out) {
    __shared__ float sval[kWaves];
    __shared__ int sidx[kWaves];
    float low;
    bool nan;
    const Best top = block_argmax<false>(logits + static_cast<int64_t>(blockIdx.x) * vocab, vocab, sval, sidx, &low, &nan);
    if (threadIdx.x == 0) out[blockIdx.x] = top.index;
}

// CUTS: some row may have a threshold.  Without, the kernel is rid of the bins (60 KB of LDS, with which a compute unit holds one
// workgroup): 380 rows of 1,000 tokens at a temperature 19 us with them, 16.5 without; 64 of 32,000 22 and 18.
template <bool CUTS>
__global__ __launch_bounds__(kThreads) void sample_kernel(const float* __restrict__ logits, int vocab,
                                                          const float* __restrict__ temperature,
                                                          const int32_t* __restrict__ top_k,
                                                          const float* __restrict__ top_p,
                                                          const double* __restrict__ uniform,
                                                          int32_t* __restrict__ out) {
    __shared__ float sval[kWaves];
    __shared__ int sidx[kWaves];
    __shared__ double run_sum[kRuns];

    const int r = blockIdx.x;
    const float* row = logits + static_cast<int64_t>(r) * vocab;
    const float temp = temperature[r];
    const int k = CUTS && top_k && top_k[r] > 0 && top_k[r] < vocab ? top_k[r] : 0;
    const float p = CUTS && top_p ? top_p[r] : 1.f;
    const bool cuts = CUTS && temp > 0.f && (k > 0 || p < 1.f);  // (only these rows need the smallest value and look for a NaN)
    float low;
    bool nan;
    const Best top = cuts ? block_argmax<true>(row, vocab, sval, sidx, &low, &nan) : block_argmax<false>(row, vocab, sval, sidx, &low, &nan);
    if (!(temp > 0.f)) {
        if (threadIdx.x == 0) out[r] = top.index;
        return;
    }
    const float mx = top.value;
    const float inv_temp = 1.0f / temp;
    uint32_t cut = 0;  // tokens with key >= cut are kept
    if constexpr (CUTS) {
        __shared__ double sdbl[kWaves];
        __shared__ Binned binned;
        if (cuts && (vocab > kMaxBinned || !(fabsf(mx) < INFINITY) || !cut_by_bins(binned, row, vocab, mx, low, nan, inv_temp, k, p, &cut))) {
            __syncthreads();
            cut = cut_by_bisection(row, vocab, mx, inv_temp, k, p, sdbl);
        }
    }

    // inverse CDF in vocabulary order.  The vocabulary is cut into kRuns runs of whole 64 tokens; a wave adds up the
    // kept weights of kRuns / kWaves neighbouring ones, kAbreast of them at a time (a run alone is a chain of one trip to
    // memory and six exchanges between lanes, 1 us), then the wave whose run holds the threshold walks it.
    const int lane = threadIdx.x & (FSIE_WAVE - 1), wave = threadIdx.x / FSIE_WAVE;
    const int rows = ((vocab + FSIE_WAVE - 1) / FSIE_WAVE + kRuns - 1) / kRuns;  // 64 tokens each
    constexpr int kRunsOfWave = kRuns / kWaves, kAbreast = 4;
    for (int q = 0; q < kRunsOfWave; q += kAbreast) {
        const int run = wave * kRunsOfWave + q;
        if (static_cast<int64_t>(run) * rows * FSIE_WAVE >= vocab) {  // (a small vocabulary has fewer runs)
            if (lane < kAbreast) run_sum[run + lane] = 0.0;
            continue;
        }
        double mine[kAbreast] = {};
        for (int j0 = 0; j0 < rows; j0 += kUnroll / kAbreast) {
            float v[kAbreast][kUnroll / kAbreast];
            const auto token = [&](int a, int u) { return (static_cast<int64_t>(run + a) * rows + j0 + u) * FSIE_WAVE + lane; };
#pragma unroll
            for (int a = 0; a < kAbreast; ++a)
#pragma unroll
                for (int u = 0; u < kUnroll / kAbreast; ++u) v[a][u] = row[min(token(a, u), static_cast<int64_t>(vocab - 1))];
#pragma unroll
            for (int a = 0; a < kAbreast; ++a)
#pragma unroll
                for (int u = 0; u < kUnroll / kAbreast; ++u)
                    if (j0 + u < rows && token(a, u) < vocab && order_key(v[a][u]) >= cut) mine[a] += token_weight(v[a][u], mx, inv_temp);
        }
#pragma unroll
        for (int off = FSIE_WAVE / 2; off > 0; off >>= 1)
#pragma unroll
            for (int a = 0; a < kAbreast; ++a) mine[a] += __shfl_xor(mine[a], off, FSIE_WAVE);
        if (lane == 0) {
#pragma unroll
            for (int a = 0; a < kAbreast; ++a) run_sum[run + a] = mine[a];
        }
    }
    __syncthreads();
    draw_from_runs(row, vocab, top, inv_temp, cut, uniform[r], run_sum, kRunsOfWave, out + r);
}

// ---- a row shared by several workgroups -------------------------------------------------------
// One workgroup a row leaves three quarters of the chip idle at 64 rows and all but one unit at one row, and a unit
// needs some 10 us for every pass over 152,064 tokens (their exponentials and the adds in float64).  From kSplitFrom
// tokens on the row's runs are dealt to up to 64 workgroups, and the passes become launches: the maximum; bins (or,
// for rows without a threshold, the draw's sums); the threshold bins' tokens; the cut; the draw's sums; the draw.
// What a launch leaves for the next lies in a workspace of the row.
// A workgroup a row takes the same time up to 256 rows and grows with the row; shared, six launches' ends cost some 30 us
// and the rest grows with the tokens of all rows.  Alone / shared, us, a fifth of the rows each greedy, plain, top k, top p and
// both, at 1, 8, 32, 64, 128 and 256 rows:
//    16,384 tokens   34 /  31    34 / 33    35 / 43    35 / 50     35 /  63     36 /  82
//    32,000          45 /  32    46 / 34    46 / 45    46 / 51     46 /  65     48 /  94
//    65,536          69 /  34    69 / 39    70 / 49    71 / 58     72 /  77     75 / 114
//   152,064         137 /  38   138 / 47   144 / 66   152 / 89    153 / 127    159 / 193
// so rows are shared from kSplitFrom tokens on while each of them has kTokensForRow for every row of the call.  Without
// thresholds it is three launches, and the same line (32,000 tokens 16 / 9, 17 / 11, 17 / 14, 17 / 17, 17 / 24, 19 / 40).
// (Without temperatures it is one pass over the row, and a workgroup a row is the faster one; with temperatures that all
// say greedy too, but that only the device knows.)
constexpr int kSplitFrom = 16384;
constexpr int kTokensForRow = 800;
constexpr int kPart = 256;          // threads of a shared row's workgroups
constexpr int kMaxParts = 64;
constexpr int kPairs = 512;         // so many listed tokens are compared with each other, more are bisected
constexpr int kKeep = 4096;         // tokens that the list holds

struct SplitRow {
    unsigned long long hi[kBins], lo[kBins];
    double run_sum[kRuns];
    unsigned int count[kBins];
    unsigned int n_listed, cut;     // (behind the bins: cleared with them)
    unsigned int pad[2];
    float listed[kKeep];
    float part_max[kMaxParts], part_low[kMaxParts];
    int part_index[kMaxParts], part_nan[kMaxParts];
};
static_assert(sizeof(SplitRow) % 16 == 0, "rows of the workspace stay aligned");

struct RowParams {
    float temp, inv_temp, p;
    int k;
    bool cuts;
};
__device__ __forceinline__ RowParams row_params(int r, int vocab, const float* temperature, const int32_t* top_k,
                                                const float* top_p) {
    RowParams q;
    q.temp = temperature[r];
    q.inv_temp = 1.0f / q.temp;
    q.k = top_k && top_k[r] > 0 && top_k[r] < vocab ? top_k[r] : 0;
    q.p = top_p ? top_p[r] : 1.f;
    q.cuts = q.temp > 0.f && (q.k > 0 || q.p < 1.f);
    return q;
}

// The row's maximum and its place, the smallest value above -inf, whether a NaN is in it: from the parts', by a wave.
struct RowTop {
    Best best;
    float low;
    bool nan;
    // whether the row's thresholds can be found by bins, and their scale
    __device__ bool binned(int vocab, float inv_temp, float* scale) const {
        const float range = fminf(best.value - low, kRange);
        if (vocab > kMaxBinned || nan || !(fabsf(best.value) < INFINITY) || !(range > 1e-30f) || !weighs(inv_temp)) return false;
        *scale = static_cast<float>(kBins - 1) / range;
        return true;
    }
};
__device__ RowTop row_top(const SplitRow* w, int parts) {
    const int lane = threadIdx.x & (FSIE_WAVE - 1), at = min(lane, parts - 1);
    RowTop t{Best{w->part_max[at], w->part_index[at]}, w->part_low[at], w->part_nan[at] != 0};
#pragma unroll
    for (int off = FSIE_WAVE / 2; off > 0; off >>= 1) {
        t.best = better(t.best, Best{__shfl_xor(t.best.value, off, FSIE_WAVE), __shfl_xor(t.best.index, off, FSIE_WAVE)});
        t.low = fminf(t.low, __shfl_xor(t.low, off, FSIE_WAVE));
    }
    t.nan = __any(t.nan);
    // A NaN is neither larger nor smaller, so lanes that met one may have ended elsewhere than the others: lane 0's answer
    // (part 0 always has tokens) is the row's, in every wave and every launch, since loops with barriers depend on it.
    t.best = Best{__shfl(t.best.value, 0, FSIE_WAVE), __shfl(t.best.index, 0, FSIE_WAVE)};
    t.low = __shfl(t.low, 0, FSIE_WAVE);
    return t;
}

// 64-token lines of a run, and the tokens of part `part`
__device__ __forceinline__ int run_lines(int vocab) {
    return ((vocab + FSIE_WAVE - 1) / FSIE_WAVE + kRuns - 1) / kRuns;
}
__device__ __forceinline__ void part_range(int vocab, int parts, int part, int* begin, int* end) {
    const int64_t tokens = static_cast<int64_t>(run_lines(vocab)) * FSIE_WAVE * (kRuns / parts);
    *begin = static_cast<int>(min(static_cast<int64_t>(vocab), tokens * part));
    *end = static_cast<int>(min(static_cast<int64_t>(vocab), tokens * (part + 1)));
}

template <typename F>
__device__ __forceinline__ void for_part(const float* __restrict__ row, int begin, int end, F body) {
    for (int i0 = begin + threadIdx.x; i0 < end; i0 += kPart * kUnroll) {
        float v[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) v[u] = row[min(i0 + u * kPart, end - 1)];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u)
            if (i0 + u * kPart < end) body(v[u], i0 + u * kPart);
    }
}

// The kept weights of the part's runs, a run a wave at a time, in the order of the lanes.
__device__ void add_runs(const float* __restrict__ row, int vocab, int parts, int part, float mx, float inv_temp,
                         uint32_t cut, double* run_sum) {
    const int lane = threadIdx.x & (FSIE_WAVE - 1), wave = threadIdx.x / FSIE_WAVE;
    const int lines = run_lines(vocab), per_part = kRuns / parts;
    for (int q = wave; q < per_part; q += kPart / FSIE_WAVE) {
        const int run = part * per_part + q;
        const int64_t first = static_cast<int64_t>(run) * lines * FSIE_WAVE + lane;
        double mine = 0.0;
        for (int j0 = 0; j0 < lines; j0 += kUnroll) {
            float v[kUnroll];
#pragma unroll
            for (int u = 0; u < kUnroll; ++u)
                v[u] = row[min(first + static_cast<int64_t>(min(j0 + u, lines - 1)) * FSIE_WAVE, static_cast<int64_t>(vocab - 1))];
#pragma unroll
            for (int u = 0; u < kUnroll; ++u)
                if (j0 + u < lines && first + static_cast<int64_t>(j0 + u) * FSIE_WAVE < vocab && order_key(v[u]) >= cut)
                    mine += token_weight(v[u], mx, inv_temp);
        }
        mine = wave_sum_f64(mine);
        if (lane == 0) run_sum[run] = mine;
    }
}

__global__ __launch_bounds__(kPart) void split_top_kernel(const float* __restrict__ logits, int vocab, int parts, SplitRow* ws) {
    __shared__ float sval[kPart / FSIE_WAVE], slow[kPart / FSIE_WAVE];
    __shared__ int sidx[kPart / FSIE_WAVE], snan[kPart / FSIE_WAVE];
    SplitRow* w = ws + blockIdx.y;
    const int part = blockIdx.x, lane = threadIdx.x & (FSIE_WAVE - 1), wave = threadIdx.x / FSIE_WAVE;
    // the bins and counters of the row are this launch's to clear
    uint32_t* bins = reinterpret_cast<uint32_t*>(w->hi);
    constexpr int kClear = static_cast<int>(offsetof(SplitRow, listed) / 4);
    for (int i = part * kPart + threadIdx.x; i < kClear; i += parts * kPart) bins[i] = 0;
    int begin, end;
    part_range(vocab, parts, part, &begin, &end);
    Best best{-INFINITY, 0x7fffffff};
    float low = INFINITY;
    bool nan = false;
    for_part(logits + static_cast<int64_t>(blockIdx.y) * vocab, begin, end, [&](float v, int i) {
        nan |= v != v;
        if (v > -INFINITY) low = fminf(low, v);
        if (best.index == 0x7fffffff || v > best.value) best = Best{v, i};
    });
#pragma unroll
    for (int off = FSIE_WAVE / 2; off > 0; off >>= 1) {
        best = better(best, Best{__shfl_xor(best.value, off, FSIE_WAVE), __shfl_xor(best.index, off, FSIE_WAVE)});
        low = fminf(low, __shfl_xor(low, off, FSIE_WAVE));
    }
    nan = __any(nan);
    if (lane == 0) {
        sval[wave] = best.value;
        sidx[wave] = best.index;
        slow[wave] = low;
        snan[wave] = nan;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < kPart / FSIE_WAVE; ++i) {
            best = better(best, Best{sval[i], sidx[i]});
            low = fminf(low, slow[i]);
            nan = nan || snan[i];
        }
        w->part_max[part] = best.value;
        w->part_index[part] = best.index;
        w->part_low[part] = low;
        w->part_nan[part] = nan;
    }
}

__global__ __launch_bounds__(kPart) void split_bins_kernel(const float* __restrict__ logits, int vocab, int parts,
                                                           const float* __restrict__ temperature,
                                                           const int32_t* __restrict__ top_k,
                                                           const float* __restrict__ top_p, SplitRow* ws) {
    __shared__ unsigned long long hi[kBins], lo[kBins];
    __shared__ unsigned int count[kBins];
    const int r = blockIdx.y;
    const RowParams q = row_params(r, vocab, temperature, top_k, top_p);
    if (!(q.temp > 0.f)) return;
    SplitRow* w = ws + r;
    const RowTop top = row_top(w, parts);
    const float* row = logits + static_cast<int64_t>(r) * vocab;
    const float mx = top.best.value;
    if (!q.cuts) {
        add_runs(row, vocab, parts, blockIdx.x, mx, q.inv_temp, 0, w->run_sum);
        return;
    }
    float scale;
    if (!top.binned(vocab, q.inv_temp, &scale)) return;
    for (int b = threadIdx.x; b < kBins; b += kPart) {
        hi[b] = lo[b] = 0;
        count[b] = 0;
    }
    __syncthreads();
    const int hi_bits = 63 - (32 - __clz(vocab));  // vocab < 2^(32 - clz): the sum of all weights stays below 2^63
    int begin, end;
    part_range(vocab, parts, blockIdx.x, &begin, &end);
    for_part(row, begin, end, [&](float v, int) {
        const int b = bin_of(v, mx, scale);
        atomicAdd(&count[b], 1u);
        if (q.p < 1.f) {
            const Limbs m = limbs_of(expf((v - mx) * q.inv_temp), hi_bits);
            if (m.hi) atomicAdd(&hi[b], m.hi);
            if (m.lo) atomicAdd(&lo[b], m.lo);
        }
    });
    __syncthreads();
    for (int b = threadIdx.x; b < kBins; b += kPart) {
        if (!count[b]) continue;
        atomicAdd(&w->count[b], count[b]);
        if (hi[b]) atomicAdd(&w->hi[b], hi[b]);
        if (lo[b]) atomicAdd(&w->lo[b], lo[b]);
    }
}

// The running sums of the bins' values from the maximum down, found by a workgroup of THREADS: where `target` is first
// reached, and the sum above that bin.
struct Found {
    int bin;       // -1: nowhere
    double above, total;
};
// `v`: the values of this thread's own kBins / THREADS neighbouring bins (read from memory once for all searches).
template <int THREADS>
__device__ Found find_in_bins(double target, const double (&v)[kBins / THREADS]) {
    constexpr int PER = kBins / THREADS;
    __shared__ double wave_sum[THREADS / FSIE_WAVE];
    __shared__ Found found;
    const int lane = threadIdx.x & (FSIE_WAVE - 1), wave = threadIdx.x / FSIE_WAVE;
    double run = 0.0;
#pragma unroll
    for (int i = 0; i < PER; ++i) run += v[i];
#pragma unroll
    for (int off = 1; off < FSIE_WAVE; off <<= 1) {
        const double other = __shfl_up(run, off, FSIE_WAVE);
        if (lane >= off) run += other;
    }
    __syncthreads();
    if (lane == FSIE_WAVE - 1) wave_sum[wave] = run;
    if (threadIdx.x == 0) found.bin = -1;
    __syncthreads();
    double base = 0.0, total = 0.0;
    for (int i = 0; i < THREADS / FSIE_WAVE; ++i) {
        if (i == wave) base = total;
        total += wave_sum[i];
    }
    const double left = __shfl_up(run, 1, FSIE_WAVE);  // (all lanes together: a shuffle reads active lanes only)
    double before = base + (lane ? left : 0.0);
    if (before < target && target <= base + run) {
        int bin = static_cast<int>(threadIdx.x) * PER;
#pragma unroll
        for (int i = 0; i < PER - 1; ++i)
            if (bin == static_cast<int>(threadIdx.x) * PER + i && target > before + v[i]) {
                before += v[i];
                ++bin;
            }
        found.bin = bin;
        found.above = before;
    }
    __syncthreads();
    const Found out{found.bin, found.above, total};
    __syncthreads();
    return out;
}

__global__ __launch_bounds__(kPart) void split_list_kernel(const float* __restrict__ logits, int vocab, int parts,
                                                           const float* __restrict__ temperature,
                                                           const int32_t* __restrict__ top_k,
                                                           const float* __restrict__ top_p, SplitRow* ws) {
    const int r = blockIdx.y;
    const RowParams q = row_params(r, vocab, temperature, top_k, top_p);
    if (!q.cuts) return;
    SplitRow* w = ws + r;
    const RowTop top = row_top(w, parts);
    float scale;
    if (!top.binned(vocab, q.inv_temp, &scale)) return;
    const int hi_bits = 63 - (32 - __clz(vocab));
    constexpr int PER = kBins / kPart;
    const int b0 = static_cast<int>(threadIdx.x) * PER;
    double counts[PER], weights[PER], some[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        counts[i] = static_cast<double>(w->count[b0 + i]);
        weights[i] = value_of(Limbs{w->hi[b0 + i], w->lo[b0 + i]}, hi_bits);
    }
    int k_bin = -1, from = 0, upto = -1;
    if (q.k > 0) k_bin = find_in_bins<kPart>(q.k, counts).bin;
    if (q.p < 1.f) {
        // top p of what top k keeps: all of the bins above its own and some of that one, so the last kept token lies
        // between the bins that the least and the most of it give
#pragma unroll
        for (int i = 0; i < PER; ++i) some[i] = k_bin < 0 || b0 + i <= k_bin ? weights[i] : 0.0;
        const double most = find_in_bins<kPart>(INFINITY, some).total;
        double least = most;
        if (k_bin >= 0) {
#pragma unroll
            for (int i = 0; i < PER; ++i) some[i] = b0 + i < k_bin ? weights[i] : 0.0;
            least = find_in_bins<kPart>(INFINITY, some).total;
        }
        const double p = static_cast<double>(q.p);
        if (p > 0.0) {
            upto = find_in_bins<kPart>(p * most, weights).bin;
            from = k_bin < 0 ? upto : find_in_bins<kPart>(p * least, weights).bin;
            from = max(0, from);
        }
    }
    int begin, end;
    part_range(vocab, parts, blockIdx.x, &begin, &end);
    for_part(logits + static_cast<int64_t>(r) * vocab, begin, end, [&](float v, int) {
        const int b = bin_of(v, top.best.value, scale);
        if (b == k_bin || (from <= b && b <= upto)) {
            const unsigned int at = atomicAdd(&w->n_listed, 1u);
            if (at < kKeep) w->listed[at] = v;
        }
    });
}

// The key of the first listed token, from the largest down, at which reached(key's tokens and all larger) holds, by
// bisection over the keys; what is summed are integers, so the list's order does not matter.
template <typename S, typename F>
__device__ uint32_t bisect_list(const uint32_t* keys, int n, uint32_t key_max, S value, F reached) {
    __shared__ unsigned long long sum_hi, sum_lo;
    uint32_t lo = 0, hi = key_max;
    while (lo < hi) {
        const uint32_t mid = lo + (hi - lo) / 2 + ((hi - lo) & 1);
        __syncthreads();
        if (threadIdx.x == 0) sum_hi = sum_lo = 0;
        __syncthreads();
        Limbs mine{0, 0};
        for (int i = threadIdx.x; i < n; i += kThreads)
            if (keys[i] >= mid) {
                const Limbs v = value(i);
                mine.hi += v.hi;
                mine.lo += v.lo;
            }
        if (mine.hi) atomicAdd(&sum_hi, mine.hi);
        if (mine.lo) atomicAdd(&sum_lo, mine.lo);
        __syncthreads();
        if (reached(Limbs{sum_hi, sum_lo})) lo = mid; else hi = mid - 1;
    }
    return lo;
}

__global__ __launch_bounds__(kThreads) void split_cut_kernel(const float* __restrict__ logits, int vocab, int parts,
                                                             const float* __restrict__ temperature,
                                                             const int32_t* __restrict__ top_k,
                                                             const float* __restrict__ top_p, SplitRow* ws) {
    __shared__ uint32_t keys[kKeep];
    __shared__ short bin_of_key[kKeep];
    __shared__ unsigned long long w_hi[kPairs], w_lo[kPairs];
    __shared__ double sdbl[kWaves];
    __shared__ unsigned long long kept_hi, kept_lo;
    __shared__ uint32_t cut_found;
    __shared__ unsigned int of_bin;
    const int r = blockIdx.x;
    const RowParams q = row_params(r, vocab, temperature, top_k, top_p);
    if (!q.cuts) return;
    SplitRow* w = ws + r;
    const RowTop top = row_top(w, parts);
    const float* row = logits + static_cast<int64_t>(r) * vocab;
    const float mx = top.best.value;
    const uint32_t key_max = order_key(mx);
    const int n = static_cast<int>(min(w->n_listed, static_cast<unsigned int>(kKeep + 1)));
    float scale = 0.f;
    bool fits = top.binned(vocab, q.inv_temp, &scale) && n <= kKeep;  // (the same in every thread)
    uint32_t cut = 0;
    if (fits) {
        const int hi_bits = 63 - (32 - __clz(vocab));
        for (int i = threadIdx.x; i < n; i += kThreads) {
            const float v = w->listed[i];
            keys[i] = order_key(v);
            bin_of_key[i] = static_cast<short>(bin_of(v, mx, scale));
            if (i < kPairs) {
                const Limbs m = limbs_of(expf((v - mx) * q.inv_temp), hi_bits);
                w_hi[i] = m.hi;
                w_lo[i] = m.lo;
            }
        }
        const auto listed_weight = [&](int i) {
            if (i < kPairs) return Limbs{w_hi[i], w_lo[i]};
            return limbs_of(expf((w->listed[i] - mx) * q.inv_temp), hi_bits);
        };
        if (threadIdx.x == 0) {
            kept_hi = kept_lo = 0;
            cut_found = 0;
            of_bin = 0;
        }
        __syncthreads();
        int k_bin = -1;
        constexpr int PER = kBins / kThreads;
        const int b0 = static_cast<int>(threadIdx.x) * PER;
        double values[PER];
        if (q.k > 0) {
#pragma unroll
            for (int i = 0; i < PER; ++i) values[i] = static_cast<double>(w->count[b0 + i]);
            const Found at = find_in_bins<kThreads>(q.k, values);
            k_bin = at.bin;
            const long long want = q.k - static_cast<long long>(at.above);
            if (k_bin < 0) {
                fits = false;
            } else if (n <= kPairs) {
                if (static_cast<int>(threadIdx.x) < n && bin_of_key[threadIdx.x] == k_bin) {
                    const uint32_t mine = keys[threadIdx.x];
                    int over = 0, upto = 0;
                    for (int j = 0; j < n; ++j) {
                        const bool same = bin_of_key[j] == k_bin;
                        over += same && keys[j] > mine;
                        upto += same && keys[j] >= mine;
                    }
                    if (over < want && want <= upto) cut_found = mine;  // (equal keys write the same)
                }
                __syncthreads();
                cut = cut_found;
            } else {
                cut = bisect_list(keys, n, key_max, [&](int i) { return Limbs{bin_of_key[i] == k_bin, 0}; },
                                  [&](Limbs s) { return static_cast<long long>(s.hi) >= want; });
            }
            if (cut == 0) fits = false;
        }
        if (fits && q.p < 1.f) {
            __syncthreads();
            Limbs kept{0, 0};  // of top k's bin
            for (int i = threadIdx.x; i < n; i += kThreads)
                if (bin_of_key[i] == k_bin && keys[i] >= cut) {
                    const Limbs m = listed_weight(i);
                    kept.hi += m.hi;
                    kept.lo += m.lo;
                }
            if (kept.hi) atomicAdd(&kept_hi, kept.hi);
            if (kept.lo) atomicAdd(&kept_lo, kept.lo);
            if (threadIdx.x == 0) cut_found = 0;
            __syncthreads();
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                const int b = b0 + i;
                values[i] = value_of(Limbs{w->hi[b], w->lo[b]}, hi_bits);
                if (k_bin >= 0 && b >= k_bin) values[i] = b == k_bin ? value_of(Limbs{kept_hi, kept_lo}, hi_bits) : 0.0;
            }
            const double target = static_cast<double>(q.p) * find_in_bins<kThreads>(INFINITY, values).total;
            if (!(target > 0.0)) {
                cut = key_max;
            } else {
                const Found at = find_in_bins<kThreads>(target, values);
                const auto counts = [&](int i) { return bin_of_key[i] == at.bin && keys[i] >= cut; };
                const auto reaches = [&](Limbs s) { return target <= at.above + value_of(s, hi_bits); };
                // (rounding may have put the target outside the bins that were listed)
                unsigned int mine_of_bin = 0;
                for (int i = threadIdx.x; i < n; i += kThreads) mine_of_bin += bin_of_key[i] == at.bin;
                if (mine_of_bin) atomicAdd(&of_bin, mine_of_bin);
                __syncthreads();
                uint32_t found = 0;
                if (at.bin < 0 || of_bin != w->count[max(at.bin, 0)]) {
                    fits = false;
                } else if (n <= kPairs) {
                    if (static_cast<int>(threadIdx.x) < n && counts(threadIdx.x)) {
                        const uint32_t mine = keys[threadIdx.x];
                        Limbs over{0, 0}, upto{0, 0};
                        for (int j = 0; j < n; ++j) {
                            if (!counts(j) || keys[j] < mine) continue;
                            upto.hi += w_hi[j];
                            upto.lo += w_lo[j];
                            if (keys[j] > mine) {
                                over.hi += w_hi[j];
                                over.lo += w_lo[j];
                            }
                        }
                        if (!reaches(over) && reaches(upto)) cut_found = mine;
                    }
                    __syncthreads();
                    found = cut_found;
                } else {
                    found = bisect_list(keys, n, key_max, [&](int i) { return counts(i) ? listed_weight(i) : Limbs{0, 0}; }, reaches);
                }
                if (found == 0) fits = false;
                cut = found;
            }
        }
    }
    if (!fits) {
        __syncthreads();
        cut = cut_by_bisection(row, vocab, mx, q.inv_temp, q.k, q.p, sdbl);
    }
    if (threadIdx.x == 0) w->cut = cut;
}

__global__ __launch_bounds__(kPart) void split_runs_kernel(const float* __restrict__ logits, int vocab, int parts,
                                                           const float* __restrict__ temperature,
                                                           const int32_t* __restrict__ top_k,
                                                           const float* __restrict__ top_p, SplitRow* ws) {
    const int r = blockIdx.y;
    const RowParams q = row_params(r, vocab, temperature, top_k, top_p);
    if (!q.cuts) return;  // (rows without a threshold have their sums already)
    SplitRow* w = ws + r;
    add_runs(logits + static_cast<int64_t>(r) * vocab, vocab, parts, blockIdx.x, row_top(w, parts).best.value, q.inv_temp,
             w->cut, w->run_sum);
}

__global__ __launch_bounds__(FSIE_WAVE) void split_draw_kernel(const float* __restrict__ logits, int vocab, int parts,
                                                               const float* __restrict__ temperature,
                                                               const int32_t* __restrict__ top_k,
                                                               const float* __restrict__ top_p,
                                                               const double* __restrict__ uniform, const SplitRow* ws,
                                                               int32_t* __restrict__ out) {
    const int r = blockIdx.x;
    const RowParams q = row_params(r, vocab, temperature, top_k, top_p);
    const SplitRow* w = ws + r;
    const Best top = row_top(w, parts).best;
    if (!(q.temp > 0.f)) {
        if (threadIdx.x == 0) out[r] = top.index;
        return;
    }
    draw_from_runs(logits + static_cast<int64_t>(r) * vocab, vocab, top, q.inv_temp, q.cuts ? w->cut : 0, uniform[r],
                   w->run_sum, -1, out + r);
}

}  // namespace

extern "C" int64_t fsie_sample_workspace(int n_rows, int vocab) {
    return vocab >= kSplitFrom && n_rows > 0 && vocab / n_rows >= kTokensForRow ? static_cast<int64_t>(n_rows) * static_cast<int64_t>(sizeof(SplitRow)) : 0;
}

extern "C" int fsie_sample(const float* logits, int n_rows, int vocab, const float* temperature,
                           const int32_t* top_k, const float* top_p, const double* uniform, int32_t* out,
                           hipStream_t stream) {
    FSIE_REQUIRE(n_rows >= 0 && vocab > 0, "sample: bad sizes rows=%d vocab=%d", n_rows, vocab);
    FSIE_REQUIRE(!temperature || uniform, "sample: temperatures given without uniform numbers");
    if (n_rows == 0) return 0;
    if (temperature && (top_k || top_p))
        sample_kernel<true><<<n_rows, kThreads, 0, stream>>>(logits, vocab, temperature, top_k, top_p, uniform, out);
    else if (temperature) sample_kernel<false><<<n_rows, kThreads, 0, stream>>>(logits, vocab, temperature, nullptr, nullptr, uniform, out);
    else sample_greedy_kernel<<<n_rows, kThreads, 0, stream>>>(logits, vocab, out);
    FSIE_CHECK_LAUNCH("sample");
    return 0;
}

extern "C" int fsie_sample_split(const float* logits, int n_rows, int vocab, const float* temperature, const int32_t* top_k,
                                 const float* top_p, const double* uniform, void* workspace, int32_t* out,
                                 hipStream_t stream) {
    FSIE_REQUIRE(n_rows > 0 && n_rows <= 65535 && vocab > 0, "sample_split: bad sizes rows=%d vocab=%d", n_rows, vocab);
    FSIE_REQUIRE(temperature && uniform, "sample_split: temperatures and uniform numbers are needed");
    FSIE_REQUIRE(workspace && reinterpret_cast<uintptr_t>(workspace) % 16 == 0,
                 "sample_split: a workspace on 16 bytes is needed");
    SplitRow* ws = static_cast<SplitRow*>(workspace);
    // a power of two of parts that gives every compute unit about four workgroups
    int parts = 1;
    while (parts < kMaxParts && n_rows * parts < 1024) parts *= 2;
    const dim3 grid(parts, n_rows);
    split_top_kernel<<<grid, kPart, 0, stream>>>(logits, vocab, parts, ws);
    split_bins_kernel<<<grid, kPart, 0, stream>>>(logits, vocab, parts, temperature, top_k, top_p, ws);
    if (top_k || top_p) {
        split_list_kernel<<<grid, kPart, 0, stream>>>(logits, vocab, parts, temperature, top_k, top_p, ws);
        split_cut_kernel<<<n_rows, kThreads, 0, stream>>>(logits, vocab, parts, temperature, top_k, top_p, ws);
        split_runs_kernel<<<grid, kPart, 0, stream>>>(logits, vocab, parts, temperature, top_k, top_p, ws);
    }
    split_draw_kernel<<<n_rows, FSIE_WAVE, 0, stream>>>(logits, vocab, parts, temperature, top_k, top_p, uniform, ws, out);
    FSIE_CHECK_LAUNCH("sample_split");
    return 0;
}
