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
// add them changes nothing.  Rows that do not fit this (a maximum that is not finite, a NaN, more than 2,048 tokens in
// the threshold's bin) are bisected over the order-preserving integer image of the logits, a pass a probe.
// What bounds it is how often a compute unit reads a row of 600 KB from the caches: 2 passes for greedy and
// plain temperature, 4 with a threshold, where the bisection alone took 32 a threshold (64 rows of 152,064, a fifth
// of them each greedy, at a temperature, top k, top p and both: 183 us, 1,504 with the bisection alone).
#include "common.h"
#include "api.h"

#include <math.h>

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
__device__ Best block_argmax(const float* row, int vocab, float* sval, int* sidx, float* low, bool* nan) {
    Best best{-INFINITY, 0x7fffffff};
    *low = INFINITY;
    *nan = false;
    auto take = [&](float v, int i) {
        *nan |= v != v;
        if (v > -INFINITY) *low = fminf(*low, v);
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
    if (odd || !(range > 1e-30f)) return false;
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

__global__ __launch_bounds__(kThreads) void sample_kernel(const float* __restrict__ logits, int vocab,
                                                          const float* __restrict__ temperature,
                                                          const int32_t* __restrict__ top_k,
                                                          const float* __restrict__ top_p,
                                                          const double* __restrict__ uniform,
                                                          int32_t* __restrict__ out) {
    __shared__ float sval[kWaves];
    __shared__ int sidx[kWaves];
    __shared__ double sdbl[kWaves];
    __shared__ double run_sum[kRuns];
    __shared__ Binned binned;

    const int r = blockIdx.x;
    const float* row = logits + static_cast<int64_t>(r) * vocab;
    float low;
    bool nan;
    const Best top = block_argmax(row, vocab, sval, sidx, &low, &nan);
    const float temp = temperature ? temperature[r] : 0.f;
    if (!(temp > 0.f)) {
        if (threadIdx.x == 0) out[r] = top.index;
        return;
    }
    const float mx = top.value;
    const float inv_temp = 1.0f / temp;
    uint32_t cut = 0;  // tokens with key >= cut are kept
    const int k = top_k && top_k[r] > 0 && top_k[r] < vocab ? top_k[r] : 0;
    const float p = top_p ? top_p[r] : 1.f;
    if (k > 0 || p < 1.f) {
        if (vocab > kMaxBinned || !(fabsf(mx) < INFINITY) || !cut_by_bins(binned, row, vocab, mx, low, nan, inv_temp, k, p, &cut)) {
            __syncthreads();
            cut = cut_by_bisection(row, vocab, mx, inv_temp, k, p, sdbl);
        }
    }

    // inverse CDF in vocabulary order.  The vocabulary is cut into kRuns runs of whole 64 tokens; a wave adds up the
    // kept weights of kRuns / kWaves neighbouring ones, then the wave whose run holds the threshold walks it.
    const int lane = threadIdx.x & (FSIE_WAVE - 1), wave = threadIdx.x / FSIE_WAVE;
    const int rows = ((vocab + FSIE_WAVE - 1) / FSIE_WAVE + kRuns - 1) / kRuns;  // 64 tokens each
    constexpr int kRunsOfWave = kRuns / kWaves;
    const auto kept_weight = [&](float v, int i) { return i < vocab && order_key(v) >= cut ? token_weight(v, mx, inv_temp) : 0.0; };
    for (int q = 0; q < kRunsOfWave; ++q) {
        const int run = wave * kRunsOfWave + q;
        double mine = 0.0;
        for (int j0 = 0; j0 < rows; j0 += kUnroll) {
            float v[kUnroll];
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) {
                const int64_t i = (static_cast<int64_t>(run) * rows + min(j0 + u, rows - 1)) * FSIE_WAVE + lane;
                v[u] = row[i < vocab ? i : vocab - 1];
            }
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) {
                const int64_t i = (static_cast<int64_t>(run) * rows + j0 + u) * FSIE_WAVE + lane;
                if (j0 + u < rows && i < vocab) mine += kept_weight(v[u], static_cast<int>(i));
            }
        }
        mine = wave_sum_f64(mine);
        if (lane == 0) run_sum[run] = mine;
    }
    __syncthreads();
    // every wave finds the run by itself: four neighbouring runs a lane
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
    const double threshold = uniform[r] * total;
    double before = __shfl_up(upto, 1, FSIE_WAVE);
    if (lane == 0) before = 0.0;
    // the first lane whose running sum passes the threshold, then the first of its runs
    const unsigned long long past = __ballot(threshold < upto);
    if (past == 0) {  // a NaN or no weight at all
        if (threadIdx.x == 0) out[r] = top.index;
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
    if (wave != run / kRunsOfWave) return;
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
            if (lane == __ffsll(hit) - 1) out[r] = static_cast<int>(i);
            return;
        }
        if (any) last_kept = static_cast<int>((static_cast<int64_t>(run) * rows + j) * FSIE_WAVE) + 63 - __clzll(any);
        cum += __shfl(w, FSIE_WAVE - 1, FSIE_WAVE);
    }
    if (lane == 0) out[r] = last_kept >= 0 ? last_kept : top.index;  // rounding at the run's end
}

}  // namespace

extern "C" int fsie_sample(const float* logits, int n_rows, int vocab, const float* temperature,
                           const int32_t* top_k, const float* top_p, const double* uniform, int32_t* out,
                           hipStream_t stream) {
    FSIE_REQUIRE(n_rows >= 0 && vocab > 0, "sample: bad sizes rows=%d vocab=%d", n_rows, vocab);
    FSIE_REQUIRE(!temperature || uniform, "sample: temperatures given without uniform numbers");
    if (n_rows == 0) return 0;
    sample_kernel<<<n_rows, kThreads, 0, stream>>>(logits, vocab, temperature, top_k, top_p, uniform, out);
    FSIE_CHECK_LAUNCH("sample");
    return 0;
}
