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
// 152,064, a fifth of them each greedy, at a temperature, top k, top p and both: 141 us, 1,504 with the bisection alone).
// Long rows are shared by several workgroups (below): 45 us for the same call.
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

// A 64-bit value moved between the lanes by the vector unit's data path (a general shuffle is a trip through LDS): lanes that get none
// have 0.  CTRL: n lanes up within sixteen (0x110 + n), the last of sixteen to the next sixteen (0x142) or to the upper half (0x143).
template <int CTRL, int ROWS, typename T>
__device__ __forceinline__ T lanes_up(T v) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned int lo = __builtin_amdgcn_update_dpp(0u, static_cast<unsigned int>(u), CTRL, ROWS, 0xf, false);
    const unsigned int hi = __builtin_amdgcn_update_dpp(0u, static_cast<unsigned int>(u >> 32), CTRL, ROWS, 0xf, false);
    return __builtin_bit_cast(T, (static_cast<unsigned long long>(hi) << 32) | lo);
}
// The sum over this lane and those below it, all 64 active; T: double or unsigned long long.
template <typename T>
__device__ __forceinline__ T wave_upto(T v) {
    v += lanes_up<0x111, 0xf>(v);
    v += lanes_up<0x112, 0xf>(v);
    v += lanes_up<0x114, 0xf>(v);
    v += lanes_up<0x118, 0xf>(v);
    v += lanes_up<0x142, 0xa>(v);
    return v + lanes_up<0x143, 0xc>(v);
}
// The value of one lane (the same in all), in all of them.
template <typename T>
__device__ __forceinline__ T of_lane(T v, int lane) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned int lo = __builtin_amdgcn_readlane(static_cast<unsigned int>(u), lane);
    const unsigned int hi = __builtin_amdgcn_readlane(static_cast<unsigned int>(u >> 32), lane);
    return __builtin_bit_cast(T, (static_cast<unsigned long long>(hi) << 32) | lo);
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
// sums of the runs (in LDS): every wave finds the run, whose 64-token lines the waves then walk side by side, one each.  (One
// wave after all of them is a chain of a trip to memory and six exchanges between lanes a line: 64 rows of 152,064
// tokens 8.2 us in a kernel of their own; and 2 so.  Up to kLinesOfOne lines are one wave's, with all their loads under way at once.)
constexpr int kLinesOfOne = 4;
__device__ void draw_from_runs(const float* __restrict__ row, int vocab, Best top, float inv_temp, uint32_t cut, double uniform,
                               const double* run_sum, int32_t* out) {
    __shared__ double line_sum[kWaves];
    __shared__ int line_hit[kWaves], line_last[kWaves];
    const int lane = threadIdx.x & (FSIE_WAVE - 1), wave = threadIdx.x / FSIE_WAVE;
    const int lines = ((vocab + FSIE_WAVE - 1) / FSIE_WAVE + kRuns - 1) / kRuns;
    const float mx = top.value;
    // four neighbouring runs a lane
    double part[kRuns / FSIE_WAVE], upto = 0.0;
#pragma unroll
    for (int q = 0; q < kRuns / FSIE_WAVE; ++q) {
        part[q] = run_sum[lane * (kRuns / FSIE_WAVE) + q];
        upto += part[q];
    }
    upto = wave_upto(upto);
    const double total = of_lane(upto, FSIE_WAVE - 1);
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
    run = __builtin_amdgcn_readlane(run, owner);
    cum = of_lane(cum, owner);
    int last_kept = -1;
    if (lines <= kLinesOfOne) {
        if (wave > 0) return;
        const int64_t first = static_cast<int64_t>(run) * lines * FSIE_WAVE;
        float v[kLinesOfOne];
#pragma unroll
        for (int q = 0; q < kLinesOfOne; ++q) v[q] = row[min(first + min(q, lines - 1) * FSIE_WAVE + lane, static_cast<int64_t>(vocab - 1))];
#pragma unroll
        for (int q = 0; q < kLinesOfOne; ++q) {
            if (q >= lines) break;
            const int64_t line = first + q * FSIE_WAVE;
            const bool kept = line + lane < vocab && order_key(v[q]) >= cut;
            const double w = wave_upto(kept ? token_weight(v[q], mx, inv_temp) : 0.0);
            const unsigned long long hit = __ballot(kept && threshold < cum + w), any = __ballot(kept);
            if (hit) {
                if (lane == 0) *out = static_cast<int>(line) + __ffsll(hit) - 1;
                return;
            }
            if (any) last_kept = static_cast<int>(line) + 63 - __clzll(any);
            cum += of_lane(w, FSIE_WAVE - 1);
        }
        if (lane == 0) *out = last_kept >= 0 ? last_kept : top.index;
        return;
    }
    for (int j0 = 0; j0 < lines; j0 += kWaves) {
        const int64_t i = (static_cast<int64_t>(run) * lines + j0 + wave) * FSIE_WAVE + lane;
        const float v = row[i < vocab ? i : vocab - 1];
        const bool kept = j0 + wave < lines && i < vocab && order_key(v) >= cut;
        const double w = wave_upto(kept ? token_weight(v, mx, inv_temp) : 0.0);
        if (j0 > 0) __syncthreads();
        if (lane == FSIE_WAVE - 1) line_sum[wave] = w;
        __syncthreads();
        double base = cum;
        for (int q = 0; q < kWaves; ++q) {
            if (q == wave) base = cum;
            cum += line_sum[q];
        }
        const unsigned long long hit = __ballot(kept && threshold < base + w), any = __ballot(kept);
        const int64_t first = i - lane;
        if (lane == 0) {
            line_hit[wave] = hit ? static_cast<int>(first) + __ffsll(hit) - 1 : -1;
            line_last[wave] = any ? static_cast<int>(first) + 63 - __clzll(any) : -1;
        }
        __syncthreads();
        for (int q = 0; q < kWaves; ++q) {
            if (line_hit[q] >= 0) {
                if (threadIdx.x == 0) *out = line_hit[q];
                return;
            }
            last_kept = max(last_kept, line_last[q]);
        }
    }
    if (threadIdx.x == 0) *out = last_kept >= 0 ? last_kept : top.index;  // rounding at the run's end
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
    draw_from_runs(row, vocab, top, inv_temp, cut, uniform[r], run_sum, out + r);
}

// ---- a row shared by several workgroups -------------------------------------------------------
// One workgroup a row leaves three quarters of the chip idle at 64 rows and all but one unit at one row, and a unit
// needs some 10 us for every pass over 152,064 tokens (their exponentials and the adds in float64).  From kSplitFrom
// tokens on the row's runs are dealt to up to 32 workgroups, and the passes become launches: the maximum; the row's bins (or,
// for rows without a threshold, the draw's sums); the tokens about the thresholds, side by side, and the draw's sums of
// those that are kept for certain; the cut among the listed tokens and the draw.  What a launch leaves for the next lies in
// a workspace of the row.
// Alone / shared, us, a fifth of the rows each greedy, plain, top k, top p and both, at 8, 64, 128, 256, 512, 2,048 and 4,096 rows:
//    16,384 tokens   37 / 23    37 / 27    38 / 29     39 /  34     71 /  51    215 / 134    405 /   243
//    32,000          46 / 23    48 / 28    48 / 33     51 /  45     96 /  71    269 / 188    516 /   419
//    65,536          71 / 24    71 / 33    74 / 43     77 /  63    147 / 107    432 / 368    794 /   692
//   152,064         138 / 25   150 / 46   152 / 70    158 / 116    303 / 211    870 / 759  1,640 / 1,424
// so where both thresholds are given rows are shared up to kMostRows of them (what was measured; their workspaces are 59 KB a row).  Where all rows ask
// for one kind, a workgroup a row is the faster one below that, up to one round of them: all rows at top k / top p / a temperature alone, alone / shared, us,
//    16,384 tokens, 16 rows  25 / 24    34 / 28    17 / 14;  40  25 / 28    34 / 33    18 / 15;  100  25 / 32    34 / 38    18 / 18;  256  27 / 29    35 / 36    19 / 22
//    32,000          40      30 / 29    45 / 35    19 / 16;  80  31 / 30    45 / 37    19 / 18;  192  32 / 36    47 / 46    20 / 24;  320  60 / 52    87 / 67    37 / 38
//    65,536          80      42 / 35    72 / 46    25 / 23; 128  43 / 37    73 / 49    26 / 28;  224  50 / 56    77 / 72    32 / 40;  512 100 / 91   152 / 121   62 / 72
//   152,064          64      87 / 40   154 / 55    50 / 29; 128  88 / 59   155 / 82    53 / 46;  224  95 / 96   159 / 128   60 / 72; 1,024 412 / 416 649 / 497 260 / 306
// and the lines lie where they meet (fsie_sample_shares).  Parameters that the first launch brings spare a copy that is 20 us of the host: such rows are always shared.
// (Without temperatures it is one pass over the row, and a workgroup a row is the faster one; with temperatures that all
// say greedy too, but that only the device knows.)
constexpr int kSplitFrom = 16384;
constexpr int kMostRows = 4096, kMostPlainRows = 160;
constexpr int kLongPlain = 98304;
constexpr int kPart = 512;          // threads of a shared row's workgroups
constexpr int kMaxParts = 32;
// Bins of a shared row.  512 are a per cent faster where the thresholds lie among few tokens (64 rows of 152,064 as above 44.7 us, 45.1 with 2,048), but
// lists then overflow, and one workgroup settles the row, where a threshold lies in a bulk of tokens far below the maximum (64 rows, normal of a
// width of 0.35, 25 below it: top k of 20,000 230 us, 52 so; top p at a temperature of 4 596 and 84; both 672 and 64).
constexpr int kCoarse = 2048;
constexpr int kFine = 1024;         // what the bin of a threshold is cut into
constexpr int kPairs = 512;         // so many tokens of a fine bin are compared with each other, more are bisected
constexpr int kKeep = 4096;         // tokens that the list holds
constexpr int kAllListed = 1024;    // up to this top k the list takes every token down to the bin of the k-th
static_assert(kRuns / kMaxParts >= kPart / FSIE_WAVE, "every wave of a part has a run");

struct SplitRow {
    unsigned int n_listed, pad;       // (in front of the bins: cleared with them)
    unsigned long long sum[kCoarse];  // weights, in units of their bin's own (RowBins)
    unsigned int count[kCoarse];
    double uniform;                   // the row's parameters, as the first launch brings them
    float temperature, top_p;
    int top_k;
    int top_index, top_nan;           // from the parts'
    float top_max, top_low;
    int k_bin, from, upto;            // the bin of top k; those that hold the last token of top p
    double above_k, above, target;    // tokens above k_bin; weight above `from`; what top p's kept weight has to reach (0: no top p alone)
    double run_sum[kRuns];
    float listed[kKeep];
    int listed_at[kKeep];
    float part_max[kMaxParts], part_low[kMaxParts];
    int part_index[kMaxParts], part_nan[kMaxParts];
};
static_assert(sizeof(SplitRow) % 8 == 0, "rows of the workspace stay aligned");

struct RowParams {
    float temp, inv_temp, p;
    int k;
    bool cuts;
};
__device__ __forceinline__ RowParams row_params(const SplitRow* w, int vocab) {
    RowParams q;
    q.temp = w->temperature;
    q.inv_temp = 1.0f / q.temp;
    q.k = w->top_k > 0 && w->top_k < vocab ? w->top_k : 0;
    q.p = w->top_p;
    q.cuts = q.temp > 0.f && (q.k > 0 || q.p < 1.f);
    return q;
}

// The rows' parameters where the first launch finds them: in arrays on the device, or among its own arguments, which the host writes (a
// copy to the device in front of the launches, with its pinned buffer and the event that guards it, is 20 us of the host, which is what bounds a call of 64 rows, and 2.4 of the device: 68 us and 45 through the sampler).
struct RowArrays {
    const float* temperature;
    const int32_t* top_k;  // or null
    const float* top_p;    // or null
    const double* uniform;
    __device__ void to(SplitRow* w, int r) const {
        w->temperature = temperature[r];
        w->top_k = top_k ? top_k[r] : 0;
        w->top_p = top_p ? top_p[r] : 1.f;
        w->uniform = uniform[r];
    }
};
constexpr int kByValue = 192;
struct RowValues {
    double uniform[kByValue];
    float temperature[kByValue], top_p[kByValue];
    int32_t top_k[kByValue];
    __device__ void to(SplitRow* w, int r) const {
        w->temperature = temperature[r];
        w->top_k = top_k[r];
        w->top_p = top_p[r];
        w->uniform = uniform[r];
    }
};
static_assert(sizeof(RowValues) + 64 <= 4096, "a launch has room for 4 KB of arguments");

// The row's bins: kCoarse equal ones over what it spans, at most kRange or 30 temperatures (43 powers of two in weight).  A bin's weights are
// summed as integers of a unit of its own, one limb: 2^-(unit + below(bin)), where below(bin) powers of two lie between
// the largest weight and the bin's.  With at most unit - 25 powers of two a bin nothing of a weight is lost; in the last one,
// which takes all that lies further down, nothing above 2^-(unit + 42); two limbs of 40 bits lose no less.  Rows so cold that a bin would be more (top p
// below a temperature of some 0.001) end their bins where it is not, far below the last weight that is not zero: what lies further down is the last
// bin's, and weighs nothing, so that a top k whose token is there binds nothing.  Top k alone weighs nothing and spans as above.  (Settled by one
// workgroup instead, 64 rows of 152,064 at 0.001: top p 119 us, 44 so, top k 97 and 38, both 138 and 40.)
// (Two limbs are twice the additions in LDS and into the row's bins, and thrice the instructions.)
struct RowBins {
    float scale, binades;
    int unit;
    bool cold;  // what the bins span ends where weights are long zero
    __device__ int bin(float v, float mx) const { return static_cast<int>(fminf((mx - v) * scale, static_cast<float>(kCoarse - 1))); }
    __device__ int below(int b) const { return static_cast<int>(static_cast<float>(b) * binades); }
    __device__ unsigned long long weight(float w, int b) const {
        const uint32_t u = __float_as_uint(w);
        const int e = static_cast<int>(u >> 23);
        const unsigned long long m = e ? (u & 0x7fffffu) | 0x800000u : 0u;
        return (m << (unit - 22)) >> min(max(128 - e - below(b), 0), 63);  // m * 2^(e - 150) in units
    }
    // no token below this lies in bin `b` or above it (a little further down, for what the bins' arithmetic rounds)
    __device__ float reach(int b, float mx) const {
        if (b >= kCoarse - 1) return -INFINITY;
        const float far = static_cast<float>(b + 1) / scale * 1.00001f;
        return mx - far - fmaxf(fabsf(mx), far) * 1e-6f;
    }
    // whether the list takes every token down to the bin of the k-th
    __device__ bool all_listed(const RowParams& q) const { return 0 < q.k && q.k <= kAllListed && !cold; }
    __device__ double value(unsigned long long sum, int b) const { return ldexp(static_cast<double>(sum), -(unit + below(b))); }
};

// The row's maximum and its place, the smallest value above -inf, whether a NaN is in it: from the parts', by a wave.
struct RowTop {
    Best best;
    float low;
    bool nan;
    // whether the row's thresholds can be found by bins
    __device__ bool binned(int vocab, const RowParams& q, RowBins* bins) const {
        bins->unit = 62 - (32 - __clz(vocab));  // 2^(32 - clz) weights of less than two of a bin's stay below 2^63
        float range = fminf(best.value - low, fmaxf(kRange, 30.f * q.temp));
        const float most = 0.999f * static_cast<float>(bins->unit - 25) * static_cast<float>(kCoarse - 1) / (q.inv_temp * 1.44269504f);
        bins->cold = q.p < 1.f && range > most;
        if (bins->cold) range = most;
        if (vocab > kMaxBinned || nan || !(fabsf(best.value) < INFINITY) || !(range > 1e-30f) || !weighs(q.inv_temp)) return false;
        bins->scale = static_cast<float>(kCoarse - 1) / range;
        bins->binades = q.inv_temp * 1.44269504f / bins->scale;
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
// The same as an earlier launch has left it.
__device__ __forceinline__ RowTop kept_top(const SplitRow* w) {
    return RowTop{Best{w->top_max, w->top_index}, w->top_low, w->top_nan != 0};
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

constexpr int kAhead = 10;  // loads of a thread in a batch; the next batch is under way while one is worked on

template <typename F>
__device__ __forceinline__ void for_part(const float* __restrict__ row, int begin, int end, F body) {
    const auto bring = [&](float (&v)[kAhead], int i0) {
#pragma unroll
        for (int u = 0; u < kAhead; ++u) v[u] = row[min(i0 + static_cast<int>(threadIdx.x) + u * kPart, end - 1)];
    };
    if (begin >= end) return;
    float v[kAhead], next[kAhead];
    bring(v, begin);
    for (int i0 = begin; i0 < end; i0 += kPart * kAhead) {
        if (i0 + kPart * kAhead < end) bring(next, i0 + kPart * kAhead);
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int i = i0 + static_cast<int>(threadIdx.x) + u * kPart;
            if (i < end) body(v[u], i);
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u) v[u] = next[u];
    }
}

// The sums of body(value, index) over the runs of part `part`, by THREADS threads: every wave takes neighbouring runs, whose
// lines it goes through as one row of them.  A run's sum does not depend on who adds it up.
template <int THREADS, typename F>
__device__ __forceinline__ void add_runs(const float* __restrict__ row, int vocab, int parts, int part, double* run_sum, F body) {
    const int lane = threadIdx.x & (FSIE_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / FSIE_WAVE);
    const int lines = run_lines(vocab), runs = kRuns / parts / (THREADS / FSIE_WAVE), all = runs * lines;
    int run = part * (kRuns / parts) + wave * runs, in_run = 0;
    const int64_t first = static_cast<int64_t>(run) * lines * FSIE_WAVE + lane;
    const auto bring = [&](float (&v)[kAhead], int j0) {
#pragma unroll
        for (int u = 0; u < kAhead; ++u) v[u] = row[min(first + static_cast<int64_t>(j0 + u) * FSIE_WAVE, static_cast<int64_t>(vocab - 1))];
    };
    float v[kAhead], next[kAhead];
    bring(v, 0);
    double mine = 0.0;
    for (int j0 = 0; j0 < all; j0 += kAhead) {
        if (j0 + kAhead < all) bring(next, j0 + kAhead);
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            if (j0 + u >= all) break;
            const int64_t i = first + static_cast<int64_t>(j0 + u) * FSIE_WAVE;
            if (i < vocab) mine += body(v[u], static_cast<int>(i));
            if (++in_run == lines) {
                mine = wave_upto(mine);
                if (lane == FSIE_WAVE - 1) run_sum[run] = mine;
                mine = 0.0;
                in_run = 0;
                ++run;
            }
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u) v[u] = next[u];
    }
}

template <typename ROWS>
__global__ __launch_bounds__(kPart) void split_top_kernel(const float* __restrict__ logits, int vocab, int parts, SplitRow* ws, ROWS rows) {
    __shared__ float sval[kPart / FSIE_WAVE], slow[kPart / FSIE_WAVE];
    __shared__ int sidx[kPart / FSIE_WAVE], snan[kPart / FSIE_WAVE];
    SplitRow* w = ws + blockIdx.y;
    const int part = blockIdx.x, lane = threadIdx.x & (FSIE_WAVE - 1), wave = threadIdx.x / FSIE_WAVE;
    if (part == 0 && threadIdx.x == 0) rows.to(w, static_cast<int>(blockIdx.y));
    // the row's bins and counter are this launch's to clear
    uint32_t* bins = reinterpret_cast<uint32_t*>(w);
    constexpr int kClear = static_cast<int>(offsetof(SplitRow, uniform) / 4);
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

// Rows without a threshold: the draw's sums.  The others: their bins, counted for top k, weighed for top p (not where the list will
// hold all that top k keeps).  What bounds it are the weighed rows' instructions, some fifty a token.
__global__ __launch_bounds__(kPart) void split_weigh_kernel(const float* __restrict__ logits, int vocab, int parts, SplitRow* ws) {
    __shared__ unsigned long long sum[kCoarse];
    __shared__ unsigned int count[kCoarse];
    const int r = blockIdx.y;
    SplitRow* w = ws + r;
    const RowParams q = row_params(w, vocab);
    const RowTop top = row_top(w, parts);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        w->top_max = top.best.value;
        w->top_index = top.best.index;
        w->top_low = top.low;
        w->top_nan = top.nan;
    }
    if (!(q.temp > 0.f)) return;
    const float* row = logits + static_cast<int64_t>(r) * vocab;
    const float mx = top.best.value;
    if (!q.cuts) {
        add_runs<kPart>(row, vocab, parts, blockIdx.x, w->run_sum, [&](float v, int) { return token_weight(v, mx, q.inv_temp); });
        return;
    }
    RowBins bins;
    if (!top.binned(vocab, q, &bins)) return;
    const bool weigh = q.p < 1.f && !bins.all_listed(q), counts = q.k > 0;
    for (int b = threadIdx.x; b < kCoarse; b += kPart) {
        sum[b] = 0;
        count[b] = 0;
    }
    __syncthreads();
    int begin, end;
    part_range(vocab, parts, blockIdx.x, &begin, &end);
    if (weigh) {
        for_part(row, begin, end, [&](float v, int) {
            const int b = bins.bin(v, mx);
            if (counts) atomicAdd(&count[b], 1u);
            const unsigned long long m = bins.weight(expf((v - mx) * q.inv_temp), b);
            if (m) atomicAdd(&sum[b], m);
        });
    } else {
        for_part(row, begin, end, [&](float v, int) { atomicAdd(&count[bins.bin(v, mx)], 1u); });
    }
    __syncthreads();
    for (int b = threadIdx.x; b < kCoarse; b += kPart) {
        if (counts && count[b]) atomicAdd(&w->count[b], count[b]);
        if (weigh && sum[b]) atomicAdd(&w->sum[b], sum[b]);
    }
}

// The running sums of the bins' values from the maximum down, over a workgroup of THREADS, and the bin in which one first
// reaches a target.  Fixed order of additions.
struct Found {
    int bin;  // -1: nowhere
    double above;
};
template <int THREADS>
struct BinScan {
    static constexpr int PER = kCoarse > THREADS ? kCoarse / THREADS : 1;  // (threads beyond the bins have none: 0)
    double v[PER];  // the values of this thread's neighbouring bins
    double before, upto, total;

    // `wave_sum`: a number a wave, in LDS, of this scan alone
    __device__ void run(double* wave_sum) {
        const int lane = threadIdx.x & (FSIE_WAVE - 1), wave = threadIdx.x / FSIE_WAVE;
        double sum = 0.0;
#pragma unroll
        for (int i = 0; i < PER; ++i) sum += v[i];
        sum = wave_upto(sum);
        if (lane == FSIE_WAVE - 1) wave_sum[wave] = sum;
        const double left = __shfl_up(sum, 1, FSIE_WAVE);  // (all lanes together: a shuffle reads active lanes only)
        __syncthreads();
        double base = 0.0;
        total = 0.0;
#pragma unroll
        for (int i = 0; i < THREADS / FSIE_WAVE; ++i) {
            if (i == wave) base = total;
            total += wave_sum[i];
        }
        before = base + (lane ? left : 0.0);
        upto = base + sum;
    }
    // `found`: in LDS, of this search alone, its bin set to -1 before the last barrier
    __device__ Found find(double target, Found* found) const {
        if (before < target && target <= upto) {
            int bin = static_cast<int>(threadIdx.x) * PER;
            double above = before;
#pragma unroll
            for (int i = 0; i < PER - 1; ++i)
                if (bin == static_cast<int>(threadIdx.x) * PER + i && target > above + v[i]) {
                    above += v[i];
                    ++bin;
                }
            *found = Found{bin, above};
        }
        __syncthreads();
        return *found;
    }
    // the sum of the bins above `bin`, and with it
    __device__ void around(int bin, double* above, double* with) const {
        __shared__ double shared[2];
        if (static_cast<int>(threadIdx.x) == bin / PER) {
            double sum = before;
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                if (bin % PER == i) {
                    shared[0] = sum;
                    shared[1] = sum + v[i];
                }
                sum += v[i];
            }
        }
        __syncthreads();
        *above = shared[0];
        *with = shared[1];
    }
};

// Every workgroup of the row finds the bins of its thresholds, lists the part's tokens of them and adds up the draw's sums
// of those above, which are kept whatever the cut among the listed ones will be.  Most tokens lie below all that: a wave lays those
// that do not side by side in LDS, so that bins and exponentials are computed of these alone (of all tokens of a line where one of them is kept:
// 9 us of a top-p row's pass over 19,008 tokens, and 3 so).
constexpr int kNear = kAhead * FSIE_WAVE + 3 * FSIE_WAVE;
static_assert(kMaxBinned <= 1 << 23 && kRuns <= 1 << 8, "a token's place and its run within the part fit 32 bits");
__global__ __launch_bounds__(kPart) void split_list_kernel(const float* __restrict__ logits, int vocab, int parts, SplitRow* ws) {
    __shared__ float near[kPart / FSIE_WAVE][kNear];
    __shared__ unsigned int near_at[kPart / FSIE_WAVE][kNear];
    __shared__ unsigned long long run_hi[kRuns], run_lo[kRuns];
    __shared__ double wave_sum[2][kPart / FSIE_WAVE];
    __shared__ Found found[3];
    const int r = blockIdx.y;
    SplitRow* w = ws + r;
    const RowParams q = row_params(w, vocab);
    if (!q.cuts) return;
    const RowTop top = kept_top(w);
    RowBins bins;
    if (!top.binned(vocab, q, &bins)) return;
    const float mx = top.best.value;
    constexpr int PER = kCoarse / kPart;
    const int b0 = static_cast<int>(threadIdx.x) * PER;
    int k_bin = -1, from = 0, upto = -1;
    double above_k = 0.0, above = 0.0, target = 0.0;
    BinScan<kPart> scan;
    for (int i = threadIdx.x; i < kRuns / parts; i += kPart) run_hi[i] = run_lo[i] = 0;
    if (threadIdx.x == 0) {
        found[0].bin = found[1].bin = found[2].bin = -1;
    }
    if (q.k > 0) {
#pragma unroll
        for (int i = 0; i < PER; ++i) scan.v[i] = static_cast<double>(w->count[b0 + i]);
        scan.run(wave_sum[0]);
        const Found at = scan.find(q.k, &found[0]);
        k_bin = at.bin;
        above_k = at.above;
        from = upto = k_bin;
    }
    const bool binds = q.k > 0 && !(bins.cold && k_bin == kCoarse - 1);  // (else top k keeps every token that weighs anything)
    if (!binds) k_bin = -1;
    if (bins.all_listed(q)) {
        from = 0;
    } else if (q.p < 1.f) {
#pragma unroll
        for (int i = 0; i < PER; ++i) scan.v[i] = bins.value(w->sum[b0 + i], b0 + i);
        scan.run(wave_sum[1]);
        const double p = static_cast<double>(q.p);
        if (k_bin >= 0) {
            // top p of what top k keeps: all of the bins above its own and some of that one, so the last kept token lies
            // between the bins that the least and the most of it give
            double least, most;
            scan.around(k_bin, &least, &most);
            upto = scan.find(p * most, &found[1]).bin;
            from = scan.find(p * least, &found[2]).bin;
        } else if (!binds) {
            target = p * scan.total;
            const Found at = scan.find(target, &found[1]);
            from = upto = at.bin;
            above = at.above;
        }
        from = max(from, 0);  // (nothing to reach: the largest token, which lies in the first bin)
        upto = max(upto, 0);
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        w->k_bin = k_bin;
        w->from = from;
        w->upto = upto;
        w->above_k = above_k;
        w->above = above;
        w->target = target;
    }
    __syncthreads();
    const float* row = logits + static_cast<int64_t>(r) * vocab;
    const int lane = threadIdx.x & (FSIE_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / FSIE_WAVE);
    const int lines = run_lines(vocab), runs = kRuns / parts / (kPart / FSIE_WAVE), all = runs * lines;
    const int first_run = blockIdx.x * (kRuns / parts), hi_bits = 63 - (32 - __clz(vocab));
    const int first = (first_run + wave * runs) * lines * FSIE_WAVE + lane;
    const float reach = bins.reach(max(k_bin, upto), mx);
    int run = wave * runs, in_run = 0, n = 0;
    // (a wave's tokens change lanes here: what the others wrote is read below, and is read before the next ones are written over it)
    const auto meet = [] {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    const auto settle = [&]() {
        meet();
        for (int at = lane; at < n; at += FSIE_WAVE) {
            const float v = near[wave][at];
            const unsigned int place = near_at[wave][at];
            const int b = bins.bin(v, mx);
            if (b == k_bin || (from <= b && b <= upto)) {
                const unsigned int slot = atomicAdd(&w->n_listed, 1u);
                if (slot < kKeep) {
                    w->listed[slot] = v;
                    w->listed_at[slot] = static_cast<int>(place & 0x7fffffu);
                }
            } else if (b < from) {
                const Limbs m = limbs_of(expf((v - mx) * q.inv_temp), hi_bits);
                if (m.hi) atomicAdd(&run_hi[place >> 23], m.hi);
                if (m.lo) atomicAdd(&run_lo[place >> 23], m.lo);
            }
        }
        meet();
        n = 0;
    };
    const auto bring = [&](float (&v)[kAhead], int j0) {
#pragma unroll
        for (int u = 0; u < kAhead; ++u) v[u] = row[min(first + (j0 + u) * FSIE_WAVE, vocab - 1)];
    };
    float v[kAhead], next[kAhead];
    bring(v, 0);
    for (int j0 = 0; j0 < all; j0 += kAhead) {
        if (j0 + kAhead < all) bring(next, j0 + kAhead);
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            if (j0 + u >= all) break;
            const int i = first + (j0 + u) * FSIE_WAVE;
            const bool is = v[u] >= reach && i < vocab;
            const unsigned long long mask = __ballot(is);
            if (mask) {
                const int slot = n + __builtin_amdgcn_mbcnt_hi(static_cast<unsigned int>(mask >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<unsigned int>(mask), 0));
                if (is) {
                    near[wave][slot] = v[u];
                    near_at[wave][slot] = static_cast<unsigned int>(run) << 23 | static_cast<unsigned int>(i);
                }
                n += __popcll(mask);
            }
            if (++in_run == lines) {
                in_run = 0;
                ++run;
            }
        }
        if (n > kNear - kAhead * FSIE_WAVE) settle();
#pragma unroll
        for (int u = 0; u < kAhead; ++u) v[u] = next[u];
    }
    settle();
    __syncthreads();
    for (int i = threadIdx.x; i < kRuns / parts; i += kPart) w->run_sum[first_run + i] = value_of(Limbs{run_hi[i], run_lo[i]}, hi_bits);
}

// What the last launch holds of a row's list: kHeld tokens a thread, in registers.
constexpr int kHeld = kKeep / kThreads;
struct Search {  // one of a key, cleared before the last barrier
    unsigned long long fine[kFine], member[kPairs], wave_sum[kWaves], before, sum;
    uint32_t member_key[kPairs], cut;
    unsigned int members, few;
    int at;
    __device__ void clear() {
        fine[threadIdx.x] = 0;
        if (threadIdx.x == 0) {
            members = 0;
            few = 0;
            cut = 0;
            at = -1;
        }
    }
};
struct Cutting {
    Search search[2];
    unsigned long long coarse[kCoarse], run_hi[kRuns], run_lo[kRuns];
    double wave_sum[kWaves];
    Found found;
};
static_assert(kFine == kThreads, "a bin a thread");

constexpr unsigned int kFew = 64;
// The key of the first token of bin `bin`, from the largest down, at which above + amount(sum of its and all larger
// tokens' values) reaches `target`; 0: none.  FEW: there may be few tokens in the bin, which are then compared with each other at once
// (two barriers instead of five, 0.9 us).  Else the bin's tokens (`in`) are dealt to kFine bins, of which one holds it; that one's few
// tokens are compared with each other, or their keys bisected.  What is summed are integers, so the list's order does not matter.
template <bool FEW, typename A>
__device__ uint32_t key_reaching(Search& s, const RowBins& bins, float mx, int bin, const float (&v)[kHeld], const bool (&in)[kHeld],
                                 const unsigned long long (&value)[kHeld], double above, double target, A amount) {
    const int lane = threadIdx.x & (FSIE_WAVE - 1), wave = threadIdx.x / FSIE_WAVE;
    const auto reaches = [&](unsigned long long sum) { return target <= above + amount(sum); };
    // among the first n members, with `before` above them
    const auto compare = [&](unsigned int n, unsigned long long before) {
        if (threadIdx.x < n) {
            const uint32_t key = s.member_key[threadIdx.x];
            unsigned long long over = before, upto = before;
            for (unsigned int j = 0; j < n; ++j) {
                if (s.member_key[j] >= key) upto += s.member[j];
                if (s.member_key[j] > key) over += s.member[j];
            }
            if (!reaches(over) && reaches(upto)) s.cut = key;  // (equal keys write the same)
        }
        __syncthreads();
        return s.cut;
    };
    const auto join = [&](unsigned int& count, int j, unsigned int most) {
        const unsigned int m = atomicAdd(&count, 1u);
        if (m < most) {
            s.member_key[m] = order_key(v[j]);
            s.member[m] = value[j];
        }
    };
    if constexpr (FEW) {
#pragma unroll
        for (int j = 0; j < kHeld; ++j)
            if (in[j]) join(s.few, j, kFew);
        __syncthreads();
        if (s.few <= kFew) return compare(s.few, 0);
    }
    int f[kHeld];
#pragma unroll
    for (int j = 0; j < kHeld; ++j) {
        f[j] = -1;
        if (!in[j]) continue;
        f[j] = static_cast<int>(fminf(fmaxf(((mx - v[j]) * bins.scale - static_cast<float>(bin)) * kFine, 0.f), static_cast<float>(kFine - 1)));
        atomicAdd(&s.fine[f[j]], value[j]);
    }
    __syncthreads();
    const unsigned long long mine = s.fine[threadIdx.x];
    unsigned long long run = wave_upto(mine);
    if (lane == FSIE_WAVE - 1) s.wave_sum[wave] = run;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kWaves; ++i) run += i < wave ? s.wave_sum[i] : 0;
    if (mine && !reaches(run - mine) && reaches(run)) {
        s.at = static_cast<int>(threadIdx.x);
        s.before = run - mine;
    }
    __syncthreads();
    const int at = s.at;
    if (at < 0) return 0;
    const unsigned long long before = s.before;
#pragma unroll
    for (int j = 0; j < kHeld; ++j)
        if (f[j] == at) join(s.members, j, kPairs);
    __syncthreads();
    if (s.members <= kPairs) return compare(s.members, before);
    uint32_t lo = 0, hi = order_key(mx);
    while (lo < hi) {
        const uint32_t mid = lo + (hi - lo) / 2 + ((hi - lo) & 1);
        __syncthreads();
        if (threadIdx.x == 0) s.sum = before;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kHeld; ++j)
            if (f[j] == at && order_key(v[j]) >= mid) atomicAdd(&s.sum, value[j]);
        __syncthreads();
        if (reaches(s.sum)) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// The key at which the row's kept set ends, from its list; 0 where the list does not tell.
__device__ uint32_t cut_of_list(Cutting& s, const SplitRow* w, const RowParams& q, const RowBins& bins, float mx,
                                const float (&v)[kHeld], int n) {
    uint32_t cut = 0;
    int bin[kHeld];
    bool in[kHeld];
    unsigned long long value[kHeld];
    const int k_bin = w->k_bin;
    const bool all_listed = bins.all_listed(q), binds = q.k > 0 && !(bins.cold && k_bin < 0);
    Found at{w->from, w->above};
    double target = w->target;
#pragma unroll
    for (int j = 0; j < kHeld; ++j)
        bin[j] = static_cast<int>(threadIdx.x) + j * kThreads < n ? bins.bin(v[j], mx) : -2;
    if (binds) {
        if (k_bin < 0) return 0;
#pragma unroll
        for (int j = 0; j < kHeld; ++j) {
            in[j] = bin[j] == k_bin;
            value[j] = 1;
        }
        cut = key_reaching<true>(s.search[0], bins, mx, k_bin, v, in, value, w->above_k, static_cast<double>(q.k),
                           [](unsigned long long sum) { return static_cast<double>(sum); });
        if (cut == 0 || !(q.p < 1.f)) return cut;
    }
#pragma unroll
    for (int j = 0; j < kHeld; ++j) value[j] = bin[j] >= 0 ? bins.weight(expf((v[j] - mx) * q.inv_temp), bin[j]) : 0;
    if (binds) {
        // the weights of what top k keeps: of its own bin from the list, of those above from the list or the row's bins
        using Scan = BinScan<kThreads>;
        const int b0 = static_cast<int>(threadIdx.x) * Scan::PER;
#pragma unroll
        for (int j = 0; j < kHeld; ++j)
            if (bin[j] >= 0 && order_key(v[j]) >= cut && (bin[j] == k_bin || all_listed)) atomicAdd(&s.coarse[bin[j]], value[j]);
        unsigned long long others[Scan::PER];
#pragma unroll
        for (int i = 0; i < Scan::PER; ++i) others[i] = !all_listed && b0 + i < k_bin ? w->sum[b0 + i] : 0;
        __syncthreads();
        Scan scan;
#pragma unroll
        for (int i = 0; i < Scan::PER; ++i) scan.v[i] = b0 + i < kCoarse ? bins.value(s.coarse[b0 + i] + others[i], b0 + i) : 0.0;
        scan.run(s.wave_sum);
        target = static_cast<double>(q.p) * scan.total;
        at = scan.find(target, &s.found);
        // (rounding may have put the target outside the bins that were listed)
        if (target > 0.0 && !(at.bin == k_bin || (w->from <= at.bin && at.bin <= w->upto))) return 0;
    }
    if (!(target > 0.0)) return order_key(mx);
    if (at.bin < 0) return 0;
#pragma unroll
    for (int j = 0; j < kHeld; ++j) in[j] = bin[j] == at.bin && order_key(v[j]) >= cut;
    const auto weight = [&](unsigned long long sum) { return bins.value(sum, at.bin); };
    return binds ? key_reaching<true>(s.search[1], bins, mx, at.bin, v, in, value, at.above, target, weight)
                   : key_reaching<false>(s.search[1], bins, mx, at.bin, v, in, value, at.above, target, weight);
}

__global__ __launch_bounds__(kThreads) void split_draw_kernel(const float* __restrict__ logits, int vocab, const SplitRow* ws,
                                                              int32_t* __restrict__ out) {
    __shared__ union {
        Cutting list;
        Binned bins;
    } s;
    __shared__ double run_sum[kRuns], sdbl[kWaves];
    const int r = blockIdx.x;
    const SplitRow* w = ws + r;
    const RowParams q = row_params(w, vocab);
    const RowTop top = kept_top(w);
    if (!(q.temp > 0.f)) {
        if (threadIdx.x == 0) out[r] = top.best.index;
        return;
    }
    const float* row = logits + static_cast<int64_t>(r) * vocab;
    const float mx = top.best.value;
    uint32_t cut = 0;  // tokens with key >= cut are kept
    double sum = threadIdx.x < kRuns ? w->run_sum[threadIdx.x] : 0.0;
    if (q.cuts) {
        RowBins bins;
        const unsigned int listed = w->n_listed;
        const int n = static_cast<int>(min(listed, static_cast<unsigned int>(kKeep)));
        float v[kHeld];
        int at[kHeld];
#pragma unroll
        for (int j = 0; j < kHeld; ++j) {
            const int i = static_cast<int>(threadIdx.x) + j * kThreads;
            v[j] = i < n ? w->listed[i] : 0.f;
            at[j] = i < n ? w->listed_at[i] : 0;
        }
        s.list.search[0].clear();
        s.list.search[1].clear();
        for (int b = threadIdx.x; b < kCoarse; b += kThreads) s.list.coarse[b] = 0;
        if (threadIdx.x < kRuns) s.list.run_hi[threadIdx.x] = s.list.run_lo[threadIdx.x] = 0;
        if (threadIdx.x == 0) s.list.found.bin = -1;
        __syncthreads();
        // (all of it the same in every thread)
        if (top.binned(vocab, q, &bins) && listed <= kKeep) cut = cut_of_list(s.list, w, q, bins, mx, v, n);
        if (cut != 0) {
            // the kept ones of the listed tokens join the sums of their runs
            const int hi_bits = 63 - (32 - __clz(vocab)), tokens = run_lines(vocab) * FSIE_WAVE;
#pragma unroll
            for (int j = 0; j < kHeld; ++j)
                if (static_cast<int>(threadIdx.x) + j * kThreads < n && order_key(v[j]) >= cut) {
                    const Limbs m = limbs_of(expf((v[j] - mx) * q.inv_temp), hi_bits);
                    const int run = at[j] / tokens;
                    if (m.hi) atomicAdd(&s.list.run_hi[run], m.hi);
                    if (m.lo) atomicAdd(&s.list.run_lo[run], m.lo);
                }
            __syncthreads();
            if (threadIdx.x < kRuns) sum += value_of(Limbs{s.list.run_hi[threadIdx.x], s.list.run_lo[threadIdx.x]}, hi_bits);
        } else {
            // a row that its list does not settle: as if it were not shared
            __syncthreads();
            if (vocab > kMaxBinned || !(fabsf(mx) < INFINITY) ||
                !cut_by_bins(s.bins, row, vocab, mx, top.low, top.nan, q.inv_temp, q.k, q.p, &cut)) {
                __syncthreads();
                cut = cut_by_bisection(row, vocab, mx, q.inv_temp, q.k, q.p, sdbl);
            }
            add_runs<kThreads>(row, vocab, 1, 0, run_sum, [&](float v, int) { return order_key(v) >= cut ? token_weight(v, mx, q.inv_temp) : 0.0; });
            __syncthreads();
            if (threadIdx.x < kRuns) sum = run_sum[threadIdx.x];
        }
    }
    if (threadIdx.x < kRuns) run_sum[threadIdx.x] = sum;
    __syncthreads();
    draw_from_runs(row, vocab, top.best, q.inv_temp, cut, w->uniform, run_sum, out + r);
}

}  // namespace

extern "C" int64_t fsie_sample_workspace(int n_rows, int vocab, int thresholds) {
    const bool shared = vocab >= kSplitFrom && vocab <= (1 << 30) && n_rows > 0 && n_rows <= (thresholds ? kMostRows : kMostPlainRows);
    return shared ? static_cast<int64_t>(n_rows) * static_cast<int64_t>(sizeof(SplitRow)) : 0;
}

extern "C" int fsie_sample_shares(int n_rows, int vocab, int top_k, int top_p) {
    if (fsie_sample_workspace(n_rows, vocab, top_k || top_p) == 0) return 0;
    if (top_k && top_p) return 1;
    if (!top_k && !top_p) return n_rows <= (vocab < kLongPlain ? 96 : 128);
    return n_rows <= (vocab - 8000) / (top_k ? 450 : 130) || n_rows > fsie_compute_units();
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

extern "C" int fsie_sample_by_value(void) { return kByValue; }

extern "C" int fsie_sample_split(const float* logits, int n_rows, int vocab, const float* temperature, const int32_t* top_k,
                                 const float* top_p, const double* uniform, int on_host, void* workspace, int32_t* out,
                                 hipStream_t stream) {
    FSIE_REQUIRE(n_rows > 0 && n_rows <= 65535 && vocab > 0 && vocab <= (1 << 30), "sample_split: bad sizes rows=%d vocab=%d", n_rows, vocab);
    FSIE_REQUIRE(temperature && uniform, "sample_split: temperatures and uniform numbers are needed");
    FSIE_REQUIRE(!on_host || n_rows <= kByValue, "sample_split: parameters of %d rows from the host, which are %d at most", n_rows, kByValue);
    FSIE_REQUIRE(workspace && reinterpret_cast<uintptr_t>(workspace) % 16 == 0,
                 "sample_split: a workspace on 16 bytes is needed");
    SplitRow* ws = static_cast<SplitRow*>(workspace);
    // a power of two of parts that gives every compute unit about two workgroups
    int parts = 1;
    while (parts < kMaxParts && n_rows * parts < 512) parts *= 2;
    const dim3 grid(parts, n_rows);
    if (on_host) {
        RowValues rows{};
        for (int r = 0; r < n_rows; ++r) {
            rows.uniform[r] = uniform[r];
            rows.temperature[r] = temperature[r];
            rows.top_k[r] = top_k ? top_k[r] : 0;
            rows.top_p[r] = top_p ? top_p[r] : 1.f;
        }
        split_top_kernel<<<grid, kPart, 0, stream>>>(logits, vocab, parts, ws, rows);
    } else {
        split_top_kernel<<<grid, kPart, 0, stream>>>(logits, vocab, parts, ws, RowArrays{temperature, top_k, top_p, uniform});
    }
    split_weigh_kernel<<<grid, kPart, 0, stream>>>(logits, vocab, parts, ws);
    if (top_k || top_p) split_list_kernel<<<grid, kPart, 0, stream>>>(logits, vocab, parts, ws);
    split_draw_kernel<<<n_rows, kThreads, 0, stream>>>(logits, vocab, ws, out);
    FSIE_CHECK_LAUNCH("sample_split");
    return 0;
}
