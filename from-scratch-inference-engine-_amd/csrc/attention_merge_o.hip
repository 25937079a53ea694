// The merge of a decode step's cut items (attention_merge, attention_scalar.hip) with the output projection behind it, for a few tokens.
//
// Such a step is bound by its launches: the merge of a few records a head is 2.3 to 4 us, nearly all of it the launch and one trip to memory, and the
// projection behind it as much.  Here a workgroup takes a kv head of a token: a wave merges a head (the arithmetic of attention_merge, and up to 32 records its order: more
// are dealt to four waves there), the heads, rounded to 16 bits where the heads are, meet in LDS, and each wave multiplies them by ROWS rows of the projection, which it has asked for behind the records.  Every workgroup of a kv head
// merges the same records again (2 KB a split for seven heads of 64), which costs less than a launch while all workgroups are on the chip at once.
// The result is float32 sums [n_kv][tokens][o_rows], a slice a kv head, for the norm that adds them up.
// 24 steps, ms, two launches / this: one request of the 0.5B shape (24 layers) behind 300 keys 16.09 / 15.12, 600 16.28 / 15.04, 2,000 18.06 / 16.70, two behind 400 16.45 / 15.69, behind
// 2,000 22.49 / 21.39; 12 layers of hidden size 1,536, 12 heads on 2 of 128, one behind 400 12.26 / 11.44; of 1,024, 16 on 4 of 64, behind 600 10.45 / 9.77.
// In front of a norm of its own (three and four requests, float32): three of the 0.5B shape behind 300 to 500 keys 18.26 / 17.74; in float32 four behind 40 to 301
// 26.66 / 25.79, one behind 1,500 35.31 / 33.76, four behind 400 to 800 42.13 / 41.23.
#include "common.h"
#include "api.h"

#include <math.h>

namespace {

constexpr int kMergeWaves = 8;
constexpr int kAhead = 8;  // records under way

// Eight values of the weight or of the heads, and their products added up in order.
template <typename T>
struct Eight;
template <>
struct Eight<bf16_t> {
    uint4 raw;
    __device__ void load(const bf16_t* p) { raw = *reinterpret_cast<const uint4*>(p); }
    __device__ void store(bf16_t* p) const { *reinterpret_cast<uint4*>(p) = raw; }
    __device__ float dot(const Eight& o) const {
        const uint32_t a[4] = {raw.x, raw.y, raw.z, raw.w}, b[4] = {o.raw.x, o.raw.y, o.raw.z, o.raw.w};
        float z = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            z = fmaf(__uint_as_float(a[i] << 16), __uint_as_float(b[i] << 16), z);
            z = fmaf(__uint_as_float(a[i] & 0xffff0000u), __uint_as_float(b[i] & 0xffff0000u), z);
        }
        return z;
    }
};
template <>
struct Eight<float> {
    float4 lo, hi;
    __device__ void load(const float* p) { lo = *reinterpret_cast<const float4*>(p), hi = *reinterpret_cast<const float4*>(p + 4); }
    __device__ void store(float* p) const { *reinterpret_cast<float4*>(p) = lo, *reinterpret_cast<float4*>(p + 4) = hi; }
    __device__ float dot(const Eight& o) const {
        float z = fmaf(lo.w, o.lo.w, fmaf(lo.z, o.lo.z, fmaf(lo.y, o.lo.y, lo.x * o.lo.x)));
        return fmaf(hi.w, o.hi.w, fmaf(hi.z, o.hi.z, fmaf(hi.y, o.hi.y, fmaf(hi.x, o.hi.x, z))));
    }
};

// T: what the heads and the weight are; DIMS = head_dim / 64.
template <typename T, int DIMS, int ROWS>
__global__ __launch_bounds__(64 * kMergeWaves) void attention_merge_o_kernel(
    const float* __restrict__ partials, const int32_t* __restrict__ merges, const T* __restrict__ heads, const T* __restrict__ o_weight,
    float* __restrict__ o_sums, int n_heads, int group, int o_rows, int64_t part_stride) {
    constexpr int HD = 64 * DIMS, LOADS = 16 * HD / 8 / 64;  // a row's loads of eight values a lane (sixteen heads at most)
    __shared__ __align__(16) T x[16 * HD];
    const int32_t* mi = merges + static_cast<int64_t>(blockIdx.z) * FSIE_ATTN_MERGE_INTS;
    const int row = mi[0], first = mi[1], n_splits = mi[2], stride = mi[3];
    const int kvh = blockIdx.y, h0 = kvh * group;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int o_first = (static_cast<int>(blockIdx.x) * kMergeWaves + wave) * ROWS, units = group * (HD / 8);

    constexpr int64_t rec_size = HD + 2;
    const int64_t rec_step = static_cast<int64_t>(stride) * n_heads * rec_size;
    const bool cut = n_splits > 0;  // (else attention has left the token's heads whole)
    // the first head's first records, then the weight
    float ms = -INFINITY, l = 0.f, v[kAhead][DIMS];
    auto ask = [&](const float* rec, int from, int n) {
#pragma unroll
        for (int j = 0; j < kAhead; ++j)
#pragma unroll
            for (int i = 0; i < DIMS; ++i) v[j][i] = rec[min(from + j, n - 1) * rec_step + lane + 64 * i];
    };
    const float* rec0 = partials + (static_cast<int64_t>(first) * n_heads + h0 + min(wave, group - 1)) * rec_size;
    if (cut) {
        ms = rec0[min(lane, n_splits - 1) * rec_step + HD];
        l = rec0[min(lane, n_splits - 1) * rec_step + HD + 1];
        ask(rec0, 0, n_splits);
    }
    Eight<T> w[ROWS][LOADS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        const T* at = o_weight + (static_cast<int64_t>(min(o_first + r, o_rows - 1)) * n_heads + h0) * HD;
#pragma unroll
        for (int u = 0; u < LOADS; ++u)
            if (u == 0 || u * 64 < units) w[r][u].load(at + min(u * 64 + lane, units - 1) * 8);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (cut) {
        for (int h = wave; h < group; h += kMergeWaves) {
            const float* rec = partials + (static_cast<int64_t>(first) * n_heads + h0 + h) * rec_size;
            const bool loaded = h == wave;
            float m = lane < n_splits && loaded ? ms : -INFINITY;
            for (int s = loaded ? lane + 64 : lane; s < n_splits; s += 64) m = fmaxf(m, rec[s * rec_step + HD]);
            m = wave_max(m);
            float denom = 0.f, a[DIMS];
#pragma unroll
            for (int i = 0; i < DIMS; ++i) a[i] = 0.f;
            for (int base = 0; base < n_splits; base += 64) {
                const int s = min(base + lane, n_splits - 1);
                const bool have = loaded && base == 0;
                const float m_s = have ? ms : rec[s * rec_step + HD], l_s = have ? l : rec[s * rec_step + HD + 1];
                const float w_s = base + lane >= n_splits || m_s == -INFINITY ? 0.f : expf(m_s - m);
                const int here = min(64, n_splits - base);
                for (int j0 = 0; j0 < here; j0 += kAhead) {
                    if (!have || j0 > 0) ask(rec + base * rec_step, j0, here);
#pragma unroll
                    for (int j = 0; j < kAhead; ++j) {
                        const int src = min(j0 + j, 63);
                        const float wj = j0 + j < here ? __shfl(w_s, src) : 0.f;
                        const float lj = __shfl(l_s, src);
                        if (wj != 0.f) {  // the same for the whole wave
                            denom += lj * wj;
#pragma unroll
                            for (int i = 0; i < DIMS; ++i) a[i] += v[j][i] * wj;
                        }
                    }
                }
            }
            const float inv = denom > 0.f ? 1.0f / denom : 0.f;
#pragma unroll
            for (int i = 0; i < DIMS; ++i) x[h * HD + lane + 64 * i] = from_float<T>(a[i] * inv);
        }
    } else {
        for (int u = threadIdx.x; u < units; u += 64 * kMergeWaves) {
            Eight<T> e;
            e.load(heads + (static_cast<int64_t>(row) * n_heads + h0) * HD + u * 8);
            e.store(x + u * 8);
        }
    }
    __syncthreads();
    float sum[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) sum[r] = 0.f;
#pragma unroll
    for (int u = 0; u < LOADS; ++u) {
        if (u > 0 && u * 64 >= units) break;  // (the same for the whole workgroup)
        const int unit = u * 64 + lane;
        Eight<T> xv;
        xv.load(x + min(unit, units - 1) * 8);
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            const float more = xv.dot(w[r][u]);
            sum[r] += unit < units ? more : 0.f;
        }
    }
    float mine = 0.f;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        const float all = wave_sum(sum[r]);
        mine = lane == r ? all : mine;
    }
    if (lane < ROWS && o_first + lane < o_rows) o_sums[kvh * part_stride + static_cast<int64_t>(row) * o_rows + o_first + lane] = mine;
}

}  // namespace

// Rows of the output projection a wave, for n_merges tokens; 0: the merge and the projection are better two launches, or there is no kernel.  As few as leave
// no more workgroups than units (which bounds the weight that is read, once a token, to 34 MB for groups of eight heads of 128 in float32).
// Groups of more than eight heads give a wave two to merge, one after the other, in every workgroup: they gain less, and lose from three tokens on, in float32
// from two, and beyond 12 heads.  16 steps behind 400 / 1,500 keys, one launch over two:
//   up to 8 heads   0.92 to 1.00 at every size and number of tokens (1,024 wide, 8 on 1 of 128, one token 0.94 / 0.94, four 0.98 / 0.98; float32 0.98 / 0.98 and 0.99 / 0.99; 2,048
//                   wide, 16 on 2 of 128, one 0.98 / 0.97; float32 2,560 wide, 8 on 1, two 1.00 / 1.00)
//   10 and 12       one token 0.93 to 0.99 (1,536 wide, 12 on 1 of 128, 0.93 / 0.94), two 0.94 to 0.99, four 1.01 / 1.01 (1,280 wide, 10 on 1) and 0.99 / 1.00; float32 one 0.98 / 0.99
//                   to 1.00, two 0.98 / 1.01, four 1.01 / 1.01
//   16              one token 0.97 to 1.01 (2,048 wide, 16 on 1 of 128, 1.01 / 1.01; 32 on 2 of 64 1.01 / 1.00; 4,096 wide, 32 on 2 of 128, 0.98 / 0.99), four 1.02 / 1.02; float32 0.99 / 1.01 to 1.00 / 1.02
extern "C" int fsie_attention_merge_o_rows(int n_merges, int n_heads, int n_kv, int head_dim, int o_rows, int dtype, int units) {
    if (n_merges <= 0 || n_heads <= 0 || n_kv <= 0 || n_heads % n_kv || o_rows <= 0 || units <= 0) return 0;
    if ((head_dim != 64 && head_dim != 128) || (dtype != FSIE_F32 && dtype != FSIE_BF16)) return 0;
    const int group = n_heads / n_kv;
    if (group > kMergeWaves && (group > 12 || n_merges > (dtype == FSIE_F32 ? 1 : 2))) return 0;
    for (int rows = 1; rows <= 4; ++rows)
        if (ceil_div64(o_rows, kMergeWaves * rows) * n_kv * n_merges <= units) return rows;
    return 0;
}

// merges [n_merges], records: as fsie_attention_merge.  A token whose merge has no splits: its heads stand whole in `heads` [tokens][n_heads head_dim].  o_weight
// [o_rows][n_heads head_dim] (rows without gaps, of the heads' type `dtype`); o_sums [n_kv][n_tokens][o_rows].
extern "C" int fsie_attention_merge_o(const float* partials, const int32_t* merges, int n_merges, int n_tokens, const void* heads, const void* o_weight,
                                      int o_rows, float* o_sums, int rows_of_wave, int n_heads, int n_kv, int head_dim, int dtype, hipStream_t stream) {
    FSIE_REQUIRE(n_merges >= 0 && n_tokens >= 0 && o_rows > 0 && n_heads > 0 && n_kv > 0 && n_heads % n_kv == 0 && n_heads / n_kv <= 16,
                 "attention_merge_o: bad sizes, %d heads on %d, %d rows", n_heads, n_kv, o_rows);
    FSIE_REQUIRE((head_dim == 64 || head_dim == 128) && rows_of_wave >= 1 && rows_of_wave <= 4, "attention_merge_o: heads of %d, %d rows a wave", head_dim, rows_of_wave);
    FSIE_REQUIRE(partials && merges && heads && o_weight && o_sums && reinterpret_cast<uintptr_t>(heads) % 16 == 0 && reinterpret_cast<uintptr_t>(o_weight) % 16 == 0,
                 "attention_merge_o: heads and weight must be 16-byte aligned");
    FSIE_REQUIRE(dtype == FSIE_F32 || dtype == FSIE_BF16, "attention_merge_o: unknown dtype %d", dtype);
    if (n_merges == 0) return 0;
    const dim3 grid(static_cast<unsigned>(ceil_div64(o_rows, kMergeWaves * rows_of_wave)), n_kv, n_merges);
#define FSIE_MERGE_O(T, D, R)                                                                                          \
    attention_merge_o_kernel<T, D, R><<<grid, 64 * kMergeWaves, 0, stream>>>(partials, merges, static_cast<const T*>(heads), static_cast<const T*>(o_weight), \
                                                                             o_sums, n_heads, n_heads / n_kv, o_rows, static_cast<int64_t>(n_tokens) * o_rows)
#define FSIE_MERGE_O_ROWS(T, D)                                                                                        \
    switch (rows_of_wave) {                                                                                            \
        case 1: FSIE_MERGE_O(T, D, 1); break;                                                                          \
        case 2: FSIE_MERGE_O(T, D, 2); break;                                                                          \
        case 3: FSIE_MERGE_O(T, D, 3); break;                                                                          \
        default: FSIE_MERGE_O(T, D, 4); break;                                                                         \
    }
    if (dtype == FSIE_F32) {
        if (head_dim == 64) FSIE_MERGE_O_ROWS(float, 1) else FSIE_MERGE_O_ROWS(float, 2)
    } else {
        if (head_dim == 64) FSIE_MERGE_O_ROWS(bf16_t, 1) else FSIE_MERGE_O_ROWS(bf16_t, 2)
    }
#undef FSIE_MERGE_O_ROWS
#undef FSIE_MERGE_O
    FSIE_CHECK_LAUNCH("attention_merge_o");
    return 0;
}
