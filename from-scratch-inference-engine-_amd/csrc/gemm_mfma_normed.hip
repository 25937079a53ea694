// Y[M, N] = norm(stream)[M, K] . W[N, K]^T for one or two rows and a short K: the RMS norm in front of a product of few rows, in
// the product's own workgroups.
//
// A decode step of one request is bound by its launches: a norm of one row of 896 values is 2 us of which the row's arithmetic is a
// tenth, and the product behind it (gemm_mfma_stream.hip) waits for one trip to memory.  Here every workgroup of the product
// asks for the row (the stream and the last product's partial sums, all of K), then for all of its W, and makes the norm while W is on its
// way: the sum over the row across the workgroup, the normed row to LDS in bfloat16, from where the waves take their fragments.
// Every workgroup adds the same numbers in the same order, as the norm's own kernel does (block_sum, a quad a thread); the first one
// writes the new stream, to another buffer than the one the others still read.
// The price is the row, (1 + partial sums) * K * 4 bytes a row and workgroup, through the caches.  One request of the 0.5B shape: five launches
// a layer where there were seven, 23.4 us -> 20.6 as traced.
#include "common.h"
#include "api.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(1))) u32x4* GlobalVec;

union Frag {
    u32x4 q;
    bf16x8 v;
};

enum Result { SUMS = 0, GATED = 1 };  // float32 [slices of K, M, N]; bfloat16 [M, N / 2] of gate and up rows in turn

struct NormedCall {
    const float *residual, *sums, *norm_weight;
    const bf16_t* w;
    float* stream;
    void* y;
    int M, N, K, n_parts, slices;
    float eps;
    int act;
    float pos, neg;
};

// WAVES waves deal the K / 32 steps (SUMS: those of slice blockIdx.y) among themselves, S consecutive ones each, for one block of 16 rows of W;
// a thread has one quad of the row (K <= 4 * 64 WAVES).  PARTS: partial sums that are asked for together (0: none, more than there are: the last again, not added).
template <int WAVES, int S, int RESULT, bool FRAGS, int ROWS, int PARTS>
__global__ __launch_bounds__(WAVES * 64) void gemm_mfma_normed_kernel(const float* residual, const float* sums, const float* norm_weight,
                                                                         const bf16_t* w, float* stream, void* y, int M, int N, int K,
                                                                         int n_parts, float eps, int act, float pos, float neg, int slice_steps) {
    __shared__ floatx4 red[WAVES * 64];
    __shared__ __align__(16) uint2 normed[ROWS][WAVES * 64];  // four bfloat16 a thread
    __shared__ float wave_sq[ROWS][16];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = lane & 15, kg = lane >> 4;
    const int steps = K / 32, slice = RESULT == SUMS ? static_cast<int>(blockIdx.y) : 0;
    const int first = slice * slice_steps + wave * S, end = min(steps, (slice + 1) * slice_steps);
    const int j = min(static_cast<int>(threadIdx.x) * 4, K - 4);
    const bool mine = static_cast<int>(threadIdx.x) * 4 < K;
    floatx4 v[ROWS], p[ROWS][PARTS > 0 ? PARTS : 1];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        const int64_t at = static_cast<int64_t>(min(r, M - 1)) * K + j;
        v[r] = *reinterpret_cast<const floatx4*>(residual + at);
#pragma unroll
        for (int s = 0; s < PARTS; ++s)
            p[r][s] = *reinterpret_cast<const floatx4*>(sums + static_cast<int64_t>(min(s, n_parts - 1)) * M * K + at);
    }
    const floatx4 nw = *reinterpret_cast<const floatx4*>(norm_weight + j);
    __builtin_amdgcn_sched_barrier(0);  // (the row first: it is waited for while W is under way)
    Frag a[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int k = min(first + s, steps - 1);
        if constexpr (FRAGS)
            a[s].q = __builtin_nontemporal_load((GlobalVec)(w + (static_cast<int64_t>(blockIdx.x) * steps + k) * 512 + lane * 8));
        else
            a[s].q = *(GlobalVec)(w + static_cast<int64_t>(min(static_cast<int>(blockIdx.x) * 16 + row, N - 1)) * K + k * 32 + kg * 8);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        if constexpr (PARTS > 0) {
            floatx4 d = p[r][0];
#pragma unroll
            for (int s = 1; s < PARTS; ++s)
                if (s < n_parts) d += p[r][s];
            v[r] += d;
        }
        const float sq = wave_sum(mine ? v[r][0] * v[r][0] + v[r][1] * v[r][1] + v[r][2] * v[r][2] + v[r][3] * v[r][3] : 0.f);
        if (lane == 0) wave_sq[r][wave] = sq;
        if (PARTS > 0 && blockIdx.x == 0 && slice == 0 && mine && r < M) *reinterpret_cast<floatx4*>(stream + static_cast<int64_t>(r) * K + j) = v[r];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        const float total = sum_of_sixteen((lane & 15) < WAVES ? wave_sq[r][lane & 15] : 0.f);
        const float scale = inverse_sqrt(total / static_cast<float>(K) + eps);
        normed[r][threadIdx.x] = uint2{pack2_bf16((v[r][0] * scale) * nw[0], (v[r][1] * scale) * nw[1]),
                                       pack2_bf16((v[r][2] * scale) * nw[2], (v[r][3] * scale) * nw[3])};
    }
    __syncthreads();
    floatx4 acc = floatx4{0.f, 0.f, 0.f, 0.f};
    Frag b[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        b[s].q = u32x4{0, 0, 0, 0};
        if (row < ROWS && row < M) b[s].q = *reinterpret_cast<const u32x4*>(&normed[row][min(first + s, steps - 1) * 8 + kg * 2]);
    }
#pragma unroll
    for (int s = 0; s < S; ++s)
        if (first + s < end) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[s].v, b[s].v, acc, 0, 0, 0);
    // the waves' shares, added in the order of the waves
    red[wave * 64 + lane] = acc;
    __syncthreads();
    if (wave > 0) return;
    floatx4 sum = red[lane];
#pragma unroll
    for (int i = 1; i < WAVES; ++i) sum += red[i * 64 + lane];
    // lane holds D[n + r][m = row]
    const int n = blockIdx.x * 16 + kg * 4, m = row;
    if (m >= M || n >= N) return;
    if constexpr (RESULT == GATED) {  // rows n .. n + 3: gate, up, gate, up (N is a multiple of 4)
        uint32_t* out = static_cast<uint32_t*>(y);
        out[(static_cast<int64_t>(m) * (N / 2) + n / 2) / 2] = pack2_bf16(gate_pair(sum[0], sum[1], act, pos, neg), gate_pair(sum[2], sum[3], act, pos, neg));
    } else {  // (N is a multiple of 4)
        *reinterpret_cast<floatx4*>(static_cast<float*>(y) + (static_cast<int64_t>(slice) * M + m) * N + n) = sum;
    }
}

template <int WAVES, int S, int RESULT, bool FRAGS, int ROWS, int PARTS>
int launch(const NormedCall& c, hipStream_t stream) {
    const dim3 grid((c.N + 15) / 16, c.slices);
    gemm_mfma_normed_kernel<WAVES, S, RESULT, FRAGS, ROWS, PARTS><<<grid, WAVES * 64, 0, stream>>>(
        c.residual, c.sums, c.norm_weight, c.w, c.stream, c.y, c.M, c.N, c.K, c.n_parts, c.eps, c.act, c.pos, c.neg,
        (c.K / 32 + c.slices - 1) / c.slices);
    FSIE_CHECK_LAUNCH("gemm_mfma_normed");
    return 0;
}

template <int WAVES, int S, int RESULT, bool FRAGS, int ROWS>
int launch_parts(const NormedCall& c, hipStream_t stream) {
    if (c.n_parts == 0) return launch<WAVES, S, RESULT, FRAGS, ROWS, 0>(c, stream);
    if (c.n_parts == 1) return launch<WAVES, S, RESULT, FRAGS, ROWS, 1>(c, stream);
    return c.n_parts <= 4 ? launch<WAVES, S, RESULT, FRAGS, ROWS, 4>(c, stream) : launch<WAVES, S, RESULT, FRAGS, ROWS, 8>(c, stream);
}

template <int WAVES, int S, int RESULT, bool FRAGS>
int launch_rows(const NormedCall& c, hipStream_t stream) {
    if (c.M == 1) return launch_parts<WAVES, S, RESULT, FRAGS, 1>(c, stream);
    return launch_parts<WAVES, S, RESULT, FRAGS, 2>(c, stream);
}

template <int RESULT, bool FRAGS>
int launch_shape(const NormedCall& c, hipStream_t stream) {
    const int steps = c.K / 32;
    if constexpr (RESULT == SUMS)
        if (c.slices == 2) return steps <= 32 ? launch_rows<4, 4, RESULT, FRAGS>(c, stream) : launch_rows<8, 4, RESULT, FRAGS>(c, stream);
    if (steps <= 28) return launch_rows<4, 7, RESULT, FRAGS>(c, stream);
    if (steps <= 32) return launch_rows<4, 8, RESULT, FRAGS>(c, stream);
    if (steps <= 48) return launch_rows<8, 6, RESULT, FRAGS>(c, stream);
    return launch_rows<8, 8, RESULT, FRAGS>(c, stream);
}

}  // namespace

// Whether this is the faster way, and one this kernel has: the slices of K that SUMS takes (GATED: 1), or 0.  Two slices where their
// workgroups are no more than the units: one row of N = 1152, K = 896 2.8 us, in one slice 3.1; N = 2560, K = 2048 5.0 and 4.4.
// Norm and product alone / this kernel, us, cold weights, with 1, 4 and 7 partial sums.
// SUMS (the product alone in its slices of K), one row: N = 1152, K = 896 4.5 / 2.7, 4.6 / 2.8, 4.2 / 2.9; N = 2048, K = 1536 5.3 / 3.6, 5.5 / 3.9, 5.7 / 4.1;
// N = 2560, K = 2048 5.7 / 4.0, 6.0 / 4.4, 6.5 / 4.7; two rows 4.2 / 3.0, 4.6 / 3.2, 4.2 / 3.6 to 5.9 / 4.5, 6.2 / 4.8, 6.4 / 5.4;
// three and four rows as fast and slower.  GATED, one row: N = 9728, K = 896 7.0 / 5.3, 7.0 / 5.6, 7.0 / 6.1; N = 17920, K = 1536 13.2 / 11.5,
// 13.2 / 11.7, 13.0 / 12.9; N = 16384, K = 2048 15.3 / 12.6, 14.9 / 13.5, 15.3 / 14.3; two rows 7.1 / 5.6, 7.5 / 6.4, 7.4 / 7.3; 12.9 / 11.6,
// 13.1 / 13.8, 13.1 / 15.6; 14.9 / 13.4, 15.2 / 15.1, 15.4 / 16.7: its many workgroups read the row from 9,000 values on longer than a launch takes.
extern "C" int fsie_gemm_mfma_normed_takes(int M, int N, int K, int result, int n_parts) {
    const int units = fsie_compute_units();
    if (M < 1 || M > 2 || N < 4 || N % 4 || K < 64 || K % 32 || K > 2048 || n_parts < 0 || n_parts > 8 || units <= 0) return 0;
    if (result == GATED) return (1 + n_parts) * M * K <= 9000 ? 1 : 0;
    return result == SUMS ? ((N + 15) / 16 * 2 <= units ? 2 : 1) : 0;
}

extern "C" int fsie_gemm_mfma_normed(const float* residual, const float* sums, int n_parts, const float* norm_weight, float eps,
                                     float* new_stream, const void* w, void* y, int M, int N, int K, int result, int slices,
                                     int frags, int act, float pos, float neg, hipStream_t stream) {
    FSIE_REQUIRE(M >= 1 && M <= 2 && N >= 4 && N % 4 == 0 && K >= 64 && K % 32 == 0 && K <= 2048 && n_parts >= 0 && n_parts <= 8 &&
                     (slices == 1 || (slices == 2 && result == SUMS)) && (result == SUMS || result == GATED),
                 "gemm_mfma_normed: M=%d N=%d K=%d result %d, %d partial sums, %d slices", M, N, K, result, n_parts, slices);
    FSIE_REQUIRE(result != GATED || FSIE_PAIR_KNOWN(act), "gemm_mfma_normed: unknown activation %d", act);
    FSIE_REQUIRE(n_parts == 0 || (sums && new_stream && new_stream != residual), "gemm_mfma_normed: partial sums need a new stream");
    FSIE_REQUIRE(reinterpret_cast<uintptr_t>(residual) % 16 == 0 && reinterpret_cast<uintptr_t>(sums) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(norm_weight) % 16 == 0 && reinterpret_cast<uintptr_t>(new_stream) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(w) % 16 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0,
                 "gemm_mfma_normed: operands must be 16-byte aligned");
    const NormedCall c{residual, sums, norm_weight, static_cast<const bf16_t*>(w), new_stream, y, M, N, K, n_parts, slices, eps, act, pos, neg};
    if (result == GATED) return frags ? launch_shape<GATED, true>(c, stream) : launch_shape<GATED, false>(c, stream);
    return frags ? launch_shape<SUMS, true>(c, stream) : launch_shape<SUMS, false>(c, stream);
}
