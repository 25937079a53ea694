// Y[M, N] = X[M, K] . W[N, K]^T of a hundred to some thousand rows where the tiles of gemm_mfma_tile.hip would leave most of the chip idle: matrices
// of one to some ten MB, a step's portion of a prompt at a time.  bfloat16 operands in rows, on the matrix cores; the result in
// bfloat16 with the bias added before the one rounding, or float32 partial sums of slices of K for the norm that adds them up.
//
// A workgroup of four waves makes a tile of 64 x 64, 64 x 128 or 128 x 128 rows of X and W, a wave a quarter of it.  Both operands go
// through LDS, 64 values of K at a time, straight from memory, in three stages: one is read, one has arrived or is about to, one is
// asked for behind the barrier that says that every wave has read it.  One barrier a step.
// What bounds it: how much a unit can have under way.  A step takes 0.235, 0.305 and 0.53 us for the three tiles, which is 60 to 79 GB/s a
// unit of 140 that it draws from its L2 at most; without its loads it takes 0.2 to 0.4, without its products or its reads of LDS as long as
// with them.  Stages beyond three (eight of 64 x 64) and the next step's fragments read ahead into registers changed nothing, two stages
// and twice the workgroups a unit lost (0.6 us).  At 1,375 rows, cold weights: N = 1152, K = 896 8.1 us where the library's product takes 9.6, N = K = 896
// 7.6 and 9.2; at 512 rows 6.0 and 8.3, 5.9 and 8.1; 1,000 of N = K = 2048 14.6 and 16.9.  A call of the library's is 21 us of the host besides, one of this 13.
#include "common.h"
#include "api.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kStep = 64;  // values of K a stage
constexpr int kRowBytes = kStep * 2;

enum Result { kPlain = 0, kSums = 1 };  // bfloat16 [M, N] with a bias; float32 [splits, M, N]

// A tile: 32 T rows of X by 32 J rows of W, a wave of four a quarter of it.
template <int T, int J>
struct Shape {
    static constexpr int kRows = 32 * T, kCols = 32 * J;
    static constexpr int kStage = (kRows + kCols) * kRowBytes;  // W, then X
    static constexpr int kLoads = T + J;                        // a wave's, of eight rows each: J of W, T of X
    static constexpr int kStages = 3;
};

// 16 bytes a lane from memory to LDS, lane i's at lds + 16 i (m0 is an operand; the wait state behind its write is not the compiler's to
// put inside an asm statement).
__device__ __forceinline__ void load_to_lds(u32x4 rsrc, uint32_t lds, uint32_t offset, uint32_t k_offset) {
    asm volatile(
        "s_nop 0\n\t"
        "buffer_load_dwordx4 %1, %2, %3 offen lds"
        :
        : "{m0}"(lds), "v"(offset), "s"(rsrc), "s"(k_offset)
        : "memory");
}
#define FSIE_BLOCK_FENCE() __builtin_amdgcn_sched_barrier(0)

__device__ __forceinline__ u32x4 rows_from(const bf16_t* base, uint32_t bytes) {
    const uint64_t at = reinterpret_cast<uint64_t>(base);
    u32x4 r;
    r[0] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(at));
    r[1] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(at >> 32));
    r[2] = __builtin_amdgcn_readfirstlane(bytes);
    r[3] = 0x00020000u;
    return r;
}

// The permutation of a row's eight 16-byte units in LDS: W's rows are read 16 at a time as 4 runs of 4 that lie 4 J apart, X's as 16
// neighbours; in both any eight lanes in a row meet eight different units.
template <int J>
__device__ __forceinline__ int w_key(int row) { return (row >> 1 & 1) | (row % (16 * J) / (4 * J)) << 1; }
__device__ __forceinline__ int x_key(int row) { return row >> 1 & 7; }

template <int RESULT, int T, int J>
__global__ __launch_bounds__(256, 1) void gemm_block_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                            const float* __restrict__ bias, void* __restrict__ y, int M, int N, int K,
                                                            int m_tiles, int n_tiles, int splits, int n_outside) {
    using S = Shape<T, J>;
    extern __shared__ char lds[];
    // a die (the workgroup's number modulo 8) takes neighbouring tiles: of the larger operand its own eighth, of the other one all
    const int tiles = m_tiles * n_tiles * splits, a_die = (tiles + 7) / 8;
    const int id = static_cast<int>(blockIdx.x & 7) * a_die + static_cast<int>(blockIdx.x >> 3);
    if (id >= tiles) return;
    int m_tile, n_tile, slice;
    if (n_outside) {
        m_tile = id % m_tiles;
        n_tile = id / m_tiles % n_tiles;
        slice = id / m_tiles / n_tiles;
    } else {
        n_tile = id % n_tiles;
        m_tile = id / n_tiles % m_tiles;
        slice = id / n_tiles / m_tiles;
    }
    const int m0 = m_tile * S::kRows, n0 = n_tile * S::kCols;
    const int all_steps = K / kStep;
    const int first_step = static_cast<int>(static_cast<int64_t>(all_steps) * slice / splits);
    const int steps = static_cast<int>(static_cast<int64_t>(all_steps) * (slice + 1) / splits) - first_step;

    const int lane = threadIdx.x & (FSIE_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / FSIE_WAVE);
    const int mw = wave >> 1, nw = wave & 1;
    const int row = lane & 15, kg = lane >> 4;

    // what this wave brings of a stage: a quarter of the rows of W and of X, eight rows a load; rows past the end repeat the last one
    // and are never written
    const u32x4 x_rows = rows_from(x, static_cast<uint32_t>(M) * static_cast<uint32_t>(K) * 2u);
    const u32x4 w_rows = rows_from(w, static_cast<uint32_t>(N) * static_cast<uint32_t>(K) * 2u);
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds);
    uint32_t w_from[J], x_from[T];
#pragma unroll
    for (int i = 0; i < J; ++i) {
        const int r = (wave * J + i) * 8 + (lane >> 3);
        w_from[i] = static_cast<uint32_t>(min(n0 + r, N - 1)) * static_cast<uint32_t>(K) * 2u + ((lane & 7) ^ w_key<J>(r)) * 16u;
    }
#pragma unroll
    for (int i = 0; i < T; ++i) {
        const int r = (wave * T + i) * 8 + (lane >> 3);
        x_from[i] = static_cast<uint32_t>(min(m0 + r, M - 1)) * static_cast<uint32_t>(K) * 2u + ((lane & 7) ^ x_key(r)) * 16u;
    }
    uint32_t bring_to = 0, read_from = 0;  // the stages' places, in turn
    const auto bring = [&](int step) {
        const uint32_t k = static_cast<uint32_t>(first_step + min(step, steps - 1)) * kRowBytes, to = lds0 + bring_to;
#pragma unroll
        for (int i = 0; i < J; ++i) load_to_lds(w_rows, to + (wave * J + i) * 1024u, w_from[i], k);
#pragma unroll
        for (int i = 0; i < T; ++i) load_to_lds(x_rows, to + S::kCols * kRowBytes + (wave * T + i) * 1024u, x_from[i], k);
        bring_to = bring_to == (S::kStages - 1) * S::kStage ? 0 : bring_to + S::kStage;
    };

    // Fragments: A = 16 rows of W, B = 16 rows of X, a lane 8 values of K (16 bytes).  Row r of tile j of W is row
    // (r / 4) * 4 J + j * 4 + r % 4 of the wave's 16 J, so that a lane's results of the J tiles are 4 J neighbours.
    const int w_row = (row >> 2) * 4 * J + (row & 3);
    const int w_at = (nw * 16 * J + w_row) * kRowBytes, wk = w_key<J>(w_row);  // (the same for all j)
    const int x_at = S::kCols * kRowBytes + (mw * 16 * T + row) * kRowBytes, xk = x_key(row);

    floatx4 acc[J][T];
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
        for (int t = 0; t < T; ++t) acc[j][t] = floatx4{0.f, 0.f, 0.f, 0.f};

    bring(0);
    bring(1);
    for (int step = 0; step < steps; ++step) {
        // all but the youngest stage's loads have arrived, and what this wave has read of the stage before is in its registers
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(S::kLoads) : "memory");
        FSIE_BLOCK_FENCE();
        __builtin_amdgcn_s_barrier();
        FSIE_BLOCK_FENCE();
        bring(step + 2);  // into the stage that was read before the barrier
        const char* stage = lds + read_from;
        read_from = read_from == (S::kStages - 1) * S::kStage ? 0 : read_from + S::kStage;
        bf16x8 a[J][2], b[T][2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int j = 0; j < J; ++j)
                a[j][h] = *reinterpret_cast<const bf16x8*>(stage + w_at + j * 4 * kRowBytes + (((h * 4 + kg) ^ wk) * 16));
#pragma unroll
            for (int t = 0; t < T; ++t)
                b[t][h] = *reinterpret_cast<const bf16x8*>(stage + x_at + t * 16 * kRowBytes + (((h * 4 + kg) ^ xk) * 16));
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int j = 0; j < J; ++j) acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[j][h], b[t][h], acc[j][t], 0, 0, 0);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (no load may still write LDS when the workgroup's is given away)

    // lane holds, for every tile t of 16 rows of X, the results of 4 J neighbouring rows of W from n on
    const int n = n0 + nw * 16 * J + kg * 4 * J;
    if (n >= N) return;  // (N is a multiple of 16: 4 J neighbours are all in or all out)
    floatx4 add[J];
    if (RESULT == kPlain) {
#pragma unroll
        for (int j = 0; j < J; ++j) add[j] = bias ? *reinterpret_cast<const floatx4*>(bias + n + 4 * j) : floatx4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const int m = m0 + mw * 16 * T + t * 16 + row;
        if (m >= M) continue;
        if (RESULT == kSums) {
            float* to = static_cast<float*>(y) + (static_cast<int64_t>(slice) * M + m) * N + n;
#pragma unroll
            for (int j = 0; j < J; ++j) *reinterpret_cast<floatx4*>(to + 4 * j) = acc[j][t];
        } else {
            uint32_t out[2 * J];
#pragma unroll
            for (int j = 0; j < J; ++j) {
                const floatx4 v = acc[j][t] + add[j];
                out[2 * j] = pack2_bf16(v[0], v[1]);
                out[2 * j + 1] = pack2_bf16(v[2], v[3]);
            }
            uint4* to = reinterpret_cast<uint4*>(static_cast<bf16_t*>(y) + static_cast<int64_t>(m) * N + n);
#pragma unroll
            for (int j = 0; j < J; j += 2) to[j / 2] = uint4{out[2 * j], out[2 * j + 1], out[2 * j + 2], out[2 * j + 3]};
        }
    }
}

struct Call {
    const bf16_t *x, *w;
    const float* bias;
    void* y;
    int M, N, K, splits;
    hipStream_t stream;
};

template <int RESULT, int T, int J>
int launch(const Call& c) {
    using S = Shape<T, J>;
    const int m_tiles = (c.M + S::kRows - 1) / S::kRows, n_tiles = (c.N + S::kCols - 1) / S::kCols;
    const unsigned groups = static_cast<unsigned>((m_tiles * n_tiles * c.splits + 7) / 8 * 8);
    static const hipError_t allowed = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_block_kernel<RESULT, T, J>),
                                                          hipFuncAttributeMaxDynamicSharedMemorySize, S::kStages * S::kStage);
    FSIE_REQUIRE(allowed == hipSuccess, "gemm_mfma_block: %d bytes of LDS: %s", S::kStages * S::kStage, hipGetErrorString(allowed));
    gemm_block_kernel<RESULT, T, J><<<groups, 256, S::kStages * S::kStage, c.stream>>>(c.x, c.w, c.bias, c.y, c.M, c.N, c.K, m_tiles, n_tiles,
                                                                                   c.splits, c.N >= c.M);
    FSIE_CHECK_LAUNCH("gemm_mfma_block");
    return 0;
}

template <int RESULT>
int launch_shape(int tile, const Call& c) {
    switch (tile) {
        case 0: return launch<RESULT, 2, 2>(c);
        case 1: return launch<RESULT, 2, 4>(c);
        default: return launch<RESULT, 4, 4>(c);
    }
}

}  // namespace

// Which tile, and in how many slices of K, M rows of this product are best taken; -1: the library's product is faster or the sizes are not
// the kernel's.  Returns tile + 256 * slices.
// The rule is the time that a count of steps gives: fixed + steps * a step's, workgroups that share a unit taking turns (0.92 and 1.05 of a
// step each, as many as the unit's LDS holds), weights that come from HBM, at its latency, up to 1.35 and 1.1 of that; partial sums count their
// bytes here and in the norm at 4.5 TB/s.  It has to be 0.92 of the library's 6.5 us and 0.95 PFLOP/s, or 3 us and its weights at 2.5 TB/s: the least that
// it took at 24 matrices of 1 to 33 MB and 19 numbers of rows from 70 to 4,096.  Of these 456 and as many with slices and the norm the rule takes 237,
// at a median of 0.77 of the library's time, the largest 1.04 (this / the library and the norm: 96 rows of N = 896, K = 4864 8.8 / 12.4, 256 12.0 / 14.6; 96 of
// N = 2048, K = 8192 17.7 / 24.3, 129 20.6 / 29.6; 96 of N = K = 3584 16.4 / 23.3; whole, 256 of N = 3072, K = 1024 6.6 / 9.1; 850 of N = K = 2048 14.1 / 15.8).
extern "C" int fsie_gemm_mfma_block_plan(int M, int N, int K, int result, int units) {
    if (M <= 0 || N <= 0 || K <= 0 || units <= 0 || N % 16 || K % kStep || (result != kPlain && result != kSums)) return -1;
    if (static_cast<int64_t>(M) * K * 2 >= (int64_t{1} << 31) || static_cast<int64_t>(N) * K * 2 >= (int64_t{1} << 31)) return -1;
    const int rows[3] = {64, 64, 128}, cols[3] = {64, 128, 128};
    const double us_a_step[3] = {0.235, 0.305, 0.58}, fixed[3] = {2.3, 2.6, 3.4};
    const int64_t steps = K / kStep;
    const double weights = 2.0 * N * static_cast<double>(K), flops = 2.0 * M * static_cast<double>(N) * K;
    double best = 1e30;
    int choice = -1;
    for (int tile = 0; tile < 3; ++tile) {
        for (int slices = 1; slices <= (result == kSums ? 8 : 1); ++slices) {
            if (slices > 1 && steps / slices < 4) break;
            const int64_t groups = ceil_div64(M, rows[tile]) * ceil_div64(N, cols[tile]) * slices, deep = ceil_div64(groups, units);
            if (deep > 3 - tile) continue;  // (so many a unit's LDS holds)
            const double from_memory = weights < 10e6 ? 0.0 : weights < 16e6 ? 0.7 : 1.0;
            const double step = us_a_step[tile] * (1.0 + from_memory * (tile == 2 ? 0.1 : 0.35)) * (deep > 1 ? (tile == 0 ? 0.92 : 1.05) * deep : 1.0);
            double us = fixed[tile] + static_cast<double>(ceil_div64(steps, slices)) * step;
            if (result == kSums) us += 8.0 * slices * M * static_cast<double>(N) / 4.5e6;
            if (us < best) {
                best = us;
                choice = tile + 256 * slices;
            }
        }
    }
    const double product = 6.5 + flops / 0.95e9, read = 3.0 + weights / 2.5e6;
    return choice >= 0 && best <= 0.92 * (product > read ? product : read) ? choice : -1;
}

extern "C" int fsie_gemm_mfma_block(const void* x, const void* w, const float* bias, void* y, int M, int N, int K, int result, int splits,
                                    int tile, hipStream_t stream) {
    FSIE_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm_mfma_block: bad sizes M=%d N=%d K=%d", M, N, K);
    FSIE_REQUIRE(N % 16 == 0 && K % kStep == 0, "gemm_mfma_block: N=%d must be a multiple of 16, K=%d of %d", N, K, kStep);
    FSIE_REQUIRE(result == kPlain || result == kSums, "gemm_mfma_block: unknown result %d", result);
    FSIE_REQUIRE(splits >= 1 && splits <= K / kStep && (splits == 1 || result == kSums), "gemm_mfma_block: %d slices", splits);
    FSIE_REQUIRE(!bias || result == kPlain, "gemm_mfma_block: partial sums take no bias");
    FSIE_REQUIRE(tile >= 0 && tile <= 2, "gemm_mfma_block: unknown tile %d", tile);
    FSIE_REQUIRE(static_cast<int64_t>(M) * K * 2 < (int64_t{1} << 31) && static_cast<int64_t>(N) * K * 2 < (int64_t{1} << 31),
                 "gemm_mfma_block: operands of %d x %d and %d x %d are more than the kernel's 32-bit offsets take", M, K, N, K);
    FSIE_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(y) % 16 == 0 && reinterpret_cast<uintptr_t>(bias) % 16 == 0,
                 "gemm_mfma_block: operands must be 16-byte aligned");
    if (M == 0) return 0;
    const Call c{static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(w), bias, y, M, N, K, splits, stream};
    return result == kSums ? launch_shape<kSums>(tile, c) : launch_shape<kPlain>(tile, c);
}
