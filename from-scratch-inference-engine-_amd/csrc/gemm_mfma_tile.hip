// Y[M, N] = X[M, K] . W[N, K]^T of many rows (prompts), bfloat16 operands, on the matrix cores, with what follows the
// product in its epilogue: gate and up values of neighbouring rows of W multiplied, or float32 partial sums of slices
// of K for the norm that adds them up.
//
// A workgroup of eight waves makes a tile of 256 rows of X by 256 of W, a wave 128 by 64 of it (128 accumulators a
// lane).  Both operands go through LDS, 64 values of K at a time, in two stages of 64 KB, straight from memory
// (buffer loads that write LDS); a row's eight 16-byte units lie permuted by the row, so that the fragments' reads of
// eight rows meet eight different groups of banks.
// Two waves share a SIMD, and what one of them reads from LDS takes about as long as the other's matrix instructions:
// so the waves go in two groups, one a phase behind the other.  A wave's step of K is four phases, each ended by a
// barrier of the whole workgroup:
//   M1  all fragments of its 64 rows of W, those of the first 64 of its 128 rows of X      C1  32 matrix instructions
//   M2  the fragments of the other 64 rows of X                                            C2  32 matrix instructions
// and while one group is in an M phase the other is in a C phase.  What M1 reads of a stage (W and half of X) is free
// for the step after next as soon as both groups have read it, the other half of X a phase pair later: each is asked for
// then, four phases (some 2,000 cycles) before it is waited for.  A wave has the same number of loads under way at
// every wait (the last steps' are asked for again when there are no more), so "all but the last kUnderWay of the shape" is
// what has to have arrived.
// What bounds it: a step of 256 x 256 x 64 takes 1.38 us where its matrix instructions alone take 1.04 (v_mfma_f32_16x16x32
// at 2.07 PFLOP/s over the chip); the LDS is busy for nine tenths of that (24 KB of fragments a wave and step, 64 KB
// written).  On zeros a step takes 1.09 us (2,048 x 8192 x 18944 332 us, 431 on random values): the clock gives way to the power that data costs, so a better order
// of the same reads and products would gain little.  1,320 TFLOP/s at 2,048 x 37888 x 3584 with gate and up multiplied.  The instruction
// of 32 x 32 x 16, faster by itself, reads the same bytes in a worse pattern: 1,150.
#include "common.h"
#include "api.h"
#include "lds_loads.h"

namespace {

using namespace fsie_lds;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kStep = 64;  // values of K a stage
constexpr int kRowBytes = kStep * 2;

// A tile: T = tiles of 16 rows of X in each half of a wave's rows (4: 256 rows a workgroup, 2: 128), J = tiles of 16 rows of
// W a wave (64 J rows a workgroup).
template <int T, int J>
struct Shape {
    static constexpr int kRows = 64 * T, kCols = 64 * J;
    static constexpr int kWBytes = kCols * kRowBytes;        // a stage: W, then the first and the second halves of the waves' X rows
    static constexpr int kXHalf = kRows / 2 * kRowBytes;
    static constexpr int kStage = kWBytes + 2 * kXHalf;
    static constexpr int kXLoads = T / 2;                    // a wave's loads of 8 rows: of a half of X, of W
    static constexpr int kWLoads = J;
    static constexpr int kUnderWay = kWLoads + 2 * kXLoads;  // loads that are younger than those a wait is for
};

enum Result { kPair = 1, kSums = 2 };

#define FSIE_TILE_FENCE() __builtin_amdgcn_sched_barrier(0)

// The permutation of a row's 16-byte units.  W's rows are read 16 at a time as 4 runs of 4 that lie 16 apart (see the
// fragments below), X's as 16 neighbours: in both any eight lanes in a row see eight values.
template <int J>
__device__ __forceinline__ int w_key(int row) { return (row & 3) | ((row % (16 * J) / (4 * J) & 1) << 2); }
__device__ __forceinline__ int x_key(int row) { return row & 7; }

template <int RESULT, int ACT, int T, int J>
__global__ __launch_bounds__(512, 2) void gemm_tile_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                           void* __restrict__ y, int M, int N, int K, int m_tiles, int n_tiles,
                                                           int splits, float act_pos, float act_neg) {
    using S = Shape<T, J>;
    extern __shared__ char lds[];
    // workgroups of one tile of W lie side by side on one die (their number modulo 8), whose L2 then reads that tile once
    const int die = blockIdx.x & 7, at = blockIdx.x >> 3;
    const int m_tile = at % m_tiles, column = (at / m_tiles) * 8 + die;
    if (column >= n_tiles * splits) return;
    const int slice = column / n_tiles;
    const int m0 = m_tile * S::kRows, n0 = (column - slice * n_tiles) * S::kCols;
    const int all_steps = K / kStep;
    const int first_step = static_cast<int>(static_cast<int64_t>(all_steps) * slice / splits);
    const int steps = static_cast<int>(static_cast<int64_t>(all_steps) * (slice + 1) / splits) - first_step;

    const int lane = threadIdx.x & (FSIE_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / FSIE_WAVE);
    const int mw = wave >> 2, nw = wave & 3;
    const int row = lane & 15, kg = lane >> 4;

    // what this wave brings of a stage: an eighth of the rows of W and of each half of X, eight rows a load;
    // rows past the end repeat the last one and are never written
    const u32x4 x_rows = rows_from(x, static_cast<uint32_t>(M) * static_cast<uint32_t>(K) * 2u);
    const u32x4 w_rows = rows_from(w, static_cast<uint32_t>(N) * static_cast<uint32_t>(K) * 2u);
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds);
    uint32_t w_from[S::kWLoads], x_from[2][S::kXLoads];
#pragma unroll
    for (int i = 0; i < S::kWLoads; ++i) {
        const int r = (wave * S::kWLoads + i) * 8 + (lane >> 3);
        w_from[i] = static_cast<uint32_t>(min(n0 + r, N - 1)) * static_cast<uint32_t>(K) * 2u + ((lane & 7) ^ w_key<J>(r)) * 16u;
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < S::kXLoads; ++i) {
            const int r = (wave * S::kXLoads + i) * 8 + (lane >> 3);  // row of the half: 16 T of each of the waves' 32 T
            const int m = m0 + r / (16 * T) * (32 * T) + h * (16 * T) + r % (16 * T);
            x_from[h][i] = static_cast<uint32_t>(min(m, M - 1)) * static_cast<uint32_t>(K) * 2u + ((lane & 7) ^ x_key(r)) * 16u;
        }
    const auto k_of = [&](int step) { return static_cast<uint32_t>(first_step + min(step, steps - 1)) * kRowBytes; };
    const auto stage_of = [&](int step) { return lds0 + static_cast<uint32_t>(step & 1) * S::kStage; };
    const auto bring_first = [&](int step) {  // W and the first half of X
        const uint32_t k = k_of(step), to = stage_of(step);
#pragma unroll
        for (int i = 0; i < S::kWLoads; ++i) load_to_lds(w_rows, to + (wave * S::kWLoads + i) * 1024u, w_from[i], k);
#pragma unroll
        for (int i = 0; i < S::kXLoads; ++i)
            load_to_lds(x_rows, to + S::kWBytes + (wave * S::kXLoads + i) * 1024u, x_from[0][i], k);
    };
    const auto bring_second = [&](int step) {
        const uint32_t k = k_of(step), to = stage_of(step);
#pragma unroll
        for (int i = 0; i < S::kXLoads; ++i)
            load_to_lds(x_rows, to + S::kWBytes + S::kXHalf + (wave * S::kXLoads + i) * 1024u, x_from[1][i], k);
    };

    // Fragments: A = 16 rows of W, B = 16 rows of X, a lane 8 values of K (16 bytes).  Row r of tile j of W is row
    // (r / 4) * 4 J + j * 4 + r % 4 of the wave's 16 J, so that a lane's results of the J tiles are 4 J neighbours.
    const int w_at = (nw * 16 * J + (row >> 2) * 4 * J + (row & 3)) * kRowBytes;
    const int wk = w_key<J>((row >> 2) * 4 * J + (row & 3));  // (the same for all j)
    const int x_at = S::kWBytes + (mw * 16 * T + row) * kRowBytes;
    const int xk = x_key(row);

    floatx4 acc[J][2 * T];
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
        for (int t = 0; t < 2 * T; ++t) acc[j][t] = floatx4{0.f, 0.f, 0.f, 0.f};

    bring_first(0);
    bring_second(0);
    bring_first(1);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(S::kUnderWay) : "memory");
    FSIE_TILE_FENCE();
    __builtin_amdgcn_s_barrier();
    if (wave >= 4) __builtin_amdgcn_s_barrier();  // the second group is a phase behind
    FSIE_TILE_FENCE();

    bf16x8 a[J][2], b[T][2];
    for (int step = 0; step < steps; ++step) {
        const char* stage = lds + (step & 1) * S::kStage;
        // ---- M1
        bring_second(step + 1);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int j = 0; j < J; ++j)
                a[j][h] = *reinterpret_cast<const bf16x8*>(stage + w_at + j * 4 * kRowBytes + (((h * 4 + kg) ^ wk) * 16));
#pragma unroll
            for (int t = 0; t < T; ++t)
                b[t][h] = *reinterpret_cast<const bf16x8*>(stage + x_at + t * 16 * kRowBytes + (((h * 4 + kg) ^ xk) * 16));
        }
        FSIE_TILE_FENCE();
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(S::kUnderWay) : "memory");
        __builtin_amdgcn_s_barrier();
        FSIE_TILE_FENCE();
        // ---- C1
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int j = 0; j < J; ++j) acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[j][h], b[t][h], acc[j][t], 0, 0, 0);
        __builtin_amdgcn_s_setprio(0);
        FSIE_TILE_FENCE();
        __builtin_amdgcn_s_barrier();
        FSIE_TILE_FENCE();
        // ---- M2
        bring_first(step + 2);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int t = 0; t < T; ++t)
                b[t][h] = *reinterpret_cast<const bf16x8*>(stage + x_at + S::kXHalf + t * 16 * kRowBytes + (((h * 4 + kg) ^ xk) * 16));
        FSIE_TILE_FENCE();
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(S::kUnderWay) : "memory");
        __builtin_amdgcn_s_barrier();
        FSIE_TILE_FENCE();
        // ---- C2
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int j = 0; j < J; ++j)
                    acc[j][T + t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[j][h], b[t][h], acc[j][T + t], 0, 0, 0);
        __builtin_amdgcn_s_setprio(0);
        FSIE_TILE_FENCE();
        __builtin_amdgcn_s_barrier();
        FSIE_TILE_FENCE();
    }
    if (wave < 4) __builtin_amdgcn_s_barrier();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (no load may still write LDS when the workgroup's is given away)

    // lane holds, for every tile t of 16 rows of X, the results of 4 J neighbouring rows of W from n on
    const int n = n0 + nw * 16 * J + kg * 4 * J;
#pragma unroll
    for (int t = 0; t < 2 * T; ++t) {
        const int m = m0 + mw * 32 * T + t * 16 + row;
        if (m >= M) continue;
        if (RESULT == kSums) {
            float* to = static_cast<float*>(y) + (static_cast<int64_t>(slice) * M + m) * N + n;
#pragma unroll
            for (int j = 0; j < J; ++j)
                if (n + 4 * j < N) *reinterpret_cast<floatx4*>(to + 4 * j) = acc[j][t];
        } else {
            uint32_t out[J];  // two values each, of 4 rows of W
#pragma unroll
            for (int j = 0; j < J; ++j) {
                // gate and up are rounded to 16 bits first, as the library's product leaves them for the pass that
                // multiplies them: what a token of a prompt gets does not depend on which of the two its portion takes, up to the
                // order of the float32 sums (which now and then round to neighbouring 16-bit values)
                const uint32_t a = pack2_bf16(acc[j][t][0], acc[j][t][1]), b = pack2_bf16(acc[j][t][2], acc[j][t][3]);
                out[j] = pack2_bf16(gate_pair(__uint_as_float(a << 16), __uint_as_float(a & 0xffff0000u), ACT, act_pos, act_neg),
                                    gate_pair(__uint_as_float(b << 16), __uint_as_float(b & 0xffff0000u), ACT, act_pos, act_neg));
            }
            uint32_t* to = reinterpret_cast<uint32_t*>(static_cast<bf16_t*>(y) + static_cast<int64_t>(m) * (N / 2) + n / 2);
            if constexpr (J % 4 == 0) {  // (N is a multiple of 16: 16 neighbours are all in or all out)
#pragma unroll
                for (int j = 0; j < J; j += 4)
                    if (n + 4 * j < N) *reinterpret_cast<uint4*>(to + j) = uint4{out[j], out[j + 1], out[j + 2], out[j + 3]};
            } else {
#pragma unroll
                for (int j = 0; j < J; ++j)
                    if (n + 4 * j < N) to[j] = out[j];
            }
        }
    }
}

struct Call {
    const bf16_t *x, *w;
    void* y;
    int M, N, K, splits;
    float act_pos, act_neg;
    hipStream_t stream;
};

template <int RESULT, int ACT, int T, int J>
int launch(const Call& c) {
    using S = Shape<T, J>;
    const int m_tiles = (c.M + S::kRows - 1) / S::kRows, n_tiles = (c.N + S::kCols - 1) / S::kCols;
    const unsigned groups = static_cast<unsigned>((n_tiles * c.splits + 7) / 8 * 8) * static_cast<unsigned>(m_tiles);
    static const hipError_t allowed = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_tile_kernel<RESULT, ACT, T, J>),
                                                          hipFuncAttributeMaxDynamicSharedMemorySize, 2 * S::kStage);
    FSIE_REQUIRE(allowed == hipSuccess, "gemm_mfma_tile: %d bytes of LDS: %s", 2 * S::kStage, hipGetErrorString(allowed));
    gemm_tile_kernel<RESULT, ACT, T, J><<<groups, 512, 2 * S::kStage, c.stream>>>(c.x, c.w, c.y, c.M, c.N, c.K, m_tiles, n_tiles,
                                                                                 c.splits, c.act_pos, c.act_neg);
    FSIE_CHECK_LAUNCH("gemm_mfma_tile");
    return 0;
}

template <int RESULT, int ACT>
int launch_shape(int tile, const Call& c) {
    switch (tile) {
        case 0: return launch<RESULT, ACT, 2, 4>(c);
        case 1: return launch<RESULT, ACT, 4, 3>(c);
        case 2: return launch<RESULT, ACT, 4, 4>(c);
        default: return launch<RESULT, ACT, 4, 5>(c);
    }
}

}  // namespace

// Which tile, and how many slices of K, a product of M rows should take; -1: the library's product (and the pass that
// follows it) is faster, or the sizes are not the kernel's.  Returns tile + 256 * slices.
//
// The rule is the time that a count of rounds gives: workgroups (one a compute unit) in rounds over the units of a die, which
// gets every eighth column of tiles with all of its tiles of X (20 columns of 12 tiles are 36 workgroups for the 32 units of four
// of the dies: two rounds, not one), a step of
// 64 values of K in 0.90, 1.10, 1.38 and 1.78 us for the tiles of 128 x 256, 256 x 192, 256 x 256 and 256 x 320, and 8 us
// a round for filling the stages and writing the result (each within 8 % of what 11 numbers of rows from 144 to 4,096 took
// at N x K = 37888 x 3584, 27648 x 5120, 28672 x 4096, 16384 x 2048 and 9728 x 896).
// Gate and up: against the library's product at 1.2 PFLOP/s (or its weights at 5.5 TB/s) and 8 us, and the pass that
// multiplies gate and up (3 bytes an output of the product at 4.8 TB/s, and 3 us): the two together took 554 us at 2,048 x
// 37888 x 3584 where this kernel takes 423, 316 / 213 at 978 rows, 149 / 108 at 512; 121 / 106 at 2,048 x 16384 x 2048; but
// 48 / 63 at 144 x 28672 x 4096, 25 / 32 at 144 x 16384 x 2048, where the tiles do not fill the chip.  Over 14 matrices and 18
// numbers of rows from 129 to 4,096 the choice takes 0.89 of the library's time, and at none more than 1.03.
// Partial sums: the library has to cut a long K as well and does it badly.  With the norm that follows, library / this kernel, us:
// 378 / 243 at 2,048 x 3584 x 18944, 281 / 197 at 1,500 rows, 204 / 81 at 512, 106 / 51 at 129; 288 / 140 at 512 x 5120 x
// 27648.  At K = 14336 and below it is the faster one (208 / 226 at 2,048 x 4096 x 14336), and at K = 16384 from some 32 tiles of
// 256 x 256 on (2,048 x 2048 136 / 145, 4,096 x 1024 133 / 152; 1,024 x 2048 97 / 86).  Up to half as many tiles as units
// this kernel is the faster one (K = 18944 to 28672, N = 1536 to 8192, 576 to 5,000 rows: 0.4 to 0.9 of the library's time, 1.03 once).
// Beyond, the library fills the chip by itself and runs at 1.2 to 1.45 PFLOP/s at most numbers of rows: only a plan of one round
// is as fast (2,560 x 3584 x 18944 in two slices 280, 542; 2,048 x 5120 x 27648 412 / 455), not one of two (2,816 x 3584 x 18944
// 362 / 310, 2,560 x 4096 339 / 309, 2,816 x 4096 419 / 348, 2,304 x 5120 x 27648 547 / 504; where the library's choice is a slow
// one, two rounds would still gain: 3,072 x 3584 373 / 573), and from three quarters as many tiles as units on only in one slice that
// promises 1.25 (4,096 x 3584 x 18944 446 / 563; 3,840 x 4096 440 / 410).
// The sums' own bytes, written here and read by the norm, count at 4.5 TB/s.
extern "C" int fsie_gemm_mfma_tile_plan(int M, int N, int K, int result, int units) {
    if (M <= 0 || N <= 0 || K <= 0 || units <= 0 || N % 16 || K % kStep || (result != kPair && result != kSums)) return -1;
    if (static_cast<int64_t>(M) * K * 2 >= (int64_t{1} << 31) || static_cast<int64_t>(N) * K * 2 >= (int64_t{1} << 31)) return -1;
    const int rows[4] = {128, 256, 256, 256}, cols[4] = {256, 192, 256, 320};
    const double us_a_step[4] = {0.90, 1.10, 1.38, 1.78};
    const int64_t steps = K / kStep;
    const int64_t tiles = ceil_div64(M, 256) * ceil_div64(N, 256);
    if (result == kSums && (K < 16384 || tiles >= units || (K < 17408 && tiles > 32))) return -1;
    const bool one_round = result == kSums && 2 * tiles > units;
    double best = 1e30;
    int choice = -1;
    for (int tile = 0; tile < 4; ++tile) {
        for (int slices = 1; slices <= (result == kSums ? 16 : 1); ++slices) {
            const int64_t columns = ceil_div64(ceil_div64(N, cols[tile]) * slices, 8);  // of a die
            const int64_t rounds = ceil_div64(columns * ceil_div64(M, rows[tile]), ceil_div64(units, 8));
            if (one_round && rounds > 1) continue;
            double us = static_cast<double>(rounds) * (static_cast<double>(ceil_div64(steps, slices)) * us_a_step[tile] + 8.0);
            if (result == kSums) us += 8.0 * slices * M * static_cast<double>(N) / 4.5e6;
            if (us < best) {
                best = us;
                choice = tile + 256 * slices;
            }
        }
    }
    const double flops = 2.0 * M * static_cast<double>(N) * K;
    if (choice < 0 || (one_round && flops / best < (choice / 256 > 1 ? 1.05e9 : 1.25e9))) return -1;
    if (result == kSums && 4 * tiles >= 3 * static_cast<int64_t>(units) && choice / 256 > 1) return -1;
    if (result == kPair) {
        const double weights = 2.0 * N * static_cast<double>(K);
        const double product = flops / 1.2e9 > weights / 5.5e6 ? flops / 1.2e9 : weights / 5.5e6;
        if (best > product + 8.0 + 3.0 * M * static_cast<double>(N) / 4.8e6 + 3.0) return -1;
    }
    return choice;
}

extern "C" int fsie_gemm_mfma_tile(const void* x, const void* w, void* y, int M, int N, int K, int result, int splits,
                                   int tile, int act, float act_pos, float act_neg, hipStream_t stream) {
    FSIE_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm_mfma_tile: bad sizes M=%d N=%d K=%d", M, N, K);
    FSIE_REQUIRE(N % 16 == 0 && K % kStep == 0, "gemm_mfma_tile: N=%d must be a multiple of 16, K=%d of %d", N, K, kStep);
    FSIE_REQUIRE(result == kPair || result == kSums, "gemm_mfma_tile: unknown result %d", result);
    FSIE_REQUIRE(splits >= 1 && splits <= K / kStep && (splits == 1 || result == kSums), "gemm_mfma_tile: %d slices", splits);
    FSIE_REQUIRE(tile >= 0 && tile <= 3, "gemm_mfma_tile: unknown tile %d", tile);
    FSIE_REQUIRE(result != kPair || FSIE_PAIR_KNOWN(act), "gemm_mfma_tile: unknown activation %d", act);
    FSIE_REQUIRE(static_cast<int64_t>(M) * K * 2 < (int64_t{1} << 31) && static_cast<int64_t>(N) * K * 2 < (int64_t{1} << 31),
                 "gemm_mfma_tile: operands of %d x %d and %d x %d are more than the kernel's 32-bit offsets take", M, K, N, K);
    FSIE_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(y) % 16 == 0, "gemm_mfma_tile: operands must be 16-byte aligned");
    if (M == 0) return 0;
    const Call c{static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(w), y, M, N, K, splits, act_pos, act_neg, stream};
    if (result == kSums) return launch_shape<kSums, 0>(tile, c);
    switch (act) {
        case FSIE_ACT_SILU: return launch_shape<kPair, FSIE_ACT_SILU>(tile, c);
        case FSIE_ACT_GELU_TANH: return launch_shape<kPair, FSIE_ACT_GELU_TANH>(tile, c);
        case FSIE_ACT_RELU: return launch_shape<kPair, FSIE_ACT_RELU>(tile, c);
        default: return launch_shape<kPair, FSIE_PAIR_CLIPPED>(tile, c);
    }
}
