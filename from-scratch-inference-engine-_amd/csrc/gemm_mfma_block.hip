// Y[M, N] = X[M, K] . W[N, K]^T of some twenty to some thousand rows where the tiles of gemm_mfma_tile.hip would leave most of the chip idle: matrices
// of one to some ten MB, a step's portion of a prompt at a time.  bfloat16 operands in rows, on the matrix cores; the result in
// bfloat16 with the bias added before the one rounding, or float32 partial sums of slices of K for the norm that adds them up.
//
// A workgroup of four waves makes a tile of 64 x 64, 64 x 128 or 128 x 128 rows of X and W, a wave a quarter of it.  Both operands go
// through LDS, 64 values of K at a time, straight from memory, in three stages: one is read, one has arrived or is about to, one is
// asked for behind the barrier that says that every wave has read it.  One barrier a step.
// What bounds it: how much a unit can have under way, and where W lies.  Weights are read once a pass and come from HBM, 1.4 us away; the
// loads of a unit return in order, so that the tiles took 0.34, 0.41 and 0.55 us a step where weights in the caches took 0.24, 0.30 and 0.36.
// So a workgroup first asks for its share of the W that the workgroups of its die will read (see below): at 1,375 rows, cold weights, N = 1152,
// K = 896 took 8.7 us without and takes 7.5, 1,000 rows of N = K = 3584 35.2 and 30.4, 1,375 of N = K = 2048 20.7 and 17.0.  Where all tiles of
// 64 x 64 are on the chip at once six stages fit: 512 rows of N = 1024, K = 4096 15.0 us instead of 18.6, 512 of N = K = 2048 9.7 as with three.
// A step of 128 x 128 took 0.53 us with its loads, its reads of LDS and its products each in a row, and takes 0.36 with them in turns.
// Without gain: more stages for the larger tiles, two stages and twice the workgroups a unit, other permutations in LDS, two steps' lines of a row
// asked for together; a fifth wave that asks for W along the way (it holds up the other four's loads).
// The library's product takes 11.3 us of the first size above, 36.9 and 21.7 of the others; a call of the library's is 21 us of the host besides,
// one of this 13.
#include "common.h"
#include "api.h"
#include "lds_loads.h"

namespace {

using namespace fsie_lds;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kStep = 64;  // values of K a stage
constexpr int kRowBytes = kStep * 2;

constexpr int kTouched = FSIE_WAVE * 4;  // a wave's values of lines that it only asks for

enum Result { kPlain = 0, kSums = 1 };  // bfloat16 [M, N] with a bias; float32 [splits, M, N]

// A tile: 32 T rows of X by 32 J rows of W, a wave of four a quarter of it.
template <int T, int J, int STAGES>
struct Shape {
    static constexpr int kRows = 32 * T, kCols = 32 * J;
    static constexpr int kStage = (kRows + kCols) * kRowBytes;  // W, then X
    static constexpr int kLoads = T + J;                        // a wave's, of eight rows each: J of W, T of X
    static constexpr int kStages = STAGES;
    static constexpr int kLds = kStages * kStage + 4 * kTouched;
};

#define FSIE_BLOCK_FENCE() __builtin_amdgcn_sched_barrier(0)

// The permutation of a row's eight 16-byte units in LDS: W's rows are read 16 at a time as 4 runs of 4 that lie 4 J apart, X's as 16
// neighbours; in both any eight lanes in a row meet eight different units.
template <int J>
__device__ __forceinline__ int w_key(int row) { return (row >> 1 & 1) | (row % (16 * J) / (4 * J)) << 1; }
__device__ __forceinline__ int x_key(int row) { return row >> 1 & 7; }

template <int RESULT, int T, int J, int STAGES>
__global__ __launch_bounds__(256, 1) void gemm_block_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                            const float* __restrict__ bias, void* __restrict__ y, int M, int N, int K,
                                                            int m_tiles, int n_tiles, int splits) {
    using S = Shape<T, J, STAGES>;
    extern __shared__ char lds[];
    // a die (the workgroup's number modulo 8) takes neighbouring tiles: of W its own eighth, of X all
    const int tiles = m_tiles * n_tiles * splits, a_die = (tiles + 7) / 8;
    const int id = static_cast<int>(blockIdx.x & 7) * a_die + static_cast<int>(blockIdx.x >> 3);
    if (id >= tiles) return;
    const int m_tile = id % m_tiles, n_tile = id / m_tiles % n_tiles, slice = id / m_tiles / n_tiles;
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
    const auto next_stage = [](uint32_t at) { return at == (S::kStages - 1) * S::kStage ? 0u : at + S::kStage; };
    const auto k_of = [&](int step) { return static_cast<uint32_t>(first_step + min(step, steps - 1)) * kRowBytes; };
    const auto load = [&](int i, uint32_t k) {  // the i-th of this wave's loads of a stage
        if (i < J) load_to_lds(w_rows, lds0 + bring_to + (wave * J + i) * 1024u, w_from[i], k);
        else load_to_lds(x_rows, lds0 + bring_to + S::kCols * kRowBytes + (wave * T + i - J) * 1024u, x_from[i - J], k);
    };

    // What of W the stages at the start leave is asked for at once, a value a line, and goes nowhere: the workgroups of this tile of W and
    // slice, on one die but for few, share its steps.  From HBM a line is 1.4 us away, and three stages would wait for it at every step.
    if (m_tiles > 2) {
        for (int step = S::kStages + 4 * m_tile + wave; step < steps; step += 4 * m_tiles) {
#pragma unroll
            for (int c = 0; c < S::kCols / FSIE_WAVE; ++c)
                touch(w_rows, lds0 + S::kStages * S::kStage + wave * kTouched,
                      static_cast<uint32_t>(min(n0 + c * FSIE_WAVE + lane, N - 1)) * static_cast<uint32_t>(K) * 2u, k_of(step));
        }
    }

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

    bf16x8 a[2][J][2], b[2][T][2];  // this step's fragments and the next one's
    const auto read = [&](int i, bf16x8 (&to_a)[J][2], bf16x8 (&to_b)[T][2]) {  // the i-th of a stage's 2 (J + T) fragments
        const char* stage = lds + read_from;
        const int h = i / (J + T), f = i % (J + T);
        if (f < J) to_a[f][h] = *reinterpret_cast<const bf16x8*>(stage + w_at + f * 4 * kRowBytes + (((h * 4 + kg) ^ wk) * 16));
        else to_b[f - J][h] = *reinterpret_cast<const bf16x8*>(stage + x_at + (f - J) * 16 * kRowBytes + (((h * 4 + kg) ^ xk) * 16));
    };
    // A step: the next stage has arrived (all loads but the youngest stage's) and this step's fragments are in every wave's registers,
    // so its stage is free for the one after the next two.  A load, two fragments of the next step and this step's products go in
    // turns: eight loads in a row are waited for in the units' address queue as long as the products take, and reads in a row in the LDS's.
    const auto go = [&](int step, const bf16x8 (&fa)[J][2], const bf16x8 (&fb)[T][2], bf16x8 (&next_a)[J][2], bf16x8 (&next_b)[T][2]) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((S::kStages - 2) * S::kLoads) : "memory");
        FSIE_BLOCK_FENCE();
        __builtin_amdgcn_s_barrier();
        FSIE_BLOCK_FENCE();
        const uint32_t k = k_of(step + S::kStages);
#pragma unroll
        for (int c = 0; c < J + T; ++c) {
            constexpr int kProducts = 2 * J * T;
#pragma unroll
            for (int q = c * kProducts / (J + T); q < (c + 1) * kProducts / (J + T); ++q) {
                const int h = q / (J * T), t = q / J % T, j = q % J;
                acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[j][h], fb[t][h], acc[j][t], 0, 0, 0);
            }
            read(2 * c, next_a, next_b);
            read(2 * c + 1, next_a, next_b);
            load(c, k);
            FSIE_BLOCK_FENCE();
        }
        bring_to = next_stage(bring_to);
        read_from = next_stage(read_from);
    };
#pragma unroll
    for (int i = 0; i < S::kStages; ++i) {
        const uint32_t k = k_of(i);
#pragma unroll
        for (int c = 0; c < J + T; ++c) load(c, k);
        bring_to = next_stage(bring_to);
    }
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S::kStages - 1) * S::kLoads) : "memory");
    FSIE_BLOCK_FENCE();
    __builtin_amdgcn_s_barrier();
    FSIE_BLOCK_FENCE();
#pragma unroll
    for (int i = 0; i < 2 * (J + T); ++i) read(i, a[0], b[0]);
    read_from = next_stage(read_from);
    for (int step = 0; step < steps; step += 2) {
        go(step, a[0], b[0], a[1], b[1]);
        if (step + 1 >= steps) break;
        go(step + 1, a[1], b[1], a[0], b[0]);
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

template <int RESULT, int T, int J, int STAGES>
int launch(const Call& c) {
    using S = Shape<T, J, STAGES>;
    const int m_tiles = (c.M + S::kRows - 1) / S::kRows, n_tiles = (c.N + S::kCols - 1) / S::kCols;
    const unsigned groups = static_cast<unsigned>((m_tiles * n_tiles * c.splits + 7) / 8 * 8);
    static const hipError_t allowed = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_block_kernel<RESULT, T, J, STAGES>),
                                                          hipFuncAttributeMaxDynamicSharedMemorySize, S::kLds);
    FSIE_REQUIRE(allowed == hipSuccess, "gemm_mfma_block: %d bytes of LDS: %s", S::kLds, hipGetErrorString(allowed));
    gemm_block_kernel<RESULT, T, J, STAGES><<<groups, 256, S::kLds, c.stream>>>(c.x, c.w, c.bias, c.y, c.M, c.N, c.K, m_tiles, n_tiles,
                                                                                   c.splits);
    FSIE_CHECK_LAUNCH("gemm_mfma_block");
    return 0;
}

template <int RESULT>
int launch_shape(int tile, const Call& c) {
    switch (tile) {
        case 0: return launch<RESULT, 2, 2, 3>(c);
        case 1: return launch<RESULT, 2, 4, 3>(c);
        case 2: return launch<RESULT, 4, 4, 3>(c);
        default: return launch<RESULT, 2, 2, 6>(c);
    }
}

}  // namespace

// Which tile, and in how many slices of K, M rows of this product are best taken; -1: the library's product is faster or the sizes are not
// the kernel's.  Returns tile + 256 * slices.
// The rule is the time that a count of steps gives: fixed + steps * a step's, workgroups that share a unit taking turns (so many as the unit's LDS
// holds; a second round of 128 x 128 was up to 1.36 of the library's time and is not taken), the weights from HBM at 6.7 to 9 TB/s more; no less than the
// eight dies' reads of x take; a whole product's bytes or the slices' sums here and in the norm at 3 TB/s.  It has to be no more than the library's 8.3 us, 1.64 PFLOP/s,
// weights at 3 TB/s and x at 2.2, the best fit of what it took with weights from HBM (slices: 0.95 of that and the norm's reading).
// Measured with weights from HBM at 2,241 sizes that it takes, 17 to 4,096 rows of 0.02 to 53 MB for the most part, it is at a median of 0.7 of the library's time; 56 are beyond 1.02,
// of which 100 rows of N = K = 4096 1.10, 385 of N = 6144, K = 4096 1.17, 1,009 of N = 160, K = 3072 1.21 (this / the library, us: 17 rows of
// N = K = 768 5.1 / 5.0, 64 of them 5.2 / 7.0, 64 of N = 512, K = 896 5.0 / 7.7, 1,375 of N = 1152,
// K = 896 7.5 / 11.3, 512 of N = 4608, K = 3584 28.9 / 33.3, 1,000 of N = K = 3584 30.4 / 36.9, 2,048 of N = 2048, K = 8192 67.7 / 75.5, 256 of N = 3072, K = 1024 6.9 / 11.9; with
// the norm, 96 rows of N = 896, K = 4864 in seven slices 9.2 / 15.4, 96 of N = 2048, K = 8192 in four 16.3 / 24.0).  What it leaves out besides:
// - beyond kBeyond, where the estimate tells nothing (129 rows of N = K = 8192 66.6 / 46.4, 384 79.9 / 62.1), all but slices
//   of a K no shorter than N for up to 512 rows (N = 4096, K = 14336 0.44 to 0.79 of the library's time, 0.95 to 1.06 from 300 rows on; N = 5120, K = 13824 0.49 to 0.97 and 1.06) and, from 129
//   rows on, tiles of 128 x 128 that leave few units idle, K up to 8192, 6144 beyond 256 rows (N = 16384, K = 5120 0.90 to 1.01, N = 14336, K = 8192 0.87 to 1.04): 74 sizes,
//   median 0.90, at most 1.06 (of 53 to 80 MB 170 sizes, median 0.93, 41 beyond 1.02, at most 1.25, 129 rows of N = 8192, K = 4096);
// - slices of more than 8,192 rows of W (65 rows of N = 10240, K = 2048 and the norm 59.9 / 50.3).
// 129 to 159 rows of N above 6,400 to 10,240 and K from 2048, where the library is at its best and a third of these tiles' rows are none, are taken all the same
// (N = 8192, K = 2048 18.3 / 15.9, N = 10240 19.9 / 17.7, N = 7168, K = 3072 24.2 / 22.1; with K = 1536 or N = 6144 0.72): such portions of a prompt are bound by the
// host, for which the library's call is 21 us and the bias behind it a launch more, this one 13 (Romepel, 9 layers, prompts of 129 to 159 tokens 1.29 ms, 1.43 so).
// Of matrices of 8 to 40 MB and 320 to 2,600 rows the fit is some fifth too good to the library, whose choice of a kernel goes by other things than the time
// counted here: up to 1.3 of it is taken (K to 6 N), in slices up to 1.1 where the fit has no whole product that is as fast.  4,295 sizes from the library to
// these tiles, weights from HBM: whole 0.82 of its time, with the norm 0.84, slices with the norm 0.80; 107 beyond 1.02, 37 beyond 1.05, at most 1.17 (525 rows of
// N = 912, K = 5120 19.2 / 16.4).  1,375 rows of N = 896, K = 4864 and the norm 27.7 / 32.1, 513 of N = 2048, K = 8192 39.6 / 47.2, 1,025 of N = K = 2048 21.8 / 24.9, 640 of
// N = K = 3584 33.8 / 37.8.  200 to 320 rows are the library's at up to 1.4 (251 of N = 880, K = 4608 15.6 / 11.0), and so are a longer K (1,895 of N = 1088, K = 11008 92.5 / 75.5).
// The dies' reads of x: 1,845 rows of N = 512, K = 6656 33.7 / 29.4, 2,284 of N = 432, K = 11776 57.6 / 49.6, which the steps alone put at 22.8 and 37.7.
constexpr double kBeyond = 80e6;   // bytes of weights
constexpr double kDiesRead = 6.5e6;  // bytes a us of x by all dies

extern "C" int fsie_gemm_mfma_block_plan(int M, int N, int K, int result, int units) {
    if (M <= 0 || N <= 0 || K <= 0 || units <= 0 || N % 16 || K % kStep || (result != kPlain && result != kSums)) return -1;
    if (static_cast<int64_t>(M) * K * 2 >= (int64_t{1} << 31) || static_cast<int64_t>(N) * K * 2 >= (int64_t{1} << 31)) return -1;
    const int rows[4] = {64, 64, 128, 64}, cols[4] = {64, 128, 128, 64}, at_once[4] = {3, 2, 1, 1};
    const double us_a_step[4] = {0.228, 0.295, 0.405, 0.182}, fixed[4] = {2.5, 3.2, 4.2, 3.1}, us_a_mb[4] = {0.15, 0.15, 0.13, 0.11};
    const double turns[4][4] = {{0, 1, 1.55, 2.6}, {0, 1, 1.9}, {0, 1}, {0, 1}};  // workgroups on a unit: a step's time of one alone
    const int64_t steps = K / kStep;
    const double weights = 2.0 * N * static_cast<double>(K), flops = 2.0 * M * static_cast<double>(N) * K;
    const double rows_bytes = 2.0 * M * static_cast<double>(K);
    const bool large = weights > kBeyond;
    if (large && (result == kSums ? M > 512 || K < N : M <= 128 || K > (M <= 256 ? 8192 : 6144))) return -1;
    if (result == kSums && N > 8192) return -1;
    const double whole = 4.0 * M * static_cast<double>(N) / 3e6;  // the delta in bfloat16, out and into the norm
    double best = 1e30, best_plain = 1e30;
    int choice = -1;
    bool fills = false;  // (nearly all units)
    for (int tile = 0; tile < 4; ++tile) {
        for (int slices = 1; slices <= (result == kSums ? 8 : 1); ++slices) {
            if (slices > 1 && steps / slices < 4) break;
            const int64_t m_tiles = ceil_div64(M, rows[tile]), n_tiles = ceil_div64(N, cols[tile]), groups = m_tiles * n_tiles * slices;
            const int64_t deep = ceil_div64(groups, units), a_die = ceil_div64(groups, 8);
            if (deep > at_once[tile]) continue;
            double us = fixed[tile] + static_cast<double>(ceil_div64(steps, slices)) * us_a_step[tile] * turns[tile][deep] + weights * 1e-6 * us_a_mb[tile];
            // (of one slice's x a die reads the rows of its tiles, of a second one where its tiles go on into that)
            const double of_slice = a_die < m_tiles ? static_cast<double>(a_die) / m_tiles : 1.0, slices_read = static_cast<double>(a_die) / (m_tiles * n_tiles);
            const double share = (of_slice > slices_read ? of_slice : slices_read) / slices, read = 8.0 * rows_bytes * (share < 1.0 ? share : 1.0) / kDiesRead;
            if (us < read) us = read;
            if (slices == 1 && us < best_plain) best_plain = us;
            if (result == kSums) us += (slices == 1 ? whole : 2.0 * slices * whole);
            if (us < best) {
                best = us;
                choice = tile + 256 * slices;
                fills = 8 * groups >= 7 * units;
            }
        }
    }
    const double library = 8.3 + flops / 1.64e9 + weights / 3e6 + rows_bytes / 2.2e6;
    if (large && result == kPlain && (choice % 256 != 2 || !fills)) return -1;
    if (choice < 0) return -1;
    const bool middle = weights >= 8e6 && weights <= 40e6 && M >= 320 && M <= 2600 && N >= 800;
    if (result == kSums)
        return best <= 0.95 * (library + whole) ||
                       (middle && (N <= 2560 || M >= 500) && best <= 1.1 * (library + whole) && best_plain > library) ? choice : -1;
    return best <= (middle && K <= 6 * static_cast<int64_t>(N) ? 1.3 : 1.0) * library ? choice : -1;
}

extern "C" int fsie_gemm_mfma_block(const void* x, const void* w, const float* bias, void* y, int M, int N, int K, int result, int splits,
                                    int tile, hipStream_t stream) {
    FSIE_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm_mfma_block: bad sizes M=%d N=%d K=%d", M, N, K);
    FSIE_REQUIRE(N % 16 == 0 && K % kStep == 0, "gemm_mfma_block: N=%d must be a multiple of 16, K=%d of %d", N, K, kStep);
    FSIE_REQUIRE(result == kPlain || result == kSums, "gemm_mfma_block: unknown result %d", result);
    FSIE_REQUIRE(splits >= 1 && splits <= K / kStep && (splits == 1 || result == kSums), "gemm_mfma_block: %d slices", splits);
    FSIE_REQUIRE(!bias || result == kPlain, "gemm_mfma_block: partial sums take no bias");
    FSIE_REQUIRE(tile >= 0 && tile <= 3, "gemm_mfma_block: unknown tile %d", tile);
    FSIE_REQUIRE(static_cast<int64_t>(M) * K * 2 < (int64_t{1} << 31) && static_cast<int64_t>(N) * K * 2 < (int64_t{1} << 31),
                 "gemm_mfma_block: operands of %d x %d and %d x %d are more than the kernel's 32-bit offsets take", M, K, N, K);
    FSIE_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(y) % 16 == 0 && reinterpret_cast<uintptr_t>(bias) % 16 == 0,
                 "gemm_mfma_block: operands must be 16-byte aligned");
    if (M == 0) return 0;
    const Call c{static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(w), bias, y, M, N, K, splits, stream};
    return result == kSums ? launch_shape<kSums>(tile, c) : launch_shape<kPlain>(tile, c);
}
