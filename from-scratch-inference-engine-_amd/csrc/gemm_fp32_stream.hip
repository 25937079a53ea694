// Y[M, N] = X[M, K] . W[N, K]^T (+ bias) in true float32 for up to 64 rows of X, from a copy of W in the order of the matrix instruction's
// operands (fsie_fragment_order on the matrix as 2 K columns of 16 bits: 16 rows and 16 values of K lie together, 1 KB, in the order of the lanes).
//
// The product of few rows that reads rows of W (gemm_mfma_fp32.hip) asks for four steps of 16 values of K a wave, 16 pieces of 64 bytes each,
// waits, multiplies, and asks again: K = 896 in two waves is seven trips to memory, one after the other.  Here a load is one piece of 1 KB
// by streaming loads, and a workgroup's waves, eight or sixteen for its 16 rows of W, deal the steps among themselves, so that a wave has all of its up to
// eight steps under way at once: one trip.  A longer K goes four steps at a time with the next four under way.  The waves' shares meet in LDS and are
// added in the order of the waves; a share is at most eight steps, 128 values, before it is added to the ones behind it, which leaves half the rounding
// errors of runs of 512 (relative error of K = 896 3.9e-7 -> 2.0e-7, K = 4864 in eight slices 2.2e-7 -> 1.7e-7).
// As there a row's sums depend on N, K, the number of tiles of 16 rows and whether the step has one or two rows (the plan below), never on what the other rows hold.
//
// MI355X, us, cold weights, rows of W before / this, 4 rows: gate and up with their product N = 9728, K = 896 (35 MB) 11.2 / 9.2, N = 16384, K = 2048 39.3 / 26.2,
// N = 37888, K = 3584 104 / 91; sums with the norm that adds them up N = 896, K = 4864 9.3 / 7.6, N = 896, K = 896 5.7 / 5.0, N = 2048, K = 8192 22.8 / 15.9,
// N = 3584, K = 18944 55.7 / 49.9; whole N = 1152, K = 896 5.1 / 4.2, N = 6208, K = 2048 16.4 / 12.8, N = 151936, K = 896 111 / 83.  One row, against the vector
// kernel: 10.1 / 9.3 and 12.8 / 5.4 of the first and fourth size, 89 / 80 of the last.  32 rows 20.4 / 17.2 and 14.9 / 11.6; 64 rows, where the matrix
// instruction (a quarter of the rate of half the rows) is the bound, 20.0 / 18.3 of the fourth.
#include "common.h"
#include "api.h"

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(1))) u32x4* GlobalVec;

constexpr int kStep = 16;          // values of K a step: 1 KB of 16 rows of W
constexpr int kMostSteps = 8;      // of a wave, all under way at once
constexpr int kTogether = 4;       // beyond: so many at a time, and the next as many under way

// float32 [slices][M, N] with a bias (one slice); float32 [M, N / 2] of gate and up rows in turn
enum Result { PLAIN = 0, GATED = 1 };

struct StreamCall {
    const float *x, *w, *bias;
    float* y;
    int M, N, K, slice_steps, slices, act;
    float limit, slope;
};

// MT tiles of 16 rows of X; WAVES waves deal the steps of slice blockIdx.y among themselves, `S` consecutive ones each (LONG: any number, S at
// a time), for block blockIdx.x of 16 rows of W.  A step past the end reads the last one of K again and is not multiplied.
template <int MT, int WAVES, int S, bool LONG, int RESULT>
__global__ __launch_bounds__(WAVES * 64) void gemm_fp32_stream_kernel(const float* x, const float* w, float* y, int M, int N, int K, int slice_steps,
                                                                      const float* bias, int act, float limit, float slope) {
    __shared__ floatx4 red[WAVES * MT * 64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = lane & 15, kg = lane >> 4;  // row of the A tile (n) and column of the B tile (m); which 4 of a step's 16 values
    const int steps = K / kStep, slice = blockIdx.y;
    const int run = LONG ? (slice_steps + WAVES - 1) / WAVES : S;
    const int first = slice * slice_steps + wave * run;
    const int end = min(min(steps, (slice + 1) * slice_steps), first + run);  // may be `first` or less: the same for the whole wave
    // (rows of x that are not there: past the buffer's end, zeros, and no request)
    const __amdgpu_buffer_rsrc_t x_rows = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(x), 0, M * K * 4, 0x00020000);
    struct Set {
        u32x4 a[S], b[S][MT];
    };
    auto load = [&](Set& v, int at) {
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int k = min(at + s, steps - 1);
#pragma unroll
            for (int t = 0; t < MT; ++t) v.b[s][t] = __builtin_amdgcn_raw_buffer_load_b128(x_rows, ((t * 16 + row) * K + k * kStep + kg * 4) * 4, 0, 0);
        }
#pragma unroll
        for (int s = 0; s < S; ++s)
            v.a[s] = __builtin_nontemporal_load((GlobalVec)(w + (static_cast<int64_t>(blockIdx.x) * steps + min(at + s, steps - 1)) * 256 + lane * 4));
    };
    floatx4 acc[MT], total[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = total[t] = floatx4{0.f, 0.f, 0.f, 0.f};
    auto products = [&](const Set& v, int at) {
#pragma unroll
        for (int s = 0; s < S; ++s) {
            if (at + s < end) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int t = 0; t < MT; ++t)
                        acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(v.a[s][j]), __uint_as_float(v.b[s][t][j]), acc[t], 0, 0, 0);
            }
        }
    };
    if constexpr (LONG) {
        Set even, odd;
        load(even, first);
        for (int at = first; at < end; at += 2 * S) {
            load(odd, at + S);
            products(even, at);
            load(even, at + 2 * S);
            products(odd, at + S);
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                total[t] += acc[t];
                acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
            }
        }
    } else {
        Set all;
        load(all, first);
        products(all, first);
#pragma unroll
        for (int t = 0; t < MT; ++t) total[t] = acc[t];
    }
#pragma unroll
    for (int t = 0; t < MT; ++t) red[(wave * MT + t) * 64 + lane] = total[t];
    __syncthreads();
    if (wave >= MT) return;
    floatx4 sum = red[wave * 64 + lane];
#pragma unroll
    for (int i = 1; i < WAVES; ++i) sum += red[(i * MT + wave) * 64 + lane];
    // lane holds D[n + r][m]
    const int n = blockIdx.x * 16 + kg * 4, m = wave * 16 + row;
    if (m >= M) return;
    if constexpr (RESULT == GATED) {  // rows n .. n + 3: gate, up, gate, up (N is even)
#pragma unroll
        for (int r = 0; r < 4; r += 2)
            if (n + r < N) y[static_cast<int64_t>(m) * (N / 2) + (n + r) / 2] = gate_pair(sum[r], sum[r + 1], act, limit, slope);
    } else {
        float* out = y + (static_cast<int64_t>(slice) * M + m) * N + n;
        if (N % 4 == 0) {  // (four neighbours are all in or all out)
            if (n >= N) return;
            if (bias) sum += floatx4{bias[n], bias[n + 1], bias[n + 2], bias[n + 3]};
            *reinterpret_cast<floatx4*>(out) = sum;
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (n + r < N) out[r] = bias ? sum[r] + bias[n + r] : sum[r];
        }
    }
}

template <int MT, int WAVES, int S, bool LONG, int RESULT>
int launch(const StreamCall& c, hipStream_t stream) {
    gemm_fp32_stream_kernel<MT, WAVES, S, LONG, RESULT><<<dim3((c.N + 15) / 16, c.slices), WAVES * 64, 0, stream>>>(
        c.x, c.w, c.y, c.M, c.N, c.K, c.slice_steps, c.bias, c.act, c.limit, c.slope);
    FSIE_CHECK_LAUNCH("gemm_fp32_stream");
    return 0;
}

// LEAST: steps a wave; fewer are taken as so many
template <int MT, int WAVES, int LEAST, int RESULT>
int launch_steps(int s, const StreamCall& c, hipStream_t stream) {
    if constexpr (LEAST < kMostSteps)
        if (s > LEAST) return launch_steps<MT, WAVES, LEAST + 1, RESULT>(s, c, stream);
    return launch<MT, WAVES, LEAST, false, RESULT>(c, stream);
}

template <int MT, int RESULT>
int launch_waves(int waves, int s, const StreamCall& c, hipStream_t stream) {
    if (waves == 4) return launch<MT, 4, kTogether, true, RESULT>(c, stream);
    if (waves == 8) return s <= kMostSteps ? launch_steps<MT, 8, 2, RESULT>(s, c, stream) : launch<MT, 8, kTogether, true, RESULT>(c, stream);
    // (sixteen waves leave a lane 128 registers: two tiles of X)
    if constexpr (MT <= 2) return s <= kMostSteps ? launch_steps<MT, 16, 5, RESULT>(s, c, stream) : launch<MT, 16, kTogether, true, RESULT>(c, stream);
    fsie_set_error("gemm_fp32_stream: sixteen waves take up to 32 rows");
    return 1;
}

template <int MT>
int launch_result(bool gated, int waves, int s, const StreamCall& c, hipStream_t stream) {
    return gated ? launch_waves<MT, GATED>(waves, s, c, stream) : launch_waves<MT, PLAIN>(waves, s, c, stream);
}

}  // namespace

// How M rows of this product are best taken, or -1 where the kernels that read rows of W are the better ones: waves + 256 * slices of K.  By N, K,
// the tiles of 16 rows, and of one or two rows whether the vector kernel is the better one.  result 0: whole; 1: gate and up in turn; 2: partial sums for a norm that adds them up, or whole (one slice).
// Whole: eight waves where they hold K at once (K up to 1,024), else sixteen where the units have no workgroup each (N = 3072, K = 1536 6.0 us, with four 6.5;
// N = 4096, K = 2048 8.1 / 8.3), else four, of which a unit holds several (N = 16384, K = 2048 26.2, with 16 27.8; N = 37888, K = 3584 91 / 118;
// N = 3584, K = 3584 11.5 / 13.0).  From 33 rows on the matrix instruction bounds a short K and this is no faster (N = 9728, K = 896 25.8 / 24.7 at 48
// rows, 31.8 / 30.8 at 64; K = 2048 22.0 / 25.3).  One and two rows of some workgroups more than the units, which leave them an uneven second round, stay
// with the vector kernel (one row of N = 4608, K = 3584 17.6 / 14.4; N = 37888 87 / 98).
// Sums: whole where that gives four in five of the units a workgroup of a K long enough to fill it (with the norm N = 3584, K = 3584, 16 rows 15.9, in eight
// slices 17.6; K = 18944, four rows 49.9 / 55 and more; N = 4096, K = 2048, 16 rows 11.8 / 12.2; but N = 3072, K = 1536 9.7 / 9.3); else slices of 32 steps, up to eight, and
// more of 8 steps and longer until the units have a workgroup each (N = 896, K = 896 in four 5.0 us, whole 6.5).
extern "C" int fsie_gemm_fp32_stream_plan(int M, int N, int K, int result) {
    const int units = fsie_compute_units();
    if (M < 1 || M > FSIE_GEMM_MFMA_SKINNY_MAX_M || N < 1 || K < 64 || K % kStep || units <= 0 || (result == 1 && N % 2)) return -1;
    const int steps = K / kStep, blocks = (N + 15) / 16;
    if (result == 2 && blocks * 5 < units * 4) {
        int slices = (steps + 31) / 32;
        if (slices > 8) slices = 8;
        while (slices < 8 && blocks * slices * 5 < units * 4 && steps / (slices + 1) >= 8) ++slices;
        while (slices > 1 && (steps + slices - 1) / slices * (slices - 1) >= steps) --slices;  // (no empty slice)
        if (slices > 1) return 8 + 256 * slices;
    }
    if (M > 32 && K < 1536) return -1;
    if (M <= 2 && result != 2 && blocks > units && blocks < 4 * units) return -1;
    const int waves = steps <= 8 * kMostSteps ? 8 : blocks <= units && M <= 32 && steps <= 16 * kMostSteps ? 16 : blocks * 2 < units ? (M <= 32 ? 16 : 8) : 4;
    return waves + 256;
}

// x float32 [M, K], up to 64 rows, K a multiple of 16; w the copy; plan: what fsie_gemm_fp32_stream_plan said.  gated: the rows of w are gate and up in turn (N even), y
// [M, N / 2], act a FsieGateAct or FsieGatePair with its limit and slope.  Else y [slices, M, N], bias (one slice) or null.  x and w 16-byte aligned, y of a
// whole product of N % 4 == 0 too.
extern "C" int fsie_gemm_fp32_stream(const float* x, const float* w, const float* bias, float* y, int M, int N, int K, int gated, int plan, int act,
                                     float limit, float slope, hipStream_t stream) {
    const int waves = plan & 255, slices = plan >> 8;
    FSIE_REQUIRE(M >= 0 && M <= FSIE_GEMM_MFMA_SKINNY_MAX_M && N > 0 && K >= kStep && K % kStep == 0, "gemm_fp32_stream: bad sizes M=%d N=%d K=%d", M, N, K);
    FSIE_REQUIRE(plan > 0 && (waves == 4 || waves == 8 || (waves == 16 && M <= 32)) && slices >= 1 && slices <= FSIE_GEMM_MAX_SPLITS &&
                     (slices == 1 || (!gated && !bias)) && (!gated || (N % 2 == 0 && !bias)),
                 "gemm_fp32_stream: no such plan %d of %d rows", plan, M);
    FSIE_REQUIRE(!gated || FSIE_PAIR_KNOWN(act), "gemm_fp32_stream: unknown activation %d", act);
    FSIE_REQUIRE(static_cast<int64_t>(M) * K * 4 < (int64_t{1} << 31), "gemm_fp32_stream: x of %d x %d is more than the kernel's 32-bit offsets take", M, K);
    FSIE_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0,
                 "gemm_fp32_stream: operands must be 16-byte aligned");
    const int steps = K / kStep, slice = (steps + slices - 1) / slices, s = (slice + waves - 1) / waves;
    FSIE_REQUIRE(slice * (slices - 1) < steps, "gemm_fp32_stream: K=%d in %d slices", K, slices);
    if (M == 0) return 0;
    const StreamCall c{x, w, bias, y, M, N, K, slice, slices, act, limit, slope};
    if (M <= 16) return launch_result<1>(gated != 0, waves, s, c, stream);
    if (M <= 32) return launch_result<2>(gated != 0, waves, s, c, stream);
    if (M <= 48) return launch_result<3>(gated != 0, waves, s, c, stream);
    return launch_result<4>(gated != 0, waves, s, c, stream);
}
