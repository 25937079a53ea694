// Y[M, N] = X[M, K] . W[N, K]^T for bfloat16 operands and up to 16 rows of X: few rows, and a K so short that every load
// of a wave is under way at once.
//
// As in the other products of few rows, D[n, m] = sum_k W[n, k] X[m, k]: W streams from HBM straight into the A registers of
// v_mfma_f32_16x16x32_bf16.  A product of 3 to 30 MB is not bound by the memory's rate but by the trips to it: the kernel that
// shares X through LDS makes one for every 128 values of K, each behind a barrier, with 8 KB of W a workgroup under way.
// Here a workgroup owns one or two blocks of 16 rows of W and its waves deal the steps of 32 values of K among themselves, up
// to eight consecutive ones each: X's fragments (a buffer descriptor ends behind the last row, so rows that are not there cost
// nothing), then W's, all asked for before the first product; the waves' shares meet in LDS, one barrier, and are added in the
// order of the waves.  One trip to memory, 28 KB and more of W a unit under way.
//
// The price is X: every block of rows of W reads all of it (through the caches), so from three rows on the widest gate and up
// matrices stay with the kernel that shares it.  Measured on MI355X, us, cold weights in fragment order, this kernel / the one
// before, at 1, 8 and 16 rows: gate and up of N = 9728, K = 896 5.2 / 6.7, 5.8 / 6.7, 6.7 / 6.8; N = 16384, K = 2048 13.0 / 14.1,
// 13.0 / 13.1, 14.1 / 13.1; an activation of single values, N = 8192, K = 2048 7.9 / 10.6, 8.0 / 10.5, 8.6 / 10.7; plain, against
// the kernel of few rows on rows, N = 6208, K = 2048 6.4 / 8.9, 6.8 / 9.2, 7.5 / 10.4; sums with the norm that adds them up,
// N = 896, K = 4864 in 4 slices 5.9 / 7.2, 6.4 / 7.5, 6.7 / 7.9 (8 slices), N = K = 2048 in 2 (two norms) 6.8 / 7.8, 7.3 / 8.3,
// 7.7 / 8.7, N = 2048, K = 8192 in 4 11.3 / 12.3, 11.8 / 12.4, 12.5 / 12.9 (13), N = K = 3584 in 2 9.2 / 10.0, 9.9 / 10.3,
// 10.7 / 11.2 (7), N = 1536, K = 8960 in 5 9.3 / 11.6, 10.2 / 11.9, 10.9 / 12.6 (14).
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

constexpr int kMostSteps = 8;  // steps of 32 values of K a wave

// SUMS: float32 partial sums [slices][M][N]; GATED: bfloat16 [M, N / 2] of gate and up rows in turn; POINT: bfloat16 [M, N],
// act(sum + bias)
enum Result { SUMS = 0, GATED = 1, POINT = 2 };
constexpr int kPlanOne = 4;
constexpr int kPlanActivation = 3;  // to the plan alone: POINT where the kernel that shares X has the activation in its epilogue too
struct StreamCall {
    const bf16_t* x;
    const bf16_t* w;
    void* y;
    int M, N, K, slice_steps;
    int act;
    float pos, neg;
    const float* bias;
};

// WAVES waves a workgroup deal the steps of a slice of K among themselves, S consecutive ones each, for NB blocks of 16 rows
// of W.  blockIdx.y: the slice.  Steps past the slice's end read the last step of K again and are not multiplied; rows of W past
// the end repeat the last one (a fragment-ordered copy is filled up to whole blocks) and are not written.
template <int WAVES, int S, int NB, int RESULT, bool FRAGS>
__global__ __launch_bounds__(WAVES * 64) void gemm_mfma_stream_kernel(const bf16_t* x, const bf16_t* w, void* y, int M, int N, int K,
                                                                         int slice_steps, int act, float pos, float neg,
                                                                         const float* bias) {
    const StreamCall c{x, w, y, M, N, K, slice_steps, act, pos, neg, bias};  // (one by one they come with the launch, a struct would not)
    __shared__ floatx4 red[WAVES * NB * 64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = lane & 15, kg = lane >> 4;
    const int steps = c.K / 32;
    const int slice_end = min(steps, (static_cast<int>(blockIdx.y) + 1) * c.slice_steps);
    const int first = blockIdx.y * c.slice_steps + wave * S;
    const int here = min(S, slice_end - first);  // may be zero or less: the same for the whole wave
    const __amdgpu_buffer_rsrc_t x_rows = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<bf16_t*>(c.x), 0, c.M * c.K * static_cast<int>(sizeof(bf16_t)), 0x00020000);
    const int xo = row * c.K * static_cast<int>(sizeof(bf16_t)) + kg * 16;
    const int b0 = blockIdx.x * NB, last_block = (c.N - 1) / 16;
    Frag a[S][NB], b[S];
#pragma unroll
    for (int s = 0; s < S; ++s)
        b[s].q = __builtin_amdgcn_raw_buffer_load_b128(x_rows, xo + min(first + s, steps - 1) * 64, 0, 0);
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int k = min(first + s, steps - 1);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            if constexpr (FRAGS)
                a[s][nb].q = __builtin_nontemporal_load(
                    (GlobalVec)(c.w + (static_cast<int64_t>(min(b0 + nb, last_block)) * steps + k) * 512 + lane * 8));
            else
                a[s][nb].q = *(GlobalVec)(c.w + static_cast<int64_t>(min((b0 + nb) * 16 + row, c.N - 1)) * c.K + k * 32 + kg * 8);
        }
    }
    floatx4 acc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[nb] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < S; ++s) {
        if (s < here) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[s][nb].v, b[s].v, acc[nb], 0, 0, 0);
        }
    }
    // the waves' shares, added in the order of the waves, a block of the result a wave
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) red[(wave * NB + nb) * 64 + lane] = acc[nb];
    __syncthreads();
    if (wave >= NB) return;
    floatx4 sum = red[wave * 64 + lane];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) {
        const floatx4 v = red[(w * NB + wave) * 64 + lane];
#pragma unroll
        for (int r = 0; r < 4; ++r) sum[r] += v[r];
    }
    // lane holds D[n + r][m = row]
    const int n = (b0 + wave) * 16 + kg * 4, m = row;
    if (m >= c.M || n >= c.N) return;
    if constexpr (RESULT == GATED) {  // rows n .. n + 3: gate, up, gate, up (N is a multiple of 4)
        uint32_t* out = static_cast<uint32_t*>(c.y);
        out[(static_cast<int64_t>(m) * (c.N / 2) + n / 2) / 2] =
            pack2_bf16(gate_pair(sum[0], sum[1], c.act, c.pos, c.neg), gate_pair(sum[2], sum[3], c.act, c.pos, c.neg));
    } else if constexpr (RESULT == POINT) {  // (N is a multiple of 4)
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = point_act<false>(sum[r] + (c.bias ? c.bias[n + r] : 0.f), c.act, c.pos, c.neg);
        static_cast<uint2*>(c.y)[(static_cast<int64_t>(m) * c.N + n) / 4] = uint2{pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3])};
    } else {
        float* part = static_cast<float*>(c.y) + (static_cast<int64_t>(blockIdx.y) * c.M + m) * c.N;
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (n + r < c.N) part[n + r] = sum[r];
    }
}

template <int WAVES, int S, int NB, int RESULT, bool FRAGS>
int launch(const StreamCall& c, hipStream_t stream) {
    const int blocks = (c.N + 15) / 16;
    const dim3 grid((blocks + NB - 1) / NB, (c.K / 32 + c.slice_steps - 1) / c.slice_steps);
    gemm_mfma_stream_kernel<WAVES, S, NB, RESULT, FRAGS><<<grid, WAVES * 64, 0, stream>>>(c.x, c.w, c.y, c.M, c.N, c.K, c.slice_steps, c.act,
                                                                                       c.pos, c.neg, c.bias);
    FSIE_CHECK_LAUNCH("gemm_mfma_stream");
    return 0;
}

// LEAST: the fewest steps a wave that a plan asks for with so many waves; fewer are taken as so many (the waves past the last step
// multiply nothing).
template <int WAVES, int LEAST, int NB, int RESULT, bool FRAGS>
int launch_steps(int s, const StreamCall& c, hipStream_t stream) {
    if constexpr (LEAST < kMostSteps)
        if (s > LEAST) return launch_steps<WAVES, LEAST + 1, NB, RESULT, FRAGS>(s, c, stream);
    return launch<WAVES, LEAST, NB, RESULT, FRAGS>(c, stream);
}

// (four waves: whole products, and sums on rows of W; sums on a fragment-ordered W: eight.  Two blocks of rows a workgroup: of eight waves, on a
// fragment-ordered W; what else is asked for in twos goes one by one)
template <int RESULT, bool FRAGS>
int launch_waves(int waves, int nb, int s, const StreamCall& c, hipStream_t stream) {
    constexpr int LEAST = RESULT == SUMS ? 4 : 5;
    if constexpr (FRAGS)
        if (waves == 8 && nb == 2) return launch_steps<8, LEAST, 2, RESULT, FRAGS>(s, c, stream);
    if constexpr (RESULT != SUMS || FRAGS)
        if (waves == 8) return launch_steps<8, LEAST, 1, RESULT, FRAGS>(s, c, stream);
    if constexpr (RESULT != SUMS)
        return waves == 4 ? launch_steps<4, 1, 1, RESULT, FRAGS>(s, c, stream) : launch_steps<16, LEAST, 1, RESULT, FRAGS>(s, c, stream);
    if constexpr (RESULT == SUMS && !FRAGS)
        if (waves == 4) return launch_steps<4, 5, 1, RESULT, FRAGS>(s, c, stream);
    fsie_set_error("gemm_mfma_stream: sums take eight waves a workgroup, on rows four");
    return 1;
}

}  // namespace

// How M rows of this product are best taken, or -1 where another kernel is the better one or this one does not take them:
// waves + 256 * blocks of rows a workgroup + 65536 * slices of K.  frags: W is the copy in fragment order.
// Whole products (GATED, POINT): as few waves as hold K in eight steps each.  Two blocks of rows a workgroup, which share X's
// fragments, where one would leave the units an uneven second round or X's reads weigh (N = 6208, K = 2048 in 194 workgroups
// 6.4 us, in 388 6.7; N = 4096 in 256 5.2 at 8 rows, in 128 6.1; N = 8192 at 8 rows in 256 8.1, in 512 8.7).
// Beyond 24 MB gate and up of one and two rows only, and to 72 MB (N = 17920, K = 1536, two rows 10.7 us, four 11.2, eight 12.3;
// the kernel that shares X 11.3, 11.1, 11.1; N = 22016, K = 2048, two rows 16.8 / 16.5), below it not more than two workgroups a unit
// for nine rows and more (N = 11264, K = 1024, 16 rows 7.9 / 7.4); an activation beyond 64 MB up to four rows (N = 14336,
// K = 4096, four 23.5 / 23.4, eight 25.9 / 23.3).  Rows of W that are no copy up to a workgroup a unit (against the few-rows kernel,
// 8 rows, N = 2048, K = 1280 4.6 / 5.2, N = 1552, K = 2048 5.6 / 6.1, N = 4096, K = 896 4.2 / 5.0), beyond 28 MB up to eight rows
// (N = K = 4096, eight 10.4 / 11.1, 13 11.9 / 11.2, 16 12.6 / 11.5; N = K = 3584, 16 9.6 / 10.2).
// Sums: the fewest slices that a workgroup of eight waves holds, then as many more as leave a wave four steps and the workgroups
// no more than the units: a second round costs what it hides (N = 4608, K = 3584 8.1 us against 7.0 in seven slices), and the
// norm pays for every slice.
// kPlanOne: sums of one slice, for a norm that the next product makes itself (gemm_mfma_normed.hip), whose every workgroup reads them.
// Rows of W in four waves: N = K = 896, one and two rows 2.9 us, in seven slices 2.4; gate and up with the norm behind them 5.3 and 5.6, 6.1 and 7.3.
extern "C" int fsie_gemm_mfma_stream_plan(int M, int N, int K, int result, int frags) {
    const int units = fsie_compute_units();
    if (M < 1 || M > 16 || N < 1 || K < 32 || K % 32 || units <= 0) return -1;
    const int steps = K / 32, groups = (N + 15) / 16;
    const int64_t bytes = static_cast<int64_t>(N) * K * 2;
    if (result == kPlanOne) return !frags && M <= 2 && steps > 4 * 4 && steps <= 4 * kMostSteps && groups <= units ? 4 + 256 + 65536 : -1;
    if (result == SUMS) {
        if (!frags || K < 1024) return -1;
        int splits = (steps + 8 * kMostSteps - 1) / (8 * kMostSteps);
        if (splits > FSIE_GEMM_MAX_SPLITS) return -1;  // (K beyond 32,768: more partial sums than the norm takes)
        const int blocks = groups * splits > units ? 2 : 1;
        const int across = (groups + blocks - 1) / blocks;
        if (across * splits > units) return -1;
        while (splits < FSIE_GEMM_MAX_SPLITS && across * (splits + 1) <= units && steps / (splits + 1) >= 32) ++splits;
        while (splits > 1 && (steps + splits - 1) / splits * (splits - 1) >= steps) --splits;  // (no empty slice)
        if ((steps + splits - 1) / splits > 8 * kMostSteps) return -1;
        return 8 + 256 * blocks + 65536 * splits;
    }
    if (N % 4 || steps > 16 * kMostSteps) return -1;
    const int waves = steps <= 4 * kMostSteps ? 4 : steps <= 8 * kMostSteps ? 8 : 16;
    int blocks = 1;
    if (waves == 8 && groups > units && (M > 4 || (groups + 1) / 2 <= units)) blocks = 2;
    constexpr int64_t MB = 1024 * 1024;
    if (result == GATED && (!frags || (bytes > 24 * MB && (M > 2 || bytes > 72 * MB)) || (M > 8 && groups > 2 * units))) return -1;
    if (result == kPlanActivation && frags && M > 4 && bytes > 64 * MB) return -1;
    if (result != GATED && !frags && (groups > units || (M > 8 && bytes > 28 * MB))) return -1;
    return waves + 256 * blocks + 65536;
}

// x [M, K], M up to 16, K a multiple of 32; w [N, K] or (frags) its copy in fragment order.  result 0: y float32 partial sums
// [splits, M, N] (one slice: [M, N]); 1: w's rows are gate and up in turn, y bfloat16 [M, N / 2], act a FsieGateAct or FsieGatePair with
// limit pos and slope neg; 2: y bfloat16 [M, N] = act(sum + bias), act a FsiePointAct with its constants, bias float32 or null.
// N a multiple of 4 for 1 and 2, one slice.  plan: what fsie_gemm_mfma_stream_plan said.  x and w 16-byte aligned.
extern "C" int fsie_gemm_mfma_stream(const void* x, const void* w, const float* bias, void* y, int M, int N, int K, int result,
                                     int plan, int frags, int act, float pos, float neg, hipStream_t stream) {
    const int waves = plan & 255, blocks = plan >> 8 & 255, splits = plan >> 16;
    FSIE_REQUIRE(M >= 0 && M <= 16 && N > 0 && K > 0 && K % 32 == 0, "gemm_mfma_stream: bad sizes M=%d N=%d K=%d", M, N, K);
    FSIE_REQUIRE(result == SUMS || ((result == GATED || result == POINT) && N % 4 == 0 && splits == 1),
                 "gemm_mfma_stream: result %d of N=%d in %d slices", result, N, splits);
    FSIE_REQUIRE(result != GATED || FSIE_PAIR_KNOWN(act), "gemm_mfma_stream: unknown activation %d", act);
    FSIE_REQUIRE(result != POINT || FSIE_POINT_KNOWN(act), "gemm_mfma_stream: unknown activation %d", act);
    FSIE_REQUIRE(plan > 0 && (waves == 4 || waves == 8 || waves == 16) && (blocks == 1 || (blocks == 2 && waves > 4)) && splits >= 1 &&
                     splits <= FSIE_GEMM_MAX_SPLITS && (result != SUMS || (frags ? waves == 8 : waves == 4 && splits == 1)) && (result != GATED || frags),
                 "gemm_mfma_stream: no such plan %d for result %d", plan, result);
    const int steps = K / 32, slice = (steps + splits - 1) / splits, s = (slice + waves - 1) / waves;
    FSIE_REQUIRE(slice * (splits - 1) < steps && s <= kMostSteps, "gemm_mfma_stream: K=%d in %d slices of %d waves", K, splits, waves);
    FSIE_REQUIRE(static_cast<int64_t>(M) * K * 2 <= 0x7fffffff, "gemm_mfma_stream: K=%d is more than 32-bit offsets into x take", K);
    FSIE_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0 && reinterpret_cast<uintptr_t>(y) % 8 == 0,
                 "gemm_mfma_stream: operands must be 16-byte aligned, the result 8-byte");
    if (M == 0) return 0;
    const StreamCall c{static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(w), y, M, N, K, slice, act, pos, neg, bias};
    if (result == GATED) return launch_waves<GATED, true>(waves, blocks, s, c, stream);
    if (result == SUMS) return frags ? launch_waves<SUMS, true>(waves, blocks, s, c, stream) : launch_waves<SUMS, false>(waves, blocks, s, c, stream);
    return frags ? launch_waves<POINT, true>(waves, blocks, s, c, stream) : launch_waves<POINT, false>(waves, blocks, s, c, stream);
}
