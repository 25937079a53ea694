// Y[M, N] = X[M, K] . W[N, K]^T (+ bias) in true float32 on the matrix cores, for up to 64 rows
// (the 32-bit path's decoding): v_mfma_f32_16x16x4_f32 multiplies and adds float32 values as they
// are, no reduced-precision mode.  As in the bfloat16 product for few rows, the product is
// computed transposed, D[n, m] = sum_k W[n, k] X[m, k]: W streams from HBM straight into the A
// operands (16 bytes, four values of k, per lane), X comes from cache through a buffer descriptor
// that ends with its last row, the waves of a workgroup split K and their partial tiles are added
// through LDS in the fixed order of the waves: a row's sums depend on K and on the launch shape
// that N, K and the number of tiles of 16 rows give (runs of a length for up to 32 rows, of half of it beyond), never on
// what the other rows hold.
#include "common.h"
#include "api.h"
#include "lds_loads.h"

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// What stands in the place of the plain sums: the rows of W are gate and up in turn and y is [M, N / 2], their product of
// values (gate_pair), without bias.  As a pass of its own behind the product it was 4.5 us a layer and step of few rows.
struct Gate {
    int act;
    float limit, slope;
};

// MT tiles of 16 rows of X; WAVES waves split K in steps of 16 values (4 per lane group), U steps in flight.
template <int MT, int WAVES, bool GATED>
__global__ __launch_bounds__(WAVES * FSIE_WAVE) void gemm_mfma_fp32_kernel(const float* __restrict__ x,
                                                                          const float* __restrict__ w,
                                                                          const float* __restrict__ bias,
                                                                          float* __restrict__ y, int M, int N, int K,
                                                                          int slice_steps, Gate gate) {
    constexpr int U = MT >= 3 ? 2 : 4;
    __shared__ float red[WAVES > 1 ? (WAVES - 1) * MT * FSIE_WAVE * 4 : 1];
    const int lane = threadIdx.x & (FSIE_WAVE - 1);
    const int wave = threadIdx.x / FSIE_WAVE;
    const int row = lane & 15;  // row of the A tile (n) and column of the B tile (m)
    const int kg = lane >> 4;   // which 4 of a step's 16 k values this lane holds
    const int n0 = blockIdx.x * 16;
    const float* wp = w + static_cast<int64_t>(min(n0 + row, N - 1)) * K;  // rows past the end repeat the last; never written
    const __amdgpu_buffer_rsrc_t x_rows = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(x), 0, M * K * static_cast<int>(sizeof(float)), 0x00020000);
    int xo[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) xo[t] = (t * 16 + row) * K * static_cast<int>(sizeof(float));
    // two levels of float32 sums: a run of kFlush passes of the loop (some hundreds of products) is
    // summed on its own and then added to the total, so that the rounding error grows with the
    // square roots of the run and of the number of runs, not of K (K reaches 18944 in a 7B model)
    constexpr int kFlush = 8;
    floatx4 acc[MT], total[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = total[t] = floatx4{0.f, 0.f, 0.f, 0.f};

    // blockIdx.y: a slice of K of `slice_steps` steps, whose sums are a plane of y of their own
    const int first_step = blockIdx.y * slice_steps;
    const int n_steps = min((K + 15) / 16, first_step + slice_steps);
    const int k_end = min(K, n_steps * 16);
    y += static_cast<int64_t>(blockIdx.y) * M * N;
    int pass = 0;
    for (int s0 = first_step + wave; s0 < n_steps; s0 += WAVES * U, ++pass) {
        if (pass > 0 && pass % kFlush == 0) {
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                total[t] += acc[t];
                acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
            }
        }
        float4 a[U];
        u32x4 b[U][MT];
        bool ok[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k0 = (s0 + u * WAVES) * 16 + kg * 4;
            ok[u] = k0 < k_end;  // K is a multiple of 4: a lane's four values are all in or all out
            const int k0c = ok[u] ? k0 : 0;
            a[u] = *reinterpret_cast<const float4*>(wp + k0c);
#pragma unroll
            for (int t = 0; t < MT; ++t)
                b[u][t] = __builtin_amdgcn_raw_buffer_load_b128(x_rows, xo[t] + k0c * static_cast<int>(sizeof(float)), 0, 0);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (!ok[u]) a[u] = float4{0.f, 0.f, 0.f, 0.f};
            const float av[4] = {a[u].x, a[u].y, a[u].z, a[u].w};
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int t = 0; t < MT; ++t)
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[j], __uint_as_float(b[u][t][j]), acc[t], 0, 0, 0);
        }
    }
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] += total[t];
    if (WAVES > 1) {
        if (wave > 0) {
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) red[(((wave - 1) * MT + t) * 4 + r) * FSIE_WAVE + lane] = acc[t][r];
        }
        __syncthreads();
        if (wave > 0) return;
        for (int wv = 0; wv < WAVES - 1; ++wv)
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[t][r] += red[((wv * MT + t) * 4 + r) * FSIE_WAVE + lane];
    }
    // lane holds D[n0 + 4 kg + r][m = 16 t + row]
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const int m = t * 16 + row;
        if (m >= M) continue;
        if constexpr (GATED) {
#pragma unroll
            for (int r = 0; r < 4; r += 2) {
                const int nn = n0 + kg * 4 + r;
                if (nn < N) y[static_cast<int64_t>(m) * (N / 2) + nn / 2] = gate_pair(acc[t][r], acc[t][r + 1], gate.act, gate.limit, gate.slope);
            }
            continue;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int nn = n0 + kg * 4 + r;
            if (nn < N) y[static_cast<int64_t>(m) * N + nn] = bias ? acc[t][r] + bias[nn] : acc[t][r];
        }
    }
}

template <int MT, bool GATED>
int launch_mt(int waves, const float* x, const float* w, const float* bias, float* y, int M, int N, int K, int splits, Gate gate,
              hipStream_t stream) {
    const int steps = (K + 15) / 16, slice = (steps + splits - 1) / splits;
    const dim3 groups(static_cast<unsigned>((N + 15) / 16), static_cast<unsigned>(splits));
    switch (waves) {
        case 1: gemm_mfma_fp32_kernel<MT, 1, GATED><<<groups, 64, 0, stream>>>(x, w, bias, y, M, N, K, slice, gate); break;
        case 2: gemm_mfma_fp32_kernel<MT, 2, GATED><<<groups, 128, 0, stream>>>(x, w, bias, y, M, N, K, slice, gate); break;
        case 4: gemm_mfma_fp32_kernel<MT, 4, GATED><<<groups, 256, 0, stream>>>(x, w, bias, y, M, N, K, slice, gate); break;
        default: gemm_mfma_fp32_kernel<MT, 8, GATED><<<groups, 512, 0, stream>>>(x, w, bias, y, M, N, K, slice, gate); break;
    }
    FSIE_CHECK_LAUNCH("gemm_mfma_fp32");
    return 0;
}

// ---- many rows (prompts) ----------------------------------------------------------------------
// A workgroup of four waves makes 64 rows of X by 64 of W, a wave 32 by 32; 32 values of K at a time go through LDS, a row's eight 16-byte
// units permuted by the row so that the rows' reads meet different banks.  A wave's read of 16 bytes a lane feeds four instructions of 32
// cycles each, so the matrix cores are the bound, and the small tile is what fills the chip: N = 896 at 682 rows makes 154 of them (in slices
// of K as many times that).  Two levels of float32 sums as above, runs of kTileFlush values of K.
// Through registers and two stages (the first kernel, for K that is no multiple of 32) the matrix cores were busy in 0.66 to 0.71 of the
// units' cycles: 682 x 9728 x 896 132 us, 682 x 3584 x 18944 1,116, 300 x 1152 x 896 27.8, 128 x 4608 x 3584 102, in seven slices 300 x 896 x 4864
// 41.7, weights from HBM.  Straight to LDS, the loads, the reads and the products of three stages in turns (the second kernel): 114, 894, 21.2, 74
// and 34.4; 117 TFLOP/s at 1,500 x 9728 x 896 (96 before), where the library reaches 154 at 8,192 cubed.  Six stages where every workgroup has a unit
// to itself, whose step of 0.43 us would else not cover the way from HBM; three leave room for three workgroups a unit.
constexpr int kTileEdge = 64, kTileK = 32, kTileFlush = 256;

enum Whole { PLAIN = 0, SUMS = 1, GATED = 2 };

// A lane holds D[n .. n + 4][m] of a wave's 2 x 2 tiles; m and n: of the first.
template <int RESULT>
__device__ __forceinline__ void write_tile(const floatx4 (&acc)[2][2], const floatx4 (&total)[2][2], float* __restrict__ y, const float* __restrict__ bias,
                                           const Gate& gate, int M, int N, int m_first, int n_first, int slice) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int m = m_first + 16 * t;
        if (m >= M) continue;
        float* to = RESULT == GATED ? y + static_cast<int64_t>(m) * (N / 2) : y + (static_cast<int64_t>(RESULT == SUMS ? slice : 0) * M + m) * N;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int n = n_first + 16 * j;
            const floatx4 v = acc[j][t] + total[j][t];
            if constexpr (RESULT == GATED) {
#pragma unroll
                for (int i = 0; i < 4; i += 2)
                    if (n + i < N) to[(n + i) / 2] = gate_pair(v[i], v[i + 1], gate.act, gate.limit, gate.slope);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (n + i < N) to[n + i] = RESULT == PLAIN && bias ? v[i] + bias[n + i] : v[i];
            }
        }
    }
}

template <int RESULT>
__global__ __launch_bounds__(256) void gemm_fp32_tile_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                            const float* __restrict__ bias, float* __restrict__ y, int M,
                                                            int N, int K, int k_slice, Gate gate) {
    __shared__ float4 lds[2][2][kTileEdge][kTileK / 4];
    const int lane = threadIdx.x & (FSIE_WAVE - 1), wave = threadIdx.x / FSIE_WAVE;
    const int n0 = blockIdx.x * kTileEdge, m0 = blockIdx.y * kTileEdge;
    const int k_begin = blockIdx.z * k_slice, k_end = min(K, k_begin + k_slice);
    // this thread's units of a stage: rows r and r + 32 of W and of X, values 4 u .. 4 u + 4
    const int r = threadIdx.x >> 3, u = threadIdx.x & 7;
    const float* from[4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {  // rows past the end repeat the last one and are never written
        from[i] = w + static_cast<int64_t>(min(n0 + r + 32 * i, N - 1)) * K;
        from[2 + i] = x + static_cast<int64_t>(min(m0 + r + 32 * i, M - 1)) * K;
    }
    float4 held[4];
    const auto bring = [&](int k0) {
        const int k = k0 + 4 * u;  // K and the slices are multiples of 4: four values are all in or all out
        const bool in = k < k_end;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            held[i] = *reinterpret_cast<const float4*>(from[i] + (in ? k : k_begin));
            if (!in) held[i] = float4{0.f, 0.f, 0.f, 0.f};
        }
    };
    const int row = lane & 15, kg = lane >> 4;
    const int nw = (wave & 1) * 32, mw = (wave >> 1) * 32;
    floatx4 acc[2][2], total[2][2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[j][t] = total[j][t] = floatx4{0.f, 0.f, 0.f, 0.f};
    bring(k_begin);
    int buf = 0, run = 0;
    for (int k0 = k_begin; k0 < k_end; k0 += kTileK, buf ^= 1) {
#pragma unroll
        for (int i = 0; i < 4; ++i) lds[buf][i >> 1][r + 32 * (i & 1)][u ^ (r & 7)] = held[i];
        __syncthreads();  // (one a step: the stage written next was read before the last one)
        if (k0 + kTileK < k_end) bring(k0 + kTileK);
        float4 a[2][2], b[2][2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                a[j][h] = lds[buf][0][nw + 16 * j + row][(4 * h + kg) ^ (row & 7)];
                b[j][h] = lds[buf][1][mw + 16 * j + row][(4 * h + kg) ^ (row & 7)];
            }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int t = 0; t < 2; ++t)
                        acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(reinterpret_cast<const float*>(&a[j][h])[i],
                                                                        reinterpret_cast<const float*>(&b[t][h])[i], acc[j][t], 0, 0, 0);
        if (++run == kTileFlush / kTileK) {
            run = 0;
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    total[j][t] += acc[j][t];
                    acc[j][t] = floatx4{0.f, 0.f, 0.f, 0.f};
                }
        }
    }
    write_tile<RESULT>(acc, total, y, bias, gate, M, N, m0 + mw + row, n0 + nw + 4 * kg, static_cast<int>(blockIdx.z));
}

// The same tiles where K is a whole number of steps: both operands go to LDS straight from memory, STAGES - 1 steps ahead, and a wave reads the
// next step's fragments, asks for its share of a later stage and multiplies this step's in turns.  The order of every sum is that of the kernel
// above, and so are its bits.
template <int RESULT, int STAGES>
__global__ __launch_bounds__(256) void gemm_fp32_block_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                             const float* __restrict__ bias, float* __restrict__ y, int M, int N, int K,
                                                             int k_slice, int m_tiles, int n_tiles, int abreast, Gate gate) {
    constexpr int kRowBytes = kTileK * 4, kHalf = kTileEdge * kRowBytes, kStage = 2 * kHalf, kLoads = 4;  // a stage: W, then X
    extern __shared__ char lds[];
    // A die (the workgroup's number modulo 8) takes neighbouring tiles: of W its own eighth, of X all.  The slices are laid side by side and dealt so, a
    // die few of them (abreast == splits), or dealt one by one, a die some tiles of each (abreast == 1).
    const int tiles = m_tiles * n_tiles, dealt = tiles * abreast, a_die = (dealt + 7) / 8, turn = static_cast<int>(blockIdx.x >> 3);
    const int id = static_cast<int>(blockIdx.x & 7) * a_die + turn % a_die;
    if (id >= dealt) return;
    const int slice = turn / a_die + id / tiles, m_tile = id % m_tiles, n_tile = id % tiles / m_tiles;
    const int m0 = m_tile * kTileEdge, n0 = n_tile * kTileEdge;
    const int first_step = slice * k_slice / kTileK, steps = min(K - slice * k_slice, k_slice) / kTileK;
    const int lane = threadIdx.x & (FSIE_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / FSIE_WAVE);
    const int row = lane & 15, kg = lane >> 4;
    const int nw = (wave & 1) * 32, mw = (wave >> 1) * 32;

    // a wave's loads of a stage: 16 rows of W and of X, eight a load; a row's eight 16-byte units lie permuted by the row
    const u32x4 w_rows = fsie_lds::rows_from(w, static_cast<uint32_t>(N) * static_cast<uint32_t>(K) * 4u);
    const u32x4 x_rows = fsie_lds::rows_from(x, static_cast<uint32_t>(M) * static_cast<uint32_t>(K) * 4u);
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds);
    uint32_t from[4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {  // rows past the end repeat the last one and are never written
        const int r = (wave * 2 + i) * 8 + (lane >> 3);
        const uint32_t unit = ((lane & 7) ^ (r >> 1 & 7)) * 16u;
        from[i] = static_cast<uint32_t>(min(n0 + r, N - 1)) * static_cast<uint32_t>(K) * 4u + unit;
        from[2 + i] = static_cast<uint32_t>(min(m0 + r, M - 1)) * static_cast<uint32_t>(K) * 4u + unit;
    }
    uint32_t bring_to = 0, read_from = 0;  // the stages' places, in turn
    const auto next_stage = [](uint32_t at) { return at == (STAGES - 1) * kStage ? 0u : at + kStage; };
    const auto k_of = [&](int step) { return static_cast<uint32_t>(first_step + min(step, steps - 1)) * kRowBytes; };
    const auto load = [&](int i, uint32_t k) {
        fsie_lds::load_to_lds(i < 2 ? w_rows : x_rows, lds0 + bring_to + (i >> 1) * kHalf + (wave * 2 + (i & 1)) * 1024u, from[i], k);
    };
    floatx4 acc[2][2], total[2][2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[j][t] = total[j][t] = floatx4{0.f, 0.f, 0.f, 0.f};
    floatx4 f[2][4][2];  // this step's fragments and the next one's: [W 0, 1, X 0, 1][half of the step]
    const auto read = [&](int i, floatx4 (&to)[4][2]) {  // the i-th of a stage's eight
        const int h = i >> 2, at = i & 3;
        const int r = (at < 2 ? nw : mw) + (at & 1) * 16 + row;
        to[at][h] = *reinterpret_cast<const floatx4*>(lds + read_from + (at >> 1) * kHalf + r * kRowBytes + (((4 * h + kg) ^ (row >> 1 & 7)) * 16));
    };
    const auto go = [&](int step, const floatx4 (&now)[4][2], floatx4 (&next)[4][2]) {
        // the next stage has arrived, and this step's fragments are in every wave's registers: its stage is free
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((STAGES - 2) * kLoads) : "memory");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t k = k_of(step + STAGES);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
#pragma unroll
            for (int q = 2 * c; q < 2 * c + 2; ++q)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int t = 0; t < 2; ++t)
                        acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(now[j][q >> 2][q & 3], now[2 + t][q >> 2][q & 3], acc[j][t], 0, 0, 0);
            read(2 * c, next);
            read(2 * c + 1, next);
            load(c, k);
            __builtin_amdgcn_sched_barrier(0);
        }
        bring_to = next_stage(bring_to);
        read_from = next_stage(read_from);
    };
#pragma unroll
    for (int i = 0; i < STAGES; ++i) {
        const uint32_t k = k_of(i);
#pragma unroll
        for (int c = 0; c < 4; ++c) load(c, k);
        bring_to = next_stage(bring_to);
    }
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((STAGES - 1) * kLoads) : "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 8; ++i) read(i, f[0]);
    read_from = next_stage(read_from);
    constexpr int kRun = kTileFlush / kTileK;
    for (int step = 0; step < steps; step += 2) {
        go(step, f[0], f[1]);
        if (step + 1 < steps) go(step + 1, f[1], f[0]);
        if ((step + 2) % kRun == 0) {  // (kRun is even; the last run is short of a step where there is an odd number: added below all the same)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    total[j][t] += acc[j][t];
                    acc[j][t] = floatx4{0.f, 0.f, 0.f, 0.f};
                }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (no load may still write LDS when the workgroup's is given away)
    write_tile<RESULT>(acc, total, y, bias, gate, M, N, m0 + mw + row, n0 + nw + 4 * kg, slice);
}

struct TileCall {
    const float *x, *w, *bias;
    float* y;
    Gate gate;
    int M, N, K, slice, m_tiles, n_tiles, splits;
    hipStream_t stream;
};

// Whether slices are dealt to the dies one by one.  Side by side a die reads its slices' part of X alone, which is up to 8 per cent faster (200 rows of N = 2048,
// K = 8192 in four 74 us, 80 one by one); but a short last slice leaves its dies idle: 2,048 rows of N = 1024, K = 640, slices of 512 and 128,
// took 42.6 us (36.3 in the kernel above, whose workgroups go to the dies in turn; 32.4 one by one), 512 rows of N = 896, K = 4864 in seven 58.3, 47.6 one by one.  So where
// a die's workgroups make fewer rounds over its units one by one, and always where two slices are of different lengths.
bool dealt_one_by_one(const TileCall& c) {
    if (c.splits == 1 || c.K == static_cast<int64_t>(c.slice) * c.splits) return false;
    if (c.splits == 2) return true;
    const int units = fsie_compute_units(), a_die = units > 8 ? units / 8 : 1;
    const int64_t tiles = static_cast<int64_t>(c.m_tiles) * c.n_tiles;
    return ceil_div64(ceil_div64(tiles, 8) * c.K, static_cast<int64_t>(c.slice) * a_die) < ceil_div64(ceil_div64(tiles * c.splits, 8), a_die);
}

template <int RESULT, int STAGES>
int launch_block(const TileCall& c) {
    constexpr int kLds = STAGES * 2 * kTileEdge * kTileK * 4;
    static const hipError_t allowed = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_fp32_block_kernel<RESULT, STAGES>),
                                                          hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    FSIE_REQUIRE(allowed == hipSuccess, "gemm_fp32_tile: %d bytes of LDS: %s", kLds, hipGetErrorString(allowed));
    const int abreast = dealt_one_by_one(c) ? 1 : c.splits;
    const unsigned groups = static_cast<unsigned>((static_cast<int64_t>(c.m_tiles) * c.n_tiles * abreast + 7) / 8 * 8 * (c.splits / abreast));
    gemm_fp32_block_kernel<RESULT, STAGES><<<groups, 256, kLds, c.stream>>>(c.x, c.w, c.bias, c.y, c.M, c.N, c.K, c.slice, c.m_tiles, c.n_tiles, abreast, c.gate);
    FSIE_CHECK_LAUNCH("gemm_fp32_tile");
    return 0;
}

}  // namespace

// float32 operands and result, any number of rows, K a multiple of 4, x and w 16-byte aligned.  splits > 1: y holds
// that many partial sums [splits][M][N] of slices of K, without bias.
static int tile_product(const float* x, const float* w, const float* bias, float* y, int M, int N, int K, int splits,
                        const Gate* gate, hipStream_t stream) {
    FSIE_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm_fp32_tile: bad sizes M=%d N=%d K=%d", M, N, K);
    FSIE_REQUIRE(K % 4 == 0, "gemm_fp32_tile: K=%d must be a multiple of 4", K);
    FSIE_REQUIRE(splits >= 1 && splits <= 64 && (splits == 1 || !bias), "gemm_fp32_tile: %d slices", splits);
    FSIE_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0,
                 "gemm_fp32_tile: operands must be 16-byte aligned");
    if (M == 0) return 0;
    const int64_t tiles_m = ceil_div64(M, kTileEdge);
    FSIE_REQUIRE(tiles_m <= 65535, "gemm_fp32_tile: %d rows", M);
    // slices of whole flushes where K gives them, so that a slice's runs are those of the uncut sum; else of whole steps
    int64_t slice = ceil_div64(ceil_div64(K, splits), kTileFlush) * kTileFlush;
    if (slice * (splits - 1) >= K) slice = ceil_div64(ceil_div64(K, splits), kTileK) * kTileK;
    FSIE_REQUIRE(splits == 1 || slice * (splits - 1) < K, "gemm_fp32_tile: K=%d does not give %d slices", K, splits);
    const int64_t tiles_n = ceil_div64(N, kTileEdge), groups = tiles_m * tiles_n * splits;
    if (splits == 1) slice = ceil_div64(K, kTileK) * kTileK;
    // (from four steps on: what a workgroup asks for ahead is past the end else, 65 rows of N = 151936, K = 64 59 us, through registers 48; N = 1024 6.1 and 5.6;
    // K = 128 as fast or faster but for the first of these, 78 and 73)
    if (K % kTileK == 0 && slice >= 4 * kTileK && static_cast<int64_t>(M) * K * 4 < (int64_t{1} << 31) && static_cast<int64_t>(N) * K * 4 < (int64_t{1} << 31) &&
        groups < (int64_t{1} << 30)) {
        const TileCall c{x, w, bias, y, gate ? *gate : Gate{}, M, N, K, static_cast<int>(slice), static_cast<int>(tiles_m), static_cast<int>(tiles_n), splits, stream};
        const bool few = groups <= fsie_compute_units();  // (a unit each)
        if (splits > 1) return few ? launch_block<SUMS, 6>(c) : launch_block<SUMS, 3>(c);
        if (gate) return few ? launch_block<GATED, 6>(c) : launch_block<GATED, 3>(c);
        return few ? launch_block<PLAIN, 6>(c) : launch_block<PLAIN, 3>(c);
    }
    const dim3 grid(static_cast<unsigned>((N + kTileEdge - 1) / kTileEdge), static_cast<unsigned>(tiles_m), static_cast<unsigned>(splits));
    if (splits > 1)
        gemm_fp32_tile_kernel<SUMS><<<grid, 256, 0, stream>>>(x, w, nullptr, y, M, N, K, static_cast<int>(slice), Gate{});
    else if (gate)
        gemm_fp32_tile_kernel<GATED><<<grid, 256, 0, stream>>>(x, w, nullptr, y, M, N, K, static_cast<int>(slice), *gate);
    else
        gemm_fp32_tile_kernel<PLAIN><<<grid, 256, 0, stream>>>(x, w, bias, y, M, N, K, static_cast<int>(slice), Gate{});
    FSIE_CHECK_LAUNCH("gemm_fp32_tile");
    return 0;
}

extern "C" int fsie_gemm_fp32_tile(const float* x, const float* w, const float* bias, float* y, int M, int N, int K, int splits,
                                   hipStream_t stream) {
    return tile_product(x, w, bias, y, M, N, K, splits, nullptr, stream);
}

// float32 operands and result.  1 <= M <= 64, K a multiple of 4, x and w 16-byte aligned.
// waves: 1, 2, 4 or 8 waves of a workgroup split K; 0 = choose.  splits > 1: y = partial sums [splits][M][N] of slices of K,
// no bias.
static int few_rows(const float* x, const float* w, const float* bias, float* y, int M, int N, int K, int waves, int splits,
                    const Gate* gate, hipStream_t stream) {
    FSIE_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm_mfma_fp32: bad sizes M=%d N=%d K=%d", M, N, K);
    FSIE_REQUIRE(M <= FSIE_GEMM_MFMA_SKINNY_MAX_M, "gemm_mfma_fp32: at most %d rows, got %d",
                 FSIE_GEMM_MFMA_SKINNY_MAX_M, M);
    FSIE_REQUIRE(K % 4 == 0, "gemm_mfma_fp32: K=%d must be a multiple of 4", K);
    FSIE_REQUIRE(static_cast<int64_t>(M) * K * 4 < (int64_t{1} << 31),
                 "gemm_mfma_fp32: x of %d x %d is more than the kernel's 32-bit offsets take", M, K);
    FSIE_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0,
                 "gemm_mfma_fp32: operands must be 16-byte aligned");
    FSIE_REQUIRE(waves == 0 || waves == 1 || waves == 2 || waves == 4 || waves == 8,
                 "gemm_mfma_fp32: waves must be 0, 1, 2, 4 or 8");
    const int steps = (K + 15) / 16;
    FSIE_REQUIRE(splits >= 1 && splits <= FSIE_GEMM_MAX_SPLITS &&
                     (splits == 1 || ((steps + splits - 1) / splits) * (splits - 1) < steps),
                 "gemm_mfma_fp32: K=%d does not give %d slices", K, splits);
    if (M == 0) return 0;
    if (waves == 0) {
        const int groups = (N + 15) / 16 * splits;
        waves = 1;
        while (waves < 8 && groups * waves < 1024) waves *= 2;
        while (waves > 1 && steps / splits < 4 * waves) waves /= 2;
    }
    switch ((M + 15) / 16) {
        case 1: return gate ? launch_mt<1, true>(waves, x, w, bias, y, M, N, K, splits, *gate, stream)
                             : launch_mt<1, false>(waves, x, w, bias, y, M, N, K, splits, Gate{}, stream);
        case 2: return gate ? launch_mt<2, true>(waves, x, w, bias, y, M, N, K, splits, *gate, stream)
                             : launch_mt<2, false>(waves, x, w, bias, y, M, N, K, splits, Gate{}, stream);
        case 3: return gate ? launch_mt<3, true>(waves, x, w, bias, y, M, N, K, splits, *gate, stream)
                             : launch_mt<3, false>(waves, x, w, bias, y, M, N, K, splits, Gate{}, stream);
        default: return gate ? launch_mt<4, true>(waves, x, w, bias, y, M, N, K, splits, *gate, stream)
                             : launch_mt<4, false>(waves, x, w, bias, y, M, N, K, splits, Gate{}, stream);
    }
}

extern "C" int fsie_gemm_mfma_fp32(const float* x, const float* w, const float* bias, float* y, int M, int N, int K,
                                   int waves, hipStream_t stream) {
    return few_rows(x, w, bias, y, M, N, K, waves, 1, nullptr, stream);
}

extern "C" int fsie_gemm_mfma_fp32_sums(const float* x, const float* w, float* y, int M, int N, int K, int splits,
                                        hipStream_t stream) {
    return few_rows(x, w, nullptr, y, M, N, K, 0, splits, nullptr, stream);
}

// The rows of w are gate and up in turn (N even): y [M, N / 2] is their product of values, act a FsieGateAct or FsieGatePair
// with its limit and slope.  Any number of rows; otherwise as the two products above, whose bits its sums have.
extern "C" int fsie_gemm_fp32_gated(const float* x, const float* w, float* y, int M, int N, int K, int act, float limit, float slope,
                                    hipStream_t stream) {
    FSIE_REQUIRE(N % 2 == 0, "gemm_fp32_gated: N=%d rows of gate and up in turn", N);
    FSIE_REQUIRE(FSIE_PAIR_KNOWN(act), "gemm_fp32_gated: unknown activation %d", act);
    const Gate gate{act, limit, slope};
    return M <= FSIE_GEMM_MFMA_SKINNY_MAX_M ? few_rows(x, w, nullptr, y, M, N, K, 0, 1, &gate, stream)
                                            : tile_product(x, w, nullptr, y, M, N, K, 1, &gate, stream);
}
