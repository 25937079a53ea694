// Gated linear attention of a step of one token a request, from the projections to what the output projection reads, in one
// launch: the decays' second product, the update of every head's state, o, its norm and its gate.
//
//   z = W_a2 a + b,  alpha = sigmoid(z)^(1/tau),  S <- diag(alpha) S + k v^T,  o = S^T q,
//   y = rmsnorm(o; weight) * act(g)
//
// A step of few tokens is bound by its launches and by the trips to memory inside them: the product of the decays, the
// operands' layout, the update, and the norm with the gate were four launches that each wrote what the next one read.  All of it
// depends on one token and head only.  A workgroup of sixteen waves has a head of a request: the state, dim x vdim floats, is read
// and written once, a wave DIM / 16 rows of it, a lane VDIM / 64 columns, all of it under way while the decays are computed.
// What a state of 128 KB costs a unit is then the bound.
#include "common.h"
#include "api.h"
#include "chunk_scan_impl.h"
#include "log_sigmoid.h"

#include <math.h>

namespace {

constexpr int kStepWaves = 16;
constexpr int kStepThreads = 64 * kStepWaves;

struct StepCall {
    const bf16_t* proj;  // [n_tokens][proj_stride]: q, k, v, g and the decays' bottleneck a of every token
    int64_t proj_stride;
    int q_off, k_off, v_off, g_off, a_off, rank;
    const bf16_t* a2;     // [heads * dim][rank]
    const float* a2_bias; // [heads * dim]
    float* state;         // [n_slots][heads][dim][vdim]
    const int32_t* q_starts;
    const int32_t* seq_slots;
    const float* norm;  // [vdim]
    bf16_t* out;        // [n_tokens][heads * vdim]
    int heads, n_slots;
    float q_scale, inv_tau, eps;
    int act;
};

// The products of eight pairs of bfloat16 added to z.
__device__ __forceinline__ float dot8(uint4 a, uint4 b, float z) {
    const uint32_t x[4] = {a.x, a.y, a.z, a.w}, y[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        z = fmaf(__uint_as_float(x[i] << 16), __uint_as_float(y[i] << 16), z);
        z = fmaf(__uint_as_float(x[i] & 0xffff0000u), __uint_as_float(y[i] & 0xffff0000u), z);
    }
    return z;
}

// CPL consecutive floats, one access
template <int CPL>
struct alignas(4 * CPL) Cols {
    float f[CPL];
};

// ROWS = dim / 16 (key channels a wave), CPL = vdim / 64 (value columns a lane).  grid = (requests, heads)
template <int ROWS, int CPL>
__global__ __launch_bounds__(kStepThreads) void gla_step_kernel(
    const int32_t* q_starts, const int32_t* seq_slots, const bf16_t* proj, int64_t proj_stride, const bf16_t* a2, float* state,
    int n_slots, int heads, int rank, int a_off, int q_off, int k_off, int v_off, int g_off, const float* a2_bias,
    const float* norm, bf16_t* out, float q_scale, float inv_tau, float eps, int act) {
    // (one by one the first of them come with the launch, a struct would not)
    const StepCall c{proj, proj_stride, q_off, k_off, v_off, g_off, a_off, rank, a2, a2_bias, state, q_starts, seq_slots,
                     norm, out, heads, n_slots, q_scale, inv_tau, eps, act};
    constexpr int DIM = 16 * ROWS, VDIM = 64 * CPL;
    typedef Cols<CPL> Vec;
    __shared__ float s_q[DIM], s_k[DIM], s_a[DIM];
    __shared__ float s_part[kStepWaves][VDIM];
    __shared__ float s_sum[CPL];
    const int seq = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int t = c.q_starts[seq];
    const int slot = c.seq_slots[seq];
    if (c.q_starts[seq + 1] != t + 1 || slot < 0 || slot >= c.n_slots) return;  // the same for the whole workgroup
    const bf16_t* row = c.proj + static_cast<int64_t>(t) * c.proj_stride;

    // What the decays need: eight threads a channel, eight values of the bottleneck each.  Asked for before the state, which is
    // under way while they are computed.
    constexpr int ROUNDS = (DIM * 8 + kStepThreads - 1) / kStepThreads;
    const int part = tid & 7;
    uint4 a8[ROUNDS], w8[ROUNDS];
    const bf16_t* ap = row + c.a_off;
    const bf16_t* wp = c.a2 + static_cast<int64_t>(h) * DIM * c.rank;
#pragma unroll
    for (int i = 0; i < ROUNDS; ++i) {
        const int ch = min(i * (kStepThreads / 8) + (tid >> 3), DIM - 1), r = part * 8 < c.rank ? part * 8 : 0;
        a8[i] = *reinterpret_cast<const uint4*>(ap + r);
        w8[i] = *reinterpret_cast<const uint4*>(wp + ch * c.rank + r);
    }
    const int ch0 = min(tid, DIM - 1), col = min(tid, VDIM - 1);
    const float q = to_float(row[c.q_off + h * DIM + ch0]) * c.q_scale, k = to_float(row[c.k_off + h * DIM + ch0]);
    const float bias = c.a2_bias[h * DIM + ch0];
    float* mine = c.state + ((static_cast<int64_t>(slot) * c.heads + h) * DIM + wave * ROWS) * VDIM + lane * CPL;
    Vec S[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) S[r] = *reinterpret_cast<const Vec*>(mine + r * VDIM);
    float v[CPL];
#pragma unroll
    for (int j = 0; j < CPL; ++j) v[j] = to_float(row[c.v_off + h * VDIM + lane * CPL + j]);
    const float gate = to_float(row[c.g_off + h * VDIM + col]), weight = c.norm[col];

#pragma unroll
    for (int i = 0; i < ROUNDS; ++i) {
        const int ch = i * (kStepThreads / 8) + (tid >> 3);
        float z = part * 8 < c.rank ? dot8(a8[i], w8[i], 0.f) : 0.f;
        for (int r = 64 + part * 8; r < c.rank; r += 64)
            z = dot8(*reinterpret_cast<const uint4*>(ap + r), *reinterpret_cast<const uint4*>(wp + min(ch, DIM - 1) * c.rank + r), z);
        z = sum_of_eight(z);
        if (part == 0 && ch < DIM) s_a[ch] = z;
    }
    lds_barrier();
    if (tid < DIM) {
        s_a[tid] = expf(c.inv_tau * log_sigmoid(s_a[tid] + bias));
        s_q[tid] = q;
        s_k[tid] = k;
    }
    lds_barrier();

    float o[CPL];
#pragma unroll
    for (int j = 0; j < CPL; ++j) o[j] = 0.f;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        const float ar = s_a[wave * ROWS + r], kr = s_k[wave * ROWS + r], qr = s_q[wave * ROWS + r];
        Vec out;
#pragma unroll
        for (int j = 0; j < CPL; ++j) {
            const float s = fmaf(ar, S[r].f[j], kr * v[j]);
            o[j] = fmaf(s, qr, o[j]);
            out.f[j] = s;
        }
        *reinterpret_cast<Vec*>(mine + r * VDIM) = out;
    }
#pragma unroll
    for (int j = 0; j < CPL; ++j) s_part[wave][lane * CPL + j] = o[j];
    lds_barrier();
    // a column of o a thread, the waves' shares in their order; then the norm over the head and the gate
    float sum = 0.f;
    if (tid < VDIM) {
#pragma unroll
        for (int w = 0; w < kStepWaves; ++w) sum += s_part[w][tid];
        const float squares = wave_sum(sum * sum);
        if (lane == 0) s_sum[wave] = squares;
    }
    lds_barrier();
    if (tid < VDIM) {
        float total = s_sum[0];
#pragma unroll
        for (int w = 1; w < CPL; ++w) total += s_sum[w];
        const float by = inverse_sqrt(total / static_cast<float>(VDIM) + c.eps);
        c.out[(static_cast<int64_t>(t) * c.heads + h) * VDIM + tid] = from_float<bf16_t>(((sum * by) * weight) * gate_act(gate, c.act));
    }
}

template <int ROWS, int CPL>
void launch_step(const StepCall& c, int n_seqs, hipStream_t stream) {
    gla_step_kernel<ROWS, CPL><<<dim3(n_seqs, c.heads), kStepThreads, 0, stream>>>(
        c.q_starts, c.seq_slots, c.proj, c.proj_stride, c.a2, c.state, c.n_slots, c.heads, c.rank, c.a_off, c.q_off, c.k_off,
        c.v_off, c.g_off, c.a2_bias, c.norm, c.out, c.q_scale, c.inv_tau, c.eps, c.act);
}

template <int ROWS>
void launch_step_cols(int cpl, const StepCall& c, int n_seqs, hipStream_t stream) {
    if (cpl == 1) launch_step<ROWS, 1>(c, n_seqs, stream);
    else if (cpl == 2) launch_step<ROWS, 2>(c, n_seqs, stream);
    else launch_step<ROWS, 4>(c, n_seqs, stream);
}
}  // namespace

// Whether fsie_gla_step takes layers of these sizes.
extern "C" int fsie_gla_step_takes(int heads, int dim, int vdim, int rank) {
    const bool rows = dim == 16 || dim == 32 || dim == 64 || dim == 128 || dim == 256;
    return heads > 0 && heads <= 65535 && rows && (vdim == 64 || vdim == 128 || vdim == 256) && rank > 0 && rank % 8 == 0;
}

// A step of one token a request (every other request of the step is left alone, its rows of out unwritten): proj
// [n_tokens][proj_stride] bfloat16 holds every token's q, k (heads x dim), v, g (heads x vdim) and the decays' bottleneck (rank
// values) from the columns q_off, k_off, v_off, g_off and a_off; a2 [heads * dim][rank] bfloat16 and a2_bias float32 make the decays
// before the sigmoid of the bottleneck; state, q_starts, seq_slots, q_scale and inv_tau as for fsie_gla_scan; out [n_tokens][heads *
// vdim] = the heads' o, normed over vdim (weight `norm`) times act(g).  proj, a2 and state 16-byte aligned, a_off and
// proj_stride multiples of 8.
extern "C" int fsie_gla_step(const void* proj, int64_t proj_stride, int q_off, int k_off, int v_off, int g_off, int a_off, int rank,
                             const void* a2, const float* a2_bias, float* state, const int32_t* q_starts, const int32_t* seq_slots,
                             int n_seqs, const float* norm, void* out, int heads, int dim, int vdim, float q_scale, float inv_tau,
                             float eps, int act, int n_slots, hipStream_t stream) {
    FSIE_REQUIRE(n_seqs >= 0 && n_slots > 0 && fsie_gla_step_takes(heads, dim, vdim, rank),
                 "gla_step: heads of %d x %d, %d of them, a bottleneck of %d", dim, vdim, heads, rank);
    FSIE_REQUIRE(proj && a2 && a2_bias && state && q_starts && seq_slots && norm && out, "gla_step: missing operand");
    FSIE_REQUIRE(FSIE_ACT_KNOWN(act), "gla_step: unknown activation %d", act);
    const int64_t kw = static_cast<int64_t>(heads) * dim, vw = static_cast<int64_t>(heads) * vdim;
    FSIE_REQUIRE(q_off >= 0 && k_off >= 0 && v_off >= 0 && g_off >= 0 && a_off >= 0 && q_off + kw <= proj_stride && k_off + kw <= proj_stride &&
                     v_off + vw <= proj_stride && g_off + vw <= proj_stride && a_off + rank <= proj_stride,
                 "gla_step: the columns do not fit a row of %lld", static_cast<long long>(proj_stride));
    FSIE_REQUIRE(proj_stride % 8 == 0 && a_off % 8 == 0 && reinterpret_cast<uintptr_t>(proj) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(a2) % 16 == 0 && reinterpret_cast<uintptr_t>(state) % 16 == 0,
                 "gla_step: the bottleneck, its matrix and the state must be 16-byte aligned");
    if (n_seqs == 0) return 0;
    const StepCall c{static_cast<const bf16_t*>(proj), proj_stride, q_off, k_off, v_off, g_off, a_off, rank, static_cast<const bf16_t*>(a2),
                     a2_bias, state, q_starts, seq_slots, norm, static_cast<bf16_t*>(out), heads, n_slots, q_scale, inv_tau, eps, act};
    const int cpl = vdim / 64;
    switch (dim) {
        case 16: launch_step_cols<1>(cpl, c, n_seqs, stream); break;
        case 32: launch_step_cols<2>(cpl, c, n_seqs, stream); break;
        case 64: launch_step_cols<4>(cpl, c, n_seqs, stream); break;
        case 128: launch_step_cols<8>(cpl, c, n_seqs, stream); break;
        default: launch_step_cols<16>(cpl, c, n_seqs, stream); break;
    }
    FSIE_CHECK_LAUNCH("gla_step");
    return 0;
}
