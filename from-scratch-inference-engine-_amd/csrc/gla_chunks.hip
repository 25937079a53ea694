// Gated linear attention over portions of prompts: chunks of sixteen tokens on the float32 matrix instruction, runs of eight
// to 32 chunks (segments) side by side.  The recurrence and what a chunk makes of it stand in linear_attention.hip; with B_t the
// sum of log alpha over the chunk's tokens up to and including t, per channel,
//   o_t   = (q_t * exp(B_t))^T S_in + sum_{j <= t} A[t][j] v_j,   A[t][j] = sum_c q_t[c] k_j[c] exp(B_t[c] - B_j[c]),
//   S_out = diag(exp(B_last)) S_in + sum_j (k_j * exp(B_last - B_j)) v_j^T.
// A first kernel lays the scaled q and k, the chunk's decay and A out for every chunk and head.  The walk over a portion's chunks
// is a chain, 128 chunks for a prompt of 2,048 tokens; it is cut into segments, in two launches:
//   1  a portion's first segment, whole, from the request's state; of the segments between first and last what they
//      make of a state: S_end = diag(G) S_begin + L, with L their walk from zero and G the product of their decays
//   2  the segments after the first, each from the state that the ones before it leave, L + G (L' + G' (..)), and the last one's end
//      is the request's state.
// A wave has sixteen value columns and all key channels of a head, or half of them from 129 on: tiles of S in accumulators, whose
// layout is that of the instruction's second operand if step i of a tile takes the channels 4 g + i (g = 0 .. 3).  A chunk is 68
// instructions of 32 cycles for a wave and 128 channels, 0.9 us; its operands, which other dies have written, take some 2 us to come.
// So a chunk's record lies in memory as the waves read it and goes straight to LDS, two chunks ahead in three stages, for all waves of
// a workgroup together.  (In registers, three chunks ahead, the operands are 400 of them a lane and the copies between the two halves of
// the register file took longer than the products; one ahead, a chunk waited 1.7 us.)
// A chunk takes 1.25 us: what is not products is the barrier and the first reads behind it.  It was 1.6 with a wait that counted the
// stores of o among the next chunk's loads, all reads and loads in front of the first product, and S copied once a chunk.
// Two workgroups share a unit, whose matrix cores are then busy most of the time.  With the kernel in front and the norm behind, us,
// fixed decays (retention), one wave per sixteen channels and columns with all chunks in a row / this: 8 heads of 128 x 256,
// 100 tokens 27.8 / 22.6, 200 32.8 / 30.5, 256 35.2 / 34.5, 300 38.0 / 37.0, 500 49 / 43, 2,048 126 / 73, eight prompts of 40 to 200
// 82 / 41; 4 of 64 x 64, 256 25.7 / 22.2, 2,048 94 / 34; 4 of 256 x 512, 256 79 / 60, 2,048 232 / 124; 2 of 256 x 256, 256 55.1 / 54.3,
// three of 5 to 14, which went token by token, 20.0 / 21.1.  With the decays of every channel given: 8 of 128 x 256, 200 33.0 / 32.2,
// 256 35.3 / 36.2, 300 38.1 / 38.9, 500 49.0 / 43.9 (where a bottleneck makes them, the product that goes is 16 us).
#include "common.h"
#include "api.h"
#include "log_sigmoid.h"

#include <math.h>
#include <type_traits>

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kChunk = 16;     // tokens of a chunk: one tile of the matrix instruction
constexpr int kLeastSegment = 8;  // chunks of the shortest segment

// Chunks of a segment of a portion of n chunks, by that number alone: the chain is a segment in each launch, and a segment of the
// second one starts with a pass over the records of those before it.  Up to sixteen chunks one segment: a second launch costs
// more than the half of the chain that it spares (300 tokens, 19 chunks, of 8 heads of 128 x 256 in segments 37.0 us, whole 39.0).
constexpr int kWhole = 16;
__device__ __forceinline__ int segment_of(int n) { return n <= kWhole ? n : n <= 128 ? kLeastSegment : (n <= 512 ? 16 : 32); }
constexpr int kPrepThreads = 256;

__device__ __forceinline__ int chunks_of(int len, int slot, int n_slots) {
    return (len > 0 && slot >= 0 && slot < n_slots) ? (len + kChunk - 1) / kChunk : 0;
}

// The sum over this lane and those below it, of a wave with all lanes active: within rows of sixteen, then over the rows.
__device__ __forceinline__ int sum_up_to_lane(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // from one lane below, two, four, eight; zero beyond the row
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // rows 1 and 3: the last lane of the row before
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // rows 2 and 3: lane 31
    return v;
}

// The requests' portions laid out one after the other, entries(chunks) places each: the request that has a place.
struct Place {
    int seq;     // -1: none
    int chunks;  // of its portion
    int before;  // places of the requests before it
    int first;   // and their chunks
};

// Every wave for itself, all lanes active, the result the same for all lanes.  More than a few requests are read four a lane and added up
// by lanes: one after the other, in every workgroup of both kernels, a step in which 255 requests decode beside a portion of two
// tokens took 960 us a layer of 8 heads of 128 x 256.
template <typename Entries>
__device__ __forceinline__ Place place_of(int place, const int32_t* __restrict__ q_starts, const int32_t* __restrict__ seq_slots, int n_seqs,
                                          int n_slots, Entries entries) {
    constexpr int kSerial = 8, kEach = 4;
    int before = 0, first = 0;
    if (n_seqs <= kSerial) {
        for (int s = 0; s < n_seqs; ++s) {
            const int chunks = chunks_of(q_starts[s + 1] - q_starts[s], seq_slots[s], n_slots), here = entries(chunks);
            if (place < before + here) return Place{s, chunks, before, first};
            before += here, first += chunks;
        }
        return Place{-1, 0, 0, 0};
    }
    const int lane = threadIdx.x & 63;
    for (int s0 = 0; s0 < n_seqs; s0 += 64 * kEach) {
        int starts[kEach + 1], slots[kEach], chunks[kEach], places = 0, sum = 0;
#pragma unroll
        for (int i = 0; i <= kEach; ++i) starts[i] = q_starts[min(s0 + lane * kEach + i, n_seqs)];
#pragma unroll
        for (int i = 0; i < kEach; ++i) slots[i] = seq_slots[min(s0 + lane * kEach + i, n_seqs - 1)];
#pragma unroll
        for (int i = 0; i < kEach; ++i) {  // (past the last request: no tokens)
            chunks[i] = chunks_of(starts[i + 1] - starts[i], slots[i], n_slots);
            places += entries(chunks[i]), sum += chunks[i];
        }
        const int places_to = sum_up_to_lane(places), sum_to = sum_up_to_lane(sum);
        const uint64_t beyond = __ballot(place < before + places_to);
        if (beyond) {
            const int at = __builtin_ctzll(beyond);  // the lane that has the request
            before += __builtin_amdgcn_readlane(places_to - places, at), first += __builtin_amdgcn_readlane(sum_to - sum, at);
            Place found{-1, 0, 0, 0};
#pragma unroll
            for (int i = 0; i < kEach; ++i) {
                const int n = __builtin_amdgcn_readlane(chunks[i], at), here = entries(n);
                if (found.seq < 0 && place < before + here) found = Place{s0 + at * kEach + i, n, before, first};
                before += here, first += n;
            }
            return found;
        }
        before += __builtin_amdgcn_readlane(places_to, 63), first += __builtin_amdgcn_readlane(sum_to, 63);
    }
    return Place{-1, 0, 0, 0};
}

// Work array of one chunk and head, each operand as the lanes 16 g + n of a wave read it, four floats a lane: q * exp(B_t)
// [channels / 16][g][n][4], the token n and the channels 4 g ..; k * exp(B_last - B_t) [channels / 16][g][n][4], the channel n and the
// tokens 4 g ..; exp(B_last) [channels]; A (zero above the diagonal) [g][n][4], the token n and the earlier ones 4 g ..; from a
// multiple of 256 floats on v in float32, [columns / 16][g][n][4], the column n and the tokens 4 g ..
__host__ __device__ constexpr int operand_floats_of(int dp) { return ((2 * kChunk + 1) * dp + kChunk * kChunk + 255) / 256 * 256; }
__host__ __device__ inline int64_t chunk_floats_of(int dp, int vdim) { return operand_floats_of(dp) + (vdim + 15) / 16 * 256; }
__device__ __forceinline__ int a_place(int t, int j) { return ((j >> 2) * 16 + t) * 4 + (j & 3); }
// ... and of a segment: L as the accumulators lie, and G.
__host__ __device__ inline int64_t segment_floats_of(int dp, int vdim) { return static_cast<int64_t>(dp) * ((vdim + 15) / 16 * 16) + dp; }

// Where the decays come from a bottleneck (bfloat16), z = W_a2 a + b: the chunk's own kernel multiplies, 16 tokens by a head's channels
// by rank; as a product of its own that was 16 us a layer of a prompt of 2,048 tokens, and z in memory twice.  a2 null: z is given.
struct Bottleneck {
    const bf16_t* a;      // [n_tokens][a_stride]
    const bf16_t* a2;     // [heads * dim][rank], rank a multiple of 32
    const float* bias;    // [heads * dim]
    int64_t a_stride;
    int rank;
};

struct ChunksCall {
    const void *proj, *qk;
    int64_t proj_stride, qk_stride;
    int q_off, k_off, v_off;
    const float* z;
    float *work, *state, *out;
    const int32_t *q_starts, *seq_slots;
    int n_seqs, n_tokens, max_chunks, heads, dim, vdim, n_slots;
    float q_scale, inv_tau;
    const float* head_decay;
    const float2* cos_sin;
    int pairs;
    Bottleneck from;
    hipStream_t stream;
};

// grid = (heads, upper bound of the step's chunks): a head's records are written on the die (workgroup number modulo 8) that reads
// them.  The logarithms are kept to the base two (the hardware's exponential is
// 2^x).  Every load of a thread goes out before the first is used (the trips one after the other were most of the kernel).  A's
// pairs below the diagonal are two threads each, the diagonal (exponents of zero) the last sixteen threads.
template <typename T, int DP>
__global__ __launch_bounds__(kPrepThreads) void gla_chunk_prep_kernel(
    const int32_t* __restrict__ q_starts, const int32_t* __restrict__ seq_slots, const T* __restrict__ rows, int64_t row_stride,
    const float* __restrict__ z, float* __restrict__ work, int n_seqs, int n_slots, int q_off, int k_off, int heads, int dim,
    const T* __restrict__ v_rows, int64_t v_stride, int vdim, float q_scale, float inv_tau, const float* __restrict__ head_decay, const float2* __restrict__ cos_sin, int pairs, Bottleneck from) {
    constexpr int LD = DP + 4, PER = kChunk * DP / kPrepThreads;
    __shared__ __attribute__((aligned(16))) float qs[kChunk * LD], ks[kChunk * LD], bs[kChunk * LD];
    const int h = blockIdx.x, chunk = blockIdx.y, tid = threadIdx.x;
    const Place at = place_of(chunk, q_starts, seq_slots, n_seqs, n_slots, [](int chunks) { return chunks; });
    const int seq = at.seq, first = at.first;
    if (seq < 0) return;  // the same for the whole workgroup
    const int t0 = q_starts[seq] + (chunk - first) * kChunk;
    const int nt = min(kChunk, q_starts[seq + 1] - t0);
    float* w = work + (static_cast<int64_t>(h) * gridDim.y + chunk) * chunk_floats_of(DP, vdim);
    float* kdT = w + kChunk * DP;
    float* g = kdT + kChunk * DP;
    float* A = g + DP;
    const float to_log2 = inv_tau * 1.44269504088896340736f;

    T q_read[PER], k_read[PER];
    float la[PER];
    const float decay = head_decay ? head_decay[h] : 1.f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {  // (places past the portion's end or the head read a neighbour's value and are zeroed below)
        const int e = tid + i * kPrepThreads, t = t0 + min(e / DP, nt - 1), c = min(e % DP, dim - 1);
        const T* row = rows + static_cast<int64_t>(t) * row_stride + h * dim + c;
        q_read[i] = row[q_off];
        k_read[i] = row[k_off];
        la[i] = head_decay || from.a2 ? 0.f : z[(static_cast<int64_t>(t) * heads + h) * dim + c];
    }
    if constexpr (sizeof(T) == 2) {
        if (from.a2) {
            // D[channel][token], a tile of sixteen channels a wave at a time
            const int lane = tid & 63, n = lane & 15, g4 = lane >> 4;
            const bf16_t* a = from.a + static_cast<int64_t>(t0 + min(n, nt - 1)) * from.a_stride + 8 * g4;
            for (int tile = tid >> 6; tile < DP / 16; tile += kPrepThreads / 64) {
                const bf16_t* w2 = from.a2 + static_cast<int64_t>(h * dim + min(16 * tile + n, dim - 1)) * from.rank + 8 * g4;
                floatx4 sum{0.f, 0.f, 0.f, 0.f}, b4, out;
#pragma unroll
                for (int i = 0; i < 4; ++i) b4[i] = from.bias[h * dim + min(16 * tile + 4 * g4 + i, dim - 1)];
#pragma unroll 2
                for (int s = 0; s < from.rank; s += 32)
                    sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(w2 + s),
                                                                 *reinterpret_cast<const bf16x8*>(a + s), sum, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    out[i] = n < nt && 16 * tile + 4 * g4 + i < dim ? to_log2 * log_sigmoid(sum[i] + b4[i]) : 0.f;
                *reinterpret_cast<floatx4*>(bs + n * LD + 16 * tile + 4 * g4) = out;
            }
        }
    }
    float q[PER], k[PER];
    if (cos_sin) {
        // the first 2 * pairs channels of a head are turned, channel c with channel c + pairs, by (cos, sin); float32.  (No branch a
        // channel: each would be a trip to memory of its own.)
        T q_other[PER], k_other[PER];
        float2 turn[PER];
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int e = tid + i * kPrepThreads, t = t0 + min(e / DP, nt - 1), c = min(e % DP, dim - 1);
            const T* other = rows + static_cast<int64_t>(t) * row_stride + h * dim + (c < pairs ? c + pairs : c < 2 * pairs ? c - pairs : c);
            q_other[i] = other[q_off];
            k_other[i] = other[k_off];
            turn[i] = cos_sin[static_cast<int64_t>(t) * pairs + (c < pairs ? c : min(c - pairs, pairs - 1))];
        }
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int c = min((tid + i * kPrepThreads) % DP, dim - 1);
            const float q1 = to_float(q_read[i]), k1 = to_float(k_read[i]);
            const float q_by = to_float(q_other[i]) * turn[i].y, k_by = to_float(k_other[i]) * turn[i].y;
            q[i] = c < 2 * pairs ? fmaf(q1, turn[i].x, c < pairs ? -q_by : q_by) : q1;
            k[i] = c < 2 * pairs ? fmaf(k1, turn[i].x, c < pairs ? -k_by : k_by) : k1;
        }
    } else {
#pragma unroll
        for (int i = 0; i < PER; ++i) q[i] = to_float(q_read[i]), k[i] = to_float(k_read[i]);
    }
    for (int c = tid; c < (vdim + 15) / 16 * 16; c += kPrepThreads) {  // v, a column a thread
        const T* from = v_rows + static_cast<int64_t>(t0) * v_stride + h * vdim + min(c, vdim - 1);
        float v[kChunk];
#pragma unroll
        for (int t = 0; t < kChunk; ++t) v[t] = to_float(from[min(t, nt - 1) * v_stride]);
        floatx4* to = reinterpret_cast<floatx4*>(w + operand_floats_of(DP)) + (c >> 4) * 64 + (c & 15);
#pragma unroll
        for (int t = 0; t < kChunk; t += 4) {
            floatx4 v4;
#pragma unroll
            for (int u = 0; u < 4; ++u) v4[u] = t + u < nt && c < vdim ? v[t + u] : 0.f;
            to[t * 4] = v4;
        }
    }
    const float log2_decay = log2f(decay);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int e = tid + i * kPrepThreads, t = e / DP, c = e % DP;
        const bool is = t < nt && c < dim;
        qs[t * LD + c] = is ? q[i] * q_scale : 0.f;
        ks[t * LD + c] = is ? k[i] : 0.f;
        if (from.a2) continue;
        bs[t * LD + c] = !is ? 0.f : head_decay ? log2_decay : to_log2 * log_sigmoid(la[i]);
    }
    __syncthreads();
    if (tid < DP) {
        float b[kChunk], sum = 0.f;
#pragma unroll
        for (int t = 0; t < kChunk; ++t) b[t] = bs[t * LD + tid];
#pragma unroll
        for (int t = 0; t < kChunk; ++t) {
            sum += b[t];
            bs[t * LD + tid] = sum;
        }
        float whole = __builtin_amdgcn_exp2f(sum);
        if (head_decay && tid < dim) {
            // a fixed decay: the chunk's decay is its power, by multiplications (it is what the state carries from
            // chunk to chunk, so its rounding adds up over a long prompt)
            whole = 1.f;
#pragma unroll
            for (int t = 0; t < kChunk; ++t) whole *= t < nt ? decay : 1.f;
        }
        g[tid] = whole;
    }
    __syncthreads();
#pragma unroll
    for (int e = tid; e < kChunk * DP / 4; e += kPrepThreads) {  // four neighbouring channels of a token
        const int t = e & 15, c = (e >> 6) * 16 + ((e >> 4) & 3) * 4;
        const floatx4 q4 = *reinterpret_cast<const floatx4*>(qs + t * LD + c), b4 = *reinterpret_cast<const floatx4*>(bs + t * LD + c);
        floatx4 v;
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = q4[u] * __builtin_amdgcn_exp2f(b4[u]);
        *reinterpret_cast<floatx4*>(w + 4 * e) = v;
    }
#pragma unroll
    for (int e = tid; e < kChunk * DP / 4; e += kPrepThreads) {  // four neighbouring tokens of a channel
        const int c = (e >> 6) * 16 + (e & 15), t4 = ((e >> 4) & 3) * 4;
        const float last = bs[(kChunk - 1) * LD + c];
        floatx4 v;
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = ks[(t4 + u) * LD + c] * __builtin_amdgcn_exp2f(last - bs[(t4 + u) * LD + c]);
        *reinterpret_cast<floatx4*>(kdT + 4 * e) = v;
    }
    if (tid < 240) {
        // pair p = tid / 2 of the rows and columns i > j, this thread every other four channels
        const int p = tid >> 1, half = tid & 1;
        int i = static_cast<int>((1.f + sqrtf(static_cast<float>(1 + 8 * p))) * 0.5f);
        i = i * (i - 1) / 2 > p ? i - 1 : ((i + 1) * i / 2 <= p ? i + 1 : i);
        const int j = p - i * (i - 1) / 2;
        float a = 0.f;
        if (head_decay) {  // (one decay for all channels: half the reads of LDS, which are what this takes)
#pragma unroll 4
            for (int c = 4 * half; c < DP; c += 8) {
                const floatx4 q4 = *reinterpret_cast<const floatx4*>(qs + i * LD + c), k4 = *reinterpret_cast<const floatx4*>(ks + j * LD + c);
#pragma unroll
                for (int u = 0; u < 4; ++u) a = fmaf(q4[u], k4[u], a);
            }
            a *= __builtin_amdgcn_exp2f(bs[i * LD] - bs[j * LD]);
        } else {
#pragma unroll 4
            for (int c = 4 * half; c < DP; c += 8) {  // (channels past dim, tokens past the end: q = k = 0)
                const floatx4 q4 = *reinterpret_cast<const floatx4*>(qs + i * LD + c), k4 = *reinterpret_cast<const floatx4*>(ks + j * LD + c);
                const floatx4 x4 = *reinterpret_cast<const floatx4*>(bs + i * LD + c) - *reinterpret_cast<const floatx4*>(bs + j * LD + c);
#pragma unroll
                for (int u = 0; u < 4; ++u) a = fmaf(q4[u] * k4[u], __builtin_amdgcn_exp2f(x4[u]), a);
            }
        }
        a += lane_of<kLaneNeighbour>(a);
        if (half == 0) A[a_place(i, j)] = i < nt ? a : 0.f;
        else A[a_place(j, i)] = 0.f;  // above the diagonal
    } else {
        const int i = tid - 240;
        float a = 0.f;
#pragma unroll 4
        for (int c = 0; c < DP; c += 4) {
            const floatx4 q4 = *reinterpret_cast<const floatx4*>(qs + i * LD + c), k4 = *reinterpret_cast<const floatx4*>(ks + i * LD + c);
#pragma unroll
            for (int u = 0; u < 4; ++u) a = fmaf(q4[u], k4[u], a);
        }
        A[a_place(i, i)] = i < nt ? a : 0.f;
    }
}

// 16 bytes a lane from memory to LDS, lane i's at lds + 16 i.  The instruction takes the LDS address from m0, which is an
// operand here and written by the compiler; the wait state between that and the load is not, inside an asm statement.
__device__ __forceinline__ void load_to_lds(u32x4 rsrc, uint32_t lds, uint32_t offset, uint32_t base) {
    asm volatile(
        "s_nop 0\n\t"
        "buffer_load_dwordx4 %1, %2, %3 offen lds"
        :
        : "{m0}"(lds), "v"(offset), "s"(rsrc), "s"(base)
        : "memory");
}

constexpr int kStores = 4;                 // of a chunk's o, a wave: a lane has four tokens of a column
constexpr uint32_t kNowhere = 0x7fff0000u;  // behind the end of any sixteen rows of o, also with four rows added to it

template <int NT, int HALVES>
struct Stages {
    static constexpr int kWaves = 4 * HALVES;
    static constexpr int kOperands = operand_floats_of(16 * NT * HALVES) / 256;  // loads of 1 KB (256 floats) of a chunk's record: the operands,
    static constexpr int kLoads = (kOperands + 4 + kWaves - 1) / kWaves;         // v of four tiles; a wave's share (the last ones twice)
    static constexpr int kFloats = kWaves * kLoads * 256;                        // a stage
    static constexpr int kStages = 3;  // (two workgroups of 72 KB a unit for heads of 128, one of 128 KB for 256)
    static constexpr int kSwap = HALVES == 1 ? 0 : 2 * 4 * 256;  // floats: the second halves' o of two chunks
    static constexpr int kBytes = (kStages * kFloats + kSwap) * 4;
};

// grid = (heads, value columns / 64, upper bound of the launch's segments), a wave sixteen columns: workgroups without a segment come
// last (one in two among the others, they left half of every die's units to them, and the rest in two rounds).  NT: a wave's tiles of
// sixteen channels.  HALVES 2: heads of more than 128 channels, four waves more with the other half of the channels; their o goes to
// the first four through LDS, behind the next chunk's barrier.  LATER: the second launch.
template <int NT, int HALVES, bool LATER>
__global__ __launch_bounds__(256 * HALVES, 2) void gla_segment_kernel(
    const int32_t* __restrict__ q_starts, const int32_t* __restrict__ seq_slots, const float* __restrict__ work, float* segments,
    float* __restrict__ state, float* __restrict__ out, int n_seqs, int n_slots, int max_chunks, int heads, int dim, int vdim) {
    constexpr int DP = 16 * NT * HALVES;
    using St = Stages<NT, HALVES>;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int h = blockIdx.x, place = blockIdx.z, lane = threadIdx.x & 63, n = lane & 15, g4 = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int half = wave / 4, column = wave % 4, ch0 = half * 16 * NT;  // (this wave's tile of columns, its first channel)
    const int tiles = (vdim + 15) / 16, tile0 = static_cast<int>(blockIdx.y) * 4, tile = min(tile0 + column, tiles - 1);
    const int col = tile * 16 + n;
    const bool tile_ok = tile0 + column < tiles;  // (waves past the last tile repeat it and write nothing)
    const bool col_ok = tile_ok && col < vdim;
    // the request and the segment
    const Place at = place_of(place, q_starts, seq_slots, n_seqs, n_slots, [](int chunks) {
        const int len = max(1, segment_of(chunks)), segs = (chunks + len - 1) / len;
        return LATER ? max(0, segs - 1) : (segs > 1 ? segs - 1 : segs);
    });
    const int seq = at.seq, seg = place - at.before + (LATER ? 1 : 0), n_chunks = at.chunks, first = at.first;
    if (seq < 0) return;  // the same for the whole workgroup
    const int length = segment_of(n_chunks), begin = seg * length, end = min(n_chunks, begin + length);
    const bool last = end == n_chunks;
    const bool whole = LATER || seg == 0;  // o too, not only what the segment makes of a state
    const int lo = q_starts[seq], hi = q_starts[seq + 1], slot = seq_slots[seq];

    // the chunks' records to LDS: this wave's share of the loads
    const int64_t per_chunk = chunk_floats_of(DP, vdim);
    const float* w = work + (static_cast<int64_t>(h) * max_chunks + first) * per_chunk;
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds);
    uint32_t from[St::kLoads];
#pragma unroll
    for (int i = 0; i < St::kLoads; ++i) {
        const int j = wave * St::kLoads + i;
        from[i] = (j < St::kOperands ? j : St::kOperands + min(tile0 + j - St::kOperands, tiles - 1)) * 1024u + lane * 16u;
    }
    // a chunk's record (past the end the last one's once more) to stage `stage`, in loads that may be asked for one by one
    u32x4 rsrc;
    uint32_t to;
    auto bring_from = [&](int ci, int stage) {
        const uint64_t from_w = reinterpret_cast<uint64_t>(w + min(ci, end - 1) * per_chunk);
        rsrc[0] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(from_w));
        rsrc[1] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(from_w >> 32));
        rsrc[2] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(chunk_floats_of(DP, vdim) * 4));
        rsrc[3] = 0x00020000u;
        to = lds0 + static_cast<uint32_t>(stage) * (St::kFloats * 4) + wave * St::kLoads * 1024u;
    };
    auto bring_load = [&](int i) { load_to_lds(rsrc, to + i * 1024u, from[i], 0u); };
    auto bring_first = [&]() {
#pragma unroll
        for (int u = 0; u < St::kStages - 1; ++u) {
            bring_from(begin + u, u);
#pragma unroll
            for (int i = 0; i < St::kLoads; ++i) bring_load(i);
        }
    };

    // Segment records: that of the segment that starts at chunk c of the step is number c / 8 (segments that are not a portion's
    // last are eight chunks and longer, so no two have the same).
    const int64_t record = segment_floats_of(DP, vdim);
    const int64_t my_l = ((static_cast<int64_t>(tile) * HALVES + half) * NT * 64 + lane) * 4, my_g = static_cast<int64_t>(tiles) * 16 * DP + ch0 + 4 * g4;
    auto record_of = [&](int s) { return segments + (static_cast<int64_t>((first + s * length) / kLeastSegment) * heads + h) * record; };
    float* my_state = state + (static_cast<int64_t>(slot) * heads + h) * dim * vdim + min(col, vdim - 1);
    floatx4 S[NT];  // the channels ch0 + 16 t + 4 g4 + i of the column n
    if (LATER || !whole) bring_first();
    if (!LATER && whole) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) S[t][i] = my_state[static_cast<int64_t>(min(ch0 + 16 * t + 4 * g4 + i, dim - 1)) * vdim];
        // (every load stands for itself: left to the choice between it and zero, it would move behind it, a branch and a trip each)
#pragma unroll
        for (int t = 0; t < NT; ++t) asm volatile("" : "+v"(S[t]));
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) S[t][i] = (col_ok && ch0 + 16 * t + 4 * g4 + i < dim) ? S[t][i] : 0.f;
        __builtin_amdgcn_sched_barrier(0);
        bring_first();
    } else if (!LATER) {
#pragma unroll
        for (int t = 0; t < NT; ++t) S[t] = floatx4{0.f, 0.f, 0.f, 0.f};
    } else {
        const float* r = record_of(0) + my_l;
#pragma unroll
        for (int t = 0; t < NT; ++t) S[t] = *reinterpret_cast<const floatx4*>(r + t * 256);
#pragma unroll 2
        for (int s = 1; s < seg; ++s) {
            const float* of = record_of(s);
            floatx4 l4[NT], d4[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                l4[t] = *reinterpret_cast<const floatx4*>(of + my_l + t * 256);
                d4[t] = *reinterpret_cast<const floatx4*>(of + my_g + 16 * t);
            }
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) S[t][i] = fmaf(d4[t][i], S[t][i], l4[t][i]);
        }
    }
    floatx4 decays[NT];  // of the chunks so far (a segment between first and last)
#pragma unroll
    for (int t = 0; t < NT; ++t) decays[t] = floatx4{1.f, 1.f, 1.f, 1.f};

    const int64_t out_stride = static_cast<int64_t>(heads) * vdim;
    const uint32_t row_bytes = static_cast<uint32_t>(out_stride) * 4u;
    const uint32_t my_out = col_ok ? 4u * g4 * row_bytes + static_cast<uint32_t>(h * vdim + col) * 4u : kNowhere;
    // The walk, one for segments that leave o (WHOLE) and one for the others: in one loop with a branch S would be copied from
    // register to register once a chunk
    auto walk = [&](auto leaves_o) {
        constexpr bool WHOLE = decltype(leaves_o)::value;
        // o of chunk ci: kStores stores, whatever the lanes; the descriptor ends behind the portion's last token, or the chunk's
        auto store_o = [&](int ci, floatx4 sum) {
            const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(
                out + (lo + static_cast<int64_t>(ci) * kChunk) * out_stride, 0, min(kChunk, hi - lo - ci * kChunk) * row_bytes, 0x00020000);
#pragma unroll
            for (int i = 0; i < kStores; ++i)
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(sum[i]), rows, my_out + i * row_bytes, 0, 0);
        };
        float* swap = lds + St::kStages * St::kFloats + column * 256 + 4 * lane;
        floatx4 mine{0.f, 0.f, 0.f, 0.f};  // HALVES 2: this half's o of the chunk before
        auto both_halves = [&](int ci) { return mine + *reinterpret_cast<const floatx4*>(swap + (ci & 1) * 1024); };
        int stage = 0;
        for (int ci = begin; ci < end; ++ci) {
            // This chunk's loads have arrived: everything but what was asked for after them, the loads of kStages - 2 chunks and the
            // kStores stores of a chunk (none yet in front of the first, of the first two with halves).  The counter goes down in the
            // order of issue, so to leave the stores out would be to wait for most of the next chunk's loads too
            if (WHOLE && half == 0 && ci >= begin + HALVES)
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(St::kLoads * (St::kStages - 2) + kStores) : "memory");
            else
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(St::kLoads * (St::kStages - 2)) : "memory");
            bring_from(ci + St::kStages - 1, stage == 0 ? St::kStages - 1 : stage - 1);  // the stage that every wave has read before this barrier
            const float* c = lds + stage * St::kFloats;
            stage = stage == St::kStages - 1 ? 0 : stage + 1;
            if (WHOLE && HALVES == 2 && half == 0 && ci > begin) store_o(ci - 1, both_halves(ci - 1));
            // The operands of o asked for first; those of S, and the loads of the chunk after next, while o's products run (74 KB of
            // reads and 24 loads of a workgroup in front of the first product were a quarter of a chunk's time)
            floatx4 k4[NT], g[NT];
            const floatx4 v4 = *reinterpret_cast<const floatx4*>(c + St::kOperands * 256 + column * 256 + 4 * lane);
            auto read_of_state = [&](int t) {
                g[t] = *reinterpret_cast<const floatx4*>(c + 2 * kChunk * DP + ch0 + 16 * t + 4 * g4);
                k4[t] = *reinterpret_cast<const floatx4*>(c + kChunk * (DP + ch0) + t * 256 + 4 * lane);
            };
            floatx4 o[2] = {floatx4{0.f, 0.f, 0.f, 0.f}, floatx4{0.f, 0.f, 0.f, 0.f}};  // two sums that do not wait for each other
            if constexpr (WHOLE) {
                floatx4 q4[NT];
#pragma unroll
                for (int t = 0; t < NT; ++t) q4[t] = *reinterpret_cast<const floatx4*>(c + kChunk * ch0 + t * 256 + 4 * lane);
                const floatx4 a4 = *reinterpret_cast<const floatx4*>(c + (2 * kChunk + 1) * DP + 4 * lane);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int t = 0; t < NT; ++t) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) o[i & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(q4[t][i], S[t][i], o[i & 1], 0, 0, 0);
                    read_of_state(t);
#pragma unroll
                    for (int i = t * St::kLoads / NT; i < (t + 1) * St::kLoads / NT; ++i) bring_load(i);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (half == HALVES - 1) {  // (one half's; the first has the stores)
#pragma unroll
                    for (int m = 0; m < 4; ++m) o[m & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a4[m], v4[m], o[m & 1], 0, 0, 0);
                }
            } else {
#pragma unroll
                for (int t = 0; t < NT; ++t) read_of_state(t);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < St::kLoads; ++i) bring_load(i);
#pragma unroll
                for (int t = 0; t < NT; ++t) decays[t] *= g[t];
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) S[t] *= g[t];
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int t = 0; t < NT; ++t) S[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(k4[t][m], v4[m], S[t], 0, 0, 0);
            if constexpr (WHOLE) {
                mine = o[0] + o[1];
                if (HALVES == 1) store_o(ci, mine);
                else if (half == 1) *reinterpret_cast<floatx4*>(swap + (ci & 1) * 1024) = mine;
            }
        }
        if (WHOLE && HALVES == 2) {
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            if (half == 0) store_o(end - 1, both_halves(end - 1));
        }
    };
    if (LATER || whole) walk(std::true_type{});
    else walk(std::false_type{});
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (no load may still write LDS when the workgroup's is given away)
    if (!tile_ok) return;
    if (last) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = ch0 + 16 * t + 4 * g4 + i;
                if (col_ok && row < dim) my_state[static_cast<int64_t>(row) * vdim] = S[t][i];
            }
    } else if (!LATER) {
        float* of = record_of(seg);
#pragma unroll
        for (int t = 0; t < NT; ++t) *reinterpret_cast<floatx4*>(of + my_l + t * 256) = S[t];
        if (!whole && tile == 0 && n == 0) {
#pragma unroll
            for (int t = 0; t < NT; ++t) *reinterpret_cast<floatx4*>(of + my_g + 16 * t) = decays[t];
        }
    }
}

template <int NT, int HALVES, bool LATER>
int launch_segments(const ChunksCall& c, int n) {
    constexpr int bytes = Stages<NT, HALVES>::kBytes;
    static const hipError_t allowed = hipFuncSetAttribute(reinterpret_cast<const void*>(&gla_segment_kernel<NT, HALVES, LATER>),
                                                          hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    FSIE_REQUIRE(allowed == hipSuccess, "gla_scan: %d bytes of LDS: %s", bytes, hipGetErrorString(allowed));
    gla_segment_kernel<NT, HALVES, LATER><<<dim3(c.heads, (c.vdim + 63) / 64, n), 256 * HALVES, bytes, c.stream>>>(
        c.q_starts, c.seq_slots, c.work, c.work + c.max_chunks * chunk_floats_of(16 * NT * HALVES, c.vdim) * c.heads, c.state, c.out, c.n_seqs,
        c.n_slots, c.max_chunks, c.heads, c.dim, c.vdim);
    return 0;
}

template <typename T, int NT, int HALVES>
int launch(const ChunksCall& c) {
    constexpr int DP = 16 * NT * HALVES;
    const T* rows = static_cast<const T*>(c.qk ? c.qk : c.proj);
    gla_chunk_prep_kernel<T, DP><<<dim3(c.heads, c.max_chunks), kPrepThreads, 0, c.stream>>>(
        c.q_starts, c.seq_slots, rows, c.qk ? c.qk_stride : c.proj_stride, c.z, c.work, c.n_seqs, c.n_slots, c.q_off, c.k_off, c.heads,
        c.dim, static_cast<const T*>(c.proj) + c.v_off, c.proj_stride, c.vdim, c.q_scale, c.inv_tau, c.head_decay, c.cos_sin, c.pairs,
        c.from);
    // segments that are not a portion's last are eight chunks and longer: at most max_chunks / 8 of them, and none where no
    // portion can have more than sixteen chunks
    const int inner = c.n_tokens > kWhole * kChunk ? c.max_chunks / kLeastSegment : 0;
    int status = launch_segments<NT, HALVES, false>(c, c.n_seqs + inner);
    if (status == 0 && inner > 0) status = launch_segments<NT, HALVES, true>(c, inner);
    if (status) return status;
    FSIE_CHECK_LAUNCH("gla_chunks");
    return 0;
}

// Channels of a head as they are computed: a wave's one to eight sixteens, twice as many from 129 on (in one wave the chain of a chunk is
// 132 instructions: 4 heads of 256 x 512, 256 tokens 79 us, 2,048 160; in two 60 and 124).  Six sixteens, where eight would be a quarter
// of zeros: 12 heads of 96 x 192, 300 tokens 41 us padded to 128, 35 so.
int padded_dim(int dim) {
    for (int dp : {16, 32, 64, 96, 128, 192})
        if (dim <= dp) return dp;
    return 256;
}

template <typename T>
int launch_dim(const ChunksCall& c) {
    switch (padded_dim(c.dim)) {
        case 16: return launch<T, 1, 1>(c);
        case 32: return launch<T, 2, 1>(c);
        case 64: return launch<T, 4, 1>(c);
        case 96: return launch<T, 6, 1>(c);
        case 128: return launch<T, 8, 1>(c);
        case 192: return launch<T, 6, 2>(c);
        default: return launch<T, 8, 2>(c);
    }
}

}  // namespace

// Floats of work that a chunk of sixteen tokens needs for a layer of these sizes, its share of the segments' records included.
extern "C" int64_t fsie_gla_chunk_floats(int heads, int dim, int vdim) {
    const int dp = padded_dim(dim);
    return heads * chunk_floats_of(dp, vdim) + (heads * segment_floats_of(dp, vdim) + kLeastSegment - 1) / kLeastSegment;
}

// All portions of the step, chunk by chunk, for fsie_gla_scan (which has checked the operands): work has room for max_chunks
// chunks, out is [n_tokens][heads * vdim].  a2 (or null): the decays before the sigmoid are made here, z is not read.
extern "C" int fsie_gla_chunks(const void* proj, int64_t proj_stride, int q_off, int k_off, int v_off, const float* z, float* state,
                               const int32_t* q_starts, const int32_t* seq_slots, int n_seqs, int n_tokens, float* out, float* work,
                               int max_chunks, int heads, int dim, int vdim, float q_scale, float inv_tau, int n_slots, int dtype,
                               const float* head_decay, const void* qk, int64_t qk_stride, const float* cos_sin, int rot_pairs,
                               const void* a, int64_t a_stride, const void* a2, const float* a2_bias, int rank, hipStream_t stream) {
    FSIE_REQUIRE(max_chunks >= n_tokens / kChunk + n_seqs, "gla_scan: room for %d chunks, the step may have %d", max_chunks,
                 n_tokens / kChunk + n_seqs);
    FSIE_REQUIRE(n_seqs <= 65535 && heads <= 65535 && (vdim + 63) / 64 <= 65535, "gla_scan: too many requests, heads or columns");
    FSIE_REQUIRE(static_cast<int64_t>(heads) * vdim * 4 * kChunk < kNowhere, "gla_scan: a row of o of %d x %d values", heads, vdim);
    FSIE_REQUIRE(reinterpret_cast<uintptr_t>(work) % 16 == 0 && dim <= 256, "gla_scan: the work array must be 16-byte aligned");
    FSIE_REQUIRE(!a2 || (dtype == FSIE_BF16 && !head_decay && a && a2_bias && rank > 0 && rank % 32 == 0 && a_stride >= rank && a_stride % 8 == 0 &&
                         (reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(a2)) % 16 == 0),
                 "gla_scan: a bottleneck of %d in rows of %lld: bfloat16, a multiple of 32, on 16 bytes", rank, static_cast<long long>(a_stride));
    const ChunksCall c{proj, qk, proj_stride, qk_stride, q_off, k_off, v_off, z, work, state, out, q_starts, seq_slots, n_seqs,
                       n_tokens, n_tokens / kChunk + n_seqs, heads, dim, vdim, n_slots, q_scale, inv_tau, head_decay,
                       rot_pairs > 0 ? reinterpret_cast<const float2*>(cos_sin) : nullptr, rot_pairs,
                       Bottleneck{static_cast<const bf16_t*>(a), static_cast<const bf16_t*>(a2), a2_bias, a_stride, rank}, stream};
    return dtype == FSIE_F32 ? launch_dim<float>(c) : launch_dim<bf16_t>(c);
}
