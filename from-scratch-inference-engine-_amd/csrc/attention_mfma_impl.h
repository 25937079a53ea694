// Causal grouped-query attention over the pages of the cache on the matrix cores (bfloat16).
//
// One workgroup per work item and kv head (chunk).  Everything is computed transposed so that no
// operand ever has to change lanes or pass through LDS:
//
//   S^T[key, row] = K[key, :] . Q[row, :]      A = K rows from the cache (16 B per lane),
//                                              B = Q rows, kept in registers for the whole item
//   softmax over the keys of a column: 8 keys per lane, the rest by two lane swaps (16, 32)
//   O^T[d, row]  += V^T[d, key] . P^T[key, row] A = V^T from the cache, which stores values
//                                              transposed ([head_dim][slot]: 8 consecutive keys of
//                                              one dimension are one 16-byte load),
//                                              B = P^T, which is exactly the layout in which the
//                                              first product left S^T
//
// Keys are walked in blocks of 32, scored as two tiles of 16.  Row c of tile t is key
// 8 (c / 4) + 4 t + c % 4 of the block: lane group G then holds, over the two tiles, the scores of
// the keys 8 G .. 8 G + 7 in order, which is the B operand of one v_mfma_f32_16x16x32_bf16 over
// the block's 32 keys.
//
// The running maximum and sum of a query row and its accumulators live in the same lanes
// (column = lane % 16), so the online-softmax rescale is lane-local.  Scores use
// v_mfma_f32_16x16x32_bf16 over the head dimension (16x16x16 steps when head_dim is an odd
// multiple of 16, on an accumulator of their own).
//
// HDT = head_dim / 16, NT = column tiles of 16 query rows per wave (rows = tokens x heads of the
// kv head's group).  Requires page_size % 4 == 0; with a page size that is a multiple of 8 a
// lane's 8 values of a dimension come with one load instead of two.
//
// One query tile: an item's blocks are dealt to the waves of its workgroup, a block a wave where the item is short, and the
// waves' results meet in LDS, in the fixed order of the waves, behind one barrier.  Decoding against a long context needs
// neither partial records in memory nor a second kernel, and the result does not depend on timing.
// Such a step is bound by the chain inside a workgroup: the item, the block table, the keys, one trip to memory each, then
// products and exponentials that wait for each other.  So no wave takes two blocks where another has none (unless the workgroups are
// more than the units anyway, where the memory's rate bounds it and fewer waves a workgroup keep more of them under way), masks are selects (no
// branch a value), and little code is run once: 10 KB of instructions, not 31.  One request of the 0.5B shape and 60 to 110
// keys 7.2 -> 4.5 us from a workgroup's first instruction to its last, eight of the 7B shape and 64 to 550 6.6 -> 5.0.
// Several query tiles (NT > 1, up to 4 waves): a wave per 512 keys, combined by the first wave.
//
// QKV: the variant for steps of one token a request takes q, k and v as the float32 partial sums
// that a product in slices of K leaves, and finishes them itself: every workgroup adds up the
// heads it needs (its queries, and its kv head's key and value), adds the bias, rotates queries
// and key, and the workgroup whose keys end with the new one scores it from registers and writes
// it and its value into the pools.  That spares the launch between the product and attention.
//
// OROWS > 0: the same with the output projection behind it, for one or two tokens whose items are short and whole.  Such a step is
// bound by its launches and by the chain inside each; the projection's own kernel was 3.9 us a layer, of which its chain is a trip for the weight.
// So every workgroup makes the whole attention of a kv head (a few tens of keys, from the caches) and then multiplies the heads, rounded to
// 16 bits in LDS, by a few rows of the projection, which it has asked for in front of the first barrier: float32 sums
// [n_kv][tokens][o_rows], one slice a kv head, for the norm that adds them up.  One request of the 0.5B shape and 30 to 100 keys: attention and
// projection 8.6 -> 6.8 us a layer, the step 565 -> 520; two requests 591 -> 562.  Where the workgroups are more than the units attention is made
// in turns and the two launches are faster (the rule is fsie_attention_mfma_qkv_o_rows), and so it is with items of more waves (600
// keys 17.3 ms for 24 steps, 16.1 cut and merged).  The widest form (heads of 128, four rows a wave: a unit holds five waves, so 256 registers a wave, and 64 of
// them are the weight's) keeps 16 registers in scratch, 36 bytes a lane; it is faster than the two launches all the same: 16 steps of one request, ms, 2,048 wide, 16 on 2 of
// 128 6.49 / 6.35, 2,560 wide, 20 on 2 7.03 / 6.89, 1,024 wide, 16 on 4 5.95 / 5.58, two requests 2,560 wide, 8 on 1 6.96 / 6.80.
#pragma once

#include "common.h"
#include "api.h"

#include <limits.h>
#include <math.h>

namespace fsie_attn {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short shortx4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

union F16B {
    uint4 raw;
    bf16x8 v;
};
union F8B {
    uint2 raw;
    shortx4 v;
};

__device__ __forceinline__ uint4 ld16(const bf16_t* p) { return *reinterpret_cast<const uint4*>(p); }
// the same as a streaming load: for data that is read once and whose whole lines one load of a wave covers
__device__ __forceinline__ uint4 ld16_once(const bf16_t* p) {
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    const u4 v = __builtin_nontemporal_load(reinterpret_cast<const u4*>(p));
    return uint4{v[0], v[1], v[2], v[3]};
}
__device__ __forceinline__ uint2 ld8(const bf16_t* p) { return *reinterpret_cast<const uint2*>(p); }

// What the QKV variant reads and writes beside the kernel's other operands.
struct QkvSums {
    const float* sums;     // [n_parts][n_tokens][width], width = (n_heads + 2 n_kv) head_dim
    const float* bias;     // [width], or null
    const float* cos_sin;  // [n_tokens][head_dim / 2] pairs (cos, sin) of each token's position, or null: no rotation
    const int32_t* slots;  // [n_tokens] slot of a token's key and value in the pools (negative: nowhere); the kernel has it in the place of q
    bf16_t* k_out;         // the pools again, to write
    bf16_t* v_out;
    int64_t part_stride;   // n_tokens * width
    int64_t pool_slots;
    int n_parts, width;
    const float* sinks;    // [n_heads] or null: exp(sink) joins every row's denominator (any variant)
    float softcap;         // > 0: the scaled scores become softcap * tanh(score / softcap) (any variant); 0: as they are
    const float* slopes;     // [n_heads] or null: slopes[h] * (query position - key position) is taken off the (capped)
                             // scores of head h (any variant)
    const float* row_scale;  // [n_tokens] or null: a factor on all scores of a token, before the cap (any variant)
    // the variant with the output projection: its weight [o_rows][n_heads head_dim] in rows, and the sums that it leaves [n_kv][n_tokens][o_rows]
    const bf16_t* o_weight;
    float* o_sums;
    int64_t o_part_stride;   // n_tokens * o_rows
    int o_rows;
    int group;               // heads a kv head (any variant)
    uint32_t page_magic;     // 2^32 / page_size, rounded up: a key's page by one multiplication (any variant)
};

inline uint32_t magic_of(int page_size) { return 0xFFFFFFFFu / static_cast<uint32_t>(page_size) + 1u; }

// Element d of a head after the rotation of the pairs (i, i + HD / 2) by the angles whose
// cosines and sines are cs[i].  One fixed sequence of roundings, whoever asks: the key that a
// step scores from registers and its copy in the cache are the same numbers.
__device__ __forceinline__ float rotated_by(float a, float b, float cosine, float sine, bool hi) {
    const float bs = __fmul_rn(b, sine);
    return __fmaf_rn(a, cosine, hi ? bs : -bs);
}
template <int HD>
__device__ __forceinline__ float rotated(const float* head, const float2* cs, int d) {
    constexpr int half = HD / 2;
    const bool hi = d >= half;
    const float2 t = cs[hi ? d - half : d];
    return rotated_by(head[d], head[hi ? d - half : d + half], t.x, t.y, hi);
}
// The same for the elements d0 .. d0 + 7 (d0 a multiple of 8), as two bfloat16 a register: 16-byte reads.
template <int HD>
__device__ __forceinline__ uint4 rotated8(const float* head, const float2* cs, int d0) {
    constexpr int half = HD / 2;
    const bool hi = d0 >= half;
    const float4* a = reinterpret_cast<const float4*>(head + d0);
    const float4* b = reinterpret_cast<const float4*>(head + (hi ? d0 - half : d0 + half));
    const float4* t = reinterpret_cast<const float4*>(cs + (hi ? d0 - half : d0));
    const float4 a0 = a[0], a1 = a[1], b0 = b[0], b1 = b[1], t0 = t[0], t1 = t[1], t2 = t[2], t3 = t[3];
    return uint4{pack2_bf16(rotated_by(a0.x, b0.x, t0.x, t0.y, hi), rotated_by(a0.y, b0.y, t0.z, t0.w, hi)),
                 pack2_bf16(rotated_by(a0.z, b0.z, t1.x, t1.y, hi), rotated_by(a0.w, b0.w, t1.z, t1.w, hi)),
                 pack2_bf16(rotated_by(a1.x, b1.x, t2.x, t2.y, hi), rotated_by(a1.y, b1.y, t2.z, t2.w, hi)),
                 pack2_bf16(rotated_by(a1.z, b1.z, t3.x, t3.y, hi), rotated_by(a1.w, b1.w, t3.z, t3.w, hi))};
}

// A bit for each of eight consecutive keys that is among the first n (n of any sign).
__device__ __forceinline__ uint32_t keys_below(int n) { return (1u << min(max(n, 0), 8)) - 1u; }

constexpr int kFarBelow = INT_MIN / 2;  // below every key

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

template <int HDT>
constexpr int max_waves() {
    return HDT <= 4 ? 16 : (HDT <= 8 ? 8 : 4);  // registers per wave grow with the head size
}
// The variant for items of up to four blocks of keys (what a step with idle compute units is cut into): a wave a block, and
// with QKV one more for the new key.
constexpr int kShortWaves = 4;

// BIASED false: no distance bias and no factor a token, known when the kernel is compiled (the QKV variants have no
// registers to spare for them); true: whatever slopes and row_scale say.
// ONCE: values by streaming loads: where several waves walk long runs of keys, and where more workgroups than units read more than
// the caches hold; the short items of a few workgroups are slower with them.
// OROWS > 0: each wave multiplies the heads of the workgroup by so many rows of the output projection (below).
template <int HDT, int NT, int MAXW, bool V16, bool QKV = false, bool BIASED = true, bool ONCE = (MAXW > kShortWaves + 1), int OROWS = 0>
__global__ __launch_bounds__(64 * MAXW) __attribute__((amdgpu_waves_per_eu(MAXW == 1 && NT > 1 ? 2 : 1))) void attention_mfma_kernel(
    const bf16_t* __restrict__ q, int64_t q_stride, const bf16_t* __restrict__ k_pool,
    const bf16_t* __restrict__ v_pool, const int32_t* __restrict__ block_tables, int max_pages,
    const int32_t* __restrict__ items, bf16_t* __restrict__ out, float* __restrict__ partials, int n_heads,
    int n_kv, int page_size, int window, float scale, int gh, QkvSums f) {
    static_assert(!QKV || (NT == 1 && HDT % 2 == 0), "the QKV variant: one query tile, head_dim a multiple of 32");
    static_assert(OROWS == 0 || (QKV && HDT <= 8), "the output projection: behind the QKV variant, whose heads in LDS make room for the result");
    constexpr int HD = HDT * 16;
    // scores: 32-wide steps over the head dimension when head_dim is a multiple of 32, else
    // 16-wide steps throughout (the two shapes are never chained on one accumulator)
    constexpr bool X32 = (HDT % 2) == 0;
    constexpr int S32 = X32 ? HDT / 2 : 0;
    constexpr int S16 = X32 ? 0 : HDT;
    constexpr int S32A = S32 > 0 ? S32 : 1;
    constexpr int S16A = S16 > 0 ? S16 : 1;

    const int32_t* item = items + static_cast<int64_t>(OROWS > 0 ? blockIdx.z : blockIdx.x) * FSIE_ATTN_ITEM_INTS;
    // (the item in one scalar load: its fields one by one are trips of their own, each behind the last one's use)
    typedef int ItemInts __attribute__((ext_vector_type(8), aligned(4)));
    static_assert(FSIE_ATTN_ITEM_INTS == 8, "an item is eight numbers");
    const ItemInts it = *reinterpret_cast<const ItemInts*>(item);
    // (the arguments beyond those that come with the launch on the same trip: left alone, the compiler asks for them behind the item, where they are used,
    // on three trips more.  One request of the 0.5B shape 520 us a step, 515 so)
    if constexpr (QKV)
        asm volatile("" ::"s"(f.sums), "s"(f.bias), "s"(f.cos_sin), "s"(f.k_out), "s"(f.v_out), "s"(f.part_stride), "s"(f.n_parts), "s"(f.width),
                     "s"(f.group), "s"(f.page_magic), "s"(n_heads), "s"(n_kv), "s"(page_size), "s"(window), "s"(gh), "s"(scale));
    const int seq = it[FSIE_ATTN_ITEM_SEQ];
    const int q_row0 = it[FSIE_ATTN_ITEM_QROW];
    const int n_q = it[FSIE_ATTN_ITEM_NQ];
    const int pos0 = it[FSIE_ATTN_ITEM_POS];
    const int key_begin = it[FSIE_ATTN_ITEM_KBEGIN];
    int key_end = it[FSIE_ATTN_ITEM_KEND];
    const int partial_base = it[FSIE_ATTN_ITEM_PARTIAL];
    if (n_q <= 0) return;  // padding item
    // The first keys of the request that a window keeps: seen whatever the window says.  An item told to
    // (FSIE_ATTN_KEEP_WALK) reads those that lie before its own range too, [0, prefix_end), as blocks of
    // their own ahead of the range's blocks.
    const int keep = it[FSIE_ATTN_ITEM_KEEP] & ~FSIE_ATTN_KEEP_WALK;
    const int prefix_end = (it[FSIE_ATTN_ITEM_KEEP] & FSIE_ATTN_KEEP_WALK) ? min(keep, key_begin) : 0;
    // QKV: the item whose keys end with the request's new one walks the cache up to it and takes
    // the new key and value from the sums
    const bool owner = QKV && pos0 >= key_begin && pos0 < key_end;
    if (owner) key_end = pos0;
    int new_slot = -1;
    if constexpr (QKV) new_slot = reinterpret_cast<const int32_t*>(q)[q_row0];  // (there are no queries: what stands there is where tokens go)

    const int group = f.group;
    const int kvh = blockIdx.y, chunk = OROWS > 0 ? 0 : blockIdx.z;
    const int gh_here = min(gh, group - chunk * gh);
    const int h_base = kvh * group + chunk * gh;
    const int n_rows = n_q * gh;

    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    // (one tile: always launched so.  blockDim is a load that the keys of a wave wait for: 1 request of 100 keys of 64 values and 8 of
    // 64 to 550 of 128, 5.5 and 6.6 us with it, 5.2 and 6.1 without)
    const int n_waves = NT == 1 ? MAXW : static_cast<int>(blockDim.x) >> 6;
    const int c = lane & 15;  // column of S^T and O^T (query row of a tile); row of the A tiles
    const int G = lane >> 4;  // lane group: which 4 (or 8) of the reduction indices this lane holds
    const int32_t* table = block_tables + static_cast<int64_t>(seq) * max_pages;
    const float scale2 = scale * kLog2e;  // scores in units of log2 e: exp() becomes exp2()
    // capped scores: softcap * tanh(product * scale / softcap), in the same units
    const bool capped = !QKV && f.softcap > 0.f;
    const float cap2 = f.softcap * kLog2e, cap_in = capped ? scale / f.softcap : scale2;
    // the distance bias, in the same units: slope (key - query), added to the scaled scores
    const bool sloped = BIASED && f.slopes != nullptr;

    // LDS: the accumulators that the waves hand over at the end; and in the QKV variant the heads added up from
    // the sums (up to 16 of queries, a key, a value) and the cosines and sines, which a wave may still read when another
    // hands over: apart, where a unit's LDS holds two workgroups of both, else in the same place behind a barrier
    constexpr int kCombine = MAXW == 1 ? 0 : NT == 1 ? MAXW * HDT * 64 : (MAXW - 1) * NT * HDT * 64;
    // a head's row in LDS is four floats longer than the head, so that the 16 rows that a wave reads
    // at once, 16 bytes each, fall into different banks
    constexpr int RS = HD + 4;
    constexpr int kHeads = QKV ? (18 * RS + HD) / 4 : 0;
    constexpr bool kApart = HDT <= 8;
    constexpr int kLds = kApart ? kCombine + kHeads : (kCombine > kHeads ? kCombine : kHeads);
    __shared__ floatx4 s_o[kLds > 0 ? kLds : 1];
    float* s_row = reinterpret_cast<float*>(s_o + (kApart ? kCombine : 0));
    float2* s_cs = reinterpret_cast<float2*>(s_row + 18 * RS);
    // The heads this workgroup needs, added up over the slices, with the bias, into LDS.  In two
    // steps: first all the reads of up to eight slices, in straight-line code (a slice past the last
    // reads the last one again, a thread without a column reads column 0), so that they are under
    // way together, and with the reads of the first keys; then the
    // additions.  A loop of one read and one addition a slice would be a trip to memory a slice.
    constexpr int NJ = QKV ? (18 * HD / 4 + 64 * MAXW - 1) / (64 * MAXW) : 1;  // columns of four a thread
    constexpr int PC = NJ <= 3 ? 8 : 4;                                              // slices read at once
    float4 part[NJ][PC], bias_of[NJ];
    float2 angle = float2{1.f, 0.f};
    int lds_at[NJ];
    const float* col_at[NJ];
    const int sum_thread = static_cast<int>(threadIdx.x), sum_threads = 64 * n_waves;
    auto issue_sums = [&]() {
        const int q_dim = n_heads * HD, kv_dim = n_kv * HD;
        const int n_cols = (gh_here + 2) * HD;
        const float* row = f.sums + static_cast<int64_t>(q_row0) * f.width;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            if (j > 0 && j * sum_threads * 4 >= n_cols) {  // (the same for the whole workgroup: no thread has such a column)
                lds_at[j] = -1;
                continue;
            }
            const int i = (sum_thread + j * sum_threads) * 4;
            const bool has = i < n_cols;
            const int ic = has ? i : 0;
            const int seg = ic / HD, d = ic - seg * HD;
            lds_at[j] = has ? seg * RS + d : -1;
            const int col = seg < gh_here ? (h_base + seg) * HD + d : q_dim + (seg - gh_here) * kv_dim + kvh * HD + d;
            col_at[j] = row + col;
#pragma unroll
            for (int u = 0; u < PC; ++u)
                part[j][u] = *reinterpret_cast<const float4*>(col_at[j] + min(u, f.n_parts - 1) * f.part_stride);
            bias_of[j] = *reinterpret_cast<const float4*>(f.bias ? f.bias + col : col_at[j]);
        }
        if (f.cos_sin) {
            const float2* cs = reinterpret_cast<const float2*>(f.cos_sin) + static_cast<int64_t>(q_row0) * (HD / 2);
            angle = cs[min(sum_thread, HD / 2 - 1)];
        }
    };
    auto finish_sums = [&]() {
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            if (j > 0 && j * sum_threads * 4 >= (gh_here + 2) * HD) continue;
            float4 a{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int u = 0; u < PC; ++u)
                if (u < f.n_parts)
                    a = float4{a.x + part[j][u].x, a.y + part[j][u].y, a.z + part[j][u].z, a.w + part[j][u].w};
            for (int s = PC; s < f.n_parts; ++s) {  // (more slices than are read at once: a trip each)
                const float4 v = *reinterpret_cast<const float4*>(col_at[j] + s * f.part_stride);
                a = float4{a.x + v.x, a.y + v.y, a.z + v.z, a.w + v.w};
            }
            if (f.bias) a = float4{a.x + bias_of[j].x, a.y + bias_of[j].y, a.z + bias_of[j].z, a.w + bias_of[j].w};
            if (lds_at[j] >= 0) *reinterpret_cast<float4*>(s_row + lds_at[j]) = a;
        }
        for (int i = sum_thread; i < HD / 2; i += sum_threads) {
            if (i == sum_thread || !f.cos_sin) s_cs[i] = angle;  // (without a table: cosine 1, sine 0)
            else s_cs[i] = (reinterpret_cast<const float2*>(f.cos_sin) + static_cast<int64_t>(q_row0) * (HD / 2))[i];
        }
    };

    // The output projection's rows of this wave, the columns of this kv head's heads: eight values a lane and load
    constexpr int OU = OROWS > 0 ? HDT / 2 : 1;  // loads a row (sixteen heads at most)
    const int o_first = (static_cast<int>(blockIdx.x) * MAXW + wave) * OROWS, o_units = gh_here * (HD / 8);
    uint4 o_w[OROWS > 0 ? OROWS : 1][OU];
    auto issue_o = [&]() {
#pragma unroll
        for (int r = 0; r < OROWS; ++r) {
            const bf16_t* w = f.o_weight + (static_cast<int64_t>(min(o_first + r, f.o_rows - 1)) * n_heads + h_base) * HD;
#pragma unroll
            for (int u = 0; u < OU; ++u)
                if (u == 0 || u * 64 < o_units) o_w[r][u] = ld16_once(w + min(u * 64 + lane, o_units - 1) * 8);
        }
        __builtin_amdgcn_sched_barrier(0);
    };

    // ---- the item's queries: B operands, kept for the whole item
    bool rvalid[NT];
    int rpos[NT], rtok[NT], rhead[NT];
    float r_in[NT], r_slope[NT];  // the row's factor from products to scores, and its head's slope
    F16B qf[NT][S32A];
    F8B qt[NT][S16A];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        const int rg = nt * 16 + c;
        const int tq = QKV ? 0 : rg / gh, hh = rg - tq * gh;
        rvalid[nt] = rg < n_rows && hh < gh_here;
        rtok[nt] = tq;
        rhead[nt] = h_base + hh;
        rpos[nt] = pos0 + tq;
        r_in[nt] = BIASED && f.row_scale ? cap_in * f.row_scale[q_row0 + (rvalid[nt] ? tq : 0)] : cap_in;
        r_slope[nt] = sloped ? f.slopes[rvalid[nt] ? rhead[nt] : h_base] * kLog2e : 0.f;
        if constexpr (!QKV) {
            const bf16_t* qp = q + static_cast<int64_t>(q_row0 + (rvalid[nt] ? tq : 0)) * q_stride +
                               static_cast<int64_t>(rvalid[nt] ? rhead[nt] : h_base) * HD;
#pragma unroll
            for (int s = 0; s < S32; ++s) qf[nt][s].raw = ld16(qp + s * 32 + 8 * G);  // a row that does not exist reads
#pragma unroll
            for (int s = 0; s < S16; ++s) qt[nt][s].raw = ld8(qp + s * 16 + 4 * G);   // the item's first row: masked later
        }
    }

    float m_run[NT], l_run[NT];
    floatx4 acc[NT][HDT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        m_run[nt] = -INFINITY;
        l_run[nt] = 0.f;
#pragma unroll
        for (int dt = 0; dt < HDT; ++dt) acc[nt][dt] = floatx4{0.f, 0.f, 0.f, 0.f};
    }

    // QKV: the queries (one token: row c of the tile is head c of the group) from the heads in LDS
    auto build_queries = [&]() {
        const float* head = s_row + (rvalid[0] ? c : 0) * RS;
#pragma unroll
        for (int s = 0; s < S32; ++s) qf[0][s].raw = rotated8<HD>(head, s_cs, s * 32 + 8 * G);
    };

    const int64_t head_stride = static_cast<int64_t>(page_size) * HD;  // one kv head of one page
    // key / page_size as one multiplication (the host has checked that keys * page_size < 2^32): a
    // division by a size known only at run time costs some thirty vector instructions
    const uint32_t page_magic = f.page_magic;
    // this wave's run of key blocks
    const int kb_first = key_begin & ~31;
    // The walk runs over block coordinates: from kb_first on a coordinate is the key itself; the blocks of
    // the kept first keys stand before that, from walk_first on, and coordinate u there is key u - walk_first.
    const int pre_len = (prefix_end + 31) & ~31;
    const int walk_first = kb_first - pre_len;
    const int n_blocks = ((key_end - kb_first + 31) >> 5) + (pre_len >> 5);
    // One query tile: an item's blocks are dealt to as many waves as it has blocks, up to what the head size allows, in runs
    // of equal length; several tiles: a wave per 16 blocks (512 keys).  By the items' lengths the variant for short items is taken only where
    // every wave has a block of its own either way: then how an item's keys are split depends on the item alone.
    constexpr int kKeyWaves = QKV && MAXW == kShortWaves + 1 ? kShortWaves : MAXW;
    const int n_run_of = NT == 1 ? (n_blocks + kKeyWaves - 1) / kKeyWaves : 0;
    const int n_active = NT == 1 ? max(1, n_run_of > 0 ? (n_blocks + n_run_of - 1) / n_run_of : 1) : min(n_waves, max(1, (n_blocks + 15) / 16));
    const int per_wave = NT == 1 ? n_run_of : (n_blocks + n_active - 1) / n_active;
    // QKV: the request's new key is a run of its own, for a wave that the keys of the cache leave
    // idle if there is one (else for the first); n_runs = waves whose results are combined
    const int new_key_wave = owner && n_active < n_waves ? n_active : 0;
    const int n_runs = owner && n_active < n_waves ? n_active + 1 : n_active;
    const int kb_begin = walk_first + wave * per_wave * 32;
    const int kb_end = min(key_end, kb_begin + per_wave * 32);
    // the keys (A operand of the scores) and values (A operand of the second product) of a block
    struct Block {
        F16B kf[2][S32A];
        F8B kt[2][S16A];
        F16B vf[HDT];
    };
    // V16: the page size is a multiple of 8, so the keys 8 G .. 8 G + 7 of a block lie in one page,
    // 16-byte aligned (a template flag: a run-time branch around the loads costs a third of the speed)
    // Where a block's keys lie: for the scores the two tiles of 16 keys (one key per lane, c), for the second product the two
    // runs of 4 consecutive keys per lane group (never across a page: page_size % 4 == 0; with V16 eight keys from a multiple
    // of eight on lie in one page, so one table entry serves both runs).  A key without a page (past the end, or behind a
    // window) points at page 0: what is read there is finite and its probability is zero; so it is with the keys behind the
    // last one in that one's page.
    constexpr int RUN = V16 ? 1 : 2;
    struct Where {
        int64_t k[RUN], v[RUN];  // element offsets into the pools
    };
    struct Asked {
        int page[2 * RUN], idx[2 * RUN], key[2 * RUN];
        int limit;  // keys from here on do not belong to the block's range
    };
    auto ask_pages = [&](int kb, Asked& p) {
        const int of_range = key_end, of_kept = prefix_end;
        p.limit = kb >= kb_first ? of_range : of_kept;
        kb = kb >= kb_first ? kb : kb - walk_first;
#pragma unroll
        for (int t = 0; t < RUN; ++t) {
            p.key[t] = kb + 8 * (c >> 2) + 4 * t;
            p.key[RUN + t] = kb + 8 * G + 4 * t;
        }
#pragma unroll
        for (int i = 0; i < 2 * RUN; ++i) {  // the table reads go out together
            p.idx[i] = static_cast<int>(__umulhi(static_cast<uint32_t>(p.key[i]), page_magic));
            p.page[i] = table[min(p.idx[i], max_pages - 1)];
        }
    };
    const int64_t page_stride = n_kv * head_stride, kv_base = kvh * head_stride;
    auto place = [&](const Asked& p, Where& at) {
#pragma unroll
        for (int i = 0; i < 2 * RUN; ++i) {
            const bool ok = (p.key[i] < p.limit) & (p.idx[i] < max_pages) & (p.page[i] >= 0);
            const int64_t head = static_cast<int64_t>(static_cast<uint32_t>(ok ? p.page[i] : 0)) * page_stride + kv_base;
            const int off = ok ? p.key[i] - p.idx[i] * page_size : 0;
            if (i < RUN) at.k[i] = head + static_cast<uint32_t>((off + (c & 3)) * HD + (X32 ? 8 : 4) * G);
            else at.v[i - RUN] = head + static_cast<uint32_t>(off + c * page_size);
        }
    };
    auto locate = [&](int kb, Where& at) {
        Asked p;
        ask_pages(kb, p);
        place(p, at);
    };
    auto load_block = [&](const Where& at, Block& blk) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const bf16_t* kp = k_pool + at.k[V16 ? 0 : t] + (V16 ? 4 * t * HD : 0);
#pragma unroll
            for (int s = 0; s < S32; ++s) blk.kf[t][s].raw = ld16(kp + s * 32);
#pragma unroll
            for (int s = 0; s < S16; ++s) blk.kt[t][s].raw = ld8(kp + s * 16);
        }
        const bf16_t* v0 = v_pool + at.v[0];
        if (V16) {
#pragma unroll
            for (int dt = 0; dt < HDT; ++dt) {
                const bf16_t* vp = v0 + static_cast<int64_t>(dt * 16) * page_size;
                blk.vf[dt].raw = ONCE ? ld16_once(vp) : ld16(vp);
            }
        } else {
            const bf16_t* v1 = v_pool + at.v[RUN - 1];
#pragma unroll
            for (int dt = 0; dt < HDT; ++dt) {
                const uint2 lo = ld8(v0 + static_cast<int64_t>(dt * 16) * page_size);
                const uint2 hi = ld8(v1 + static_cast<int64_t>(dt * 16) * page_size);
                blk.vf[dt].raw = uint4{lo.x, lo.y, hi.x, hi.y};
            }
        }
    };
    auto compute_block = [&](int kb, const Block& blk) {
        const bool kept_block = kb < kb_first;  // a block of the kept first keys (the same for the whole wave)
        if (kept_block) kb -= walk_first;
        const int of_range = key_end, of_kept = prefix_end;  // (values: a choice between the variables themselves is one of addresses)
        const int range_begin = kept_block ? 0 : key_begin, range_end = kept_block ? of_kept : of_range;
        const bool full = !kept_block && kb >= key_begin && kb + 32 <= key_end && kb + 31 <= pos0 &&
                          (window <= 0 || kb > pos0 + n_q - 1 - window);  // the same for the whole wave
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            // ---- S^T for 32 keys x 16 rows
            floatx4 st[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                st[t] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = 0; s < S32; ++s)
                    st[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(blk.kf[t][s].v, qf[nt][s].v, st[t], 0, 0, 0);
#pragma unroll
                for (int s = 0; s < S16; ++s)
                    st[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(blk.kt[t][s].v, qt[nt][s].v, st[t], 0, 0, 0);
            }
            // ---- scores, mask, running maximum; no branch a value (a mask of 64 branches was 3 of the 8.5 us of a step of one
            // request: each an exec mask and cold instructions).  A block that every row of the item sees whole (below the
            // diagonal, inside the key range and the window) needs no mask; in a long portion that is nearly every block.
            float sv[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) sv[i] = st[i >> 2][i & 3] * r_in[nt];
            if (capped) {  // (the same for the whole launch)
#pragma unroll
                for (int i = 0; i < 8; ++i) sv[i] = cap2 * tanh_by_exp(sv[i]);
            }
            const int first = kb + 8 * G;  // this lane's keys: first .. first + 7
            if (sloped) {  // (the same for the whole launch)
                const float at_first = r_slope[nt] * static_cast<float>(first - rpos[nt]);
#pragma unroll
                for (int i = 0; i < 8; ++i) sv[i] += fmaf(r_slope[nt], static_cast<float>(i), at_first);
            }
            if (!full) {
                // of the block's range, up to the row's own position: the keys inside the window, and the kept first ones
                const int upto = min(range_end, rpos[nt] + 1), hi = rvalid[nt] ? upto : kFarBelow;
                const int in_window = rpos[nt] - window + 1, seen = window > 0 ? in_window : kFarBelow;
                const uint32_t vis = keys_below(hi - first) & ~keys_below(range_begin - first) &
                                     (~keys_below(seen - first) | keys_below(keep - first));
#pragma unroll
                for (int i = 0; i < 8; ++i) sv[i] = (vis & (1u << i)) != 0u ? sv[i] : -INFINITY;
            }
            float m_loc = sv[0];
#pragma unroll
            for (int i = 1; i < 8; ++i) m_loc = fmaxf(m_loc, sv[i]);
            m_loc = max_xor32(max_xor16(m_loc));
            const float m_new = fmaxf(m_run[nt], m_loc);
            const float m_of = m_new == -INFINITY ? 0.f : m_new;  // (a row without a key so far: all its probabilities zero)
            const float corr = (m_run[nt] == -INFINITY) ? 1.f : __builtin_amdgcn_exp2f(m_run[nt] - m_of);
            float p[8];
            float p_sum = 0.f;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                p[i] = __builtin_amdgcn_exp2f(sv[i] - m_of);
                p_sum += p[i];
            }
            l_run[nt] = l_run[nt] * corr + p_sum;  // this lane's keys only; lane groups are summed at the end
            m_run[nt] = m_new;
            F16B pb;  // P^T for the keys 8 G .. 8 G + 7 of the block
            pb.raw = uint4{pack2_bf16(p[0], p[1]), pack2_bf16(p[2], p[3]), pack2_bf16(p[4], p[5]), pack2_bf16(p[6], p[7])};
            // the accumulators shrink only when some row's maximum moved (rare after the first blocks)
            if (__any(corr != 1.f)) {
#pragma unroll
                for (int dt = 0; dt < HDT; ++dt) {
                    acc[nt][dt][0] *= corr;
                    acc[nt][dt][1] *= corr;
                    acc[nt][dt][2] *= corr;
                    acc[nt][dt][3] *= corr;
                }
            }
            // ---- O^T += V^T P^T
#pragma unroll
            for (int dt = 0; dt < HDT; ++dt)
                acc[nt][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(blk.vf[dt].v, pb.v, acc[nt][dt], 0, 0, 0);
        }
    };
    // The table reads of a block go out one block ahead, so that its data reads never wait for
    // an address.  One query tile and a moderate head size leave registers for a second block:
    // its data is in flight while the matrix cores work on the present one (few waves run here,
    // so occupancy does not hide the latency).
    constexpr bool PREFETCH = NT == 1 && HDT <= 8;
    // (the variant for short items has one block a wave, as a rule)
    constexpr bool SHORT = NT == 1 && MAXW <= kShortWaves + 1 && HDT <= 8;
    // QKV: the new key and value, from the sums: a block of their own whose first key they are (the
    // mask hides the rest), and into the pools for the steps to come.  An idle wave does it, or the
    // first one before its walk, while its first keys from the cache are under way.
    // The stores into the pools (2 bytes a dimension for the value) are not ordered against the loads of
    // other waves and workgroups that read the 16 bytes around that slot: those lanes are masked
    // (probability zero), so the result does not depend on which bytes they see, provided they are
    // finite either way.  That is the pools' invariant: a slot at or after a request's length holds a
    // finite value (a page is zeroed by the step that takes it; the null page is never written).
    auto score_new_key = [&]() {
        if (!(owner && wave == new_key_wave)) return;
        key_end = pos0 + 1;
        const float* kh = s_row + gh_here * RS;
        const float* vh = kh + RS;
        Block nb;
#pragma unroll
        for (int s = 0; s < S32; ++s) {
            const uint4 r = rotated8<HD>(kh, s_cs, s * 32 + 8 * G);
            nb.kf[0][s].raw = c == 0 ? r : uint4{0u, 0u, 0u, 0u};
            nb.kf[1][s].raw = uint4{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int dt = 0; dt < HDT; ++dt)
            nb.vf[dt].raw = uint4{G == 0 ? pack2_bf16(vh[dt * 16 + c], 0.f) : 0u, 0u, 0u, 0u};
        compute_block(pos0, nb);
        key_end = pos0;
    };
    // ... and into the pools, by a wave that has the least to do
    auto keep_new_key = [&]() {
        if (!(owner && chunk == 0 && (OROWS == 0 || blockIdx.x == 0) && new_slot >= 0 && new_slot < f.pool_slots)) return;
        const float* kh = s_row + gh_here * RS;
        const float* vh = kh + RS;
        const int page = new_slot / page_size;
        const int off = new_slot - page * page_size;
        bf16_t* kd = f.k_out + ((static_cast<int64_t>(page) * n_kv + kvh) * page_size + off) * HD;
        for (int d = 2 * lane; d < HD; d += 128)
            *reinterpret_cast<uint32_t*>(kd + d) = pack2_bf16(rotated<HD>(kh, s_cs, d), rotated<HD>(kh, s_cs, d + 1));
        bf16_t* vd = f.v_out + (static_cast<int64_t>(page) * n_kv + kvh) * head_stride + off;
        for (int d = lane; d < HD; d += 64) vd[static_cast<int64_t>(d) * page_size] = from_float<bf16_t>(vh[d]);
    };

    // QKV: the block table (warm in the L2) is read first, then the reads of the sums (which come from
    // further away) and of the first keys go out together; the queries are built from LDS while the keys
    // are under way
    {
        const bool any = kb_begin < kb_end;
        Where at;
        Block cur, nxt;
        // (QKV: the reads of the sums, which come from further away than the table, go out before the
        // wait for the table)
        Asked first;
        // (a wave without keys asks all the same, for what lies at the start of page 0: behind a branch around these loads the compiler
        // cannot know how many are under way, and waits for the keys where it needs the sums)
        const bool ask = QKV || any;
        if (ask) ask_pages(kb_begin, first);
        if constexpr (QKV) issue_sums();
        if (ask) place(first, at);
        if (PREFETCH && ask) {
            load_block(at, cur);
            if (!SHORT) locate(kb_begin + 32, at);
        }
        if constexpr (OROWS > 0) issue_o();  // (behind all that attention itself waits for: a wave's loads return in order)
        if constexpr (QKV) {
            finish_sums();
            __syncthreads();
            build_queries();
            score_new_key();
            if (wave == (new_key_wave == n_waves - 1 ? 0 : n_waves - 1)) keep_new_key();
            if (!kApart) __syncthreads();
        }
        constexpr bool IN_TURN = QKV && MAXW <= 8;  // (16 waves a workgroup have 128 registers each: not enough)
        if (SHORT && any) {
            for (int kb = kb_begin;;) {
                compute_block(kb, cur);
                kb += 32;
                if (kb >= kb_end) break;
                locate(kb, at);
                load_block(at, cur);
            }
        } else if (PREFETCH && any && !IN_TURN) {
            for (int kb = kb_begin; kb < kb_end; kb += 32) {
                if (kb + 32 < kb_end) {
                    load_block(at, nxt);
                    locate(kb + 64, at);
                }
                compute_block(kb, cur);
                cur = nxt;
            }
        } else if (PREFETCH && any) {
            // two blocks in turn, each in registers of its own: while one is computed the other's
            // data is under way (with one name for "this block" the copy from the next one's
            // registers at the end of a pass waits for that data).  A per cent of a step with long
            // contexts; the variants that would spill registers this way keep the loop above
            for (int kb = kb_begin;;) {
                if (kb + 32 < kb_end) {
                    load_block(at, nxt);
                    locate(kb + 64, at);
                }
                compute_block(kb, cur);
                kb += 32;
                if (kb >= kb_end) break;
                if (kb + 32 < kb_end) {
                    load_block(at, cur);
                    locate(kb + 64, at);
                }
                compute_block(kb, nxt);
                kb += 32;
                if (kb >= kb_end) break;
            }
        } else if (any) {
            for (int kb = kb_begin; kb < kb_end; kb += 32) {
                load_block(at, cur);
                locate(kb + 32, at);
                compute_block(kb, cur);
            }
        }
    }

    // ---- one query tile: every wave with keys lays its accumulators, maxima and sums into LDS, and behind a barrier
    // the waves deal the sixteens of the head's values among themselves, each adding the runs up in their fixed order, relative to the
    // common maximum, and writing its part of the result (one barrier, no atomics).  By the first wave alone, behind two
    // barriers, the runs of eight waves would be 64 reads of LDS in a row.
    if constexpr (NT == 1) {
        constexpr int MW = (MAXW + 3) / 4 * 4;
        __shared__ float s_m1[16][MW + 4], s_l1[16][MW + 4];  // [column][wave]: a lane reads its column's waves four at a time
        if (wave < n_runs) {
#pragma unroll
            for (int dt = 0; dt < HDT; ++dt) s_o[(wave * HDT + dt) * 64 + lane] = acc[0][dt];
        }
        const float l_w = sum_xor32(sum_xor16(l_run[0]));
        if (G == 0) {  // (a wave without keys: minus infinity and zero)
            s_m1[c][wave] = m_run[0];
            s_l1[c][wave] = l_w;
        }
        __syncthreads();
        if (OROWS == 0 && !rvalid[0]) return;
        float m_of_run[MW], l_of_run[MW], factor[MW];
#pragma unroll
        for (int w = 0; w < MW; w += 4) {
            const floatx4 m4 = *reinterpret_cast<const floatx4*>(&s_m1[c][w]), l4 = *reinterpret_cast<const floatx4*>(&s_l1[c][w]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const bool is = w + i < MAXW && w + i < n_runs;
                m_of_run[w + i] = is ? m4[i] : -INFINITY;
                l_of_run[w + i] = is ? l4[i] : 0.f;
            }
        }
        float m_all = m_of_run[0];
#pragma unroll
        for (int w = 1; w < MAXW; ++w) m_all = fmaxf(m_all, m_of_run[w]);
        const float m_of = m_all == -INFINITY ? 0.f : m_all;
        float denom = 0.f;
#pragma unroll
        for (int w = 0; w < MW; ++w) {
            factor[w] = __builtin_amdgcn_exp2f(m_of_run[w] - m_of);
            denom = fmaf(l_of_run[w], factor[w], denom);
        }
        float inv = 1.f;
        if (partial_base < 0) {
            float whole = denom;
            if (!QKV && f.sinks && m_all != -INFINITY) whole += __builtin_amdgcn_exp2f(f.sinks[rhead[0]] * kLog2e - m_all);
            inv = whole > 0.f ? 1.0f / whole : 0.f;
        }
        bf16_t* o = out + (static_cast<int64_t>(q_row0 + rtok[0]) * n_heads + rhead[0]) * HD + 4 * G;
        // (a cut item's record: unnormalised sums, their maximum in natural units and denominator, for attention_merge)
        float* rec = partials + (static_cast<int64_t>(max(partial_base, 0) + rtok[0]) * n_heads + rhead[0]) * (HD + 2);
        for (int dt = wave; dt < HDT; dt += n_waves) {
            // lane holds O^T[d = 16 dt + 4 G + r][row c]
            floatx4 a{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w0 = 0; w0 < MAXW; w0 += 4) {
                if (w0 >= n_runs) break;  // (the same for the whole workgroup)
                floatx4 v[4];  // four at once, past the last run the last one again, not added
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = s_o[(min(w0 + i, n_runs - 1) * HDT + dt) * 64 + lane];
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r) a[r] = w0 + i < n_runs ? fmaf(v[i][r], factor[w0 + i], a[r]) : a[r];
            }
            if constexpr (OROWS > 0) {  // (into the place of the heads in LDS, which were last read in front of the barrier)
                if (rvalid[0])
                    *reinterpret_cast<uint2*>(reinterpret_cast<bf16_t*>(s_row) + c * HD + dt * 16 + 4 * G) =
                        uint2{pack2_bf16(a[0] * inv, a[1] * inv), pack2_bf16(a[2] * inv, a[3] * inv)};
            } else if (partial_base < 0) {
                *reinterpret_cast<uint2*>(o + dt * 16) = uint2{pack2_bf16(a[0] * inv, a[1] * inv), pack2_bf16(a[2] * inv, a[3] * inv)};
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) rec[dt * 16 + 4 * G + r] = a[r];
            }
        }
        if constexpr (OROWS > 0) {
            __syncthreads();
            float sum[OROWS];
#pragma unroll
            for (int r = 0; r < OROWS; ++r) sum[r] = 0.f;
#pragma unroll
            for (int u = 0; u < OU; ++u) {
                if (u > 0 && u * 64 >= o_units) break;  // (the same for the whole workgroup)
                const int unit = u * 64 + lane;
                const uint4 x = *reinterpret_cast<const uint4*>(reinterpret_cast<const bf16_t*>(s_row) + min(unit, o_units - 1) * 8);
                const uint32_t xs[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
                for (int r = 0; r < OROWS; ++r) {
                    const uint32_t ws[4] = {o_w[r][u].x, o_w[r][u].y, o_w[r][u].z, o_w[r][u].w};
                    float more = 0.f;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        more = fmaf(__uint_as_float(xs[i] << 16), __uint_as_float(ws[i] << 16), more);
                        more = fmaf(__uint_as_float(xs[i] & 0xffff0000u), __uint_as_float(ws[i] & 0xffff0000u), more);
                    }
                    sum[r] += unit < o_units ? more : 0.f;
                }
            }
            float mine = 0.f;
#pragma unroll
            for (int r = 0; r < OROWS; ++r) {
                const float all = wave_sum(sum[r]);
                mine = lane == r ? all : mine;
            }
            if (lane < OROWS && o_first + lane < f.o_rows)
                f.o_sums[kvh * f.o_part_stride + static_cast<int64_t>(q_row0) * f.o_rows + o_first + lane] = mine;
            return;
        }
        if (partial_base >= 0 && wave == 0 && G == 0) {
            rec[HD] = m_all * kLn2;
            rec[HD + 1] = denom;
        }
        return;
    }

    // ---- several query tiles: the denominator and maximum of every query row; several waves combine inside the
    // workgroup: maxima and sums through LDS, then the waves after the first lay their
    // accumulators, rescaled to the common maximum, into LDS, and the first wave adds them to its
    // own in the fixed order of the waves and writes the result (two barriers, no atomics)
    float l_tot[NT], m_fin[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        float l_w = l_run[nt];
        l_w = sum_xor32(sum_xor16(l_w));
        l_tot[nt] = l_w;
        m_fin[nt] = m_run[nt];
    }
    if (MAXW > 1 && n_waves > 1) {
        __shared__ float s_m[NT][MAXW][16], s_l[NT][MAXW][16];
        if (G == 0) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                s_m[nt][wave][c] = m_run[nt];
                s_l[nt][wave][c] = l_tot[nt];
            }
        }
        __syncthreads();
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            float m_all = -INFINITY;
            for (int w = 0; w < n_runs; ++w) m_all = fmaxf(m_all, s_m[nt][w][c]);
            float denom = 0.f;
            for (int w = 0; w < n_runs; ++w) {
                const float mw = s_m[nt][w][c];
                if (mw != -INFINITY) denom += s_l[nt][w][c] * __builtin_amdgcn_exp2f(mw - m_all);
            }
            const float mine = (m_run[nt] == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(m_run[nt] - m_all);
#pragma unroll
            for (int dt = 0; dt < HDT; ++dt) {
                acc[nt][dt][0] *= mine;
                acc[nt][dt][1] *= mine;
                acc[nt][dt][2] *= mine;
                acc[nt][dt][3] *= mine;
            }
            if (wave > 0 && wave < n_runs) {
#pragma unroll
                for (int dt = 0; dt < HDT; ++dt) s_o[(((wave - 1) * NT + nt) * HDT + dt) * 64 + lane] = acc[nt][dt];
            }
            l_tot[nt] = denom;
            m_fin[nt] = m_all;
        }
        __syncthreads();
        if (wave > 0) return;
        for (int w = 1; w < n_runs; ++w) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int dt = 0; dt < HDT; ++dt) {
                    const floatx4 v = s_o[(((w - 1) * NT + nt) * HDT + dt) * 64 + lane];
                    acc[nt][dt][0] += v[0];
                    acc[nt][dt][1] += v[1];
                    acc[nt][dt][2] += v[2];
                    acc[nt][dt][3] += v[3];
                }
        }
    }

    // ---- results: lane holds O^T[d = 16 dt + 4 G + r][row c], relative to the maximum m_fin
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        if (!rvalid[nt]) continue;
        if (partial_base < 0) {
            float denom = l_tot[nt];
            if (f.sinks && m_fin[nt] != -INFINITY) denom += __builtin_amdgcn_exp2f(f.sinks[rhead[nt]] * kLog2e - m_fin[nt]);
            const float inv = denom > 0.f ? 1.0f / denom : 0.f;
            bf16_t* o = out + (static_cast<int64_t>(q_row0 + rtok[nt]) * n_heads + rhead[nt]) * HD + 4 * G;
#pragma unroll
            for (int dt = 0; dt < HDT; ++dt) {
                uint2 w;
                w.x = pack2_bf16(acc[nt][dt][0] * inv, acc[nt][dt][1] * inv);
                w.y = pack2_bf16(acc[nt][dt][2] * inv, acc[nt][dt][3] * inv);
                *reinterpret_cast<uint2*>(o + dt * 16) = w;
            }
        } else {
            // the item is one of several that share a query's keys: unnormalised sums, their
            // maximum (in natural units) and denominator, for attention_merge
            float* rec = partials + (static_cast<int64_t>(partial_base + rtok[nt]) * n_heads + rhead[nt]) * (HD + 2);
#pragma unroll
            for (int dt = 0; dt < HDT; ++dt)
#pragma unroll
                for (int r = 0; r < 4; ++r) rec[dt * 16 + 4 * G + r] = acc[nt][dt][r];
            if (G == 0) {
                rec[HD] = m_fin[nt] * kLn2;
                rec[HD + 1] = l_tot[nt];
            }
        }
    }
}

template <int HDT, int NT>
int launch(const void* q, int64_t q_stride, const void* k_pool, const void* v_pool, const int32_t* block_tables,
           int max_pages, const int32_t* items, int n_items, void* out, float* partials, int n_heads, int n_kv,
           int page_size, int window, float scale, int waves, const float* sinks, float softcap, const float* slopes,
           const float* row_scale, hipStream_t stream) {
    constexpr int MAXW = NT == 1 ? max_waves<HDT>() : 4;
    QkvSums scores{};
    scores.sinks = sinks;
    scores.softcap = softcap;
    scores.slopes = slopes;
    scores.row_scale = row_scale;
    const int group = n_heads / n_kv;
    const int rows = 16 * NT;
    const int gh = group < rows ? group : rows;
    const int head_chunks = (group + gh - 1) / gh;
    const dim3 grid(n_items, n_kv, head_chunks);
    scores.group = group;
    scores.page_magic = magic_of(page_size);
    const bool few = waves == 0;  // (one tile: the variant for short items whatever their length, values by streaming loads)
    if (waves < 1) waves = 1;
    if (waves > MAXW) waves = MAXW;
    // Several query tiles: a launch of one wave per workgroup takes the instantiation without the LDS of the
    // combination, which would otherwise limit how many workgroups a compute unit holds.  One: the variant for short items,
    // or all the waves the kernel has
#define FSIE_ATTN_LAUNCH(W, THREADS, V) FSIE_ATTN_LAUNCH_ONCE(W, THREADS, V, (W > kShortWaves + 1))
#define FSIE_ATTN_LAUNCH_ONCE(W, THREADS, V, ONCE)                                                                   \
    attention_mfma_kernel<HDT, NT, W, V, false, true, ONCE><<<grid, THREADS, 0, stream>>>(                                              \
        static_cast<const bf16_t*>(q), q_stride, static_cast<const bf16_t*>(k_pool), static_cast<const bf16_t*>(v_pool), \
        block_tables, max_pages, items, static_cast<bf16_t*>(out), partials, n_heads, n_kv, page_size, window, scale, \
        gh, scores)
    const bool v16 = page_size % 8 == 0;
    if constexpr (NT == 1) {
        if (few && v16 && HDT <= 8) {  // (wider heads have this many waves and no more)
            FSIE_ATTN_LAUNCH_ONCE(kShortWaves, 64 * kShortWaves, true, (HDT <= 8));
        } else if (waves == 1) {
            if (v16) FSIE_ATTN_LAUNCH(kShortWaves, 64 * kShortWaves, true);
            else FSIE_ATTN_LAUNCH(kShortWaves, 64 * kShortWaves, false);
        } else {
            if (v16) FSIE_ATTN_LAUNCH(MAXW, 64 * MAXW, true);
            else FSIE_ATTN_LAUNCH(MAXW, 64 * MAXW, false);
        }
    } else if (waves == 1) {
        if (v16) FSIE_ATTN_LAUNCH(1, 64, true);
        else FSIE_ATTN_LAUNCH(1, 64, false);
    } else {
        if (v16) FSIE_ATTN_LAUNCH(MAXW, 64 * waves, true);
        else FSIE_ATTN_LAUNCH(MAXW, 64 * waves, false);
    }
#undef FSIE_ATTN_LAUNCH
#undef FSIE_ATTN_LAUNCH_ONCE
    FSIE_CHECK_LAUNCH("attention_mfma");
    return 0;
}

// The QKV variant: items of one token, head_dim a multiple of 32, page_size a multiple of 8.
template <int HDT>
int launch_qkv(const QkvSums& f, const void* k_pool, const void* v_pool, const int32_t* block_tables, int max_pages,
               const int32_t* items, int n_items, void* out, float* partials, int n_heads, int n_kv, int page_size,
               int window, float scale, int waves, hipStream_t stream) {
    constexpr int MAXW = max_waves<HDT>();
    const int group = n_heads / n_kv;
    const int gh = group < 16 ? group : 16;
    const dim3 grid(n_items, n_kv, (group + gh - 1) / gh);
#define FSIE_ATTN_LAUNCH(W, THREADS)                                                                                 \
    if (f.slopes || f.row_scale) FSIE_ATTN_LAUNCH_AS(W, THREADS, true); else FSIE_ATTN_LAUNCH_AS(W, THREADS, false)
#define FSIE_ATTN_LAUNCH_AS(W, THREADS, B)                                                                           \
    attention_mfma_kernel<HDT, 1, W, true, true, B><<<grid, THREADS, 0, stream>>>(                                      \
        reinterpret_cast<const bf16_t*>(f.slots), 0, static_cast<const bf16_t*>(k_pool), static_cast<const bf16_t*>(v_pool), block_tables, max_pages, \
        items, static_cast<bf16_t*>(out), partials, n_heads, n_kv, page_size, window, scale, gh, f)
    constexpr int SHORTW = HDT <= 8 ? kShortWaves + 1 : MAXW;
    if (waves <= 1) {
        FSIE_ATTN_LAUNCH(SHORTW, 64 * SHORTW);
    } else {
        FSIE_ATTN_LAUNCH(MAXW, 64 * MAXW);
    }
#undef FSIE_ATTN_LAUNCH_AS
#undef FSIE_ATTN_LAUNCH
    FSIE_CHECK_LAUNCH("attention_mfma_qkv");
    return 0;
}

// The same with the output projection: f.o_weight, f.o_sums; o_rows_of_wave rows of it a wave (2, 3 or 4).  No item is cut, none
// has more than kShortWaves blocks of keys, no group more than 16 heads.
template <int HDT>
int launch_qkv_o(const QkvSums& f, const void* k_pool, const void* v_pool, const int32_t* block_tables, int max_pages,
                 const int32_t* items, int n_items, int o_rows_of_wave, int n_heads, int n_kv, int page_size, int window,
                 float scale, hipStream_t stream) {
    constexpr int W = kShortWaves + 1;
#define FSIE_ATTN_LAUNCH(R)                                                                                          \
    attention_mfma_kernel<HDT, 1, W, true, true, false, false, R>                                                     \
        <<<dim3((f.o_rows + W * R - 1) / (W * R), n_kv, n_items), 64 * W, 0, stream>>>(                               \
            reinterpret_cast<const bf16_t*>(f.slots), 0, static_cast<const bf16_t*>(k_pool), static_cast<const bf16_t*>(v_pool), block_tables, max_pages, \
            items, nullptr, nullptr, n_heads, n_kv, page_size, window, scale, n_heads / n_kv, f)
    if (o_rows_of_wave == 2) FSIE_ATTN_LAUNCH(2);
    else if (o_rows_of_wave == 3) FSIE_ATTN_LAUNCH(3);
    else FSIE_ATTN_LAUNCH(4);
#undef FSIE_ATTN_LAUNCH
    FSIE_CHECK_LAUNCH("attention_mfma_qkv_o");
    return 0;
}

typedef int (*LaunchQkvOFn)(const QkvSums&, const void*, const void*, const int32_t*, int, const int32_t*, int, int, int, int, int, int,
                            float, hipStream_t);

typedef int (*LaunchQkvFn)(const QkvSums&, const void*, const void*, const int32_t*, int, const int32_t*, int, void*,
                           float*, int, int, int, int, float, int, hipStream_t);

typedef int (*LaunchFn)(const void*, int64_t, const void*, const void*, const int32_t*, int, const int32_t*, int, void*,
                        float*, int, int, int, int, float, int, const float*, float, const float*, const float*, hipStream_t);

}  // namespace fsie_attn
