// Causal grouped-query attention over the pages of the cache on the float32 matrix instruction, for float32 storage: products,
// softmax and sums in float32, no operand rounded.
//
// As in the bfloat16 kernel everything is computed transposed, so that no operand changes lanes or passes through LDS:
//   S^T[key, row] = K[key, :] . Q[row, :]       A = K, B = Q
//   O^T[d, row]  += V^T[d, key] . P^T[key, row] A = V^T (the cache stores values as [head_dim][slot]), B = P^T
// v_mfma_f32_16x16x4_f32 takes one value of four reduction indices from each lane (lane = 16 G + c: row c, index G).  Which indices
// a step of four takes is free as long as both operands agree: step i of a run of sixteen takes 4 G + i, so a lane's four values
// of a run are neighbours, one 16-byte load.  The first product leaves the scores of the keys 4 G .. 4 G + 3 in a lane, which is
// the B operand of the second one's four steps over those keys.
//
// A workgroup takes an item (a tile of up to 16 query rows, a range of keys) of a kv head; the item's blocks of 16 keys are
// dealt to its waves in runs of equal length, and the waves' sums meet in LDS, in the order of the waves, behind one barrier.
// What bounds it is the chain: the item, the block table, keys and values, a trip to memory each, then 32 matrix instructions a
// block and head of 64 at 32 cycles.  With the merge where items are cut, keys that no cache holds, us, the kernel on the vector
// units (attention_scalar) / this one: 4 requests of 300 keys, 14 heads on 2 of 64 13.4 / 7.4, 28 on 4 of 128 19.4 / 8.7, 16 on 1
// of 256 39 / 12.6; one of 100 keys 16.0 / 6.3, 24.0 / 7.7, 60 / 14.1; 32 of 700 26.9 / 12.4, 68 / 26.9, 56 / 25.8; a prompt of 300
// tokens 54 / 14.9, 94 / 30, 137 / 38, of 1,000 202 / 59, 562 / 155, 657 / 202.
//
// QKV: steps of one token a request take q, k and v as the partial sums that the product in slices of K leaves, as the bfloat16 kernel's
// variant does: a workgroup adds up the heads that it needs, with the bias, turns queries and key by the step's table, takes the new key and value from
// there where its keys end with them, and one workgroup a kv head writes them into the pools.  That spares the launch between product and
// attention (3.3 us of a layer and step; four requests of the 0.5B shape, 16 tokens each, 20.5 ms -> 20.0).  The bits are those of the kernels one after the other.
//
// More workgroups than units: four waves each whatever the head size, except over the tiles of long prompts (see launch).
// So it is for items that are cut to 64 keys: the twelve waves beside them have no keys, and asked in vain for sums (a unit takes 16 cycles for each of a wave's
// loads).  Four requests of 42 to 316 keys, 14 heads on 2 of 64, 8.1 us -> 6.1 with the loads in straight-line code besides (see `asks`); the step above 20.0 ms -> 19.6.  Longer items are no gain: at 128, 256 and 512 keys 20.7, 22.0 and 21.5 ms.
#include "common.h"
#include "api.h"

#include <limits.h>
#include <math.h>

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kFarBelow = INT_MIN / 2;  // below every key

template <int HDT>
constexpr int f32_waves() {
    return HDT <= 4 ? 16 : (HDT <= 8 ? 8 : 4);  // registers a wave grow with the head size
}

// What the QKV variant reads and writes beside the kernel's other operands.
struct F32Sums {
    const float *sums, *bias, *cos_sin;  // [n_parts][tokens][width]; [width] or null; [tokens][head_dim / 2] pairs of cosine and sine, or null: nothing is turned
    const int32_t* slots;                // [tokens]: where a token's key and value go (negative, or not below pool_slots: nowhere); the kernel has it in the place of q
    float *k_out, *v_out;                // the pools again, to write
    int64_t part_stride, pool_slots;
    int n_parts, width;
};

constexpr int kSumsHdt = 8;  // the QKV variant: heads of up to 128 (its wider ones would have no registers left)

struct F32Call {
    const float *q, *k_pool, *v_pool;
    int64_t q_stride;
    const int32_t *block_tables, *items;
    float *out, *partials;
    int n_items, max_pages, n_heads, n_kv, page_size, window, all_waves, few_waves;
    float scale, softcap;
    const float *sinks, *slopes, *row_scale;
    F32Sums sums;  // sums null: queries from q, keys and values in the pools already
};

// A pair turned by (c, s), with the roundings of the kernel that turns and writes by itself (rope_kv.hip).
__device__ __forceinline__ float turned(float first, float second, float c, float s, bool is_second) {
    return is_second ? __builtin_fmaf(first, s, second * c) : __builtin_fmaf(first, c, -(second * s));
}

template <int HDT, int W, bool QKV>
__global__ __launch_bounds__(64 * W) void attention_f32_kernel(
    const int32_t* __restrict__ items, const int32_t* __restrict__ block_tables, int max_pages, int page_size, uint32_t page_magic,
    int n_kv, const float* __restrict__ k_pool, const float* __restrict__ v_pool, const float* __restrict__ q, int64_t q_stride,
    float* __restrict__ out, float* __restrict__ partials, int n_heads, int group, int gh, int window, float scale, float softcap,
    const float* __restrict__ sinks, const float* __restrict__ slopes, const float* __restrict__ row_scale, F32Sums f) {
    constexpr int HD = HDT * 16, MW = (W + 3) / 4 * 4;
    __shared__ floatx4 s_o[W * HDT * 64];
    // QKV: up to 16 heads of queries, the key and the value (a row four floats longer than a head: 16 rows' reads fall into different banks); the table's pairs
    constexpr int RS = HD + 4;
    __shared__ __align__(16) float s_row[QKV ? 18 * RS : 1];
    __shared__ __align__(16) float2 s_cs[QKV ? HD / 2 : 1];
    __shared__ float s_m[16][MW + 4], s_l[16][MW + 4];  // [column][wave]: a lane reads its column's waves four at a time

    typedef int ItemInts __attribute__((ext_vector_type(8), aligned(4)));
    static_assert(FSIE_ATTN_ITEM_INTS == 8, "an item is eight numbers");
    const ItemInts it = *reinterpret_cast<const ItemInts*>(items + static_cast<int64_t>(blockIdx.x) * FSIE_ATTN_ITEM_INTS);
    const int seq = it[FSIE_ATTN_ITEM_SEQ], q_row0 = it[FSIE_ATTN_ITEM_QROW], n_q = it[FSIE_ATTN_ITEM_NQ], pos0 = it[FSIE_ATTN_ITEM_POS];
    const int key_begin = it[FSIE_ATTN_ITEM_KBEGIN], key_end = it[FSIE_ATTN_ITEM_KEND], partial_base = it[FSIE_ATTN_ITEM_PARTIAL];
    // (the arguments that do not come with the launch on the item's trip: left alone, the compiler asks for them behind it, where they are used)
    if constexpr (QKV)
        asm volatile("" ::"s"(n_heads), "s"(group), "s"(gh), "s"(window), "s"(scale), "s"(slopes), "s"(row_scale), "s"(f.sums), "s"(f.bias), "s"(f.cos_sin), "s"(f.k_out),
                     "s"(f.v_out), "s"(f.part_stride), "s"(f.n_parts), "s"(f.width));
    if (n_q <= 0) return;  // padding item
    // the first keys that a window keeps: seen whatever the window says, and read, as blocks ahead of the item's own
    // range, where the item is told to
    const int keep = it[FSIE_ATTN_ITEM_KEEP] & ~(FSIE_ATTN_KEEP_WALK | FSIE_ATTN_POOL_WALK);
    const int prefix_end = (it[FSIE_ATTN_ITEM_KEEP] & FSIE_ATTN_KEEP_WALK) ? min(keep, key_begin) : 0;

    const int kvh = blockIdx.y, chunk = blockIdx.z;
    const int gh_here = min(gh, group - chunk * gh), h_base = kvh * group + chunk * gh;
    const int lane = threadIdx.x & 63, c = lane & 15, G = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int32_t* table = block_tables + static_cast<int64_t>(seq) * max_pages;

    // the blocks, in coordinates that are the keys themselves from kb_first on; those of the kept first keys stand before
    const int kb_first = key_begin & ~15;
    const int pre_len = (prefix_end + 15) & ~15;
    const int walk_first = kb_first - pre_len;
    const int n_blocks = ((key_end - kb_first + 15) >> 4) + (pre_len >> 4);
    const int per_wave = (n_blocks + W - 1) / W;
    const int n_runs = per_wave > 0 ? (n_blocks + per_wave - 1) / per_wave : 1;
    const int kb_begin = walk_first + wave * per_wave * 16;
    const int kb_end = min(key_end, kb_begin + per_wave * 16);

    const int64_t head_stride = static_cast<int64_t>(page_size) * HD;
    const int64_t page_stride = n_kv * head_stride, kv_base = kvh * head_stride;
    // A key without a page (past the end, or behind a window) is read from page 0 and masked.
    struct Asked {
        int k_page, v_page, k_idx, v_idx, k_key, v_key, limit;
    };
    auto ask = [&](int kb, Asked& p) {
        p.limit = kb >= kb_first ? key_end : prefix_end;
        kb = kb >= kb_first ? kb : kb - walk_first;
        p.k_key = kb + c, p.v_key = kb + 4 * G;
        p.k_idx = static_cast<int>(__umulhi(static_cast<uint32_t>(p.k_key), page_magic));
        p.v_idx = static_cast<int>(__umulhi(static_cast<uint32_t>(p.v_key), page_magic));
        p.k_page = table[min(p.k_idx, max_pages - 1)];
        p.v_page = table[min(p.v_idx, max_pages - 1)];
    };
    struct Block {
        floatx4 k[HDT], v[HDT];
        bool v_ok;  // the keys 4 G .. 4 G + 3 have a page
    };
    auto load = [&](const Asked& p, Block& b) {
        const bool k_ok = (p.k_key < p.limit) & (p.k_idx < max_pages) & (p.k_page >= 0);
        b.v_ok = (p.v_key < p.limit) & (p.v_idx < max_pages) & (p.v_page >= 0);
        const float* kp = k_pool + static_cast<uint32_t>(k_ok ? p.k_page : 0) * page_stride + kv_base +
                          static_cast<uint32_t>((k_ok ? p.k_key - p.k_idx * page_size : 0) * HD + 4 * G);
        const float* vp = v_pool + static_cast<uint32_t>(b.v_ok ? p.v_page : 0) * page_stride + kv_base +
                          static_cast<uint32_t>((b.v_ok ? p.v_key - p.v_idx * page_size : 0) + c * page_size);
#pragma unroll
        for (int j = 0; j < HDT; ++j) b.k[j] = *reinterpret_cast<const floatx4*>(kp + 16 * j);
#pragma unroll
        for (int j = 0; j < HDT; ++j) b.v[j] = *reinterpret_cast<const floatx4*>(vp + static_cast<int64_t>(16 * j) * page_size);
    };

    const bool any = kb_begin < kb_end;
    // QKV with four waves: a wave without keys asks all the same, for what lies at the start of page 0.  Behind a branch around these loads the compiler cannot
    // know how many are under way, and waits for the keys where it needs the sums.
    const bool asks = (QKV && W == 4) || any;
    Asked asked;
    if (asks) ask(kb_begin, asked);
    Block b;
    // QKV: the heads' sums, all that are asked for at once and before the first keys; a thread has quads of columns of the heads this workgroup needs
    constexpr int NJ = QKV ? (18 * HD / 4 + 64 * W - 1) / (64 * W) : 1, PC = NJ <= 3 ? 8 : 4;
    const bool owner = QKV && pos0 >= key_begin && pos0 < key_end;  // the item whose keys end with the new one
    int slot = -1;
    if constexpr (QKV) slot = reinterpret_cast<const int32_t*>(q)[q_row0];  // (there are no queries: what stands there is where tokens go)
    if constexpr (QKV) {
        floatx4 part[NJ][PC], bias_of[NJ];
        float2 angle = float2{1.f, 0.f};
        const float* at[NJ];
        const int n_cols = (gh_here + 2) * HD, q_dim = n_heads * HD, kv_dim = n_kv * HD;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            if (j > 0 && j * 64 * W * 4 >= n_cols) continue;  // (the same for the whole workgroup, as below)
            const int i = (static_cast<int>(threadIdx.x) + j * 64 * W) * 4, ic = i < n_cols ? i : 0;
            const int seg = ic / HD, d = ic - seg * HD;
            const int col = seg < gh_here ? (h_base + seg) * HD + d : q_dim + (seg - gh_here) * kv_dim + kvh * HD + d;
            at[j] = f.sums + static_cast<int64_t>(q_row0) * f.width + col;
#pragma unroll
            for (int u = 0; u < PC; ++u) part[j][u] = *reinterpret_cast<const floatx4*>(at[j] + min(u, f.n_parts - 1) * f.part_stride);
            bias_of[j] = *reinterpret_cast<const floatx4*>(f.bias ? f.bias + col : at[j]);
        }
        const float2* table_row = reinterpret_cast<const float2*>(f.cos_sin) + static_cast<int64_t>(q_row0) * (HD / 2);
        if (f.cos_sin) angle = table_row[min(static_cast<int>(threadIdx.x), HD / 2 - 1)];
        if (asks) load(asked, b);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            if (j > 0 && j * 64 * W * 4 >= n_cols) continue;
            const int i = (static_cast<int>(threadIdx.x) + j * 64 * W) * 4;
            floatx4 a = part[j][0];
#pragma unroll
            for (int u = 1; u < PC; ++u)
                if (u < f.n_parts) a += part[j][u];
            for (int s = PC; s < f.n_parts; ++s) a += *reinterpret_cast<const floatx4*>(at[j] + s * f.part_stride);
            if (f.bias) a += bias_of[j];
            if (i < n_cols) *reinterpret_cast<floatx4*>(s_row + i / HD * RS + i % HD) = a;
        }
        // (four waves, two heads' halves of up to 128 pairs: a thread a pair)
        if (static_cast<int>(threadIdx.x) < HD / 2) s_cs[threadIdx.x] = angle;
        __syncthreads();
    }
    // four values of a head from d on, turned
    auto head_values = [&](int seg, int d, bool turn) -> floatx4 {
        const float* head = s_row + seg * RS;
        const floatx4 mine = *reinterpret_cast<const floatx4*>(head + d);
        if (!turn) return mine;
        const bool second = d >= HD / 2;
        const int i = second ? d - HD / 2 : d;
        const floatx4 other = *reinterpret_cast<const floatx4*>(head + (second ? i : i + HD / 2));
        floatx4 r;
#pragma unroll
        for (int e = 0; e < 4; ++e) r[e] = turned(second ? other[e] : mine[e], second ? mine[e] : other[e], s_cs[i + e].x, s_cs[i + e].y, second);
        return r;
    };
    // this lane's query row; a row that does not exist reads the item's first one and is masked
    const int tq = c / gh, hh = c - tq * gh;
    const bool row_ok = tq < n_q && hh < gh_here;
    const int head = h_base + (row_ok ? hh : 0), row = q_row0 + (row_ok ? tq : 0), pos = pos0 + tq;
    floatx4 qf[HDT];
    if constexpr (QKV) {
        if (any) {  // (one question for all of them: with one each every read of LDS waited for the last)
            if (f.cos_sin) {
#pragma unroll
                for (int j = 0; j < HDT; ++j) qf[j] = head_values(row_ok ? hh : 0, 16 * j + 4 * G, true);
            } else {
#pragma unroll
                for (int j = 0; j < HDT; ++j) qf[j] = head_values(row_ok ? hh : 0, 16 * j + 4 * G, false);
            }
        }
    } else if (W < 16 || any) {  // (of sixteen waves most have no key where items are short, and read nothing; eight are slower with the question)
        const float* qp = q + static_cast<int64_t>(row) * q_stride + static_cast<int64_t>(head) * HD + 4 * G;
#pragma unroll
        for (int j = 0; j < HDT; ++j) qf[j] = *reinterpret_cast<const floatx4*>(qp + 16 * j);
    }
    const float factor_in = row_scale ? scale * row_scale[row] : scale;
    const float slope = slopes ? slopes[head] : 0.f;

    float m_run = -INFINITY, l_run = 0.f;
    floatx4 acc[HDT];
#pragma unroll
    for (int j = 0; j < HDT; ++j) acc[j] = floatx4{0.f, 0.f, 0.f, 0.f};
    if constexpr (QKV) {
        // the new key and value into the pools, by the last wave
        if (owner && chunk == 0 && wave == W - 1) {
            if (slot >= 0 && slot < f.pool_slots) {
                const int page = slot / page_size, off = slot - page * page_size;
                float* kd = f.k_out + page * page_stride + kv_base + static_cast<int64_t>(off) * HD;
                float* vd = f.v_out + page * page_stride + kv_base + off;
                for (int d = 4 * lane; d < HD; d += 256) *reinterpret_cast<floatx4*>(kd + d) = head_values(gh_here, d, f.cos_sin != nullptr);
                for (int d = lane; d < HD; d += 64) vd[static_cast<int64_t>(d) * page_size] = s_row[(gh_here + 1) * RS + d];
            }
        }
    } else {
        if (any) load(asked, b);
    }
    for (int kb = kb_begin; kb < kb_end;) {
        if constexpr (QKV) {
            // (what the pools hold at the new key's place is not looked at)
            if (owner && kb >= kb_first && pos0 >= kb && pos0 < kb + 16) {
                const int new_i = pos0 - (kb + 4 * G);
                const float* value = s_row + (gh_here + 1) * RS + c;
#pragma unroll
                for (int j = 0; j < HDT; ++j) {
                    const floatx4 key = head_values(gh_here, 16 * j + 4 * G, f.cos_sin != nullptr);
                    if (kb + c == pos0) b.k[j] = key;
#pragma unroll
                    for (int i = 0; i < 4; ++i) b.v[j][i] = i == new_i ? value[16 * j] : b.v[j][i];
                }
            }
        }
        floatx4 st{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < HDT; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) st = __builtin_amdgcn_mfma_f32_16x16x4f32(b.k[j][i], qf[j][i], st, 0, 0, 0);
        const bool kept = kb < kb_first;  // a block of the kept first keys (the same for the whole wave)
        const int of_range = key_end, of_kept = prefix_end;
        const int range_begin = kept ? 0 : key_begin, range_end = kept ? of_kept : of_range;
        const int first = (kept ? kb - walk_first : kb) + 4 * G;  // this lane's keys: first .. first + 3
        const int upto = min(range_end, pos + 1), hi = (row_ok & b.v_ok) ? upto : kFarBelow;
        const int in_window = pos - window + 1, seen = window > 0 ? in_window : kFarBelow;
        float s[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            s[i] = st[i] * factor_in;
            if (softcap > 0.f) s[i] = softcap * tanhf(s[i] / softcap);  // (the same for the whole launch, as the next)
            if (slopes) s[i] = fmaf(slope, static_cast<float>(first + i - pos), s[i]);
            const int key = first + i;
            const bool vis = (key < hi) & (key >= range_begin) & ((key >= seen) | (key < keep));
            s[i] = vis ? s[i] : -INFINITY;
        }
        if (__any(!b.v_ok | (first + 3 >= range_end))) {
            // values outside the range need not be numbers: they must not meet their probabilities of zero
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const bool held = b.v_ok & (first + i < range_end);
#pragma unroll
                for (int j = 0; j < HDT; ++j) b.v[j][i] = held ? b.v[j][i] : 0.f;
            }
        }
        const float m_loc = max_xor32(max_xor16(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]))));
        const float m_new = fmaxf(m_run, m_loc);
        const float m_of = m_new == -INFINITY ? 0.f : m_new;  // (a row without a key so far: all its probabilities zero)
        const float corr = m_run == -INFINITY ? 1.f : expf(m_run - m_of);
        float p[4], p_sum = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            p[i] = expf(s[i] - m_of);
            p_sum += p[i];
        }
        l_run = l_run * corr + p_sum;  // this lane's keys only; the lane groups are summed at the end
        m_run = m_new;
        if (__any(corr != 1.f)) {
#pragma unroll
            for (int j = 0; j < HDT; ++j) acc[j] *= corr;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < HDT; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b.v[j][i], p[i], acc[j], 0, 0, 0);
        kb += 16;
        if (kb >= kb_end) break;
        ask(kb, asked);
        load(asked, b);
    }

    if (wave < n_runs) {
#pragma unroll
        for (int j = 0; j < HDT; ++j) s_o[(wave * HDT + j) * 64 + lane] = acc[j];
    }
    const float l_w = sum_xor32(sum_xor16(l_run));
    if (G == 0) {  // (a wave without keys: minus infinity and zero)
        s_m[c][wave] = m_run;
        s_l[c][wave] = l_w;
    }
    __syncthreads();
    if (!row_ok) return;
    float m_of_run[MW], l_of_run[MW], factor[MW];
#pragma unroll
    for (int w = 0; w < MW; w += 4) {
        if (W == 16 && w >= n_runs) {  // (the same for the whole workgroup, as below; what is left out adds zeros)
#pragma unroll
            for (int i = 0; i < 4; ++i) m_of_run[w + i] = -INFINITY, l_of_run[w + i] = 0.f;
            continue;
        }
        const floatx4 m4 = *reinterpret_cast<const floatx4*>(&s_m[c][w]), l4 = *reinterpret_cast<const floatx4*>(&s_l[c][w]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const bool is = w + i < n_runs;
            m_of_run[w + i] = is ? m4[i] : -INFINITY;
            l_of_run[w + i] = is ? l4[i] : 0.f;
        }
    }
    float m_all = m_of_run[0];
#pragma unroll
    for (int w = 1; w < W; ++w) m_all = fmaxf(m_all, m_of_run[w]);
    const float m_of = m_all == -INFINITY ? 0.f : m_all;
    float denom = 0.f;
#pragma unroll
    for (int w0 = 0; w0 < MW; w0 += 4) {
        if (W == 16 && w0 >= n_runs) break;
#pragma unroll
        for (int w = w0; w < w0 + 4; ++w) {
            factor[w] = expf(m_of_run[w] - m_of);
            denom = fmaf(l_of_run[w], factor[w], denom);
        }
    }
    float inv = 1.f;
    if (partial_base < 0) {
        // a sink is one more term of the denominator, exp(sink) relative to the maximum; it has no value
        const float whole = denom + ((sinks && m_all != -INFINITY) ? expf(sinks[head] - m_all) : 0.f);
        inv = whole > 0.f ? 1.0f / whole : 0.f;
    }
    float* o = out + (static_cast<int64_t>(row) * n_heads + head) * HD + 4 * G;
    // (a cut item's record: unnormalised sums, their maximum and denominator, for attention_merge)
    float* rec = partials + (static_cast<int64_t>(max(partial_base, 0) + tq) * n_heads + head) * (HD + 2);
    for (int j = wave; j < HDT; j += W) {
        floatx4 a{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w0 = 0; w0 < W; w0 += 4) {
            if (w0 >= n_runs) break;  // (the same for the whole workgroup)
            floatx4 v[4];  // four at once, past the last run the last one again, not added
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = s_o[(min(w0 + i, n_runs - 1) * HDT + j) * 64 + lane];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) a[r] = w0 + i < n_runs ? fmaf(v[i][r], factor[w0 + i], a[r]) : a[r];
        }
        if (partial_base < 0) {
            *reinterpret_cast<floatx4*>(o + 16 * j) = a * inv;
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) rec[16 * j + 4 * G + r] = a[r];
        }
    }
    if (partial_base >= 0 && wave == 0 && G == 0) {
        rec[HD] = m_all;
        rec[HD + 1] = denom;
    }
}

template <int HDT, int W>
void launch_waves(const F32Call& a, dim3 grid, int group, int gh, hipStream_t stream) {
    const uint32_t page_magic = 0xFFFFFFFFu / static_cast<uint32_t>(a.page_size) + 1u;
    if constexpr (HDT <= kSumsHdt)
        if (a.sums.sums)
            return attention_f32_kernel<HDT, W, true><<<grid, 64 * W, 0, stream>>>(
            a.items, a.block_tables, a.max_pages, a.page_size, page_magic, a.n_kv, a.k_pool, a.v_pool, reinterpret_cast<const float*>(a.sums.slots), 0, a.out, a.partials, a.n_heads, group,
                gh, a.window, a.scale, 0.f, nullptr, a.slopes, a.row_scale, a.sums);
    attention_f32_kernel<HDT, W, false><<<grid, 64 * W, 0, stream>>>(
            a.items, a.block_tables, a.max_pages, a.page_size, page_magic, a.n_kv, a.k_pool, a.v_pool, a.q, a.q_stride, a.out, a.partials, a.n_heads, group,
            gh, a.window, a.scale, a.softcap, a.sinks, a.slopes, a.row_scale, a.sums);
}

template <int HDT>
int launch(const F32Call& a, hipStream_t stream) {
    const int group = a.n_heads / a.n_kv, gh = group < 16 ? group : 16;
    const dim3 grid(a.n_items, a.n_kv, (group + gh - 1) / gh);
    constexpr int W = f32_waves<HDT>();
    // Workgroups of eight and sixteen waves share a unit by twos at most, and short items leave most of their waves without a key:
    // beyond the units four waves, the same waves in flight in smaller pieces.  Over cold keys, us, the vector units' kernel / all
    // waves / four: 64 requests of 40 keys, 16 heads on 16 of 64 17.2 / 21.5 / 9.5, 200 of 300 278 / 203 / 130; 200 of 1,000, 14 on 2
    // of 64 94 / 69 / 50; 64 of 700, 32 on 32 of 128 514 / 308 / 271; 16 prompts of 60 tokens, 32 on 4 of 32 26.8 / 31.4 / 10.4.  An
    // item of up to four blocks gives the same bits by either; a launch with longer tiles of prompts asks for all waves, since a
    // portion's sums are not to follow from what else is in the step (300 tokens, 14 on 2 of 64, 14.9 us where four took 13.2).
    const bool many = static_cast<int64_t>(grid.x) * grid.y * grid.z > fsie_compute_units();
    if (W > 4 && (many || a.few_waves) && !a.all_waves) launch_waves<HDT, 4>(a, grid, group, gh, stream);
    else launch_waves<HDT, W>(a, grid, group, gh, stream);
    FSIE_CHECK_LAUNCH("attention_f32");
    return 0;
}

template <int HDT>
int launch_from(int hdt, const F32Call& a, hipStream_t stream) {
    if (hdt == HDT) return launch<HDT>(a, stream);
    if constexpr (HDT < 16) return launch_from<HDT + 1>(hdt, a, stream);
    fsie_set_error("attention_f32: no kernel for head_dim %d", 16 * hdt);
    return 1;
}

}  // namespace

// Whether fsie_attention_f32 takes these sizes (float32 storage).
extern "C" int fsie_attention_f32_ok(int head_dim, int page_size) {
    return head_dim > 0 && head_dim % 16 == 0 && head_dim <= 256 && page_size > 0 && page_size % 4 == 0;
}

// Attention of float32 queries over float32 pools: items of at most 16 rows (tokens x heads of a group, as
// fsie_attention_scalar's), records and the other operands as there.  Rows of q, and the pools, on 16 bytes.
extern "C" int fsie_attention_f32(const float* q, int64_t q_stride, const float* k_pool, const float* v_pool,
                                  const int32_t* block_tables, int max_pages, const int32_t* items, int n_items, float* out,
                                  float* partials, int n_heads, int n_kv, int head_dim, int page_size, int window, float scale,
                                  const float* sinks, float softcap, const float* slopes, const float* row_scale, int all_waves,
                                  hipStream_t stream) {
    FSIE_REQUIRE(n_items >= 0 && n_heads > 0 && n_kv > 0 && n_heads % n_kv == 0,
                 "attention: heads %d must be a positive multiple of kv heads %d", n_heads, n_kv);
    FSIE_REQUIRE(fsie_attention_f32_ok(head_dim, page_size),
                 "attention_f32: head_dim %d must be a multiple of 16 up to 256 and page_size %d of 4", head_dim, page_size);
    FSIE_REQUIRE(max_pages > 0 && (static_cast<int64_t>(max_pages) + 8) * page_size * page_size < (int64_t{1} << 32),
                 "attention_f32: %d pages of %d keys are more than the kernel can address", max_pages, page_size);
    FSIE_REQUIRE(q && k_pool && v_pool && block_tables && items && out, "attention_f32: missing operand");
    FSIE_REQUIRE(q_stride % 4 == 0 && reinterpret_cast<uintptr_t>(q) % 16 == 0 && reinterpret_cast<uintptr_t>(k_pool) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(v_pool) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0,
                 "attention_f32: rows of q, the pools and the result must be 16-byte aligned");
    if (n_items == 0) return 0;
    F32Call a{};
    a.q = q, a.k_pool = k_pool, a.v_pool = v_pool, a.q_stride = q_stride, a.block_tables = block_tables, a.items = items;
    a.out = out, a.partials = partials, a.n_items = n_items, a.max_pages = max_pages, a.n_heads = n_heads, a.n_kv = n_kv;
    a.page_size = page_size, a.window = window, a.scale = scale, a.softcap = softcap;
    a.sinks = sinks, a.slopes = slopes, a.row_scale = row_scale, a.all_waves = all_waves;
    return launch_from<1>(head_dim / 16, a, stream);
}

// The same for a step of one token a request (every item has one query row a head), from the q/k/v product's partial sums [n_parts][n_tokens][(n_heads + 2 n_kv) head_dim]:
// adds them up, adds `bias` (or null), turns queries and keys by cos_sin [n_tokens][head_dim / 2][2] (or null: not), takes the new key and value from there and
// writes them to slots[t] of the pools (negative, or not below pool_slots: not).
extern "C" int fsie_attention_f32_qkv(const float* sums, int n_parts, int n_tokens, const float* bias, const float* cos_sin, const int32_t* slots,
                                      float* k_pool, float* v_pool, int64_t pool_slots, const int32_t* block_tables, int max_pages,
                                      const int32_t* items, int n_items, float* out, float* partials, int n_heads, int n_kv, int head_dim,
                                      int page_size, int window, float scale, int short_items, const float* slopes, const float* row_scale, hipStream_t stream) {
    FSIE_REQUIRE(n_items >= 0 && n_heads > 0 && n_kv > 0 && n_heads % n_kv == 0,
                 "attention_f32_qkv: heads %d must be a positive multiple of kv heads %d", n_heads, n_kv);
    FSIE_REQUIRE(fsie_attention_f32_ok(head_dim, page_size) && head_dim <= 16 * kSumsHdt,
                 "attention_f32_qkv: head_dim %d must be a multiple of 16 up to 128 and page_size %d of 4", head_dim, page_size);
    FSIE_REQUIRE(max_pages > 0 && (static_cast<int64_t>(max_pages) + 8) * page_size * page_size < (int64_t{1} << 32),
                 "attention_f32_qkv: %d pages of %d keys are more than the kernel can address", max_pages, page_size);
    FSIE_REQUIRE(n_parts >= 1 && n_parts <= FSIE_GEMM_MAX_SPLITS && n_tokens >= 1 && pool_slots >= 0, "attention_f32_qkv: bad sizes parts=%d T=%d", n_parts, n_tokens);
    FSIE_REQUIRE(sums && slots && k_pool && v_pool && block_tables && items && out, "attention_f32_qkv: missing operand");
    FSIE_REQUIRE(reinterpret_cast<uintptr_t>(sums) % 16 == 0 && reinterpret_cast<uintptr_t>(bias) % 16 == 0 && reinterpret_cast<uintptr_t>(cos_sin) % 8 == 0 &&
                     reinterpret_cast<uintptr_t>(k_pool) % 16 == 0 && reinterpret_cast<uintptr_t>(v_pool) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0,
                 "attention_f32_qkv: sums, bias, the pools and the result must be 16-byte aligned, the cosines and sines 8-byte");
    if (n_items == 0) return 0;
    F32Call a{};
    a.k_pool = k_pool, a.v_pool = v_pool, a.block_tables = block_tables, a.items = items;
    a.out = out, a.partials = partials, a.n_items = n_items, a.max_pages = max_pages, a.n_heads = n_heads, a.n_kv = n_kv;
    a.page_size = page_size, a.window = window, a.scale = scale, a.slopes = slopes, a.row_scale = row_scale, a.few_waves = short_items;
    a.sums = F32Sums{sums, bias, cos_sin, slots, k_pool, v_pool, 0, pool_slots, n_parts, (n_heads + 2 * n_kv) * head_dim};
    a.sums.part_stride = static_cast<int64_t>(n_tokens) * a.sums.width;
    return launch_from<1>(head_dim / 16, a, stream);
}
