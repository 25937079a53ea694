// Entry point of the matrix-core attention (bfloat16): picks the instantiation for the head size.
#include "attention_mfma_impl.h"

namespace fsie_attn {
LaunchFn table_a(int hdt, int large);
LaunchFn table_b(int hdt, int large);
LaunchFn table_c(int hdt, int large);
LaunchFn table_d(int hdt, int large);
LaunchQkvOFn table_a_qkv_o(int hdt);
LaunchQkvOFn table_b_qkv_o(int hdt);
LaunchQkvFn table_a_qkv(int hdt);
LaunchQkvFn table_b_qkv(int hdt);
LaunchQkvFn table_c_qkv(int hdt);
LaunchQkvFn table_d_qkv(int hdt);
}  // namespace fsie_attn

// Waves that a workgroup of the small variant may use to split an item's keys.
extern "C" int fsie_attention_mfma_max_waves(int head_dim) {
    if (head_dim <= 0 || head_dim % 16 || head_dim > 256) return 0;
    return head_dim <= 64 ? 16 : (head_dim <= 128 ? 8 : 4);
}

// Query tiles of 16 rows that one wave of the `large` variant holds for this head size.
extern "C" int fsie_attention_mfma_tiles(int head_dim, int large) {
    if (head_dim <= 0 || head_dim % 16 || head_dim > 256) return 0;
    if (!large) return 1;
    return 2;
}

// bfloat16 only; head_dim a multiple of 16 up to 256; page_size a multiple of 4.
// large = 0: items of at most 16 rows (tokens x heads of a group); large = 1: up to 16 * tiles rows.
// waves: of a workgroup, that split each item's keys.  large = 0: 1, the variant for items of up to four blocks of 32 keys; 0, the same for
// any items, where more workgroups than units share the memory's rate; more, as many as the head size has.  large = 1: at most 4.
// slopes [n_heads] (or null): slopes[h] * (query position - key position) is taken off head h's scores, after the cap;
// row_scale (or null): a factor a token (indexed like the rows of q) on its scores, before the cap.
extern "C" int fsie_attention_mfma(const void* q, int64_t q_stride, const void* k_pool, const void* v_pool,
                                   const int32_t* block_tables, int max_pages, const int32_t* items, int n_items,
                                   void* out, float* partials, int n_heads, int n_kv, int head_dim, int page_size,
                                   int window, float scale, int large, int waves, const float* sinks, float softcap,
                                   const float* slopes, const float* row_scale, hipStream_t stream) {
    FSIE_REQUIRE(n_items >= 0 && n_heads > 0 && n_kv > 0 && n_heads % n_kv == 0,
                 "attention_mfma: heads %d must be a positive multiple of kv heads %d", n_heads, n_kv);
    FSIE_REQUIRE(head_dim > 0 && head_dim % 16 == 0 && head_dim <= 256,
                 "attention_mfma: head_dim %d must be a multiple of 16 up to 256", head_dim);
    FSIE_REQUIRE(page_size > 0 && page_size % 4 == 0, "attention_mfma: page_size %d must be a multiple of 4", page_size);
    FSIE_REQUIRE(max_pages > 0, "attention_mfma: empty block table");
    // the kernel divides a key's position by the page size with one multiplication, exact below this
    FSIE_REQUIRE((static_cast<int64_t>(max_pages) + 8) * page_size * page_size < (int64_t{1} << 32),
                 "attention_mfma: %d pages of %d keys are more than the kernel can address", max_pages, page_size);
    FSIE_REQUIRE(q_stride % 8 == 0 && reinterpret_cast<uintptr_t>(q) % 16 == 0,
                 "attention_mfma: query rows must be 16-byte aligned");
    if (n_items == 0) return 0;
    const int hdt = head_dim / 16;
    fsie_attn::LaunchFn fn = hdt <= 4 ? fsie_attn::table_a(hdt, large)
                           : hdt <= 8 ? fsie_attn::table_b(hdt, large)
                           : hdt <= 12 ? fsie_attn::table_c(hdt, large) : fsie_attn::table_d(hdt, large);
    FSIE_REQUIRE(fn != nullptr, "attention_mfma: no kernel for head_dim %d", head_dim);
    return fn(q, q_stride, k_pool, v_pool, block_tables, max_pages, items, n_items, out, partials, n_heads, n_kv,
              page_size, window, scale, waves, sinks, softcap, slopes, row_scale, stream);
}

// Whether fsie_attention_mfma_qkv has a kernel for these sizes.
extern "C" int fsie_attention_mfma_qkv_ok(int head_dim, int page_size) {
    return head_dim > 0 && head_dim % 32 == 0 && head_dim <= 256 && page_size > 0 && page_size % 8 == 0;
}

namespace {

// What both entry points for a step's q/k/v sums check alike, and their operands as the kernel takes them.
int operands_of(fsie_attn::QkvSums& f, const float* sums, int n_parts, int n_tokens, const float* bias, const float* cos_sin,
                const int32_t* slots, void* k_pool, void* v_pool, int64_t pool_slots, const int32_t* block_tables, int max_pages,
                const int32_t* items, int n_items, int n_heads, int n_kv, int head_dim, int page_size) {
    FSIE_REQUIRE(n_items >= 0 && n_heads > 0 && n_kv > 0 && n_heads % n_kv == 0,
                 "attention_mfma_qkv: heads %d must be a positive multiple of kv heads %d", n_heads, n_kv);
    FSIE_REQUIRE(fsie_attention_mfma_qkv_ok(head_dim, page_size),
                 "attention_mfma_qkv: head_dim %d must be a multiple of 32 up to 256 and page_size %d a multiple of 8",
                 head_dim, page_size);
    FSIE_REQUIRE(max_pages > 0, "attention_mfma_qkv: empty block table");
    FSIE_REQUIRE((static_cast<int64_t>(max_pages) + 8) * page_size * page_size < (int64_t{1} << 32),
                 "attention_mfma_qkv: %d pages of %d keys are more than the kernel can address", max_pages, page_size);
    FSIE_REQUIRE(n_parts >= 1 && n_tokens >= 1 && pool_slots >= 0, "attention_mfma_qkv: bad sizes parts=%d T=%d",
                 n_parts, n_tokens);
    FSIE_REQUIRE(sums && slots && k_pool && v_pool && block_tables && items, "attention_mfma_qkv: missing operand");
    FSIE_REQUIRE(reinterpret_cast<uintptr_t>(sums) % 16 == 0 && reinterpret_cast<uintptr_t>(bias) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(cos_sin) % 8 == 0 && reinterpret_cast<uintptr_t>(k_pool) % 4 == 0,
                 "attention_mfma_qkv: sums and bias must be 16-byte aligned, the cosines and sines 8-byte");
    f.sums = sums;
    f.bias = bias;
    f.cos_sin = cos_sin;
    f.slots = slots;
    f.k_out = static_cast<bf16_t*>(k_pool);
    f.v_out = static_cast<bf16_t*>(v_pool);
    f.width = (n_heads + 2 * n_kv) * head_dim;
    f.part_stride = static_cast<int64_t>(n_tokens) * f.width;
    f.pool_slots = pool_slots;
    f.n_parts = n_parts;
    f.group = n_heads / n_kv;
    f.page_magic = fsie_attn::magic_of(page_size);
    return 0;
}

}  // namespace

// Attention for a step of one token a request (every item has one query row per head), straight from
// the q/k/v product's float32 partial sums [n_parts][n_tokens][(n_heads + 2 n_kv) head_dim]: the kernel adds
// them up, adds `bias` (or null), rotates queries and keys by cos_sin [n_tokens][head_dim / 2][2],
// scores the new key from registers and writes it and the value to slots[t] of the pools (negative,
// or not below pool_slots: not written).  cos_sin null: nothing is rotated.  slopes, row_scale: as there.
// Otherwise as fsie_attention_mfma with large = 0.
extern "C" int fsie_attention_mfma_qkv(const float* sums, int n_parts, int n_tokens, const float* bias,
                                       const float* cos_sin, const int32_t* slots, void* k_pool, void* v_pool,
                                       int64_t pool_slots, const int32_t* block_tables, int max_pages,
                                       const int32_t* items, int n_items, void* out, float* partials, int n_heads,
                                       int n_kv, int head_dim, int page_size, int window, float scale, int waves,
                                       const float* slopes, const float* row_scale, hipStream_t stream) {
    fsie_attn::QkvSums f{};
    if (const int rc = operands_of(f, sums, n_parts, n_tokens, bias, cos_sin, slots, k_pool, v_pool, pool_slots, block_tables, max_pages,
                                   items, n_items, n_heads, n_kv, head_dim, page_size))
        return rc;
    FSIE_REQUIRE(out, "attention_mfma_qkv: missing operand");
    if (n_items == 0) return 0;
    const int hdt = head_dim / 16;
    fsie_attn::LaunchQkvFn fn = hdt <= 4 ? fsie_attn::table_a_qkv(hdt)
                              : hdt <= 8 ? fsie_attn::table_b_qkv(hdt)
                              : hdt <= 12 ? fsie_attn::table_c_qkv(hdt) : fsie_attn::table_d_qkv(hdt);
    FSIE_REQUIRE(fn != nullptr, "attention_mfma_qkv: no kernel for head_dim %d", head_dim);
    f.slopes = slopes;
    f.row_scale = row_scale;
    return fn(f, k_pool, v_pool, block_tables, max_pages, items, n_items, out, partials, n_heads, n_kv, page_size,
              window, scale, waves, stream);
}

// Rows of the output projection a wave, for a step of n_items tokens whose items are whole and of at most four blocks of 32 keys; 0: the
// projection is better a launch of its own, or there is no kernel.  Every workgroup makes its kv head's attention again, so they must all be on
// the chip at once, one a unit: the fewest rows for which they are.  Steps of one and of two requests (30 to 100 keys), two launches / one, ms
// for 32 to 40 steps: 14 heads on 2 of 64, hidden size 896 23.23 / 21.60 with two rows (180 workgroups; with three 21.70, four 21.79), 24.23 / 23.06 with
// three (240; with two, 360, 24.27); 12 on 2 of 128, hidden size 1,536 14.61 / 13.66 with three (206; with two, 308, 15.42, with four, 154, 13.77), two
// requests 15.28 / 16.8 to 18.7 (308 and more); 16 on 4 of 64, hidden size 1,024 7.39 / 6.95 with four (208); 8 on 1 of 128, 1,024 7.90 / 7.39.  More rows a wave keep more heads within the units and are slower there: 16 on 8 of 64,
// hidden size 1,024 12.5 / 12.4 with eight rows (208), 15.1 / 17.0 at 2,048; 12 on 12 at 768 9.4 / 9.9.  Every token reads the weight again, which up to some 16 MB of it
// all costs less than the launch: 20 on 2 of 128, 2,560 (13 MB) 12.30 / 12.04; 16 on 1 of 128, 2,304, one token (9) 10.96 / 10.61, two (19) 11.33 / 11.43.
extern "C" int fsie_attention_mfma_qkv_o_rows(int n_items, int n_heads, int n_kv, int head_dim, int page_size, int o_rows, int units) {
    if (n_items <= 0 || n_heads <= 0 || n_kv <= 0 || n_heads % n_kv || n_heads / n_kv > 16 || o_rows <= 0 || units <= 0) return 0;
    if ((head_dim != 64 && head_dim != 128) || !fsie_attention_mfma_qkv_ok(head_dim, page_size)) return 0;
    if (2.0 * n_items * o_rows * n_heads * head_dim > 16e6) return 0;
    for (int rows = 2; rows <= 4; ++rows)
        if (ceil_div64(o_rows, (fsie_attn::kShortWaves + 1) * rows) * n_kv * n_items <= units) return rows;
    return 0;
}

// fsie_attention_mfma_qkv with the output projection behind it: the heads' results, rounded to bfloat16, times o_weight [o_rows][n_heads head_dim] (rows
// without gaps), as float32 sums o_sums [n_kv][n_tokens][o_rows] over the heads of each kv head.  Items are whole (no partial
// records); rows_of_wave as fsie_attention_mfma_qkv_o_rows says.
extern "C" int fsie_attention_mfma_qkv_o(const float* sums, int n_parts, int n_tokens, const float* bias, const float* cos_sin,
                                         const int32_t* slots, void* k_pool, void* v_pool, int64_t pool_slots, const int32_t* block_tables,
                                         int max_pages, const int32_t* items, int n_items, const void* o_weight, int o_rows, float* o_sums,
                                         int rows_of_wave, int n_heads, int n_kv, int head_dim, int page_size, int window, float scale,
                                         hipStream_t stream) {
    fsie_attn::QkvSums f{};
    if (const int rc = operands_of(f, sums, n_parts, n_tokens, bias, cos_sin, slots, k_pool, v_pool, pool_slots, block_tables, max_pages,
                                   items, n_items, n_heads, n_kv, head_dim, page_size))
        return rc;
    FSIE_REQUIRE(o_weight && o_sums && o_rows > 0 && reinterpret_cast<uintptr_t>(o_weight) % 16 == 0,
                 "attention_mfma_qkv_o: the output projection's weight must be 16-byte aligned");
    FSIE_REQUIRE(n_heads / n_kv <= 16 && rows_of_wave >= 2 && rows_of_wave <= 4, "attention_mfma_qkv_o: %d heads on %d, %d rows a wave",
                 n_heads, n_kv, rows_of_wave);
    if (n_items == 0) return 0;
    const fsie_attn::LaunchQkvOFn fn = head_dim <= 64 ? fsie_attn::table_a_qkv_o(head_dim / 16) : fsie_attn::table_b_qkv_o(head_dim / 16);
    FSIE_REQUIRE(fn != nullptr, "attention_mfma_qkv_o: no kernel for head_dim %d", head_dim);
    f.o_weight = static_cast<const bf16_t*>(o_weight);
    f.o_sums = o_sums;
    f.o_rows = o_rows;
    f.o_part_stride = static_cast<int64_t>(n_tokens) * o_rows;
    return fn(f, k_pool, v_pool, block_tables, max_pages, items, n_items, rows_of_wave, n_heads, n_kv, page_size, window, scale, stream);
}
