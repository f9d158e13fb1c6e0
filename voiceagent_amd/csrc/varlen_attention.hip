// Host side of the varlen attention: argument checks and launch dispatch
// (kernel in varlen_kernel.h, instantiated per element type and head_dim in
// varlen_{bf16,f16}_d{64,128}.hip).
#include <algorithm>

#include "varlen_kernel.h"

namespace va {

template <bool kBF16>
static bool dispatch_varlen(int D, int G, const VarlenParams& p, bool causal,
                            int64_t items_per_xcd, hipStream_t st) {
  switch (D) {
    case 64: return launch_varlen_d<kBF16, 64>(G, p, causal, items_per_xcd, st);
    case 128: return launch_varlen_d<kBF16, 128>(G, p, causal, items_per_xcd, st);
    default: return false;
  }
}

static int varlen_native(const va_varlen_args* a, void* stream);

}  // namespace va

// No launch needs a workspace: an FP8 pool's prefix rows are converted
// inside the attention kernel, tile by tile.
extern "C" size_t va_varlen_workspace_bytes(const va_varlen_args* a) {
  (void)a;
  return 0;
}

namespace va {

constexpr int64_t kMaxQBlocks = 65535 * 16;  // query blocks of a sequence

// Whether a launch can list `nqb` query blocks of every (sequence, kv head):
// list indices are 32-bit.
static bool list_fits(const va_varlen_args* a, int64_t nqb) {
  const int64_t npairs = (int64_t)a->num_seqs * a->num_kv_heads;
  return nqb <= kMaxQBlocks && npairs <= INT32_MAX / 2 &&
         (npairs + kXcds - 1) / kXcds * nqb * kXcds <= INT32_MAX;
}

// Per XCD: slots, the items with `rows` MFMA rows each, and the tiles of the
// longest item.  Without the lengths, which are on the device, an item over a
// pool may be as long as the block table is wide; max_seqlen_k, where it is a
// bound at all, says less (an eager step's table may be the model's whole
// width).  The lengths alone decide what is computed.  Slots are counted two a
// CU at head_dim 64 too, where three or four are resident: counted so, both
// rules below took more than they should (64/8 heads of 64, one prompt of 1000
// tokens 31.7 -> 40.3 us; 28 decoding sequences with 4 prompts 25.7 -> 33.6).
struct VarlenLoad {
  int64_t slots, items, longest;
};
static VarlenLoad varlen_load(const va_varlen_args* a, int rows) {
  const int BQ = rows * a->num_kv_heads / a->num_heads;
  int64_t keys = a->pool.k != nullptr ? (int64_t)a->table_width * a->pool.block_size : 0;
  if (a->max_seqlen_k >= a->max_seqlen_q) keys = std::min<int64_t>(keys, a->max_seqlen_k);
  keys = std::max<int64_t>(keys, a->max_seqlen_q);
  VarlenLoad w;
  w.slots = 2 * (int64_t)current_device_cus() / kXcds;
  w.items = (a->num_kv_heads * ((int64_t)a->total_q / BQ + a->num_seqs) + kXcds - 1) / kXcds;
  w.longest = (keys + kKeyTile - 1) / kKeyTile;
  return w;
}

// Tiles of a piece the device would choose (plan_split).
static int64_t split_piece(const VarlenLoad& w) {
  const int64_t over =
      std::min<int64_t>(std::max(w.slots - w.items / 4, (w.slots + 1) / 2), kSplitOver);
  return std::max<int64_t>(w.items * w.longest / 2 / over, kSplitMinTiles);
}

// Whether a launch gains from splitting its items, from what the host knows.
// With items of half the longest one's tiles on average, a slot's share is the
// piece the device would choose.  The pieces' partials and the merge launch
// cost 5-10 us, growing with the items, and a tile saved gives 1.2-1.5 us, so
// over a prefix the longest item has to exceed a piece by a quarter and three
// tiles and one more for each item of an XCD, up to nine.  Whole against
// split, us, 16/8 heads of 128: 30 tokens over 400 keys 15.2 / 14.6; four such
// prompts 15.8 / 17.1, at 64/8 heads 16.0 / 21.5; 64 over 1000 28.1 / 20.2.
// New prompts' own blocks fill the slots with items whose lengths fall evenly,
// which leaves splitting less to even out: one prompt of 420 tokens 15.3 /
// 18.5, of 2500 (2.86 pieces long) 59.4 / 62.1, four of 300 15.5 / 20.5, and
// at head_dim 64, 32/8 heads, 14.3 / 19.3.  It pays at 2.94 pieces and above
// (8/8 heads of 128: 3000 tokens beside eight prompts of 100 62.4 / 55.3, one
// of 4000 81.9 / 73.8), not for short ones (one of 1000 at 16/8 26.7 / 30.3).
static bool split_wanted(const va_varlen_args* a) {
  if (a->num_kv_heads <= 0 || a->num_heads % a->num_kv_heads != 0) return false;
  const int G = a->num_heads / a->num_kv_heads;
  if (G != 1 && G != 2 && G != 4 && G != 8) return false;
  if (a->head_dim != 64 && a->head_dim != 128) return false;
  if (a->num_seqs <= 0 || a->total_q <= 0) return false;
  if (!a->causal && a->pool.k == nullptr && a->max_seqlen_q <= kRowsPerWG / G) return false;  // kOnce
  const int64_t pairs = (int64_t)a->num_seqs * a->num_kv_heads;
  if ((pairs + kXcds - 1) / kXcds > 64) return false;  // the plan holds a pair per lane
  const VarlenLoad w = varlen_load(a, kRowsPerWG);
  const int64_t piece = split_piece(w);
  const int64_t prompt = ((int64_t)a->max_seqlen_q + kKeyTile - 1) / kKeyTile;
  if (w.longest > prompt)  // over a prefix
    return w.longest >= piece + piece / 4 + std::min<int64_t>(3 + w.items, 9);
  return w.longest >= 32 && 10 * w.longest >= 29 * piece;
}

// Whether a causal launch takes items of 64 rows (kHalf).  The last slot to
// end has about max(longest item, tiles / slots) tiles (a piece when split);
// with 64 rows an item's tile takes 0.8 of the time where it waits for nothing
// else (580 more tokens in one prompt, nine tiles: 11.4 us against 13.8; 0.7 in
// the rule), and there are up to twice the items, whose set-up and staging
// cost more than that once they come in more than two rounds (one and a half
// at group 8, where a tile is staged for eight positions).  So short blocks
// (decoding sequences, chunks of a few tokens) and launches that do not fill
// the slots take them; a full launch of prompts, or long prefixes over enough
// rows to fill the slots, do not.  128 against 64 rows, us, 16/8 heads of 128: one prompt of 420 tokens
// 18.1 / 15.3; 28 decoding sequences with 4 prompts 29.0 / 25.6; 8 chunks of a
// few tokens over 1K-4K, split, 41.4 / 39.9; 9 prompts of 60-594 tokens 24.1 /
// 22.5; 16 of 109-439 (three rounds of half items) 24.5 / 27.3; 64/8 heads:
// one of 700 (88 items) 28.1 / 27.1, one of 1000 (126) 38.2 / 43.0, two of 500
// 24.7 / 27.8.
// Nor does one whose max_seqlen_q (any bound of the lengths) makes more query
// blocks of half the rows than a launch takes.
static bool half_rows_wanted(const va_varlen_args* a, bool split) {
  if (!a->causal || a->prologue != nullptr) return false;
  const int BQ = kRowsPerWG / 2 * a->num_kv_heads / a->num_heads;
  if (!list_fits(a, ((int64_t)a->max_seqlen_q + BQ - 1) / BQ)) return false;
  const VarlenLoad full = varlen_load(a, kRowsPerWG), half = varlen_load(a, kRowsPerWG / 2);
  auto tiles = [&](const VarlenLoad& w) {
    const int64_t share = (w.items * w.longest / 2 + w.slots - 1) / w.slots;
    return std::max(split ? split_piece(w) : w.longest, share);
  };
  const int64_t most = a->num_heads == 8 * a->num_kv_heads ? half.slots * 3 / 2 : 2 * half.slots;
  return half.items <= most && tiles(half) * 7 < tiles(full) * 10;
}

// Workspace of a split launch: pieces' o, (m, l), heads and counts, for the
// slots its plan may spread over: what is left of those resident beside the
// fewest items there can be, or the pieces that the most and longest items make
// (a bound by the hints of varlen_load, so the plan is held to it).  At 128
// pieces of 128 rows whatever the launch, each took 68 MB at head_dim 128: 30
// tokens over 400 keys take 2.1, four prompts of 200-300 over 2K-8K 52.
struct SplitLayout {
  int over, slots;
  size_t o, ml, head, count, total;
};
static SplitLayout split_layout(const va_varlen_args* a, bool half) {
  const int rows = half ? kRowsPerWG / 2 : kRowsPerWG;
  const VarlenLoad w = varlen_load(a, rows);
  const int64_t resident = waves_per_simd(a->head_dim, half) * (int64_t)current_device_cus() / kXcds;
  const int64_t fewest = w.items - (a->num_seqs * (int64_t)a->num_kv_heads + kXcds - 1) / kXcds;
  SplitLayout l;
  l.over = (int)std::min({std::max(resident - fewest / 4, (resident + 1) / 2),
                          (w.items * (w.longest + 2) + 1) / kSplitMinTiles, (int64_t)kSplitOver});
  l.slots = split_pieces(l.over);
  const size_t pieces = (size_t)kXcds * l.slots;
  l.o = 0;
  l.ml = l.o + pieces * rows * a->head_dim * sizeof(float);
  l.head = l.ml + pieces * rows * sizeof(float2);
  l.count = l.head + pieces * sizeof(int4);
  l.total = l.count + 256;
  return l;
}

}  // namespace va

extern "C" size_t va_varlen_split_workspace_bytes(const va_varlen_args* a) {
  using namespace va;
  if (a == nullptr || a->struct_size != sizeof(va_varlen_args)) return 0;
  return split_wanted(a) ? split_layout(a, half_rows_wanted(a, true)).total : 0;
}

extern "C" int va_varlen_attention(const va_varlen_args* a, void* stream) {
  using namespace va;
  VA_CHECK_ARG(a != nullptr, "va_varlen_attention: null args");
  VA_CHECK_ARG(a->struct_size == sizeof(va_varlen_args),
               "va_varlen_attention: struct_size %u != %zu (header/library mismatch)",
               a->struct_size, sizeof(va_varlen_args));
  VA_CHECK_ARG(a->num_seqs >= 0, "va_varlen_attention: num_seqs < 0");
  if (a->num_seqs == 0 || a->total_q == 0) return VA_OK;
  const bool has_pool = a->pool.k != nullptr;
  VA_CHECK_ARG(!has_pool || a->pool.kv_format == VA_KV_NATIVE ||
                   a->pool.kv_format == VA_KV_FP8_E4M3,
               "va_varlen_attention: unknown kv_format %d", a->pool.kv_format);
  if (!has_pool || a->pool.kv_format == VA_KV_NATIVE) return varlen_native(a, stream);

  // ---- FP8 pool: attention with the prefix converted in the kernel, then
  // the quantising store of the new rows ----
  VA_CHECK_ARG(a->pool.k_scale > 0.f && a->pool.v_scale > 0.f,
               "va_varlen_attention: FP8 pool scales must be positive");
  va_varlen_args b = *a;
  b.slot_mapping = nullptr;
  int rc = varlen_native(&b, stream);
  if (rc != VA_OK || a->slot_mapping == nullptr) return rc;

  va_store_args sa{};
  sa.struct_size = sizeof(va_store_args);
  sa.dtype = a->dtype;
  sa.key = a->k;
  sa.value = a->v;
  sa.key_stride_tok = a->k_stride_tok;
  sa.key_stride_head = a->k_stride_head;
  sa.value_stride_tok = a->v_stride_tok;
  sa.value_stride_head = a->v_stride_head;
  sa.pool = a->pool;
  sa.slot_mapping = a->slot_mapping;
  sa.slot_dtype = a->slot_dtype;
  sa.num_tokens = a->total_q;
  sa.num_kv_heads = a->num_kv_heads;
  sa.head_dim = a->head_dim;
  return va_store_kvcache(&sa, stream);
}

int va::varlen_native(const va_varlen_args* a, void* stream) {
  using namespace va;
  VA_CHECK_ARG(a->dtype == VA_BF16 || a->dtype == VA_F16,
               "va_varlen_attention: dtype must be VA_BF16 or VA_F16 (MFMA path)");
  VA_CHECK_ARG(a->q && a->out && a->cu_seqlens_q && a->cu_seqlens_k,
               "va_varlen_attention: null pointer argument");
  VA_CHECK_ARG(a->num_seqs <= 65535, "va_varlen_attention: num_seqs > 65535");
  VA_CHECK_ARG(a->num_kv_heads > 0 && a->num_kv_heads <= 65535 && a->num_heads > 0 &&
                   a->num_heads % a->num_kv_heads == 0,
               "va_varlen_attention: num_heads (%d) must be a positive multiple of "
               "num_kv_heads (%d)",
               a->num_heads, a->num_kv_heads);
  const bool has_pool = a->pool.k != nullptr;
  VA_CHECK_ARG(has_pool || (a->k && a->v), "va_varlen_attention: k/v required without a pool");
  VA_CHECK_ARG(!has_pool || (a->pool.v && a->block_tables && a->pool.block_size > 0 &&
                             a->pool.num_blocks >= 0 && a->table_width >= 0),
               "va_varlen_attention: incomplete pool description");
  VA_CHECK_ARG((a->k == nullptr) == (a->v == nullptr),
               "va_varlen_attention: k and v must be given together");
  VA_CHECK_ARG(a->slot_mapping == nullptr || (has_pool && a->k),
               "va_varlen_attention: slot_mapping needs a pool and k/v");
  VA_CHECK_ARG(a->max_seqlen_q >= 0 && a->max_seqlen_k >= 0, "va_varlen_attention: max_seqlen");
  VA_CHECK_ARG(!has_pool || a->table_dtype == VA_I32 || a->table_dtype == VA_I64,
               "va_varlen_attention: table_dtype");
  VA_CHECK_ARG(a->slot_mapping == nullptr || a->slot_dtype == VA_I32 || a->slot_dtype == VA_I64,
               "va_varlen_attention: slot_dtype");
  // An FP8 pool holds one byte per element (its strides count bytes).
  const bool f8 = has_pool && a->pool.kv_format == VA_KV_FP8_E4M3;
  VA_CHECK_ARG(!f8 || a->head_dim % 16 == 0,
               "va_varlen_attention: FP8 pool head_dim must be a multiple of 16");
  const int64_t kv_eb = f8 ? 1 : 2;
  const int64_t strides[] = {a->q_stride_tok,  a->q_stride_head,      a->k_stride_tok,
                             a->k_stride_head, a->v_stride_tok,       a->v_stride_head,
                             a->out_stride_tok, a->out_stride_head};
  for (int64_t s : strides)
    VA_CHECK_ARG((s * 2) % 16 == 0, "va_varlen_attention: strides must be 16-byte multiples");
  const int64_t pstrides[] = {a->pool.stride_block, a->pool.stride_slot, a->pool.stride_head};
  for (int64_t s : pstrides)
    VA_CHECK_ARG((s * kv_eb) % 16 == 0,
                 "va_varlen_attention: pool strides must be 16-byte multiples");
  const uintptr_t ptrs[] = {(uintptr_t)a->q, (uintptr_t)a->k, (uintptr_t)a->v, (uintptr_t)a->out,
                            (uintptr_t)a->pool.k, (uintptr_t)a->pool.v};
  for (uintptr_t p : ptrs)
    VA_CHECK_ARG(p % 16 == 0, "va_varlen_attention: pointers must be 16-byte aligned");
  VA_CHECK_ARG(a->scale > 0.f && a->scale < INFINITY, "va_varlen_attention: scale must be > 0");
  if (a->k != nullptr) {
    // Per-lane DMA offsets inside a 64-key tile are 32-bit.
    const int64_t span = (int64_t)(kKeyTile - 1) * (a->k_stride_tok > a->v_stride_tok
                                                        ? a->k_stride_tok
                                                        : a->v_stride_tok) * 2 +
                         (int64_t)a->head_dim * 2;
    VA_CHECK_ARG(a->k_stride_tok >= 0 && a->v_stride_tok >= 0 && span < ((int64_t)1 << 32),
                 "va_varlen_attention: k/v token strides must be non-negative and below 64 MiB");
  }
  const int G = a->num_heads / a->num_kv_heads;
  if (!((a->head_dim == 64 || a->head_dim == 128) && (G == 1 || G == 2 || G == 4 || G == 8))) {
    set_error("va_varlen_attention: unsupported head_dim %d / group size %d (head_dim 64|128, "
              "group 1|2|4|8)",
              a->head_dim, G);
    return VA_ERR_UNSUPPORTED;
  }
  const bool split =
      a->workspace != nullptr && (uintptr_t)a->workspace % 16 == 0 && split_wanted(a) &&
      a->workspace_bytes >= split_layout(a, half_rows_wanted(a, true)).total;
  const bool half = half_rows_wanted(a, split);
  const int BQ = (half ? kRowsPerWG / 2 : kRowsPerWG) / G;
  const int nqb = (int)(((int64_t)a->max_seqlen_q + BQ - 1) / BQ);
  if (nqb == 0) return VA_OK;
  VA_CHECK_ARG(nqb <= kMaxQBlocks, "va_varlen_attention: max_seqlen_q too large");
  VA_CHECK_ARG(list_fits(a, nqb),
               "va_varlen_attention: too many (sequence, kv head, query block) items");

  VarlenParams p;
  p.q = (const char*)a->q;
  p.q_st = a->q_stride_tok * 2;
  p.q_sh = a->q_stride_head * 2;
  p.k = (const char*)a->k;
  p.k_st = a->k_stride_tok * 2;
  p.k_sh = a->k_stride_head * 2;
  p.v = (const char*)a->v;
  p.v_st = a->v_stride_tok * 2;
  p.v_sh = a->v_stride_head * 2;
  p.out = (char*)a->out;
  p.o_st = a->out_stride_tok * 2;
  p.o_sh = a->out_stride_head * 2;
  p.cu_q = a->cu_seqlens_q;
  p.cu_k = a->cu_seqlens_k;
  p.scale_log2 = a->scale * 1.4426950408889634f;
  p.has_pool = has_pool;
  p.kp = (char*)a->pool.k;
  p.vp = (char*)a->pool.v;
  p.s_blk = a->pool.stride_block * kv_eb;
  p.s_slot = a->pool.stride_slot * kv_eb;
  p.s_head = a->pool.stride_head * kv_eb;
  p.kv_f8 = f8;
  p.k_scale = f8 ? a->pool.k_scale : 1.0f;
  p.v_scale = f8 ? a->pool.v_scale : 1.0f;
  p.has_pro = a->prologue != nullptr;
  p.pro = PrologueParams{};
  if (a->prologue != nullptr) {
    const va_qk_prologue& pr = *a->prologue;
    VA_CHECK_ARG(a->causal != 0 && a->head_dim == 128 && !f8,
                 "va_varlen_attention: the fused query prologue needs a causal launch, "
                 "head_dim 128 and a 16-bit pool or none");
    VA_CHECK_ARG(pr.q_norm_weight && pr.cos_sin_cache && pr.positions && pr.max_position > 0 &&
                     pr.cos_sin_stride >= a->head_dim,
                 "va_varlen_attention: prologue weight / rotary cache / positions");
    VA_CHECK_ARG(pr.weight_dtype == VA_BF16 || pr.weight_dtype == VA_F16 ||
                     pr.weight_dtype == VA_F32,
                 "va_varlen_attention: prologue weight_dtype");
    VA_CHECK_ARG(pr.positions_dtype == VA_I32 || pr.positions_dtype == VA_I64,
                 "va_varlen_attention: prologue positions_dtype");
    VA_CHECK_ARG((uintptr_t)pr.q_norm_weight % 16 == 0 && (uintptr_t)pr.cos_sin_cache % 16 == 0 &&
                     (pr.cos_sin_stride * 4) % 16 == 0,
                 "va_varlen_attention: prologue weight and rotary cache must be 16-byte aligned "
                 "(rows too)");
    p.pro.q_w = pr.q_norm_weight;
    p.pro.k_w = pr.q_norm_weight;
    p.pro.w_dtype = pr.weight_dtype;
    p.pro.eps = pr.eps;
    p.pro.cs = pr.cos_sin_cache;
    p.pro.cs_stride = pr.cos_sin_stride;
    p.pro.max_pos = pr.max_position;
    p.pro.pos_i64 = pr.positions_dtype == VA_I64;
    p.pro.pos = pr.positions;
  }
  p.block_size = has_pool ? a->pool.block_size : 1;
  p.num_blocks = a->pool.num_blocks;
  p.table = a->block_tables;
  p.t_sb = a->table_stride_seq;
  p.table_i64 = a->table_dtype == VA_I64;
  p.table_width = a->table_width;
  p.slots = a->slot_mapping;
  p.slot_i64 = a->slot_dtype == VA_I64;
  p.num_qblocks = nqb;
  p.num_seqs = a->num_seqs;
  p.num_kv_heads = a->num_kv_heads;
  p.bs_div = make_fastdiv((uint32_t)p.block_size);
  p.hkv_div = make_fastdiv((uint32_t)a->num_kv_heads);
  p.slot_small = (int64_t)p.num_blocks * p.block_size <= ((int64_t)1 << 31);
  // A tile's 16 rows of one block are copied from one base with 32-bit offsets.
  p.block16 = has_pool && p.block_size % 16 == 0 && p.s_slot >= 0 &&
              15 * p.s_slot + a->head_dim * kv_eb < ((int64_t)1 << 31);

  p.half = half;
  p.split = split;
  p.split_over = p.split_slots = 0;
  p.part_o = nullptr;
  p.part_ml = nullptr;
  p.part_head = nullptr;
  p.part_count = nullptr;
  if (split) {
    const SplitLayout l = split_layout(a, half);
    p.split_over = l.over;
    p.split_slots = l.slots;
    char* const ws = (char*)a->workspace;
    p.part_o = (float*)(ws + l.o);
    p.part_ml = (float2*)(ws + l.ml);
    p.part_head = (int4*)(ws + l.head);
    p.part_count = (int32_t*)(ws + l.count);
  }

  // Persistent 1-D grid over kXcds interleaved item lists; see the kernel.
  const int64_t npairs = (int64_t)a->num_seqs * a->num_kv_heads;
  const int64_t items_per_xcd = (npairs + kXcds - 1) / kXcds * nqb;
  const hipStream_t st = (hipStream_t)stream;
  const bool ok =
      a->dtype == VA_BF16
          ? dispatch_varlen<true>(a->head_dim, G, p, a->causal != 0, items_per_xcd, st)
          : dispatch_varlen<false>(a->head_dim, G, p, a->causal != 0, items_per_xcd, st);
  if (!ok) {
    set_error("va_varlen_attention: unsupported configuration");
    return VA_ERR_UNSUPPORTED;
  }
  return check_launch("va_varlen_attention");
}
