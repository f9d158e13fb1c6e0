// Variable-length attention over packed sequences on CDNA4 bf16/f16 MFMA:
// causal prefill (bottom-right aligned, optionally over a paged prefix with
// the KV store fused) and non-causal block-diagonal encoder windows.
//
// Semantics (flash_attn_varlen_func as qwen_asr_vllm/layers/attention.py
// calls it, :1-11, 92-107, 121-139): sequence s owns queries
// [cu_q[s], cu_q[s+1]) and k_len = cu_k[s+1] - cu_k[s] keys.  Query i of head
// hq sees key j of kv head hq / G iff j < k_len and, when causal,
// j <= k_len - q_len + i; out = softmax(scale * q.K^T) V over visible keys
// (0 when none is visible).  The non-causal case with cu_q = cu_k is the
// block-diagonal mask of reference/modeling_qwen3_asr.py:649-667.
//
// Tiling (one workgroup = 4 wave64 = 256 lanes): an item is one
// (sequence, kv head, query block) with all G query heads of the kv group,
// so its 128 MFMA rows are BQ = 128 / G query positions x G heads, row
// r = position G + head: a short block's rows are the first ones, next to one
// another.  Wave w owns the 16-row tiles w and w + 4 (items of 64 rows, kHalf:
// tile w).
// Workgroups are persistent: the grid fills the
// GPU's workgroup slots once and each workgroup works through a list of
// items.  Keys stream through LDS in 64-key tiles (K and V row-major,
// 16-byte chunks XOR-swizzled by row against bank conflicts) over a ring of
// two stages filled by global_load_lds DMA, so one tile is in flight while
// one is reduced; the ring runs on from one item into the next.  Per tile:
//   S^T = K Q^T  with v_mfma_f32_16x16x32 (A = K rows from LDS via
//                ds_read_b128, B = Q^T held in registers for the whole loop);
//   online softmax in the exp2 domain on the S^T accumulators: each lane
//                holds 4 consecutive keys of one query row, so the row max /
//                sum need only two cross-lane steps;
//   O^T += V^T P^T with the same MFMA: P^T is the S^T accumulator converted
//                to 16-bit in place (the MFMA's k index is permuted to match),
//                and V^T comes from row-major V through ds_read_b64_tr_b16.
// With a paged pool, keys j < k_len - q_len are gathered through the block
// table while the tile is loaded; the new keys come from k/v.  The fused
// store copies an item's new K/V rows from the staged tiles to slot_mapping.
//
// Splitting.  A launch with few items, or with some much longer than the rest
// (a prompt continuing a long cached prefix, decoding sequences with long
// contexts beside prompts), would wait for its longest items with most of
// the chip idle.  Given a workspace, a launch cuts such items' keys into
// pieces of about (all tiles) / (workgroup slots) tiles (kSplit); a piece
// writes its rows' unnormalised (m, l, o) in fp32 and varlen_merge_kernel
// combines them with the log-sum-exp rule.  The plan is made on the device,
// from the lengths: every workgroup of an XCD computes the same one.
#pragma once

#include <atomic>
#include <type_traits>

#include "common.h"
#include "fastdiv.h"
#include "prologue.h"

namespace va {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4_t lds_s16x4_t;

struct VarlenParams {
  const char* q;
  int64_t q_st, q_sh;  // bytes
  const char* k;
  int64_t k_st, k_sh;
  const char* v;
  int64_t v_st, v_sh;
  char* out;
  int64_t o_st, o_sh;
  const int32_t* cu_q;
  const int32_t* cu_k;
  float scale_log2;
  int32_t has_pool;
  char* kp;
  char* vp;
  int64_t s_blk, s_slot, s_head;  // bytes
  int32_t block_size, num_blocks;
  const void* table;
  int64_t t_sb;
  int32_t table_i64, table_width;
  const void* slots;
  int32_t slot_i64;
  int32_t num_qblocks;
  int32_t num_seqs, num_kv_heads;
  int32_t split_over, split_slots;  // kSplit, below; here, in a line read at the start
                                    // (in a later one the plan waited 1 us for it)
  FastDiv bs_div, hkv_div;  // block_size, num_kv_heads
  int32_t slot_small;       // num_blocks * block_size <= 2^31: slots divide in 32 bits
  int32_t block16;          // block_size % 16 == 0: 16 rows from a multiple of 16 share a block
  float k_scale, v_scale;   // FP8 pool: element = code * scale
  int32_t kv_f8;            // the pool holds e4m3 codes (strides in bytes of codes)
  // Split items (kSplit; all null / 0 without a workspace): split_over, the most
  // slots of an XCD a plan spreads over; per XCD split_slots pieces, their
  // (m, l) and o, what they belong to, how many.
  int32_t split;  // host: take the kSplit instantiation
  int32_t half;   // host: take the kHalf instantiation
  float* part_o;
  float2* part_ml;
  int4* part_head;
  int32_t* part_count;
  int32_t has_pro;          // the Qwen3 query prologue runs on every query row
  PrologueParams pro;
};

// The launch's arguments where they are needed once per item or on uncommon
// tiles.  Read through a pointer the compiler cannot see through, they are
// reloaded there (scalar loads) instead of staying in scalar registers
// through the tile loop, which has none to spare: what is kept beyond them
// is spilled to vector lanes and read back with v_readlane on every tile.
// VarlenParams is the kernel's only argument, so it starts the segment.
typedef const __attribute__((address_space(4))) VarlenParams* ColdArgs;
__device__ inline ColdArgs cold_args() {
  ColdArgs a = (ColdArgs)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(a));
  return a;
}
__device__ inline FastDiv cold_div(const __attribute__((address_space(4))) FastDiv& d) {
  FastDiv r;
  r.mul = d.mul;
  r.shift = d.shift;
  r.d = d.d;
  return r;
}

template <bool kBF16>
struct Mma {
  __device__ static inline f32x4_t mfma(uint4 a, uint4 b, f32x4_t c) {
    if constexpr (kBF16)
      return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                     __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    else
      return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a),
                                                    __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  }
  // Two floats to a packed 16-bit pair, round to nearest even (bf16 through
  // gfx950's v_cvt_pk_bf16_f32).
  __device__ static inline uint32_t pack2(float lo, float hi) {
    if constexpr (kBF16) {
      bf16x2_t v;
      v.x = (__bf16)lo;
      v.y = (__bf16)hi;
      return __builtin_bit_cast(uint32_t, v);
    } else
      return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)lo) |
             ((uint32_t)__builtin_bit_cast(uint16_t, (_Float16)hi) << 16);
  }
};

constexpr int kVarlenThreads = 256;
constexpr int kRowsPerWG = 128;
constexpr int kKeyTile = 64;
// Stages of the K/V ring: one tile streams in while one is reduced.
constexpr int kStages = 2;
// MI355X hands workgroup i of a launch to XCD i % 8; each XCD has its own L2.
constexpr int kXcds = 8;
// Lazy-rescale slack of the online softmax, in log2 units (p <= 2^kLazy).
constexpr float kLazy = 8.0f;

// Splitting: the most slots of an XCD a plan spreads over, its pieces of split
// items at most (the reason: plan_split in the kernel), and the fewest tiles a
// piece holds.
constexpr int kSplitOver = 64;
constexpr int split_pieces(int over) { return (8 * over + 4) / 5; }
constexpr int kSplitMinTiles = 2;
constexpr int kSplitMaxTiles = 1 << 18;  // longer contexts are not split (float division)

// floor(a / b) for 0 <= a < 2^21, b >= 1, through one float product: a + 1/2
// is at least 1 / (2 b) away from any multiple of b, above the rounding error.
__device__ inline int small_div(int a, float inv_b) {
  return (int)(((float)a + 0.5f) * inv_b);
}

// Inclusive sum over the lanes of a wave (DPP row shifts and broadcasts).
__device__ inline int wave_scan(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, true);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, true);  // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, true);  // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, true);  // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false);  // row_bcast:15, rows 1 and 3
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false);  // row_bcast:31, rows 2 and 3
  return x;
}

// 16 zero bytes: the DMA source of every lane whose key row is past the end
// of the visible keys or unmapped, so every tile takes the same number of
// DMA instructions (the pipeline's vmcnt waits count them).
__device__ __align__(16) const uint4 kZeroRow = {0u, 0u, 0u, 0u};
// Pool byte offset of a row that is not there.  Any other value is an offset:
// pool strides may be negative.
constexpr int64_t kNoRow = INT64_MIN;

// LDS layout of a staged K or V tile: kKeyTile rows of 2 D bytes, unpadded;
// the 16-byte chunk c of row r sits at chunk position c ^ swz(r).  The XOR
// spreads the 16 rows of one K read (ds_read_b128, one chunk per row) and
// the 8 rows x 2 chunks of half a V read (ds_read_b64_tr_b16) over distinct
// banks.  swz depends on r % 16 only.
template <int D>
__device__ inline int swz(int row) {
  if constexpr (D == 128)
    return ((row & 7) << 1) | ((row >> 3) & 1);
  else
    return (((row >> 1) & 3) << 1) | ((row >> 3) & 1);
}

__device__ inline uint4 lds_read16(const char* base, int off) {
  return *reinterpret_cast<const uint4*>(base + off);
}

__device__ inline s16x4_t lds_read_tr(const char* base, int off) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(base + off));
}

// Workgroups the registers leave room for per CU (one wave of each per SIMD).
// head_dim 64 was left to what the compiler happened to use: at 169-172 VGPRs
// the paged kernels of groups 4 and 8 fell from three workgroups to two (32
// prompts of 50-450 tokens, 32/8 heads: 38.2 us with two, 34.0 with three and
// a few registers spilled), and 64-row items at 129-134 from four to three (28
// decoding sequences with 4 prompts, 32/8 heads: 27.7 us, 19.5 with four).
constexpr int waves_per_simd(int d, bool half) { return d == 64 ? (half ? 4 : 3) : 2; }

// kPaged: keys j < k_len - q_len come from the pool through the block table
// (launches with a pool); otherwise every key comes from k/v.  kF8 (with
// kPaged): the pool holds OCP e4m3 codes.  A tile's pool rows are copied as
// codes into a code area of LDS and converted, at the top of the tile's
// step, into the 16-bit stage as code * scale rounded to the 16-bit type
// (every e4m3 value converts exactly; the product is rounded once), before
// the next tile's copy may reuse the code area.  Rows from k/v are staged
// as 16-bit rows, as without a pool.
//
// kPro: q holds raw projections; each item's query rows are normalised and
// rotated (Qwen3's q_norm + rotary_emb, prologue.h's arithmetic) in registers
// at the item's first tile, with positions loaded beside the rows.
//
// kSplit: the launch has a workspace and may split items (an instantiation of
// its own: the plan's state costs the others scalar registers, 1 us of 41 on
// a launch of 32 prompts).
//
// kHalf: 64 MFMA rows per item, one 16-row tile per wave.  A tile's body is
// bound by the wave's own chain (S^T, softmax, O^T; ~1.5 us with two row tiles,
// ~1.25 with one, alone on a CU), so a launch that leaves slots idle, or whose
// blocks are short anyway, ends sooner on items of half the rows (the host's
// rule: half_rows_wanted).
template <bool kBF16, int D, int G, bool kCausal, bool kPaged, bool kOnce, bool kF8, bool kPro,
          bool kSplit, bool kHalf>
__global__ __launch_bounds__(kVarlenThreads, waves_per_simd(D, kHalf)) void
varlen_attention_kernel(VarlenParams p) {
  constexpr int NR = kHalf ? 1 : 2;        // 16-row tiles per wave
  constexpr int BQ = 64 * NR / G;          // query positions per workgroup
  constexpr int DS = D / 32;               // k-steps of the S^T MFMA
  constexpr int DT = D / 16;               // 16-wide d tiles of O^T
  constexpr int ROWB = D * 2;              // bytes per K/V row
  constexpr int CPR = ROWB / 16;           // 16-byte chunks per row
  constexpr int RPI = 64 / CPR;            // rows per DMA instruction (1 KiB)
  constexpr int TILE_B = kKeyTile * ROWB;  // bytes of one K (or V) tile
  constexpr int NI = TILE_B / 1024 / 4;    // DMA instructions per wave per tile, K or V
  constexpr int KT = kKeyTile / 16;        // 16-key tiles per key tile
  constexpr int KS = kKeyTile / 32;        // 32-key MFMA steps per key tile
  static_assert(!kHalf || !kPro, "the query prologue takes two row tiles");
  static_assert(NI * 4 * 1024 == TILE_B, "tile DMA split");
  using M = Mma<kBF16>;

  // Two stages of (K tile, V tile): one streams in while the other is
  // reduced.
  static_assert(kStages == 2, "the tile loop alternates two stages");
  __shared__ __align__(1024) char s_kv[kStages * 2 * TILE_B];
  // FP8 pool: the codes of one tile's pool rows (K, then V), row-major and
  // unswizzled: row r's 16-code chunk c at r D + 16 c.
  static_assert(!kF8 || kPaged, "FP8 codes come from a pool");
  constexpr int CODE_B = kKeyTile * D;     // bytes of one tile of codes, K or V
  constexpr int CCPR = D / 16;             // 16-code chunks per code row
  constexpr int CRPI = 64 / CCPR;          // code rows per DMA instruction
  constexpr int NIC = CODE_B / 1024 / 4;   // code DMA instructions per wave per tile, K or V
  static_assert(!kF8 || NIC * 4 * 1024 == CODE_B, "code DMA split");
  __shared__ __align__(1024) char s_code[kF8 ? 2 * CODE_B : 16];
  // kPro: the query norm weights as fp32, written once per workgroup here and
  // read by every item's prologue (the first tile's barrier orders them).
  __shared__ __align__(16) float s_qw[kPro ? D : 4];
  using ET = std::conditional_t<kBF16, BF16, F16>;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: addresses stay scalar
  const int lane = tid & 63;
  const int r16 = lane & 15;
  const int g4 = lane >> 4;
  if constexpr (kPro) {
    for (int i = tid; i < D; i += kVarlenThreads) s_qw[i] = load_weight(p.pro.q_w, p.pro.w_dtype, i);
  }

  // ---- persistent schedule ----
  // Workgroup 8 j + x runs on XCD x (MI355X hands workgroup i of a launch to
  // XCD i % 8, and each XCD has its own L2) and takes items from XCD x's
  // list: the query blocks of pairs x, x + 8, ... (pair = sequence *
  // num_kv_heads + kv head), so the blocks that share a pair's K/V rows
  // share one L2.  The list is level-major: every pair's last block, then
  // every pair's second to last, ... (late blocks are the heavy ones under
  // causal masking).  It is dealt to the XCD's nslots workgroups in snake
  // order: in round r workgroup j takes item r nslots + j when r is even and
  // r nslots + nslots - 1 - j when r is odd, which evens out the sums of a
  // list sorted heavy first.  A workgroup keeps its K/V ring running from
  // one item into the next: the next item's first tile, query rows and store
  // slots are loading while the current item's last tile is reduced.
  const int nqb = p.num_qblocks;
  // kOnce: one query block per sequence (the host launches it for the
  // encoder's windows), so every K/V row is read by one item only and the
  // tiles stream in non-temporally (config 4: 16.2 -> 15.5 us).  Otherwise a
  // pair's later blocks re-read them from L2, which the default policy keeps
  // them in (non-temporal there: config 3's prefill 40.6 -> 45.3 us).
  constexpr bool kv_once = kOnce;
  const int npairs = p.num_seqs * p.num_kv_heads;
  const int xcd = (int)blockIdx.x % kXcds;
  const int wslot = (int)blockIdx.x / kXcds;
  const int nslots = (int)gridDim.x / kXcds;
  const int ppx = (npairs - xcd + kXcds - 1) / kXcds;  // pairs on this XCD
  // With at most 64 pairs per XCD (lane_pairs), lane k holds pair k's
  // query and key ranges and the list is walked with wave ballots, no memory
  // access per item.  Otherwise the list holds every (pair, block), blocks
  // past a sequence's end are skipped, and lane k holds the ranges of this
  // workgroup's item 64 i + k (refilled every 64 items).
  const bool lane_pairs = ppx <= 64;
  int lq0 = 0, lql = 0, lk0 = 0, lkl = 0, lnq = 0, lpair = 0;
  auto load_ranges = [&](int pair) {
    const int ls = (int)fast_div((uint32_t)pair, p.hkv_div);
    lq0 = p.cu_q[ls];
    lql = p.cu_q[ls + 1] - lq0;
    lk0 = p.cu_k[ls];
    lkl = p.cu_k[ls + 1] - lk0;
  };
  const int64_t total = (int64_t)ppx * nqb;  // list length without lane_pairs
  auto item_index = [&](int r) -> int64_t {  // list index of this workgroup's round r
    return (int64_t)r * nslots + ((r & 1) ? nslots - 1 - wslot : wslot);
  };
  auto refill = [&](int r0) {
    const int64_t li = item_index(r0 + lane);
    lnq = -1;
    if (li < total) {
      const int li32 = (int)li;  // list indices stay below 2^31 (host check)
      lpair = xcd + kXcds * (li32 % ppx);
      lnq = nqb - 1 - li32 / ppx;  // the item's query block
      load_ranges(lpair);
    }
  };
  if (lane_pairs) {
    if (lane < ppx) {
      load_ranges(xcd + kXcds * lane);
      lnq = (lql + BQ - 1) / BQ;
    }
  } else {
    refill(0);
  }

  struct Item {
    int s, h, qb;        // sequence, kv head, query block
    int q0, ql, k0, kl;  // the sequence's first query and key, its lengths
    int t0, t1;          // its key tiles, or the piece's
    int slot, npc;       // piece of a split item: its partial's slot (-1: whole), pieces if first
  };
  // What follows from an item: the keys that come from the pool, and the end
  // of the keys its rows see (bottom-right aligned when causal).
  const bool has_k = !kPaged || p.k != nullptr;
  auto prefix_of = [&](const Item& it) { return kPaged ? (has_k ? it.kl - it.ql : it.kl) : 0; };
  auto kend_of = [&](const Item& it) {
    return kCausal ? max(0, min(it.kl, it.kl - it.ql + min(it.ql, it.qb * BQ + BQ))) : it.kl;
  };
  // ---- splitting (kSplit) ----
  // The items' tiles on this XCD over its slots (fewer where there are many
  // items, each of which costs a slot its set-up and epilogue) give the tiles
  // of a piece; an item longer than that by a quarter is cut into equal
  // pieces of at most that many plus a quarter.  tile_sum is an upper bound
  // of the tiles (prefix tiles rounded up to quarters, one per item for the
  // rest), at most split_over pieces long, and an item of n >= 2 pieces is more
  // than n - 3/4 pieces long: at most 8/5 split_over pieces in all.
  // (Stores of the plan's words are uniform, by all lanes of a wave: a branch
  // on the lane in this walk would make every value after it divergent, the
  // DMAs' scalar bases among them.)
  int piece = 0;  // tiles of a piece; 0: nothing is split
  float piece_inv = 0.f;
  auto tiles_at = [&](int ql, int kl, int lv) {
    const int kend = kCausal ? max(0, min(kl, kl - ql + min(ql, lv * BQ + BQ))) : kl;
    return (kend + kKeyTile - 1) / kKeyTile;
  };
  auto plan_split = [&]() {
    const int nt = lnq > 0 ? (lkl + kKeyTile - 1) / kKeyTile : 0;
    const int prefix = max(lkl - lql, 0);
    int sum = 0;
    if (lnq > 0)
      sum = kCausal ? lnq * ((prefix + 15) / 16) / 4 + lnq * (lnq + 1) / 2 * BQ / kKeyTile + lnq + 1
                    : lnq * nt;
    if (__builtin_amdgcn_ballot_w64(nt >= kSplitMaxTiles || lnq > 1024 || sum >= (1 << 24)) != 0) return;
    const int tile_sum = __builtin_amdgcn_readlane(wave_scan(sum), 63);
    const int items = __builtin_amdgcn_readlane(wave_scan(lnq), 63);
    const int over = min(max(nslots - items / 4, (nslots + 1) / 2), p.split_over);
    const int pc = max(__builtin_amdgcn_readfirstlane((tile_sum + over - 1) / over), kSplitMinTiles);
    if (__builtin_amdgcn_ballot_w64(nt > pc + pc / 4) != 0) {
      piece = pc;
      piece_inv = 1.f / (float)pc;
    }
  };
  if constexpr (kSplit) {
    if (lane_pairs) plan_split();
    if (piece == 0 && wslot == 0 && wave == 0) p.part_count[xcd] = 0;
  }
  int round = 0;                         // this workgroup's next round
  int lev = nqb - 1, cum = 0;            // lane_pairs walk: level and items above it
  int slots = 0;                         // pieces of split items above it
  auto next_item = [&](Item& it) -> bool {
    int ksel, qb;
    it.slot = -1;
    it.npc = 1;
    int pj = 0, pn = 1;  // this piece of its item, pieces of the item
    if (kSplit && piece > 0) {
      const int li = (int)item_index(round);
      int pc = 0, inc = 0;
      while (lev >= 0) {
        // Pieces of every pair's item at this level, and their running sums:
        // all pieces in the low half, those of split items in the high half.
        pc = lnq > lev
                 ? max(1, small_div(tiles_at(lql, lkl, lev) + piece - 1 - piece / 4, piece_inv))
                 : 0;
        inc = wave_scan(pc + (pc > 1 ? pc << 16 : 0));
        const int all = __builtin_amdgcn_readlane(inc, 63);
        if (li < cum + (all & 0xffff)) break;
        cum += all & 0xffff;
        slots += (int)((uint32_t)all >> 16);
        --lev;
      }
      if (lev < 0) {
        if (wslot == 0 && wave == 0) p.part_count[xcd] = slots;
        return false;
      }
      ++round;
      const int rem = li - cum;
      const int end = inc & 0xffff;
      ksel = __builtin_ctzll(__builtin_amdgcn_ballot_w64(rem < end && rem >= end - pc));
      pn = __builtin_amdgcn_readlane(pc, ksel);
      pj = rem - (__builtin_amdgcn_readlane(end, ksel) - pn);
      if (pn > 1) {
        it.slot = slots + (int)((uint32_t)__builtin_amdgcn_readlane(inc, ksel) >> 16) - pn + pj;
        it.npc = pj == 0 ? pn : 0;
      }
      qb = lev;
    } else if (lane_pairs) {
      const int64_t li = item_index(round);
      // Levels are walked downwards once over the workgroup's life: the
      // list indices of its rounds increase.
      int cnt = 0;
      while (lev >= 0) {
        cnt = __popcll(__builtin_amdgcn_ballot_w64(lnq > lev));
        if (li < cum + cnt) break;
        cum += cnt;
        --lev;
      }
      if (lev < 0) return false;
      ++round;
      const int rem = (int)(li - cum);
      const uint64_t live = __builtin_amdgcn_ballot_w64(lnq > lev);
      const int below = __builtin_amdgcn_mbcnt_hi((uint32_t)(live >> 32),
                                                   __builtin_amdgcn_mbcnt_lo((uint32_t)live, 0));
      ksel = __builtin_ctzll(__builtin_amdgcn_ballot_w64(lnq > lev && below == rem));
      qb = lev;
    } else {
      for (;;) {
        if (item_index(round) >= total) return false;
        if (round > 0 && (round & 63) == 0) refill(round);
        ksel = round & 63;
        ++round;
        qb = __builtin_amdgcn_readlane(lnq, ksel);
        if (qb * BQ < __builtin_amdgcn_readlane(lql, ksel)) break;  // else past the end
      }
    }
    const int pair = lane_pairs ? xcd + kXcds * ksel : __builtin_amdgcn_readlane(lpair, ksel);
    it.s = (int)fast_div((uint32_t)pair, p.hkv_div);
    it.h = pair - it.s * p.num_kv_heads;
    it.qb = qb;
    it.q0 = __builtin_amdgcn_readlane(lq0, ksel);
    it.ql = __builtin_amdgcn_readlane(lql, ksel);
    it.k0 = __builtin_amdgcn_readlane(lk0, ksel);
    it.kl = __builtin_amdgcn_readlane(lkl, ksel);
    const int nt = tiles_at(it.ql, it.kl, qb);
    it.t0 = 0;
    it.t1 = nt;
    if (kSplit && pn > 1) {
      const int q = __builtin_amdgcn_readfirstlane(small_div(nt, 1.f / (float)pn));
      const int r = nt - q * pn;
      it.t0 = pj * q + min(pj, r);
      it.t1 = it.t0 + q + (pj < r ? 1 : 0);
    }
    return true;
  };

  const uint32_t lds_base = __builtin_amdgcn_readfirstlane(
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)s_kv);
  const uint32_t code_base = __builtin_amdgcn_readfirstlane(
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)s_code);

  // ---- DMA of a key tile [kb, kb + 64) into a stage ----
  // Wave w fills 1 KiB blocks w NI .. w NI + NI - 1 of the K and V tiles,
  // which hold the tile's rows 16 w .. 16 w + 15; lane l of block i writes
  // row RPI i + l / CPR of them, chunk position l % CPR, so it reads logical
  // chunk (l % CPR) ^ swz(row) of that key.
  static_assert(NI * RPI == 16, "a wave stages 16 rows of a tile");
  // The offsets are those of k/v rows, or (off_pool) of 16 pool rows of one
  // block: a launch changes over once or twice an item, so the tile loop holds
  // one set and has one form of request.
  uint32_t koff[NI], voff[NI];  // per-lane byte offsets inside the wave's 16 rows
  bool off_pool = false;
  auto set_offsets = [&](uint32_t k_st, uint32_t v_st) {
    int ln = lane;
    asm volatile("" : "+v"(ln));
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const uint32_t row = RPI * i + ln / CPR;
      const uint32_t chunk = (ln % CPR) ^ swz<D>(row);
      koff[i] = row * k_st + chunk * 16;
      voff[i] = row * v_st + chunk * 16;
    }
  };
  // k/v token strides (below 2^27 bytes: host check), opaque so that they stay
  // in scalar registers.  With the bases formed from the arguments per tile the
  // compiler reloaded those, and waited for them, on every tile of k/v rows;
  // the cursor's pointers advance by them instead.  head_dim 128, us: 32 prompts
  // 33.5 -> 31.9, 9 prompts 19.2 -> 17.3, 28 decoding sequences with 4 prompts
  // 32.2 -> 30.7; head_dim 64, 32/8 heads, 32 prompts 32.9 -> 32.3.
  uint32_t k_st = (uint32_t)p.k_st, v_st = (uint32_t)p.v_st;
  asm volatile("" : "+s"(k_st), "+s"(v_st));
  set_offsets(k_st, v_st);
  // FP8 pool: a wave's 16 code rows (unswizzled, CRPI rows an instruction).
  const uint32_t code_lane =
      kF8 ? (uint32_t)(lane / CCPR) * (uint32_t)p.s_slot + (uint32_t)(lane % CCPR) * 16u : 0u;
  const uint32_t code_dst = code_base + (uint32_t)(wave * NIC * 1024);

  // The cursor of the tiles being requested, one step ahead of the tiles
  // being reduced: it runs through the current item's tiles and on into the
  // next item's.  A whole tile of k/v rows, or (block16: a wave's 16 rows lie
  // in one block) of pool rows, is an easy one: instruction i copies RPI rows
  // from a uniform base plus lane offsets, with no load or per-lane address
  // of its own, so it can be issued between the MFMAs.  Every other tile
  // takes issue_hard.
  struct Cursor {
    int t, end;           // next tile to request, the item's last + 1
    int prefix, kend;
    int h, s;
    const char* kb;       // tile t's first row of this wave in k and v (a key's
    const char* vb;       // row is q0 + key - prefix, or k0 + key without a pool)
    int row0;             // `rows` holds the pool rows of tiles [row0, row0 + 64)
  };
  Cursor cu;
  auto advance = [&]() {
    ++cu.t;
    cu.kb += (uint64_t)k_st * kKeyTile;
    cu.vb += (uint64_t)v_st * kKeyTile;
  };
  int64_t rows = kNoRow;
  uint2 pend = make_uint2(0u, 0u);  // raw block ids that `rows` takes next
  auto cursor_to = [&](const Item& it) {
    cu.t = it.t0;
    cu.prefix = prefix_of(it);
    cu.kend = kend_of(it);
    cu.end = it.t1;
    cu.h = it.h;
    cu.s = it.s;
    const int64_t row = (kPaged ? (int64_t)it.q0 - cu.prefix : (int64_t)it.k0) +
                        (int64_t)it.t0 * kKeyTile + 16 * wave;
    const ColdArgs ca = cold_args();
    cu.kb = uniform_ptr(ca->k + row * ca->k_st + it.h * ca->k_sh);
    cu.vb = uniform_ptr(ca->v + row * ca->v_st + it.h * ca->v_sh);
    cu.row0 = it.t0;
  };
  // ---- pool rows (block16) ----
  // Lane l of `rows` holds the pool byte offset of the wave's 16 rows of tile
  // row0 + l (kNoRow: a block id outside the pool).  Block ids are requested 64
  // tiles at a time and a tile ahead of their use, so no tile waits for them
  // (looked up as the tile was requested, each pool tile cost a second
  // dependent round trip: 4 prompts of 200-300 tokens over prefixes of 2K-8K
  // took 357 us, 2.8 us a tile, and 260 with the ids ahead); they stay raw
  // words until a later step's tile wait has passed.  Columns past the table
  // read block 0.
  auto load_ids = [&](int s, int t0, int prefix) {
    const ColdArgs ca = cold_args();
    const int tok = (t0 + lane) * kKeyTile + 16 * wave;
    const int col = (int)fast_div((uint32_t)tok, cold_div(ca->bs_div));
    if (tok < prefix && col < ca->table_width) {
      const uint32_t* const w = reinterpret_cast<const uint32_t*>(ca->table);
      const int i64 = ca->table_i64;
      const int64_t e = ((int64_t)s * ca->t_sb + col) << i64;
      pend.x = w[e];
      pend.y = w[e + i64];
    } else {
      pend = make_uint2(0u, 0u);
    }
  };
  auto take_ids = [&](int t0) {  // the requested ids are those of the cursor's tiles from t0 on
    cu.row0 = t0;
    if (cu.prefix <= t0 * kKeyTile) return;  // no pool rows there
    const ColdArgs ca = cold_args();
    const int64_t bid = ca->table_i64 ? (int64_t)(((uint64_t)pend.y << 32) | pend.x)
                                      : (int64_t)(int32_t)pend.x;
    const uint32_t tok = (uint32_t)((t0 + lane) * kKeyTile + 16 * wave);
    rows = kNoRow;
    if (bid >= 0 && bid < ca->num_blocks)
      rows = bid * ca->s_blk + (int64_t)fast_mod(tok, cold_div(ca->bs_div)) * ca->s_slot +
             cu.h * ca->s_head;
  };
  // What `rows` will need next: the item's following 64 tiles, or the next
  // item's first.
  auto request_ids = [&](bool has_next, const Item& nxt) {
    const bool more = cu.end - cu.row0 > 64;
    const int t0 = more ? cu.row0 + 64 : nxt.t0;
    const int prefix = more ? cu.prefix : (has_next ? prefix_of(nxt) : 0);
    if (prefix > t0 * kKeyTile) load_ids(more ? cu.s : nxt.s, t0, prefix);
  };

  // How the cursor's tile is requested.
  enum { kNone, kRows, kCodes };
  struct Easy {
    int kind;
    const char* kb;  // the wave's first row
    const char* vb;
  };
  const char* zero_row = reinterpret_cast<const char*>(&kZeroRow);
  auto issue_hard = [&](int64_t row, int st) {
    const ColdArgs ca = cold_args();
    const uint32_t dst0 = lds_base + (uint32_t)(st * 2 * TILE_B + wave * NI * 1024);
    const int kb = cu.t * kKeyTile;
    const FastDiv bs_div = cold_div(ca->bs_div);
    // Per-lane addresses; rows past kend or with an unmapped block read
    // kZeroRow.  The lane's first row is made opaque so that the address
    // arithmetic stays here instead of being hoisted out of the tile loop
    // into live registers.  Block ids (other block sizes; with block16 the
    // wave's 16 rows start at pool offset `row`) are loaded as raw words and widened after the last
    // load, and every address is formed before the first DMA: a register
    // still awaiting its load when a DMA has been issued would make the
    // compiler's wait for it also wait for that DMA.
    int row0 = 16 * wave + lane / CPR;
    asm volatile("" : "+v"(row0));
    // Address of the 16 bytes at byte column `c16` of token j's pool row.
    auto pool_at = [&](int j, const uint2& raw, int c16, const char*& ka, const char*& va_) {
      int64_t off = row;
      if (ca->block16) {
        if (off != kNoRow) off += (j & 15) * ca->s_slot + c16;
      } else {
        const int64_t bid = ca->table_i64 ? (int64_t)(((uint64_t)raw.y << 32) | raw.x)
                                          : (int64_t)(int32_t)raw.x;
        off = kNoRow;
        if (bid >= 0 && bid < ca->num_blocks)
          off = bid * ca->s_blk + (int64_t)fast_mod((uint32_t)j, bs_div) * ca->s_slot +
                cu.h * ca->s_head + c16;
      }
      if (off != kNoRow) {
        ka = ca->kp + off;
        va_ = ca->vp + off;
      }
    };
    auto raw_id = [&](int j, uint2& raw) {
      raw = make_uint2(0u, 0u);
      if (!ca->block16) {
        const int col = (int)fast_div((uint32_t)j, bs_div);
        if (j < cu.prefix && j < cu.kend && col < ca->table_width) {
          const int i64 = ca->table_i64;
          const int64_t e = ((int64_t)cu.s * ca->t_sb + col) << i64;
          const uint32_t* const w = reinterpret_cast<const uint32_t*>(ca->table);
          raw.x = w[e];
          raw.y = w[e + i64];
        }
      }
    };
    const char* kc[kF8 ? NIC : 1];
    const char* vc[kF8 ? NIC : 1];
    if constexpr (kF8) {
      // The tile's pool rows as codes: lane l of code instruction i copies
      // chunk l % CCPR of code row (wave NIC + i) CRPI + l / CCPR.
      int crow0 = 16 * wave + lane / CCPR;
      asm volatile("" : "+v"(crow0));
      uint2 craw[NIC];
#pragma unroll
      for (int i = 0; i < NIC; ++i) raw_id(kb + crow0 + i * CRPI, craw[i]);
#pragma unroll
      for (int i = 0; i < NIC; ++i) {
        const int j = kb + crow0 + i * CRPI;
        kc[i] = zero_row;
        vc[i] = zero_row;
        if (j < cu.prefix && j < cu.kend) pool_at(j, craw[i], (lane % CCPR) * 16, kc[i], vc[i]);
      }
    }
    uint2 braw[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      braw[i] = make_uint2(0u, 0u);
      if (kPaged && !kF8) raw_id(kb + row0 + i * RPI, braw[i]);
    }
    const char* ka[NI];
    const char* va_[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int row = row0 + i * RPI;
      const int chunk = (lane % CPR) ^ swz<D>(row);
      const int j = kb + row;
      ka[i] = zero_row;
      va_[i] = zero_row;
      if (j < cu.kend) {
        if (kPaged && j < cu.prefix) {
          // An FP8 pool row is staged by the code copy and its conversion.
          if constexpr (!kF8) pool_at(j, braw[i], chunk * 16, ka[i], va_[i]);
        } else {
          const uint32_t r = row - 16 * wave;
          ka[i] = cu.kb + (r * k_st + chunk * 16);
          va_[i] = cu.vb + (r * v_st + chunk * 16);
        }
      }
    }
    // A lane that uses no block id leaves its load pending, and the compiler
    // waits for it where the register is next written.  At head_dim 64 that was
    // behind the DMA, on every tile: a partial tile, an item's last one, was
    // waited for as soon as it was requested.  us, 32/8 heads: four prompts of
    // 300 14.6 -> 13.9, 9 of 60-594 22.5 -> 21.4, 28 decoding sequences with 4
    // prompts 20.6 -> 19.9; 64/8 heads, 32 of 50-450 69.7 -> 67.1.  (head_dim
    // 128 has other registers there and no such wait.)
    if constexpr (kPaged && !kF8 && D == 64) {
#pragma unroll
      for (int i = 0; i < NI; ++i) asm volatile("" ::"v"(braw[i].x), "v"(braw[i].y));
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      if constexpr (kv_once) {
        dma16_nt(ka[i], dst0 + i * 1024);
        dma16_nt(va_[i], dst0 + TILE_B + i * 1024);
      } else {
        dma16(ka[i], dst0 + i * 1024);
        dma16(va_[i], dst0 + TILE_B + i * 1024);
      }
    }
    if constexpr (kF8) {
      if (kb < cu.prefix) {
#pragma unroll
        for (int i = 0; i < NIC; ++i) {
          dma16(kc[i], code_dst + i * 1024);
          dma16(vc[i], code_dst + CODE_B + i * 1024);
        }
      }
    }
  };
  // Requests the cursor's tile into stage st, or, when it is an easy one,
  // says how (easy_issue then does, one instruction pair at a time).
  auto issue = [&](int st) -> Easy {
    Easy e;
    e.kind = kNone;
    e.kb = e.vb = nullptr;
    const int kb = cu.t * kKeyTile;
    if (kb >= cu.prefix && kb + kKeyTile <= cu.kend) {
      e.kind = kRows;
      if (kPaged && !kF8 && off_pool) {
        set_offsets(k_st, v_st);
        off_pool = false;
      }
      e.kb = cu.kb;
      e.vb = cu.vb;
      return e;
    }
    int64_t row = kNoRow;
    if (kPaged && kb < cu.prefix) {
      const int l = cu.t - cu.row0;
      row = (int64_t)(((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(rows >> 32), l) << 32) |
                      (uint32_t)__builtin_amdgcn_readlane((int)rows, l));
      if (kb + kKeyTile <= min(cu.prefix, cu.kend) && row != kNoRow && p.block16) {
        e.kind = kF8 ? kCodes : kRows;
        if (!kF8 && !off_pool) {
          const uint32_t slot = (uint32_t)cold_args()->s_slot;
          set_offsets(slot, slot);
          off_pool = true;
        }
        e.kb = uniform_ptr(p.kp + row);
        e.vb = uniform_ptr(p.vp + row);
        return e;
      }
    }
    issue_hard(row, st);
    return e;
  };
  auto easy_issue = [&](const Easy& e, int i, uint32_t dst) {  // 16-bit rows
    if constexpr (kv_once) {
      dma16_nt(koff[i], e.kb, dst + i * 1024);
      dma16_nt(voff[i], e.vb, dst + TILE_B + i * 1024);
    } else {
      dma16(koff[i], e.kb, dst + i * 1024);
      dma16(voff[i], e.vb, dst + TILE_B + i * 1024);
    }
  };
  auto easy_codes = [&](const Easy& e, int i) {
    const int64_t step = (int64_t)(i * CRPI) * p.s_slot;
    dma16(code_lane, e.kb + step, code_dst + i * 1024);
    dma16(code_lane, e.vb + step, code_dst + CODE_B + i * 1024);
  };
  auto issue_now = [&](const Easy& e, int st) {  // all of an easy tile at once
    const uint32_t dst = lds_base + (uint32_t)(st * 2 * TILE_B + wave * NI * 1024);
    if (e.kind == kRows) {
#pragma unroll
      for (int i = 0; i < NI; ++i) easy_issue(e, i, dst);
    }
    if constexpr (kF8) {
      if (e.kind == kCodes) {
#pragma unroll
        for (int i = 0; i < NIC; ++i) easy_codes(e, i);
      }
    }
  };

  // ---- query rows and store slots of an item ----
  // Two 16-row tiles per wave: row 16 (wave + 4 tt) + r16 of the block is
  // query position pos0 + row / G of head h G + row % G.
  uint4 qreg[NR][DS];
  // kPro: the rotary position of each of the lane's two query rows (the row
  // of the item's last query for rows past the end, whose output is unused).
  int64_t qrot[2] = {0, 0};
  auto load_q = [&](const Item& it) {
#pragma unroll
    for (int tt = 0; tt < NR; ++tt) {
      const int row = 16 * (wave + 4 * tt) + r16;
      const int qpos = it.qb * BQ + row / G;
      const int qhead = it.h * G + row % G;
      if constexpr (kPro)
        qrot[tt] = load_index(p.pro.pos, (int64_t)it.q0 + (qpos < it.ql ? qpos : it.ql - 1),
                              p.pro.pos_i64);
      const char* const src = p.q + (int64_t)(it.q0 + qpos) * p.q_st +
                              (int64_t)qhead * p.q_sh + g4 * 16;
#pragma unroll
      for (int ds = 0; ds < DS; ++ds) qreg[tt][ds] = make_uint4(0, 0, 0, 0);
      if (qpos < it.ql) {
#pragma unroll
        for (int ds = 0; ds < DS; ++ds) qreg[tt][ds] = ld16(src + 64 * ds);
      }
    }
  };
  // Fused store: the item's new rows are keys [pool_prefix + pos0,
  // pool_prefix + pos_end), which the tile loop stages in LDS anyway: each is
  // copied from there to its slot, so k/v are read once.  The block's rows
  // are BQ x CPR 16-byte chunks, e = row CPR + chunk; store step k of wave w
  // takes e = 256 k + 64 w + lane, so each step writes RPS = 64 / CPR whole
  // rows of K and the same rows of V.  Lane j < NSTEP RPS of a wave loads
  // the slot of the wave's row j (step j / RPS, row j % RPS of the step), and
  // a store step reads the slots it needs from those lanes.  The slot is
  // loaded with the item's query rows, as the raw 32-bit word(s) of the
  // mapping (all ones for no row), and widened only where it is used, once
  // the tile holding the row has landed: widening at the load would wait for
  // it there, behind the tile DMA just issued.
  constexpr int RPS = 64 / CPR;  // rows per store step
  constexpr int NSTEP = (BQ * CPR + kVarlenThreads - 1) / kVarlenThreads;
  static_assert(NSTEP * RPS <= 64, "one slot lane per row");
  const bool fused_store = kPaged && !kF8 && p.slots != nullptr;  // FP8: a launch of its own
  auto st_base = [&](int k) {  // first block row of store step k (BQ: none)
    const int e0 = k * kVarlenThreads + 64 * wave;
    return e0 < BQ * CPR ? e0 / CPR : BQ;
  };
  const int st_row = lane < NSTEP * RPS ? min(st_base(lane / RPS) + lane % RPS, BQ) : BQ;
  auto load_slot = [&](const Item& it) -> uint2 {
    uint2 raw = make_uint2(~0u, ~0u);
    if (fused_store && it.qb * BQ + st_row < min(it.ql, it.qb * BQ + BQ)) {
      const int64_t i = (int64_t)it.q0 + it.qb * BQ + st_row;
      if (p.slot_i64)
        raw = reinterpret_cast<const uint2*>(p.slots)[i];
      else
        raw.x = reinterpret_cast<const uint32_t*>(p.slots)[i];
    }
    return raw;
  };

  // Swizzled chunk positions of this lane's reads (row % 16 is fixed per lane).
  const int kswz = swz<D>(r16);
  const int vswz = swz<D>(4 * g4 + (r16 >> 2));

  Item cur, nxt = {};
  if (!next_item(cur)) return;
  cursor_to(cur);
  if (kPaged && cu.prefix > 0) {
    load_ids(cur.s, cur.t0, cu.prefix);
    take_ids(cur.t0);
  }
  if (cu.t < cu.end) {
    issue_now(issue(0), 0);
    advance();
  }
  load_q(cur);
  uint2 st_slot = load_slot(cur);
  int stage = 0;  // stage holding the current item's next tile to reduce

  for (;;) {
    const bool has_next = next_item(nxt);
    if constexpr (kPaged) request_ids(has_next, nxt);

    const int pos0 = cur.qb * BQ;
    const int nrows = (min(cur.ql, pos0 + BQ) - pos0) * G;  // MFMA rows of the block in use
    const int prefix = prefix_of(cur);
    const int kend = kend_of(cur);
    const int tend = cur.t1;
    int lim[NR];
#pragma unroll
    for (int tt = 0; tt < NR; ++tt) {
      // Visible keys per row: j < lim[tt].  Rows past the end of the
      // sequence have zero queries; their outputs are never written.
      const int qpos = pos0 + (16 * (wave + 4 * tt) + r16) / G;
      lim[tt] = kCausal ? min(kend, cur.kl - cur.ql + qpos + 1) : kend;
    }
    // Tiles ending at or below lim_lo (the smallest limit of the wave's rows)
    // need no mask.
    const int lim_lo = kCausal ? min(kend, cur.kl - cur.ql + pos0 + 16 * wave / G + 1) : kend;
    const int st_key0 = prefix + pos0;  // key of the block's first row

    float m[NR], l[NR];
    f32x4_t o[NR][DT];
#pragma unroll
    for (int tt = 0; tt < NR; ++tt) {
      m[tt] = -1.0e30f;
      l[tt] = 0.f;
    }
    // With the query prologue the accumulators are zeroed after it, at the
    // item's first tile, so they hold no registers while it runs.
    if constexpr (!kPro) {
#pragma unroll
      for (int tt = 0; tt < NR; ++tt)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) o[tt][dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }

    for (int t = cur.t0; t < tend; ++t) {
      const int kb = t * kKeyTile;
      // Tile t (and, in order, everything issued before it) has landed once
      // nothing is pending; the barrier makes every wave's part of it
      // visible and tells that every wave is done with the other stage,
      // which then takes the next tile: this item's tile t + 1, or the next
      // item's first tile.
      wait_vmcnt<0>();
      __syncthreads();
      // The query rows, the slot and block ids were loaded before the wait:
      // make the compiler's own wait for them fall here, before the next
      // DMA, where it is free (a later wait would also stall on that DMA).
#pragma unroll
      for (int tt = 0; tt < NR; ++tt)
#pragma unroll
        for (int ds = 0; ds < DS; ++ds)
          asm volatile("" ::"v"(qreg[tt][ds].x), "v"(qreg[tt][ds].y), "v"(qreg[tt][ds].z),
                       "v"(qreg[tt][ds].w));
      asm volatile("" ::"v"(st_slot.x), "v"(st_slot.y));
      if constexpr (kPaged) asm volatile("" ::"v"(pend.x), "v"(pend.y));
      // Qwen3 query prologue on the item's rows, in the B-operand layout:
      // lane (r16, g4) holds elements 32 ds + 8 g4 + e of its row (ds < DS,
      // e < 8), so element i < D/2 and its rotary partner i + D/2 sit in the
      // same lane (ds and ds + DS/2), and a row's sum of squares is the sum
      // over the four lanes r16 + 16 g4.  It runs before the next tile is
      // requested: the compiler's wait for the cos / sin loads would
      // otherwise also wait for that request.  Both rows' cos / sin are
      // requested together (one round trip per item), into the registers
      // the output accumulators take after this block; the weights come
      // from LDS.
      if constexpr (kPro) {
        if (t == cur.t0) {
          static_assert(DS % 2 == 0, "rotary halves");
          constexpr int HD = DS / 2;
          f32x4_t cv[2][HD][2], sv[2][HD][2];
#pragma unroll
          for (int tt = 0; tt < 2; ++tt) {
            int64_t P = qrot[tt];
            P = P < 0 ? 0 : (P >= p.pro.max_pos ? p.pro.max_pos - 1 : P);
            const float* crow = p.pro.cs + P * p.pro.cs_stride;
#pragma unroll
            for (int hh = 0; hh < HD; ++hh)
#pragma unroll
              for (int e4 = 0; e4 < 2; ++e4) {
                cv[tt][hh][e4] = *reinterpret_cast<const f32x4_t*>(crow + 32 * hh + 8 * g4 + 4 * e4);
                sv[tt][hh][e4] =
                    *reinterpret_cast<const f32x4_t*>(crow + D / 2 + 32 * hh + 8 * g4 + 4 * e4);
              }
          }
          // One row at a time, each called with a constant row index so that
          // qreg and the factors stay in registers.
          auto pro_row = [&](auto TT) {
            constexpr int tt = decltype(TT)::value;
            float x[DS][8];
#pragma unroll
            for (int ds = 0; ds < DS; ++ds) ET::unpack(qreg[tt][ds], x[ds]);
            // The sum of squares in va_qk_norm_rope's order, so that the
            // queries come out bit for bit as that kernel's do: there a lane
            // holds one 8-element chunk c of the row (a fused multiply-add
            // chain) and the 16 chunk sums meet in the tree
            // ((c0 + c1) + (c2 + c3)) + ((c4 + c5) + (c6 + c7)) + ...  Here
            // chunk c = 4 ds + g4 sits in lane g4 at ds: pairs (g4, g4 ^ 1)
            // are lanes l, l ^ 16, quads lanes l ^ 32, and the rest is in
            // the lane.
            static_assert(DS == 4, "the standalone kernel's tree for head_dim 128");
            float cs4[DS];
#pragma unroll
            for (int ds = 0; ds < DS; ++ds) {
              cs4[ds] = 0.f;
#pragma unroll
              for (int e = 0; e < 8; ++e) cs4[ds] = fmaf(x[ds][e], x[ds][e], cs4[ds]);
              cs4[ds] = sum_xor16(cs4[ds]);
              cs4[ds] = sum_xor32(cs4[ds]);
            }
            const float ss = (cs4[0] + cs4[1]) + (cs4[2] + cs4[3]);
            const float r = 1.0f / sqrtf(__fadd_rn(ss / (float)D, p.pro.eps));
#pragma unroll
            for (int ds = 0; ds < DS; ++ds) {
#pragma unroll
              for (int e = 0; e < 8; ++e) x[ds][e] = __fmul_rn(x[ds][e], r);
              round_to<ET>(x[ds]);
              const f32x4_t w0 = *reinterpret_cast<const f32x4_t*>(s_qw + 32 * ds + 8 * g4);
              const f32x4_t w1 = *reinterpret_cast<const f32x4_t*>(s_qw + 32 * ds + 8 * g4 + 4);
#pragma unroll
              for (int e = 0; e < 8; ++e) x[ds][e] = __fmul_rn(x[ds][e], e < 4 ? w0[e] : w1[e - 4]);
              round_to<ET>(x[ds]);
            }
            {
              // Products rounded apart before their sum (no fused multiply-add).
#pragma clang fp contract(off)
#pragma unroll
              for (int hh = 0; hh < HD; ++hh)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                  const float c = e < 4 ? cv[tt][hh][0][e] : cv[tt][hh][1][e - 4];
                  const float sn = e < 4 ? sv[tt][hh][0][e] : sv[tt][hh][1][e - 4];
                  const float a = x[hh][e], b2 = x[hh + HD][e];
                  x[hh][e] = a * c - b2 * sn;
                  x[hh + HD][e] = b2 * c + a * sn;
                }
            }
#pragma unroll
            for (int ds = 0; ds < DS; ++ds) {
#pragma unroll
              for (int e = 0; e < 8; ++e) pin(x[ds][e]);  // pack the fp32 sums
              qreg[tt][ds] = ET::pack(x[ds]);
            }
          };
          pro_row(std::integral_constant<int, 0>{});
          pro_row(std::integral_constant<int, 1>{});
#pragma unroll
          for (int tt = 0; tt < 2; ++tt)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) o[tt][dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
      }
      // FP8 pool: convert this tile's pool rows from the code area into the
      // stage (16-byte chunks at their swizzled positions), then free the
      // code area for the next tile's copy below.
      if constexpr (kF8) {
        if (kb < prefix) {
          char* const s_kt = s_kv + stage * 2 * TILE_B;
          for (int e = tid; e < 2 * kKeyTile * CCPR; e += kVarlenThreads) {
            const int is_v = e >= kKeyTile * CCPR ? 1 : 0;
            const int rc = e - is_v * kKeyTile * CCPR;
            const int r = rc / CCPR, c = rc % CCPR;
            if (kb + r < prefix) {
              const uint4 codes = lds_read16(s_code + is_v * CODE_B, r * D + c * 16);
              const float sc = is_v ? p.v_scale : p.k_scale;
              char* const dst = s_kt + is_v * TILE_B + r * ROWB;
              float f[8];
              ET::unpack(f8_dequant8<ET>(make_uint2(codes.x, codes.y)), f);
#pragma unroll
              for (int i = 0; i < 8; ++i) f[i] *= sc;
              *reinterpret_cast<uint4*>(dst + (((2 * c) ^ swz<D>(r)) << 4)) = ET::pack(f);
              ET::unpack(f8_dequant8<ET>(make_uint2(codes.z, codes.w)), f);
#pragma unroll
              for (int i = 0; i < 8; ++i) f[i] *= sc;
              *reinterpret_cast<uint4*>(dst + (((2 * c + 1) ^ swz<D>(r)) << 4)) = ET::pack(f);
            }
          }
          wait_lgkmcnt0();
          __syncthreads();
        }
      }
      // The next tile (this item's tile t + 1, or the next item's first)
      // goes to the other stage.  An easy tile is issued in pairs of DMAs
      // spread over the S^T loop below: issued back to back, they stall the
      // wave on the vector memory queue for as long as the MFMAs of half a
      // tile take.  Other tiles are issued here.
      const bool ends = cu.t == cu.end;
      if (ends && has_next) cursor_to(nxt);
      if constexpr (kPaged) {
        const bool window = !ends && cu.t - cu.row0 == 64;
        if (window || (ends && has_next)) take_ids(cu.t);
        if (window) request_ids(has_next, nxt);
      }
      const bool req = cu.t < cu.end;
      Easy e;
      e.kind = kNone;
      e.kb = e.vb = nullptr;
      if (req) {
        e = issue(stage ^ 1);
        advance();
      }
      const uint32_t n_dst = lds_base + (uint32_t)((stage ^ 1) * 2 * TILE_B + wave * NI * 1024);
      const char* s_k = s_kv + stage * 2 * TILE_B;
      const char* s_v = s_k + TILE_B;

      // Store steps run only on tiles that hold some of the block's new rows.
      // The rows go out non-temporally: nothing in the launch reads them back
      // (config 3: 40.4 -> 39.6 us per launch).
      if (fused_store && st_key0 < kb + kKeyTile && st_key0 + nrows / G > kb) {
        // Pool offset of this lane's row (kNoRow: not stored), computed in the
        // lane that holds the slot and handed to the lanes that store it.
        const int64_t cap = (int64_t)p.num_blocks * p.block_size;
        const int64_t slot = p.slot_i64 ? (int64_t)(((uint64_t)st_slot.y << 32) | st_slot.x)
                                          : (int64_t)(int32_t)st_slot.x;
        int64_t at = kNoRow;
        if (slot >= 0 && slot < cap) {
          const int64_t blk = p.slot_small
                                  ? (int64_t)fast_div((uint32_t)slot, p.bs_div)
                                  : slot / p.block_size;
          at = blk * p.s_blk + (slot - blk * p.block_size) * p.s_slot + cur.h * p.s_head;
        }
        const int c = lane % CPR;
#pragma unroll 4
        for (int k = 0; k < NSTEP; ++k) {
          const int holder = k * RPS + lane / CPR;
          const uint32_t lo = (uint32_t)__shfl((int)(uint32_t)at, holder, 64);
          const int hi = __shfl((int)(at >> 32), holder, 64);
          const int row = st_base(k) + lane / CPR;
          const int key = st_key0 + row;
          if (row < BQ && hi != (int)(kNoRow >> 32) && key >= kb && key < kb + kKeyTile) {
            const int64_t dst = (int64_t)(((uint64_t)(uint32_t)hi << 32) | lo) + c * 16;
            const int r = key - kb;
            const int off = r * ROWB + ((c ^ swz<D>(r)) << 4);
            st16_nt(p.kp + dst, lds_read16(s_k, off));
            st16_nt(p.vp + dst, lds_read16(s_v, off));
          }
        }
      }

      // On the item's last tile, once its S^T is done, the query rows are
      // dead: the next item's loads start.  Its store slot goes straight into
      // st_slot (this item's store steps ran above): a copy at the item's
      // end would have to wait for the load, and with it for every store
      // issued after it.
      auto load_next = [&]() {
        if (t + 1 == tend && has_next) {
          load_q(nxt);
          st_slot = load_slot(nxt);
        }
      };

      // The tile, as a lambda: written in place, the kernels spill up to 17 more
      // registers.
      auto reduce = [&]() {
        // ---- S^T = K Q^T ----
        // K rows of 16-key group kt + 1 are read before group kt's DMA pair:
        // no LDS read moves across a DMA.
        static_assert(KT % NI == 0 || NI % KT == 0, "DMA pairs spread evenly over the key groups");
        constexpr int PAIRS = NI >= KT ? NI / KT : 1;  // DMA pairs after each chosen group
        constexpr int EVERY = NI >= KT ? 1 : KT / NI;  // every EVERY-th group gets them
        // At head_dim 128 the lane's K offsets are rebuilt per tile from opaque
        // bases: held through the loop they make the compiler spill.
        int k0 = (g4 ^ kswz) << 4, krow = r16 * ROWB;
        if constexpr (D > 64) asm volatile("" : "+v"(k0), "+v"(krow));
        f32x4_t sacc[NR][KT];
        uint4 ka[2][DS];
#pragma unroll
        for (int ds = 0; ds < DS; ++ds) ka[0][ds] = lds_read16(s_k, krow + (k0 ^ (ds << 6)));
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) {
          if (kt + 1 < KT) {
#pragma unroll
            for (int ds = 0; ds < DS; ++ds)
              ka[(kt + 1) & 1][ds] = lds_read16(s_k, 16 * (kt + 1) * ROWB + krow + (k0 ^ (ds << 6)));
          }
#pragma unroll
          for (int tt = 0; tt < NR; ++tt) sacc[tt][kt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int ds = 0; ds < DS; ++ds)
#pragma unroll
            for (int tt = 0; tt < NR; ++tt)
              sacc[tt][kt] = M::mfma(ka[kt & 1][ds], qreg[tt][ds], sacc[tt][kt]);
          if (kt % EVERY == 0 && e.kind == kRows) {
#pragma unroll
            for (int j = 0; j < PAIRS; ++j) easy_issue(e, (kt / EVERY) * PAIRS + j, n_dst);
          }
          if constexpr (kF8) {
            if (kt < NIC && e.kind == kCodes) easy_codes(e, kt);
          }
        }
        load_next();

        // V^T goes through a window of VW operands, the first requested before
        // the softmax and each later one as an earlier one is used.  Over a pool
        // at head_dim 64 the registers of three workgroups a CU leave room for
        // one operand there, whose reads the compiler then waited for one by
        // one; requested after the softmax, when the scores are dead, there is
        // room for two.  us, 32/8 heads: one prompt of 2500 63.3 -> 59.9, 9 of
        // 60-594 21.3 -> 20.4; 28/14: four of 800 28.1 -> 26.4; 64/8: 32 over
        // prefixes of 700 185.6 -> 180.7.
        const int v0 = (((r16 >> 1) & 1) ^ vswz) << 4;
        const int vrow = (4 * g4 + (r16 >> 2)) * ROWB + ((r16 & 1) << 3);
        auto read_v = [&](int ks, int dt) -> uint4 {
          const int off = 32 * ks * ROWB + vrow + (v0 ^ (dt << 5));
          const uint2 lo = __builtin_bit_cast(uint2, lds_read_tr(s_v, off));
          const uint2 hi = __builtin_bit_cast(uint2, lds_read_tr(s_v, off + 16 * ROWB));
          return make_uint4(lo.x, lo.y, hi.x, hi.y);
        };
        constexpr bool late_v = D == 64 && kPaged;
        constexpr int VW = late_v ? DT / 2 : DT / 4;
        uint4 vf[VW];
        if constexpr (!late_v) {
#pragma unroll
          for (int dt = 0; dt < VW; ++dt) vf[dt] = read_v(0, dt);
        }

        // ---- online softmax (exp2 domain) and P^T packing ----
        // Scores stay unscaled until the exponent: p = 2^(s c - m) with
        // c = scale log2 e > 0 and m the row's running max of s c.  The max
        // used as reference is raised only when a row's new max exceeds it by
        // more than kLazy (or on the first scores); in between, p <= 2^kLazy,
        // which the fp32 sums and 16-bit P hold exactly as well.  Key masking
        // is applied only on tiles that cross a row's limit.
        const bool need_mask = kb + kKeyTile > lim_lo;
        uint4 pb[NR][KS];
#pragma unroll
        for (int tt = 0; tt < NR; ++tt) {
          float sv[KT][4];
          if (need_mask) {
            const int rel = lim[tt] - kb - 4 * g4;  // key 16 kt + i of this lane is visible iff < rel
#pragma unroll
            for (int kt = 0; kt < KT; ++kt)
#pragma unroll
              for (int i = 0; i < 4; ++i)
                sv[kt][i] = 16 * kt + i < rel ? sacc[tt][kt][i] : -INFINITY;
          } else {
#pragma unroll
            for (int kt = 0; kt < KT; ++kt)
#pragma unroll
              for (int i = 0; i < 4; ++i) sv[kt][i] = sacc[tt][kt][i];
          }
          float mx = -INFINITY;
#pragma unroll
          for (int kt = 0; kt < KT; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i) mx = fmaxf(mx, sv[kt][i]);
          mx = max_xor16(mx);
          mx = max_xor32(mx);
          const float mxs = mx * p.scale_log2;
          if (__builtin_amdgcn_ballot_w64(mxs > m[tt] + kLazy) != 0) {
            const float mnew = fmaxf(m[tt], mxs);
            const float alpha = fast_exp2(m[tt] - mnew);
            m[tt] = mnew;
            l[tt] *= alpha;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) o[tt][dt] *= alpha;
          }
          float pr[KT][4];
#pragma unroll
          for (int kt = 0; kt < KT; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              pr[kt][i] = fast_exp2(fmaf(sv[kt][i], p.scale_log2, -m[tt]));
              l[tt] += pr[kt][i];
            }
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) {
            pb[tt][ks].x = M::pack2(pr[2 * ks][0], pr[2 * ks][1]);
            pb[tt][ks].y = M::pack2(pr[2 * ks][2], pr[2 * ks][3]);
            pb[tt][ks].z = M::pack2(pr[2 * ks + 1][0], pr[2 * ks + 1][1]);
            pb[tt][ks].w = M::pack2(pr[2 * ks + 1][2], pr[2 * ks + 1][3]);
          }
        }

        // ---- O^T += V^T P^T ----
        if constexpr (late_v) {
#pragma unroll
          for (int dt = 0; dt < VW; ++dt) vf[dt] = read_v(0, dt);
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) {
            const uint4 a = vf[dt % VW];
#pragma unroll
            for (int tt = 0; tt < NR; ++tt) o[tt][dt] = M::mfma(a, pb[tt][ks], o[tt][dt]);
            const int nx = ks * DT + dt + VW;
            if (nx < KS * DT) vf[dt % VW] = read_v(nx / DT, nx % DT);
          }
      };
      reduce();
      stage ^= 1;
    }
    if (cur.t0 == tend && has_next) {
      // No visible keys in this item: its output is 0 and the next item's
      // loads start here.  `stage` is free: no wave has read it since the
      // last barrier.
      cursor_to(nxt);
      if constexpr (kPaged) take_ids(nxt.t0);
      if (cu.t < cu.end) {
        issue_now(issue(stage), stage);
        advance();
      }
      load_q(nxt);
      st_slot = load_slot(nxt);
    }

    // ---- normalise and write: lane holds O[row r16][16 dt + 4 g4 + i] ----
    // The rows go out through LDS so that each store instruction writes whole
    // rows (16 bytes per lane, CPR lanes per row) instead of 8-byte pieces of
    // 16 rows: the narrow pattern cost more per byte.  The staging area is
    // the stage of the item's last tile (the next item's first tile is
    // landing in the other one); wave w uses its own 16 NR rows of it, so the
    // only barrier needed is the one that tells every wave is done reading
    // that stage's K and V.  Chunks are XOR-swizzled by row against bank
    // conflicts.
    if (kSplit && cur.slot >= 0) {
      // A piece of a split item: unnormalised, in fp32, straight from the
      // accumulators (64-byte pieces of 16 rows an instruction).
      const int64_t ps = (int64_t)xcd * p.split_slots + cur.slot;
      if (wave == 0) p.part_head[ps] = make_int4(cur.npc, cur.q0 + pos0, nrows, cur.h);
#pragma unroll
      for (int tt = 0; tt < NR; ++tt) {
        const int row = 16 * (wave + 4 * tt) + r16;
        float lt = l[tt];
        lt = sum_xor16(lt);
        lt = sum_xor32(lt);
        if (row < nrows) {
          float* const po = p.part_o + (ps * (64 * NR) + row) * D + 4 * g4;
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<f32x4_t*>(po + 16 * dt) = o[tt][dt];
          if (g4 == 0) p.part_ml[ps * (64 * NR) + row] = make_float2(m[tt], lt);
        }
      }
    } else if (cur.t0 < tend) {
      __syncthreads();
      char* s_o = s_kv + (stage ^ 1) * 2 * TILE_B + wave * 16 * NR * ROWB;
#pragma unroll
      for (int tt = 0; tt < NR; ++tt) {
        float lt = l[tt];
        lt = sum_xor16(lt);
        lt = sum_xor32(lt);
        const float inv = lt > 0.f ? 1.f / lt : 0.f;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          uint2 w;
          w.x = M::pack2(o[tt][dt][0] * inv, o[tt][dt][1] * inv);
          w.y = M::pack2(o[tt][dt][2] * inv, o[tt][dt][3] * inv);
          const int chunk = (2 * dt + (g4 >> 1)) ^ (r16 % CPR);
          *reinterpret_cast<uint2*>(s_o + (16 * tt + r16) * ROWB + chunk * 16 + (g4 & 1) * 8) = w;
        }
      }
      __builtin_amdgcn_wave_barrier();
      constexpr int RPS = 64 / CPR;  // rows per store instruction
#pragma unroll 2
      for (int j = 0; j < 16 * NR / RPS; ++j) {
        const int rw = RPS * j + lane / CPR;  // row within the wave's 16 NR
        const int c = lane % CPR;
        const uint4 v = lds_read16(s_o, rw * ROWB + ((c ^ ((rw % 16) % CPR)) << 4));
        const int row = 16 * wave + 64 * (rw / 16) + rw % 16;  // MFMA row of the block
        if (row < nrows)
          st16_nt(p.out + (int64_t)(cur.q0 + pos0 + row / G) * p.o_st +
                      (int64_t)(cur.h * G + row % G) * p.o_sh + c * 16,
                  v);
      }
    } else {
      // No visible keys: the rows are 0 (the other stage may be receiving the
      // next item's first tile, so nothing is staged).
#pragma unroll
      for (int tt = 0; tt < NR; ++tt) {
        const int row = 16 * (wave + 4 * tt) + r16;
        if (row >= nrows) continue;
        char* dst = p.out + (int64_t)(cur.q0 + pos0 + row / G) * p.o_st +
                    (int64_t)(cur.h * G + row % G) * p.o_sh;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
          *reinterpret_cast<uint2*>(dst + (16 * dt + 4 * g4) * 2) = make_uint2(0u, 0u);
      }
    }
    if (!has_next) break;
    cur = nxt;
  }
}

// Merge of split items' pieces: workgroup (x, y) serves rows 32 y .. 32 y + 31
// of the item whose first piece is XCD x % 8's piece x / 8 (the XCD that wrote
// it), and ends at once when there is no such item.
//   out = sum_j 2^(m_j - M) o_j / sum_j 2^(m_j - M) l_j,  M = max_j m_j.
template <bool kBF16, int D, int G, bool kHalf>
__global__ __launch_bounds__(256) void varlen_merge_kernel(VarlenParams p) {
  constexpr int LPR = D / 4;       // lanes per row, four outputs each
  constexpr int RPP = 256 / LPR;   // rows per pass
  constexpr int rows = kHalf ? kRowsPerWG / 2 : kRowsPerWG;  // of a piece's partials
  const int xcd = (int)blockIdx.x % kXcds, slot = (int)blockIdx.x / kXcds;
  const int64_t ps = (int64_t)xcd * p.split_slots + slot;
  const int count = p.part_count[xcd];
  const int4 hd = p.part_head[ps];  // read whether or not it was written
  const int row0 = (int)blockIdx.y * 32;
  if (slot >= count || hd.x == 0 || row0 >= hd.z) return;
  const int col = threadIdx.x % LPR;
  for (int row = row0 + threadIdx.x / LPR; row < min(row0 + 32, hd.z); row += RPP) {
    const float* po = p.part_o + (ps * rows + row) * D + 4 * col;
    const float2* pm = p.part_ml + ps * rows + row;
    float M = -1.0e30f, L = 0.f;
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
    for (int j0 = 0; j0 < hd.x; j0 += 4) {
      f32x4_t oj[4];
      float2 ml[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int64_t at = min(j0 + j, hd.x - 1) * (int64_t)rows;
        ml[j] = pm[at];
        oj[j] = *reinterpret_cast<const f32x4_t*>(po + at * D);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (j0 + j >= hd.x) break;
        const float mn = fmaxf(M, ml[j].x);
        const float a = fast_exp2(M - mn), b = fast_exp2(ml[j].x - mn);
        acc = acc * a + oj[j] * b;
        L = L * a + ml[j].y * b;
        M = mn;
      }
    }
    const float inv = L > 0.f ? 1.f / L : 0.f;
    uint2 w;
    w.x = Mma<kBF16>::pack2(acc[0] * inv, acc[1] * inv);
    w.y = Mma<kBF16>::pack2(acc[2] * inv, acc[3] * inv);
    *reinterpret_cast<uint2*>(p.out + (int64_t)(hd.y + row / G) * p.o_st +
                              (int64_t)(hd.w * G + row % G) * p.o_sh + col * 8) = w;
  }
}

// Launch the persistent grid: per XCD, as many workgroups as the kernel
// keeps resident on one XCD's CUs, or fewer when the XCD's item list (at
// most items_per_xcd long) is shorter.
template <bool kBF16, int D, int G, bool kCausal, bool kPaged, bool kOnce, bool kF8, bool kPro,
          bool kSplit, bool kHalf>
static void launch_grid(const VarlenParams& p, int64_t items_per_xcd, hipStream_t st) {
  const auto kern = varlen_attention_kernel<kBF16, D, G, kCausal, kPaged, kOnce, kF8, kPro, kSplit, kHalf>;
  // Resident workgroups per CU, queried once (a failed query is not cached:
  // the launch then assumes 1, which is correct but leaves slots idle).
  static std::atomic<int> cached{0};
  int per_cu = cached.load(std::memory_order_relaxed);
  if (per_cu <= 0) {
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, kVarlenThreads, 0) ==
            hipSuccess &&
        per_cu > 0) {
      cached.store(per_cu, std::memory_order_relaxed);
    } else {
      (void)hipGetLastError();
      per_cu = 1;
    }
  }
  int64_t cus_per_xcd = current_device_cus() / kXcds;
  if (cus_per_xcd < 1) cus_per_xcd = 1;
  int64_t per_xcd = (int64_t)per_cu * cus_per_xcd;
  if (per_xcd > items_per_xcd && !kSplit) per_xcd = items_per_xcd;
  if (per_xcd < 1) per_xcd = 1;
  hipLaunchKernelGGL(kern, dim3((unsigned)(per_xcd * kXcds)), dim3(kVarlenThreads), 0, st, p);
  if constexpr (kSplit)
    hipLaunchKernelGGL((varlen_merge_kernel<kBF16, D, G, kHalf>),
                       dim3(p.split_slots * kXcds, kHalf ? 2 : 4), dim3(256), 0, st, p);
}

template <bool kBF16, int D, int G, bool kCausal, bool kPaged, bool kOnce = false,
          bool kF8 = false, bool kPro = false>
static void launch_persistent(const VarlenParams& p, int64_t items_per_xcd, hipStream_t st) {
  if constexpr (kCausal && !kPro) {
    if (p.half)
      return p.split ? launch_grid<kBF16, D, G, true, kPaged, false, kF8, false, true, true>(
                           p, items_per_xcd, st)
                     : launch_grid<kBF16, D, G, true, kPaged, false, kF8, false, false, true>(
                           p, items_per_xcd, st);
  }
  if constexpr (!kOnce) {
    if (p.split)
      return launch_grid<kBF16, D, G, kCausal, kPaged, false, kF8, kPro, true, false>(
          p, items_per_xcd, st);
  }
  launch_grid<kBF16, D, G, kCausal, kPaged, kOnce, kF8, kPro, false, false>(p, items_per_xcd, st);
}

template <bool kBF16, int D, int G, bool kCausal>
static void launch_varlen_c(const VarlenParams& p, int64_t items_per_xcd, hipStream_t st) {
  // The fused query prologue: causal launches at head_dim 128 over a 16-bit
  // pool or none (the host checks this before launching).
  if constexpr (kCausal && D == 128) {
    if (p.has_pro) {
      if (p.has_pool)
        launch_persistent<kBF16, D, G, true, true, false, false, true>(p, items_per_xcd, st);
      else
        launch_persistent<kBF16, D, G, true, false, false, false, true>(p, items_per_xcd, st);
      return;
    }
  }
  if (p.has_pool && p.kv_f8)
    launch_persistent<kBF16, D, G, kCausal, true, false, true>(p, items_per_xcd, st);
  else if (p.has_pool)
    launch_persistent<kBF16, D, G, kCausal, true>(p, items_per_xcd, st);
  else if (!kCausal && p.num_qblocks == 1)
    launch_persistent<kBF16, D, G, kCausal, false, true>(p, items_per_xcd, st);
  else
    launch_persistent<kBF16, D, G, kCausal, false>(p, items_per_xcd, st);
}

template <bool kBF16, int D, int G>
static void launch_varlen(const VarlenParams& p, bool causal, int64_t items_per_xcd,
                          hipStream_t st) {
  if (causal)
    launch_varlen_c<kBF16, D, G, true>(p, items_per_xcd, st);
  else
    launch_varlen_c<kBF16, D, G, false>(p, items_per_xcd, st);
}

// Launch for one 16-bit type and head_dim, instantiated in
// varlen_<type>_d<D>.hip so that they compile in parallel; false for an
// unsupported group.
template <bool kBF16, int D>
bool launch_varlen_d(int G, const VarlenParams& p, bool causal, int64_t items_per_xcd,
                     hipStream_t st);
template <>
bool launch_varlen_d<true, 64>(int, const VarlenParams&, bool, int64_t, hipStream_t);
template <>
bool launch_varlen_d<true, 128>(int, const VarlenParams&, bool, int64_t, hipStream_t);
template <>
bool launch_varlen_d<false, 64>(int, const VarlenParams&, bool, int64_t, hipStream_t);
template <>
bool launch_varlen_d<false, 128>(int, const VarlenParams&, bool, int64_t, hipStream_t);

template <bool kBF16, int D>
static bool dispatch_varlen_g(int G, const VarlenParams& p, bool causal, int64_t items_per_xcd,
                              hipStream_t st) {
  switch (G) {
    case 1: launch_varlen<kBF16, D, 1>(p, causal, items_per_xcd, st); return true;
    case 2: launch_varlen<kBF16, D, 2>(p, causal, items_per_xcd, st); return true;
    case 4: launch_varlen<kBF16, D, 4>(p, causal, items_per_xcd, st); return true;
    case 8: launch_varlen<kBF16, D, 8>(p, causal, items_per_xcd, st); return true;
    default: return false;
  }
}

}  // namespace va
