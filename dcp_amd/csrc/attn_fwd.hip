// Range-masked paged attention forward for gfx950.
//
// One workgroup (4 waves) owns 128 query rows of one (row, head); wave w owns
// rows 32w..32w+31.  It walks the key tiles (64 keys) its rows can see and
// keeps a running softmax per query row.  Everything is computed transposed:
//
//   S^T[kv, q] = K Q^T      A = K tile from LDS, B = Q held in registers
//   O^T[d,  q] = V^T P^T    A = V^T tile from LDS, B = P^T straight from the
//                           S^T accumulators
//
// With the 32x32x16 MFMA a lane holds one column of the accumulator, so in
// this orientation a lane owns one query row: the row max / row sum need no
// cross-lane reduction beyond one exchange between the two half-waves, the
// rescale factor is a per-lane scalar, and the masked range of the row lives
// in four registers.
//
// Software pipeline inside a wave: S^T of tile j+1 is multiplied while tile j is
// exponentiated, MFMA by MFMA in one instruction stream, so the matrix pipe and the
// vector ALU work at the same time instead of taking turns; O^T += V^T P^T of tile
// j follows as a dense run of MFMAs that the other wave of the SIMD can fill with
// its own arithmetic.
//
// K and V tiles go from global memory straight into LDS (global_load_lds, no
// register staging), in two stages: the next tile streams in while the current
// one is multiplied.  The row order and padding of each tile are chosen so that
// operand reads are conflict-free and every LDS address in the key loop is a
// per-lane base plus an immediate.  V^T is never materialised: the transposing
// LDS load delivers it from the V tile.
//
// Key tiles are chosen per workgroup from the hull of its rows' ranges (tiles
// no row can see are never loaded), each wave skips tiles outside its own
// rows' hull, and a tile that lies inside every row's range of the wave skips
// the per-element range test.  A tile that some rows see in part is multiplied like
// the others, in the pipeline, and masked afterwards.
#include <math.h>

#include <algorithm>

#include "attn_common.h"
#include "record.h"

namespace dcp {

// Part `part` of `n_parts` of a row's keys: an equal share of the key tiles of each of the row's work
// items.  n_parts > 1: the result goes to partial first_partial + part.
struct FwdPart {
  int row, part, n_parts, first_partial;
};

// A work item's queries (dcp_attn_fwd_items): 128 of a row, or a part of them as in FwdPart.  The other entry points
// have as many items for a row as its block has tiles, whether the row has queries for them or not, and a
// workgroup that draws one without spends 1.5-2 us on it (4476 tokens in sequences of 290 tokens and blocks of
// 1024, 8 heads of size 64: 528 of 832 items are like that, the launch takes 31.6 us with and 13.9 without them).
struct FwdTile {
  int row, q_tile, part_of, first_partial;  // part_of: part + 65536 * number of parts
};

struct AttnFwdParams {
  const void* q;
  const void* k;
  const void* v;
  void* out;
  float* lse;
  const int32_t* cu_seqlens_q;
  const int32_t* cu_seqlens_kv;
  const int32_t* attn_range;
  const int32_t* q_block_table;
  const int32_t* kv_block_table;
  const int32_t* out_block_table;
  const int32_t* row_order;
  int n_ranges;
  int batch;
  int max_kv_blocks;
  int total_q;
  int block_size;
  int n_heads_q;
  int n_heads_kv;
  int64_t kv_slot_stride;
  int64_t kv_token_stride;
  int n_out_slots;
  // element strides of a table entry: a slot of block_size tokens, or a single token when the
  // tables address the caller's unpadded tensors directly (entries are then token offsets)
  int64_t q_slot_stride;
  int64_t out_slot_stride;
  int64_t lse_head_stride;
  int64_t lse_slot_stride;
  float empty_lse;   // what the LSE of a query without a visible key reads: +inf, or the merged form -1
  int q_tiles_per_row;
  int xcd_group;     // work items per shared K/V stream
  int64_t n_items;   // batch * n_heads_q * q_tiles_per_row
  float scale_log2;  // softmax_scale * log2(e)
  int* tickets;      // of the item queue, zeroed before the launch; null: one item per workgroup
  int ticket_stride;
  // rows in parts (dcp_attn_fwd_parts): a record per launch entry, which takes the place of a row
  const FwdPart* parts;
  const FwdTile* tiles;  // the launch's items, one for all heads; null: all tiles of all rows
  float* partial_out;   // [partial][head][32-query block][D / 4][query][4]: O^T relative to the part's maximum
  float* partial_sums;  // [partial][head][32-query block][query][2]: the maximum (log2 domain) and the sum of the weights
};

// Wave priority by phase: the two waves of a SIMD come from different workgroups and drift
// through the loop independently.  Both matrix phases outrank the control code between them
// (2-3 % on the kernel), and the fused phase, whose vector work is the longer chain, outranks
// the dense one (another 1.5 %; the other way round it was 1.5 % slower).
constexpr int kPrioControl = 0, kPrioFused = 2, kPrioDense = 1;
// Ints from one counter of the item queue to the next, and in a workspace of the 64 bytes that used to be
// all there was (65536 causal tokens, 32 heads: 3.75 and 3.77 ms).
constexpr int kFwdTicketStride = 8, kFwdTicketStrideMin = DCP_ATTN_FWD_MIN_WORKSPACE_BYTES / (kNumXcd * 4);
constexpr int kFwdBN = 64;
constexpr int kFwdThreads = 256;
// The running maximum of a row is only raised (and O^T rescaled) when the tile's maximum
// exceeds it by more than this many powers of two; until then the weights of the tile are
// taken relative to the old maximum and are at most 2^kLazyMax.  With fp32 sums and
// accumulators that costs no accuracy, and it takes the rescale (64 multiplies per query
// block) out of almost every tile after a row's first few.
constexpr float kLazyMax = 8.0f;
// On the fast path a tile is exponentiated against the row's current reference without taking
// its maximum first; it is redone against a raised reference only if one lane's partial row sum
// of the tile (32 weights) reaches kMaxTileSum, i.e. if some weight might exceed it.  2^14 keeps
// every accepted weight representable in fp16 and far from overflowing the fp32 accumulators.
constexpr float kMaxTileSum = 16384.0f;

// QB = 32-row query blocks per wave: the workgroup owns 128*QB query rows.  With QB = 2 every
// K / V^T operand read from LDS feeds two matrix instructions and every tile brought into LDS
// serves twice the arithmetic; the wave then needs the whole register file (one workgroup
// per CU, accumulators in the AGPR half).
// ITEMS: what the launch is over.  kFwdParts: its rows are split along their keys.  A work item is a serial chain, a tile after the
// other (1.2-1.5 us each with a workgroup alone on its CU), and a launch of few, uneven rows lasts as long as its longest:
// see dcp_attn_fwd_parts.  kFwdTiles: its items are listed (FwdTile), as parts or whole.
enum FwdItems { kFwdRows, kFwdParts, kFwdTiles };
template <int DTYPE, int D, int QB, FwdItems ITEMS>
__device__ __forceinline__ void attn_fwd_item(KernArgs<AttnFwdParams>& p, int item) {
  constexpr bool PARTS = ITEMS != kFwdRows;
  constexpr int BN = kFwdBN;
  constexpr int BM = 128 * QB;
  constexpr int KS = D / 16;  // k-steps of S^T = K Q^T
  constexpr int DT = D / 32;  // 32-row tiles of O^T
  typedef KvTile<D> KTile;  // read as rows (A operand of S^T)
  typedef KvTile<D> VTile;  // read as columns (A operand of O^T = V^T P^T)
  // two stages of (K tile, V tile); separate arrays so the compiler can tell
  // the stage being filled from the stage being read
  __shared__ __attribute__((aligned(16))) uint16_t k_lds0[KTile::SIZE];
  __shared__ __attribute__((aligned(16))) uint16_t v_lds0[VTile::SIZE];
  __shared__ __attribute__((aligned(16))) uint16_t k_lds1[KTile::SIZE];
  __shared__ __attribute__((aligned(16))) uint16_t v_lds1[VTile::SIZE];
  __shared__ int hull_lds[4][4];
  __shared__ int slot_lds[kSlotTableCap];

  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int c = lane & 31;
  const int h = lane >> 5;

  // ---- which (row, head, q tile) ----------------------------------------
  // the query tiles and grouped heads of a row share its K/V: keep them on one XCD
  // Integer division runs on the vector unit, so its (uniform) results sit in vector registers
  // and drag every address derived from them there too: each tile load then costs three vector
  // instructions to rebuild a scalar base.  readfirstlane puts the indices back on the scalar unit.
  int wg = item, qt;
  if constexpr (ITEMS != kFwdTiles) {
    qt = __builtin_amdgcn_readfirstlane(wg % p.q_tiles_per_row);
    wg /= p.q_tiles_per_row;
  }
  const int head = __builtin_amdgcn_readfirstlane(wg % p.n_heads_q);
  const int bi = __builtin_amdgcn_readfirstlane(wg / p.n_heads_q);
  FwdPart part = {0, 0, 1, 0};
  if constexpr (ITEMS == kFwdTiles) {
    const FwdTile t = p.tiles[bi];
    part = {t.row, t.part_of & 0xffff, t.part_of >> 16, t.first_partial};
    qt = __builtin_amdgcn_readfirstlane(t.q_tile);
  } else if constexpr (ITEMS == kFwdParts) {
    part = p.parts[bi];
  }
  const int b = __builtin_amdgcn_readfirstlane(PARTS ? part.row : p.row_order ? p.row_order[bi] : bi);
  // Everything the tables say of the row in one trip to memory, and the ranges requested before Q, which nobody waits
  // for before its first product: each asked for where it is used was a chain of seven trips, and a launch of few short
  // rows is little more than that chain (1000 tokens, 8 heads, 13.8 -> 13.4 us; 5120 fp16 tokens, step, 102 -> 100).
  const int32_t* kv_table = p.kv_block_table + (int64_t)b * p.max_kv_blocks;
  int q_begin = p.cu_seqlens_q[b], q_end = p.cu_seqlens_q[b + 1], kv_begin = p.cu_seqlens_kv[b], kv_end = p.cu_seqlens_kv[b + 1];
  int q_entry = p.q_block_table[b], o_slot = p.out_block_table[b];
  int first_slots = 0;  // of the row's kv blocks, one a thread
  if (tid < min(p.max_kv_blocks, kSlotTableCap)) first_slots = kv_table[tid];
  asm volatile("" : "+v"(q_begin), "+v"(q_end), "+v"(kv_begin), "+v"(kv_end), "+v"(q_entry), "+v"(o_slot), "+v"(first_slots));
  q_begin = __builtin_amdgcn_readfirstlane(q_begin);
  q_entry = __builtin_amdgcn_readfirstlane(q_entry);
  o_slot = __builtin_amdgcn_readfirstlane(o_slot);
  const int seqlen_q = __builtin_amdgcn_readfirstlane(q_end) - q_begin;
  const int seqlen_kv = __builtin_amdgcn_readfirstlane(kv_end) - __builtin_amdgcn_readfirstlane(kv_begin);
  if (qt * BM >= seqlen_q) return;
  const int kv_head = __builtin_amdgcn_readfirstlane(head / (p.n_heads_q / p.n_heads_kv));
  const int64_t q_row_stride = (int64_t)p.n_heads_q * D;

  int q_local[QB];
  bool q_valid[QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    q_local[qb] = qt * BM + (w * QB + qb) * 32 + c;
    q_valid[qb] = q_local[qb] < seqlen_q;
  }

  int range_words[QB][4];  // start0, end0, start1, end1
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
#pragma unroll
    for (int i = 0; i < 4; ++i) range_words[qb][i] = 0;
    if (q_valid[qb]) {
      const int32_t* r = p.attn_range + q_begin + q_local[qb];
      range_words[qb][0] = r[0];
      range_words[qb][1] = r[p.total_q];
      if (p.n_ranges == 2) {
        range_words[qb][2] = r[2 * (int64_t)p.total_q];
        range_words[qb][3] = r[3 * (int64_t)p.total_q];
      }
    }
  }

  // ---- Q fragments (B operands of S^T) -------------------------------------
  u32x4 qreg[QB][KS];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const uint16_t* qp = reinterpret_cast<const uint16_t*>(p.q) +
                         (int64_t)q_entry * p.q_slot_stride + (int64_t)q_local[qb] * q_row_stride +
                         (int64_t)head * D + h * 8;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      u32x4 z = {0, 0, 0, 0};
      qreg[qb][ks] = q_valid[qb] ? *reinterpret_cast<const u32x4*>(qp + ks * 16) : z;
    }
  }

  // ---- this lane's query rows: ranges --------------------------------------
  RangePair rng[QB];
  const int big = 0x7fffffff;
  int w_lo0 = big, w_hi0 = 0, w_lo1 = big, w_hi1 = 0;            // hull: what any row of the wave can see
  int core_lo0 = 0, core_hi0 = big, core_lo1 = 0, core_hi1 = big;  // core: what every row sees that sees anything
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    RangePair r4 = {0, 0, 0, 0};
    if (q_valid[qb]) {
      const KeyRange range0 = key_range(range_words[qb][0], range_words[qb][1], seqlen_kv);
      r4.s0 = range0.start;
      r4.len0 = range0.len;
      if (p.n_ranges == 2) {
        const KeyRange range1 = key_range(range_words[qb][2], range_words[qb][3], seqlen_kv);
        r4.s1 = range1.start;
        r4.len1 = range1.len;
      }
    }
    rng[qb] = r4;
    w_lo0 = min(w_lo0, wave_min(r4.len0 > 0 ? r4.s0 : big));
    w_hi0 = max(w_hi0, wave_max(r4.len0 > 0 ? r4.s0 + r4.len0 : 0));
    w_lo1 = min(w_lo1, wave_min(r4.len1 > 0 ? r4.s1 : big));
    w_hi1 = max(w_hi1, wave_max(r4.len1 > 0 ? r4.s1 + r4.len1 : 0));
    // A row that sees nothing (a block's padding, or a query whose keys are all in other partials) gets a zero Q (below),
    // so that it may see anything on the way and its result is taken back at the end: were it taken as
    // seeing nothing, its wave would mask every tile, and its workgroup wait for it at every one.  (Rows past
    // the last query likewise, so that a row's results do not depend on what fills its wave.)
    const bool nothing = r4.len0 == 0 && r4.len1 == 0;
    core_lo0 = max(core_lo0, wave_max(r4.len0 > 0 ? r4.s0 : nothing ? 0 : big));
    core_hi0 = min(core_hi0, wave_min(r4.len0 > 0 ? r4.s0 + r4.len0 : nothing ? big : 0));
    core_lo1 = max(core_lo1, wave_max(r4.len1 > 0 ? r4.s1 : nothing ? 0 : big));
    core_hi1 = min(core_hi1, wave_min(r4.len1 > 0 ? r4.s1 + r4.len1 : nothing ? big : 0));
  }
  if (w_hi0 == 0 && w_hi1 == 0) core_hi0 = core_hi1 = 0;  // no row of the wave sees anything
  if (tid < min(p.max_kv_blocks, kSlotTableCap)) slot_lds[tid] = first_slots;
  load_slot_table(slot_lds, kv_table, p.max_kv_blocks, tid + kFwdThreads, kFwdThreads);
  if (lane == 0) {
    hull_lds[w][0] = w_lo0;
    hull_lds[w][1] = w_hi0;
    hull_lds[w][2] = w_lo1;
    hull_lds[w][3] = w_hi1;
  }
  __syncthreads();
  int g_lo0 = big, g_hi0 = 0, g_lo1 = big, g_hi1 = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    g_lo0 = min(g_lo0, hull_lds[i][0]);
    g_hi0 = max(g_hi0, hull_lds[i][1]);
    g_lo1 = min(g_lo1, hull_lds[i][2]);
    g_hi1 = max(g_hi1, hull_lds[i][3]);
  }
  // the same in every lane: say so, and the tile list, the cursor and the loop control that
  // derive from them live on the scalar unit
  g_lo0 = __builtin_amdgcn_readfirstlane(g_lo0);
  g_hi0 = __builtin_amdgcn_readfirstlane(g_hi0);
  g_lo1 = __builtin_amdgcn_readfirstlane(g_lo1);
  g_hi1 = __builtin_amdgcn_readfirstlane(g_hi1);
  const TileRuns runs(g_lo0, g_hi0, g_lo1, g_hi1, BN);
  int first_tile = 0, n_tiles = runs.count();  // where the item begins and ends in the tile list
  const int partial = PARTS && part.n_parts > 1 ? part.first_partial + part.part : -1;  // where its result goes
  if constexpr (PARTS) {
    first_tile = __builtin_amdgcn_readfirstlane(n_tiles * part.part / part.n_parts);
    n_tiles = __builtin_amdgcn_readfirstlane(n_tiles * (part.part + 1) / part.n_parts);
  }

  // ---- running state ---------------------------------------------------------
  f32x16 o_acc[QB][DT];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb)
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) o_acc[qb][dt][i] = 0.0f;
  float m_run[QB], l_run[QB];  // reference maximum (log2 domain); this half-wave's partial row sum
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    m_run[qb] = -INFINITY;
    l_run[qb] = 0.0f;
  }

  const uint16_t* kg = reinterpret_cast<const uint16_t*>(p.k) + (int64_t)kv_head * D;
  const uint16_t* vg = reinterpret_cast<const uint16_t*>(p.v) + (int64_t)kv_head * D;

  // loop-invariant per-lane pieces of every address used in the key loop
  const uint32_t kv_goff0 = KTile::lane_offset0(p.kv_token_stride, w, lane);
  const int k_rd = KTile::row_base(c, h);
  const int v_rd = VTile::col_base(lane, true);

  // The cursor runs two tiles ahead of the tile being exponentiated: it names the K
  // tile to request next.  V of a tile is requested one iteration after its K, from the
  // offset remembered then.
  const int tiles_per_block = p.block_size / BN;
  const int64_t tile_stride = (int64_t)BN * p.kv_token_stride;
  TileCursor cursor;
  auto cursor_next = [&]() {
    if (__builtin_expect(cursor.index + 1 < n_tiles, 1)) cursor.advance(runs, tiles_per_block, slot_lds, kv_table, p.kv_slot_stride, tile_stride);
    else ++cursor.index;  // past the end: nothing left to request
  };
  const uint32_t k_at0 = lds_address(k_lds0), k_at1 = lds_address(k_lds1);
  const uint32_t v_at0 = lds_address(v_lds0), v_at1 = lds_address(v_lds1);
  // does any row of this wave see key tile `tile` / does every row see all of it
  auto wave_sees = [&](int tile) -> bool {
    const int k0 = tile * BN;
    return (k0 < w_hi0 && k0 + BN > w_lo0) || (k0 < w_hi1 && k0 + BN > w_lo1);
  };
  auto wave_sees_all = [&](int tile) -> bool {
    const int k0 = tile * BN;
    return (core_lo0 <= k0 && k0 + BN <= core_hi0) || (core_lo1 <= k0 && k0 + BN <= core_hi1);
  };
  // the same test in tile numbers, for the loop's fast path: tiles [full0, full0 + n_full0) and
  // [full1, full1 + n_full1) lie inside every row's range
  const int full0 = (core_lo0 > big - BN ? big / BN : (core_lo0 + BN - 1) / BN), n_full0 = max(core_hi0 / BN - full0, 0);
  const int full1 = (core_lo1 > big - BN ? big / BN : (core_lo1 + BN - 1) / BN), n_full1 = max(core_hi1 / BN - full1, 0);
  auto tile_is_full = [&](int tile) -> bool {
    return ((unsigned)(tile - full0) < (unsigned)n_full0) | ((unsigned)(tile - full1) < (unsigned)n_full1);
  };

  // The tile loads of an iteration (this wave's share: LPW groups of K, LPW of V) are issued
  // one at a time between the matrix instructions of the S^T product: as a burst after the
  // barrier they fill the memory pipeline's queue and the wave sits at its last load until the
  // queue has drained, and issued later (spread over the O^T product too) the last one is still
  // on its way at the wait that opens the next iteration.  Both stages they fill are free from
  // the iteration's first barrier on.  They are issued unconditionally, so that the loop has no
  // branches around them: past the end of the tile list the cursor stays on the last tile,
  // which is then fetched again into a stage nobody reads any more.
  constexpr int NL = 2 * KTile::LPW;
  uint32_t fill_k = 0, fill_v = 0;
  int64_t fill_k_off = 0, fill_v_off = 0;
  auto issue_load = [&](int idx) {
    if (idx < KTile::LPW) KTile::load_group(fill_k, kg + fill_k_off, kv_goff0, p.kv_token_stride, w, idx);
    else if (idx < NL) VTile::load_group(fill_v, vg + fill_v_off, kv_goff0, p.kv_token_stride, w, idx - KTile::LPW);
  };

  // Operand i of S^T = K Q^T: key half i & 1, k-step i >> 1 (the two halves alternate so
  // that consecutive MFMAs are independent); each operand feeds QB MFMAs.
  auto k_operand = [&](const uint16_t* k_lds, int i) { return KTile::read_row(k_lds, k_rd, i & 1, i >> 1); };

  // S^T of a tile on its own.  The range mask enters as the accumulator's initial
  // value: 0 where the row may look, -inf where it may not.
  auto multiply_qk = [&](int tile, const uint16_t* k_lds, f32x16 (&s_out)[2][QB]) {
    if (wave_sees_all(tile)) {
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int qb = 0; qb < QB; ++qb)
#pragma unroll
          for (int e = 0; e < 16; ++e) s_out[nt][qb][e] = 0.0f;
    } else {
      // the keys a row may not see, as a bit mask per 32-key half (bit = key - first key of the
      // half), shifted so that element e of this lane's half h is bit 8 (e / 4) + e % 4
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) {
          const uint32_t closed = rng[qb].closed_window(tile * BN + nt * 32) >> (4 * h);
#pragma unroll
          for (int e = 0; e < 16; ++e) s_out[nt][qb][e] = masked_start(closed, 8 * (e / 4) + (e % 4));
        }
    }
    constexpr int N = 2 * KS, AHEAD = 3;
    u32x4 ka[4];
#pragma unroll
    for (int i2 = 0; i2 < AHEAD; ++i2) ka[i2] = k_operand(k_lds, i2);
#pragma unroll
    for (int i2 = 0; i2 < N; ++i2) {
      if (i2 + AHEAD < N) ka[(i2 + AHEAD) & 3] = k_operand(k_lds, i2 + AHEAD);
#pragma unroll
      for (int qb = 0; qb < QB; ++qb)
        s_out[i2 & 1][qb] = mfma_32x32x16<DTYPE>(ka[i2 & 3], qreg[qb][i2 >> 1], s_out[i2 & 1][qb]);
      if ((i2 + 1) % (N / NL) == 0) issue_load(i2 / (N / NL));
      __builtin_amdgcn_sched_barrier(0);  // keeps the operand reads from being hoisted into more registers
    }
  };

  // The mask of a tile whose S^T was multiplied without: 0 or -inf is added.
  auto add_mask = [&](int tile, f32x16 (&sc)[2][QB]) {
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        const uint32_t closed = rng[qb].closed_window(tile * BN + nt * 32) >> (4 * h);
#pragma unroll
        for (int e = 0; e < 16; ++e) sc[nt][qb][e] += masked_start(closed, 8 * (e / 4) + (e % 4));
      }
  };

  // ---- online softmax (log2 domain), in pieces so that it can be interleaved ----
  u32x4 pb[QB][4];       // P^T of the current tile, packed: the B operands of O^T += V^T P^T
  float alpha[QB];       // pending rescale of O^T (applied before the tile's P^T is multiplied in)
  bool rescale[QB];
  float m_use[QB], lsum[QB];
  // The maximum step of a tile: the row maximum, and the row's reference raised to it if needed.
  auto softmax_max = [&](const f32x16 (&sc)[2][QB]) {
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      float mx = -INFINITY;
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int e = 0; e < 16; ++e) mx = fmaxf(mx, sc[nt][qb][e]);
      mx = halves_max(mx * p.scale_log2);  // -inf stays -inf (scale > 0)
      // raise the reference maximum only when the tile exceeds it by more than kLazyMax (always
      // for a row that had none yet: -inf + kLazyMax = -inf), then for every row of the wave
      rescale[qb] = __any(mx > m_run[qb] + kLazyMax);
      const float m_new = rescale[qb] ? fmaxf(m_run[qb], mx) : m_run[qb];
      m_use[qb] = (m_new == -INFINITY) ? 0.0f : m_new;
      alpha[qb] = fast_exp2(m_run[qb] - m_use[qb]);  // m_run = -inf -> 0; 1 where the maximum stays
      l_run[qb] *= alpha[qb];
      m_run[qb] = m_new;
      lsum[qb] = 0.0f;
    }
  };
  // elements 2*c2, 2*c2+1 of the 32 this lane holds for query block qb
  auto softmax_pair = [&](const f32x16 (&sc)[2][QB], int qb, int c2) {
    const int nt = c2 >> 3, e = (c2 & 7) * 2;
    const float e0 = fast_exp2(fmaf(sc[nt][qb][e], p.scale_log2, -m_use[qb]));
    const float e1 = fast_exp2(fmaf(sc[nt][qb][e + 1], p.scale_log2, -m_use[qb]));
    lsum[qb] += e0 + e1;
    pb[qb][nt * 2 + (e >> 3)][(e & 7) >> 1] = pack2<DTYPE>(e0, e1);
  };
  auto apply_rescale = [&]() {
#pragma unroll
    for (int qb = 0; qb < QB; ++qb)
      if (__builtin_expect(rescale[qb], 0)) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int e = 0; e < 16; ++e) o_acc[qb][dt][e] *= alpha[qb];
      }
  };
  auto softmax = [&](const f32x16 (&sc)[2][QB]) {
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
#pragma unroll
      for (int c2 = 0; c2 < 16; ++c2) softmax_pair(sc, qb, c2);
      l_run[qb] += lsum[qb];
    }
  };

  // S^T of the next tile and the softmax of the current one in one instruction stream:
  // every MFMA is followed by its share of the softmax arithmetic, so that the matrix
  // pipe and the vector ALU of the SIMD are busy at the same time.  Operands are read
  // three ahead.  The softmax of a pair of elements goes through three stages an MFMA apart -- the argument of pair
  // c2 + 1, the exponential of pair c2, sum and packing of pair c2 - 1 -- so that no instruction waits for the one before
  // it: 1024 tokens, 8 heads 23.4 -> 22.2 us, 1000 tokens 13.4 -> 13.1; large launches gain less than they vary by (65536
  // causal tokens 0.8 % with the tables' reads above).
  auto multiply_qk_with_softmax = [&](const uint16_t* k_lds, f32x16 (&s_out)[2][QB], const f32x16 (&sc)[2][QB]) {
    constexpr int N = 2 * KS;     // operands, QB MFMAs each
    constexpr int AHEAD = 3;
    constexpr int PAIRS = 16 * QB;
    float arg[2][2], weight[2][2];  // [pair & 1][element]
    auto take_arg = [&](int c2) {
      const int qb = c2 / 16, nt = (c2 % 16) >> 3, el = (c2 & 7) * 2;
#pragma unroll
      for (int k = 0; k < 2; ++k) arg[c2 & 1][k] = fmaf(sc[nt][qb][el + k], p.scale_log2, -m_use[qb]);
    };
    auto take_sum = [&](int c2) {
      const int qb = c2 / 16, nt = (c2 % 16) >> 3, el = (c2 & 7) * 2;
      lsum[qb] += weight[c2 & 1][0] + weight[c2 & 1][1];
      pb[qb][nt * 2 + (el >> 3)][(el & 7) >> 1] = pack2<DTYPE>(weight[c2 & 1][0], weight[c2 & 1][1]);
    };
    auto softmax_stages = [&](int c2) {
      if (c2 > 0) take_sum(c2 - 1);
#pragma unroll
      for (int k = 0; k < 2; ++k) weight[c2 & 1][k] = fast_exp2(arg[c2 & 1][k]);
      if (c2 + 1 < PAIRS) take_arg(c2 + 1);
    };
    take_arg(0);
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int qb = 0; qb < QB; ++qb)
#pragma unroll
        for (int e = 0; e < 16; ++e) s_out[nt][qb][e] = 0.0f;
    u32x4 ka[4];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) ka[i] = k_operand(k_lds, i);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      if (i + AHEAD < N) ka[(i + AHEAD) & 3] = k_operand(k_lds, i + AHEAD);
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        s_out[i & 1][qb] = mfma_32x32x16<DTYPE>(ka[i & 3], qreg[qb][i >> 1], s_out[i & 1][qb]);
        // pairs [lo, hi) of the PAIRS this wave owes, query block 0 first
        const int lo = (i * QB + qb) * PAIRS / (N * QB);
        const int hi = (i * QB + qb + 1) * PAIRS / (N * QB);
#pragma unroll
        for (int c2 = lo; c2 < hi; ++c2) softmax_stages(c2);
      }
      if ((i + 1) % (N / NL) == 0) issue_load(i / (N / NL));
      __builtin_amdgcn_sched_barrier(0);
    }
    take_sum(PAIRS - 1);
  };

  // O^T += V^T P^T: V^T comes out of the row-major V tile by transpose loads, read
  // two operands ahead; consecutive MFMAs go to different accumulators
  auto multiply_pv = [&](const uint16_t* v_lds) {
    constexpr int N = 4 * DT;
    constexpr int AHEAD = 2;
    auto v_operand = [&](int i) { return VTile::template read_col<true>(v_lds, v_rd, i / DT, i % DT); };
    u32x4 va[4];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) va[i] = v_operand(i);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      if (i + AHEAD < N) va[(i + AHEAD) & 3] = v_operand(i + AHEAD);
#pragma unroll
      for (int qb = 0; qb < QB; ++qb)
        o_acc[qb][i % DT] = mfma_32x32x16<DTYPE>(va[i & 3], pb[qb][i / DT], o_acc[qb][i % DT]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // ---- key loop --------------------------------------------------------------------
  // Iteration j multiplies S^T of tile j+1 while it exponentiates tile j, then adds
  // tile j to O^T.  K tile j+1 and V tile j are in LDS by then; K tile j+2 and V tile
  // j+1 stream into the stages that K tile j and V tile j-1 have left.
  f32x16 s_a[2][QB], s_b[2][QB];
#pragma unroll
  for (int nt = 0; nt < 2; ++nt)
#pragma unroll
    for (int qb = 0; qb < QB; ++qb)
#pragma unroll
      for (int e = 0; e < 16; ++e) s_a[nt][qb][e] = s_b[nt][qb][e] = 0.0f;
  int tile_cur = 0, tile_nxt = 0;  // key tile numbers of list entries j and j+1
  int64_t v_off = 0;               // offset of list entry j+1 (its V is requested in iteration j)
  bool cur_full = false;           // list entry j lies inside every row's range
  bool raw = false;                // its S^T still lacks the range mask (the fast path multiplies without)
  bool pending = false;            // the maximum step of list entry j has been done already
  bool anchored = false;           // every row of the wave that sees anything has a (finite) reference maximum
  auto iteration = [&](int j, f32x16 (&s_cur)[2][QB], f32x16 (&s_nxt)[2][QB], const uint16_t* k_nxt, uint32_t k_fill,
                       const uint16_t* v_cur, uint32_t v_fill) {
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();  // K tile j+1 and V tile j are filled; nobody reads K tile j or V tile j-1 any more
    fill_k = k_fill;
    fill_v = v_fill;
    fill_k_off = cursor.off;
    fill_v_off = v_off;
    // the S^T product carries the tile loads; a wave that skips it still has its share to request
    const bool nxt_full = j + 1 < n_tiles && tile_is_full(tile_nxt);
    // Tiles that some rows see in part take the pipelined path too, and the mask is added to their S^T when it is
    // consumed (`raw`).  On the path below they cost a product, a maximum and a softmax one after the other, in every
    // wave of a workgroup that meets at each tile.  Forward, us, without and with this: 1000 tokens 15.4 -> 13.7; 4476
    // tokens in sequences of 290 17.3 -> 13.5; 32 000 tokens in short sequences, blocks of 1024, 73.8 -> 64.4; under a
    // causal mask over 64 k tokens, where few tiles are masked, 3709 -> 3689.  The tests for it stay out of an iteration
    // between two whole tiles; a test of every row's reference in each iteration below cost 3-4 % of every launch.
    bool cur = true, nxt = nxt_full, fast = cur_full && nxt_full && anchored;
    if (__builtin_expect(!fast, 0)) {
      cur = cur_full || wave_sees(tile_cur);
      nxt = nxt_full || (j + 1 < n_tiles && wave_sees(tile_nxt));
      fast = cur && nxt && anchored;
      if (raw) {
        add_mask(tile_cur, s_cur);
        raw = false;
      }
    }
    if (__builtin_expect(fast, 1)) {
      // The common case, decided by one test per iteration where this tile and the next are inside
      // every row's range: the wave sees both and every row has a reference maximum (one that sees nothing may not:
      // its zero Q gives it weights of 1 against the 0 that softmax_max left in its m_use).  The weights are taken relative
      // to that reference WITHOUT looking at the tile's own maximum first ...
      if (!pending) {
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) {
          lsum[qb] = 0.0f;
          rescale[qb] = false;
        }
      }
      __builtin_amdgcn_s_setprio(kPrioFused);
      multiply_qk_with_softmax(k_nxt, s_nxt, s_cur);
      // ... and the tile's partial row sums tell afterwards whether that was safe: every weight is
      // at most its lane's sum.  Only if a sum is out of bounds (or not a number) is the tile's
      // maximum taken, the reference raised and the tile exponentiated again.
      bool redo = false;
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) redo |= __any(!(lsum[qb] < kMaxTileSum));
      if (__builtin_expect(redo, 0)) {
        softmax_max(s_cur);
        softmax(s_cur);
      } else {
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) l_run[qb] += lsum[qb];
      }
      raw = !nxt_full;
    } else {
      if (nxt) {
        multiply_qk(tile_nxt, k_nxt, s_nxt);
      } else {
#pragma unroll
        for (int i = 0; i < NL; ++i) issue_load(i);
      }
      if (cur) {
        if (!pending) softmax_max(s_cur);
        softmax(s_cur);
        anchored |= cur_full;  // a tile every row sees gives every row a reference
      }
    }
    pending = false;
    if (__builtin_expect(cur, 1)) {
      apply_rescale();
      __builtin_amdgcn_s_setprio(kPrioDense);
      multiply_pv(v_cur);
      __builtin_amdgcn_s_setprio(kPrioControl);
    }
    cur_full = nxt_full;
    tile_cur = tile_nxt;
    tile_nxt = cursor.tile;
    v_off = cursor.off;
    cursor_next();
  };
  if (n_tiles > first_tile) {
    cursor.seek(runs, first_tile, tiles_per_block, slot_lds, kv_table, p.kv_slot_stride, tile_stride);
    tile_cur = cursor.tile;
    fill_k = k_at0;
    fill_v = v_at0;
    fill_k_off = fill_v_off = cursor.off;
#pragma unroll
    for (int i = 0; i < NL; ++i) issue_load(i);
    cursor_next();
    tile_nxt = cursor.tile;
    v_off = cursor.off;
    fill_k = k_at1;
    fill_k_off = cursor.off;
#pragma unroll
    for (int i = 0; i < KTile::LPW; ++i) issue_load(i);
    cursor_next();
#pragma unroll
    for (int qb = 0; qb < QB; ++qb)
      if (rng[qb].len0 == 0 && rng[qb].len1 == 0) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) qreg[qb][ks] = u32x4{0, 0, 0, 0};
      }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    cur_full = tile_is_full(tile_cur);
    if (wave_sees(tile_cur)) {
      multiply_qk(tile_cur, k_lds0, s_a);
      softmax_max(s_a);
      pending = true;
      // (with a causal mask every row sees the first tile's first key, though not all of the tile)
      bool without = false;
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) without |= m_run[qb] == -INFINITY && (rng[qb].len0 | rng[qb].len1) != 0;
      anchored = __builtin_amdgcn_readfirstlane(!__any(without)) != 0;
    }
    for (int j = first_tile; j < n_tiles; j += 2) {
      iteration(j, s_a, s_b, k_lds1, k_at0, v_lds0, v_at1);
      if (__builtin_expect(j + 1 >= n_tiles, 0)) break;
      iteration(j + 1, s_b, s_a, k_lds0, k_at1, v_lds1, v_at0);
    }
    wait_loads();  // the fetches past the end of the list must land before the workgroup's LDS is released
  }

  // ---- epilogue ------------------------------------------------------------------
#pragma unroll
  for (int qb = 0; qb < QB; ++qb)
    if (rng[qb].len0 == 0 && rng[qb].len1 == 0) {  // (see above)
      m_run[qb] = -INFINITY;
      l_run[qb] = 0.0f;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) o_acc[qb][dt][i] = 0.0f;
    }
  if constexpr (PARTS) {
    if (partial >= 0) {
      // 32 queries' 16-byte pieces side by side: whole 512-byte runs per store and half-wave
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        const float l_tot = halves_sum(l_run[qb]);
        const int64_t block = ((int64_t)partial * p.n_heads_q + head) * (p.q_tiles_per_row * (BM / 32)) +
                              qt * (BM / 32) + w * QB + qb;
        f32x4* dst = reinterpret_cast<f32x4*>(p.partial_out) + block * (32 * D / 4) + h * 32 + c;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const f32x4 o4 = {o_acc[qb][dt][4 * g], o_acc[qb][dt][4 * g + 1], o_acc[qb][dt][4 * g + 2], o_acc[qb][dt][4 * g + 3]};
            dst[(dt * 4 + g) * 64] = o4;
          }
        if (h == 0) {
          p.partial_sums[(block * 32 + c) * 2] = m_run[qb];
          p.partial_sums[(block * 32 + c) * 2 + 1] = l_tot;
        }
      }
      return;
    }
  }
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const float l_tot = halves_sum(l_run[qb]);
    if (!q_valid[qb]) continue;
    const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
    uint16_t* op = reinterpret_cast<uint16_t*>(p.out) +
                   (int64_t)o_slot * p.out_slot_stride + (int64_t)q_local[qb] * q_row_stride + (int64_t)head * D + 4 * h;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        u32x2 pk = {pack2<DTYPE>(o_acc[qb][dt][4 * g] * inv, o_acc[qb][dt][4 * g + 1] * inv),
                    pack2<DTYPE>(o_acc[qb][dt][4 * g + 2] * inv, o_acc[qb][dt][4 * g + 3] * inv)};
        *reinterpret_cast<u32x2*>(op + dt * 32 + 8 * g) = pk;
      }
    if (h == 0) {
      const float lse = l_tot > 0.0f ? (m_run[qb] + log2f(l_tot)) * kLn2 : p.empty_lse;
      p.lse[(int64_t)head * p.lse_head_stride + (int64_t)o_slot * p.lse_slot_stride + q_local[qb]] = lse;
    }
  }
}

// The kernel is persistent: the launch has (at most) as many workgroups as the device holds at
// once and each keeps taking the next work item until none is left (ItemQueue).  A grid of one
// workgroup per item loses a tenth of the device to dispatch: workgroup ids are dealt to the 8
// XCDs strictly in turn, so an XCD with a free slot waits until every XCD before it in the turn
// has taken its workgroup (13 us between two workgroups of a CU slot on average, against 100 us
// of work), and the last, unevenly long items leave slots empty at the end.  Rows come longest first;
// the counters are zeroed by a one-wave kernel on the stream just before.  A launch whose items all
// fit on the device at once needs no queue and no such kernel.
// But the queue costs that kernel, 4-5 us, and a launch of little work per slot wins less by it: dcp_attn_fwd_items
// takes a workgroup per item where it is told to (the caller knows the rows' lengths; figures at
// one_workgroup_each of items.py).
template <int DTYPE, int D, int QB, FwdItems ITEMS>
__global__ __launch_bounds__(kFwdThreads, QB == 1 ? 2 : 1) void attn_fwd_kernel(const AttnFwdParams p) {
  __shared__ int ticket_lds;
  int item = 0;
  {
    KernArgs<AttnFwdParams>& args = fresh_kernel_args<AttnFwdParams>();
    item = first_item({args.tickets, args.ticket_stride, args.n_items, args.xcd_group});
  }
  while (true) {
    KernArgs<AttnFwdParams>& args = fresh_kernel_args<AttnFwdParams>();
    if (item < 0) item = next_item({args.tickets, args.ticket_stride, args.n_items, args.xcd_group}, &ticket_lds);
    if (item < 0) break;
    attn_fwd_item<DTYPE, D, QB, ITEMS>(args, item);
    item = -1;
  }
}

__global__ void attn_fwd_reset_tickets_kernel(int* tickets, int stride) {
  if (threadIdx.x < kNumXcd) tickets[threadIdx.x * stride] = 0;
}

// Adds up the parts of the split rows: out = sum_i 2^(m_i - m) O_i / sum_i 2^(m_i - m) l_i, rounded once.
// A workgroup takes 32 queries of one (row, head); a lane one query and D / 32 groups of four dims, so
// that its reads of the partials are whole runs and a query's weights are the same for all of them.
struct FwdSplit {
  int row, n_parts, first_partial, unused;
};
constexpr int kMergePartsThreads = 256;
template <int DTYPE, int D>
__global__ __launch_bounds__(kMergePartsThreads) void attn_fwd_merge_parts_kernel(const AttnFwdParams p, const FwdSplit* splits) {
  const int blocks_per_row = p.q_tiles_per_row * 4;
  const int qb = blockIdx.x % blocks_per_row;
  const int head = blockIdx.x / blocks_per_row % p.n_heads_q;
  const FwdSplit split = splits[blockIdx.x / blocks_per_row / p.n_heads_q];
  const int q_begin = p.cu_seqlens_q[split.row];
  const int c = threadIdx.x & 31, q_local = qb * 32 + c;
  if (q_local >= p.cu_seqlens_q[split.row + 1] - q_begin) return;
  const int64_t block0 = ((int64_t)split.first_partial * p.n_heads_q + head) * blocks_per_row + qb;
  const int64_t block_step = (int64_t)p.n_heads_q * blocks_per_row;
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  const f32x2* sums = reinterpret_cast<const f32x2*>(p.partial_sums) + block0 * 32 + c;
  float m = -INFINITY;
  for (int i = 0; i < split.n_parts; ++i) m = fmaxf(m, sums[i * block_step * 32][0]);
  const float m_use = m == -INFINITY ? 0.0f : m;
  constexpr int PER = 32 * D / 4 / kMergePartsThreads;
  f32x4 acc[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) acc[k] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  float l = 0.0f;
  const f32x4* src = reinterpret_cast<const f32x4*>(p.partial_out) + block0 * (32 * D / 4) + threadIdx.x;
  for (int i = 0; i < split.n_parts; ++i) {
    const f32x2 ml = sums[i * block_step * 32];
    const float weight = fast_exp2(ml[0] - m_use);  // a part without a visible key: exp2(-inf) = 0, and its O is 0
    l += weight * ml[1];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const f32x4 o4 = src[i * block_step * (32 * D / 4) + k * kMergePartsThreads];
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[k][r] += weight * o4[r];
    }
  }
  const float inv = l > 0.0f ? 1.0f / l : 0.0f;
  const int o_slot = p.out_block_table[split.row];
  uint16_t* out = reinterpret_cast<uint16_t*>(p.out) + (int64_t)o_slot * p.out_slot_stride +
                  ((int64_t)q_local * p.n_heads_q + head) * D + 4 * (threadIdx.x >> 5);
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const u32x2 pk = {pack2<DTYPE>(acc[k][0] * inv, acc[k][1] * inv), pack2<DTYPE>(acc[k][2] * inv, acc[k][3] * inv)};
    *reinterpret_cast<u32x2*>(out + k * (kMergePartsThreads / 8)) = pk;
  }
  if (threadIdx.x < 32)
    p.lse[(int64_t)head * p.lse_head_stride + (int64_t)o_slot * p.lse_slot_stride + q_local] =
        l > 0.0f ? (m + log2f(l)) * kLn2 : p.empty_lse;
}

}  // namespace dcp

using namespace dcp;

extern "C" size_t dcp_attn_fwd_workspace_bytes(void) { return kNumXcd * kFwdTicketStride * sizeof(int32_t); }

extern "C" int dcp_attn_fwd(const void* q, const void* k, const void* v, void* out, float* lse,
                            const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_kv,
                            const int32_t* attn_range, int n_ranges, const int32_t* q_block_table,
                            const int32_t* kv_block_table, const int32_t* out_block_table,
                            const int32_t* row_order, int batch, int max_kv_blocks, int total_q,
                            int block_size, int n_heads_q, int n_heads_kv, int head_dim,
                            int64_t kv_slot_stride, int64_t kv_token_stride, int n_out_slots,
                            float softmax_scale, int dtype, void* workspace, size_t workspace_bytes,
                            void* stream) {
  DCP_RECORDED(dcp_attn_fwd(q, k, v, out, lse, cu_seqlens_q, cu_seqlens_kv, attn_range, n_ranges, q_block_table,
      kv_block_table, out_block_table, row_order, batch, max_kv_blocks, total_q, block_size, n_heads_q, n_heads_kv,
      head_dim, kv_slot_stride, kv_token_stride, n_out_slots, softmax_scale, dtype, workspace, workspace_bytes,
      stream));
  DCP_REQUIRE(batch == 0 || n_out_slots > 0, "attn_fwd: empty block tables");
  const int64_t slot = (int64_t)block_size * n_heads_q * head_dim;
  return dcp_attn_fwd_strided(q, k, v, out, lse, cu_seqlens_q, cu_seqlens_kv, attn_range, n_ranges, q_block_table,
                              kv_block_table, out_block_table, row_order, batch, max_kv_blocks, total_q, block_size,
                              n_heads_q, n_heads_kv, head_dim, kv_slot_stride, kv_token_stride, slot, slot,
                              (int64_t)n_out_slots * block_size, block_size, 0, softmax_scale, dtype, workspace,
                              workspace_bytes, stream);
}

// What dcp_attn_fwd_parts adds to dcp_attn_fwd_strided.
struct FwdParts {
  const int32_t* parts = nullptr;
  int n_entries = 0;
  const int32_t* splits = nullptr;
  int n_splits = 0, n_partials = 0;
  float* partials = nullptr;
  size_t partials_bytes = 0;
  const int32_t* tiles = nullptr;  // dcp_attn_fwd_items: n_entries of them instead of parts
  bool one_each = false;           // a workgroup per work item, whether the device holds them all at once or not
};

static int attn_fwd(const void* q, const void* k, const void* v, void* out, float* lse, const int32_t* cu_seqlens_q,
                    const int32_t* cu_seqlens_kv, const int32_t* attn_range, int n_ranges, const int32_t* q_block_table,
                    const int32_t* kv_block_table, const int32_t* out_block_table, const int32_t* row_order, int batch,
                    int max_kv_blocks, int total_q, int block_size, int n_heads_q, int n_heads_kv, int head_dim,
                    int64_t kv_slot_stride, int64_t kv_token_stride, int64_t q_slot_stride, int64_t out_slot_stride,
                    int64_t lse_head_stride, int64_t lse_slot_stride, int merged_form, float softmax_scale, int dtype,
                    void* workspace, size_t workspace_bytes, const FwdParts& in_parts, void* stream) {
  if (dtype != DCP_DTYPE_BF16 && dtype != DCP_DTYPE_FP16)
    return fail(DCP_ERR_UNSUPPORTED, "attn_fwd: dtype %d unsupported (bf16 and fp16 only)", dtype);
  if (head_dim != 64 && head_dim != 128)
    return fail(DCP_ERR_UNSUPPORTED, "attn_fwd: head_dim %d unsupported (64 or 128)", head_dim);
  DCP_REQUIRE(n_ranges == 1 || n_ranges == 2, "attn_fwd: n_ranges must be 1 or 2, got %d", n_ranges);
  DCP_REQUIRE(batch >= 0 && total_q >= 0, "attn_fwd: negative size");
  DCP_REQUIRE(softmax_scale > 0.0f, "attn_fwd: softmax_scale must be positive");
  if (batch == 0) return DCP_OK;
  DCP_REQUIRE(block_size > 0 && block_size % kFwdBN == 0,
              "attn_fwd: block_size %d must be a positive multiple of %d", block_size, kFwdBN);
  DCP_REQUIRE(n_heads_q > 0 && n_heads_kv > 0 && n_heads_q % n_heads_kv == 0,
              "attn_fwd: n_heads_q %d must be a multiple of n_heads_kv %d", n_heads_q, n_heads_kv);
  DCP_REQUIRE(max_kv_blocks > 0, "attn_fwd: empty block tables");
  DCP_REQUIRE(kv_token_stride % 8 == 0 && kv_slot_stride % 8 == 0 && q_slot_stride % 8 == 0 && out_slot_stride % 4 == 0,
              "attn_fwd: q, k, v strides must be multiples of 8 elements (out: 4)");
  DCP_REQUIRE(q_slot_stride > 0 && out_slot_stride > 0 && lse_head_stride > 0 && lse_slot_stride > 0,
              "attn_fwd: table strides must be positive");
  DCP_REQUIRE(q && k && v && out && lse && cu_seqlens_q && cu_seqlens_kv && attn_range &&
                  q_block_table && kv_block_table && out_block_table,
              "attn_fwd: null argument");
  DCP_REQUIRE(((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) |
                reinterpret_cast<uintptr_t>(v) | reinterpret_cast<uintptr_t>(out)) & 15) == 0,
              "attn_fwd: q/k/v/out must be 16-byte aligned");
  DCP_REQUIRE(workspace && (reinterpret_cast<uintptr_t>(workspace) & 3) == 0 &&
                  workspace_bytes >= DCP_ATTN_FWD_MIN_WORKSPACE_BYTES,
              "attn_fwd: workspace of %zu bytes is missing or smaller than the %d needed", workspace_bytes,
              DCP_ATTN_FWD_MIN_WORKSPACE_BYTES);
  if (in_parts.tiles != nullptr)
    DCP_REQUIRE(in_parts.n_entries > 0 && (reinterpret_cast<uintptr_t>(in_parts.tiles) & 15) == 0, "attn_fwd: no items, or not 16-byte aligned");
  if (in_parts.parts != nullptr || in_parts.tiles != nullptr) {
    DCP_REQUIRE((in_parts.tiles != nullptr || in_parts.n_entries >= batch) && in_parts.n_splits >= 0 && in_parts.n_splits <= batch && in_parts.n_partials >= 2 * in_parts.n_splits,
                "attn_fwd: %d entries and %d partials of %d split rows do not fit %d rows", in_parts.n_entries, in_parts.n_partials,
                in_parts.n_splits, batch);
    const size_t queries = (size_t)((block_size + 127) / 128) * 128 * n_heads_q * in_parts.n_partials;
    DCP_REQUIRE(in_parts.n_splits == 0 || (in_parts.splits && in_parts.partials && (reinterpret_cast<uintptr_t>(in_parts.partials) & 15) == 0 &&
                                           in_parts.partials_bytes >= queries * (head_dim + 2) * sizeof(float)),
                "attn_fwd: the partials are missing, not 16-byte aligned or smaller than the %zu bytes needed",
                queries * (head_dim + 2) * sizeof(float));
  }
  AttnFwdParams p;
  p.q = q;
  p.k = k;
  p.v = v;
  p.out = out;
  p.lse = lse;
  p.cu_seqlens_q = cu_seqlens_q;
  p.cu_seqlens_kv = cu_seqlens_kv;
  p.attn_range = attn_range;
  p.q_block_table = q_block_table;
  p.kv_block_table = kv_block_table;
  p.out_block_table = out_block_table;
  p.row_order = row_order;
  p.n_ranges = n_ranges;
  p.batch = batch;
  p.max_kv_blocks = max_kv_blocks;
  p.total_q = total_q;
  p.block_size = block_size;
  p.n_heads_q = n_heads_q;
  p.n_heads_kv = n_heads_kv;
  p.kv_slot_stride = kv_slot_stride;
  p.kv_token_stride = kv_token_stride;
  p.n_out_slots = 0;
  p.q_slot_stride = q_slot_stride;
  p.out_slot_stride = out_slot_stride;
  p.lse_head_stride = lse_head_stride;
  p.lse_slot_stride = lse_slot_stride;
  p.empty_lse = merged_form ? -1.0f : INFINITY;
  // One 32-row query block per wave.  (Two per wave do not pay with this compiler: it cannot
  // keep the O^T accumulators in the AGPR half of the register file without copies and spills.)
  const int bm = 128;
  p.q_tiles_per_row = (block_size + bm - 1) / bm;
  p.scale_log2 = softmax_scale * kLog2e;
  p.tiles = reinterpret_cast<const FwdTile*>(in_parts.tiles);
  p.n_items = (int64_t)(in_parts.parts || p.tiles ? in_parts.n_entries : batch) * n_heads_q * (p.tiles ? 1 : p.q_tiles_per_row);
  p.parts = reinterpret_cast<const FwdPart*>(in_parts.parts);
  p.partial_out = in_parts.partials;
  p.partial_sums = in_parts.partials + (size_t)in_parts.n_partials * n_heads_q * p.q_tiles_per_row * bm * head_dim;
  p.xcd_group = (p.tiles ? 1 : p.q_tiles_per_row) * (n_heads_q / n_heads_kv);
  DCP_REQUIRE(p.n_items < ((int64_t)1 << 31), "attn_fwd: too many work items");
  // as many workgroups as the device holds at once (two per CU), a multiple of the XCD count
  const int64_t n_slots = xcd_grid_size(2 * (int64_t)device_cu_count(), 1);
  const int64_t n_wg = in_parts.one_each ? xcd_grid_size(p.n_items, 1) : std::min<int64_t>(xcd_grid_size(p.n_items, 1), n_slots);
  p.tickets = p.n_items > n_wg ? reinterpret_cast<int*>(workspace) : nullptr;
  // (items that all have a CU to themselves start at once, in whatever order: a trip to memory less)
  if (p.n_items <= device_cu_count()) p.row_order = nullptr;
  p.ticket_stride = workspace_bytes >= dcp_attn_fwd_workspace_bytes() ? kFwdTicketStride : kFwdTicketStrideMin;
  dim3 grid((unsigned)n_wg), block(kFwdThreads);
  if (p.tickets) hipLaunchKernelGGL(attn_fwd_reset_tickets_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream, p.tickets, p.ticket_stride);
  auto launch = [&](auto kernel) {
    KernelTimer timer("attn_fwd_kernel", stream);
    hipLaunchKernelGGL(kernel, grid, block, 0, (hipStream_t)stream, p);
  };
#define DCP_FWD(DT, HD) (p.tiles   ? launch(attn_fwd_kernel<DT, HD, 1, kFwdTiles>)   \
                         : p.parts ? launch(attn_fwd_kernel<DT, HD, 1, kFwdParts>) \
                                   : launch(attn_fwd_kernel<DT, HD, 1, kFwdRows>))
  if (dtype == DCP_DTYPE_BF16) {
    if (head_dim == 128) DCP_FWD(DCP_DTYPE_BF16, 128);
    else DCP_FWD(DCP_DTYPE_BF16, 64);
  } else {
    if (head_dim == 128) DCP_FWD(DCP_DTYPE_FP16, 128);
    else DCP_FWD(DCP_DTYPE_FP16, 64);
  }
#undef DCP_FWD
  const int status = check_launch("attn_fwd_kernel");
  if (status != DCP_OK || in_parts.n_splits == 0) return status;
  const int64_t merges = (int64_t)in_parts.n_splits * n_heads_q * p.q_tiles_per_row * (bm / 32);
  DCP_REQUIRE(merges < ((int64_t)1 << 31), "attn_fwd: too many split rows");
  auto merge = [&](auto kernel) {
    KernelTimer timer("attn_fwd_merge_parts_kernel", stream);
    hipLaunchKernelGGL(kernel, dim3((unsigned)merges), dim3(kMergePartsThreads), 0, (hipStream_t)stream, p,
                       reinterpret_cast<const FwdSplit*>(in_parts.splits));
  };
  if (dtype == DCP_DTYPE_BF16) {
    if (head_dim == 128) merge(attn_fwd_merge_parts_kernel<DCP_DTYPE_BF16, 128>);
    else merge(attn_fwd_merge_parts_kernel<DCP_DTYPE_BF16, 64>);
  } else {
    if (head_dim == 128) merge(attn_fwd_merge_parts_kernel<DCP_DTYPE_FP16, 128>);
    else merge(attn_fwd_merge_parts_kernel<DCP_DTYPE_FP16, 64>);
  }
  return check_launch("attn_fwd_merge_parts_kernel");
}

extern "C" int dcp_attn_fwd_strided(const void* q, const void* k, const void* v, void* out, float* lse,
                                    const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_kv,
                                    const int32_t* attn_range, int n_ranges, const int32_t* q_block_table,
                                    const int32_t* kv_block_table, const int32_t* out_block_table,
                                    const int32_t* row_order, int batch, int max_kv_blocks, int total_q,
                                    int block_size, int n_heads_q, int n_heads_kv, int head_dim,
                                    int64_t kv_slot_stride, int64_t kv_token_stride, int64_t q_slot_stride,
                                    int64_t out_slot_stride, int64_t lse_head_stride, int64_t lse_slot_stride,
                                    int merged_form, float softmax_scale, int dtype, void* workspace,
                                    size_t workspace_bytes, void* stream) {
  DCP_RECORDED(dcp_attn_fwd_strided(q, k, v, out, lse, cu_seqlens_q, cu_seqlens_kv, attn_range, n_ranges,
      q_block_table, kv_block_table, out_block_table, row_order, batch, max_kv_blocks, total_q, block_size, n_heads_q,
      n_heads_kv, head_dim, kv_slot_stride, kv_token_stride, q_slot_stride, out_slot_stride, lse_head_stride,
      lse_slot_stride, merged_form, softmax_scale, dtype, workspace, workspace_bytes, stream));
  return attn_fwd(q, k, v, out, lse, cu_seqlens_q, cu_seqlens_kv, attn_range, n_ranges, q_block_table, kv_block_table, out_block_table,
                  row_order, batch, max_kv_blocks, total_q, block_size, n_heads_q, n_heads_kv, head_dim, kv_slot_stride, kv_token_stride,
                  q_slot_stride, out_slot_stride, lse_head_stride, lse_slot_stride, merged_form, softmax_scale, dtype, workspace,
                  workspace_bytes, FwdParts{}, stream);
}

extern "C" int dcp_attn_fwd_parts(const void* q, const void* k, const void* v, void* out, float* lse, const int32_t* cu_seqlens_q,
                    const int32_t* cu_seqlens_kv, const int32_t* attn_range, int n_ranges, const int32_t* q_block_table,
                    const int32_t* kv_block_table, const int32_t* out_block_table, const int32_t* row_order, int batch,
                    int max_kv_blocks, int total_q, int block_size, int n_heads_q, int n_heads_kv, int head_dim,
                    int64_t kv_slot_stride, int64_t kv_token_stride, int64_t q_slot_stride, int64_t out_slot_stride,
                    int64_t lse_head_stride, int64_t lse_slot_stride, int merged_form, float softmax_scale, int dtype,
                    void* workspace, size_t workspace_bytes, const int32_t* parts, int n_entries, const int32_t* splits,
                    int n_splits, int n_partials, void* partials, size_t partials_bytes, void* stream) {
  DCP_RECORDED(dcp_attn_fwd_parts(q, k, v, out, lse, cu_seqlens_q, cu_seqlens_kv, attn_range, n_ranges, q_block_table, kv_block_table,
      out_block_table, row_order, batch, max_kv_blocks, total_q, block_size, n_heads_q, n_heads_kv, head_dim, kv_slot_stride,
      kv_token_stride, q_slot_stride, out_slot_stride, lse_head_stride, lse_slot_stride, merged_form, softmax_scale, dtype, workspace,
      workspace_bytes, parts, n_entries, splits, n_splits, n_partials, partials, partials_bytes, stream));
  DCP_REQUIRE(parts != nullptr, "attn_fwd: no table of parts");
  return attn_fwd(q, k, v, out, lse, cu_seqlens_q, cu_seqlens_kv, attn_range, n_ranges, q_block_table, kv_block_table, out_block_table,
                  row_order, batch, max_kv_blocks, total_q, block_size, n_heads_q, n_heads_kv, head_dim, kv_slot_stride, kv_token_stride,
                  q_slot_stride, out_slot_stride, lse_head_stride, lse_slot_stride, merged_form, softmax_scale, dtype, workspace,
                  workspace_bytes, FwdParts{parts, n_entries, splits, n_splits, n_partials, reinterpret_cast<float*>(partials), partials_bytes}, stream);
}


extern "C" int dcp_attn_fwd_items(const void* q, const void* k, const void* v, void* out, float* lse, const int32_t* cu_seqlens_q,
                    const int32_t* cu_seqlens_kv, const int32_t* attn_range, int n_ranges, const int32_t* q_block_table,
                    const int32_t* kv_block_table, const int32_t* out_block_table, const int32_t* row_order, int batch,
                    int max_kv_blocks, int total_q, int block_size, int n_heads_q, int n_heads_kv, int head_dim,
                    int64_t kv_slot_stride, int64_t kv_token_stride, int64_t q_slot_stride, int64_t out_slot_stride,
                    int64_t lse_head_stride, int64_t lse_slot_stride, int merged_form, float softmax_scale, int dtype,
                    void* workspace, size_t workspace_bytes, const int32_t* items, int n_items, int one_each, const int32_t* splits,
                    int n_splits, int n_partials, void* partials, size_t partials_bytes, void* stream) {
  DCP_RECORDED(dcp_attn_fwd_items(q, k, v, out, lse, cu_seqlens_q, cu_seqlens_kv, attn_range, n_ranges, q_block_table, kv_block_table,
      out_block_table, row_order, batch, max_kv_blocks, total_q, block_size, n_heads_q, n_heads_kv, head_dim, kv_slot_stride,
      kv_token_stride, q_slot_stride, out_slot_stride, lse_head_stride, lse_slot_stride, merged_form, softmax_scale, dtype, workspace,
      workspace_bytes, items, n_items, one_each, splits, n_splits, n_partials, partials, partials_bytes, stream));
  DCP_REQUIRE(items != nullptr || (n_items == 0 && n_splits == 0), "attn_fwd: %d items and %d split rows, but no table of items", n_items, n_splits);
  return attn_fwd(q, k, v, out, lse, cu_seqlens_q, cu_seqlens_kv, attn_range, n_ranges, q_block_table, kv_block_table, out_block_table,
                  row_order, batch, max_kv_blocks, total_q, block_size, n_heads_q, n_heads_kv, head_dim, kv_slot_stride, kv_token_stride,
                  q_slot_stride, out_slot_stride, lse_head_stride, lse_slot_stride, merged_form, softmax_scale, dtype, workspace,
                  workspace_bytes, FwdParts{nullptr, n_items, splits, n_splits, n_partials, reinterpret_cast<float*>(partials), partials_bytes, items, one_each != 0}, stream);
}

