// The plan of a prefill launch in plain arithmetic, for the launching code, the
// kernels and host compilers alike: which kernel it takes, how its query
// tiles, key splits and ranges of equal work are cut.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

#ifdef __HIPCC__
#define VK_HD __host__ __device__ __forceinline__
#else
#define VK_HD inline
#endif

namespace vk {

template <typename T>
VK_HD constexpr T pf_min(T a, T b) { return a < b ? a : b; }
template <typename T>
VK_HD constexpr T pf_max(T a, T b) { return a > b ? a : b; }

// The keys [lo, hi] that the query at position p sees.
VK_HD void key_range(int32_t p, int32_t len_k, int32_t wl, int32_t wr, int32_t& lo, int32_t& hi) {
  lo = wl >= 0 ? pf_max(0, p - wl) : 0;
  hi = wr >= 0 ? pf_min(len_k - 1, p + wr) : len_k - 1;
}

// How a launch's items are ordered (prefill_item says why).
constexpr uint32_t kLine = 128;  // bytes of an L2 line
constexpr uint32_t kPfSortSeqs = 64;
constexpr uint32_t kPfSortItems = 256;  // one per CU
constexpr uint32_t kPfFewHeads = 2;
constexpr uint32_t kPfClassItems = 1024;
constexpr uint32_t kPfSortRounds = 3;
constexpr uint32_t kPfPartsRounds = 4;
constexpr uint32_t kPfShortKeys = 128;
constexpr uint32_t kPfShortTileKeys = 64;
enum PfOrder : uint32_t {
  kPfListOrder,  // as the list has them
  kPfListParts,  // the same, in contiguous parts per XCD
  kPfSequences,  // sequences from the longest context to the shortest
  kPfParts,      // the same; equal contexts in contiguous parts per XCD
  kPfByClass,    // as kPfParts, or by classes of work
};
// `keys`: the most that an item walks; `row`: bytes of a head's row; `slots`:
// workgroups the GPU runs at once. f32 launches keep the list's order with one
// tile per sequence and walk several: their steps take 2.5 times as long, and
// parts of the list end later (10 fresh sequences of 9-63 tokens, 64 q / 8 kv
// heads: 15.9 us walked, 23.7 in parts; 40 of 8-128, 16 q / 8 kv heads: 33.9 as
// listed, 38.5 in parts).
inline PfOrder prefill_order(uint32_t n_seqs, uint32_t kvh, uint32_t qtiles, uint64_t items,
                             uint32_t n_split, uint64_t keys, uint32_t row, uint32_t slots,
                             bool f32) {
  const uint64_t wgs = items * n_split;
  if (n_seqs <= 1) return kPfListOrder;
  if (qtiles <= 1) {
    if (n_split > 1 || f32) return kPfListOrder;
    if (wgs <= slots) return kPfListParts;
    if (keys <= kPfShortKeys)
      return row % kLine || wgs <= kPfPartsRounds * (uint64_t)slots ? kPfListParts : kPfListOrder;
    return n_seqs <= kPfSortSeqs && wgs <= kPfSortRounds * (uint64_t)slots ? kPfSequences
                                                                           : kPfListOrder;
  }
  if (keys <= kPfShortTileKeys && n_split == 1 && !f32) return kPfListParts;
  if (n_seqs > kPfSortSeqs || wgs <= kPfSortItems) return kPfListOrder;
  if (kvh > kPfFewHeads || n_split > 1) return kPfSequences;
  return items <= kPfClassItems ? kPfByClass : kPfParts;
}

// Workgroup -> work item. The hardware deals workgroups round-robin to the
// 8 XCDs (linear id % 8); each XCD here gets a contiguous range of work
// items, so the q-tiles of one (sequence, kv head), which read the same K/V,
// run at the same time under one L2. (deal_remap: over `parts` XCDs, of items
// dealt to them in turn.)
VK_HD uint32_t deal_remap(uint32_t lin, uint32_t n, uint32_t parts) {
  const uint32_t x = lin % parts, i = lin / parts;
  const uint32_t per = n / parts, extra = n % parts;  // part x gets per + (x < extra)
  return x * per + pf_min(x, extra) + i;
}
VK_HD uint32_t xcd_remap(uint32_t lin, uint32_t n) {
  constexpr uint32_t kXcds = 8;
  return deal_remap(lin, n, kXcds);
}

// Item i of a launch in kPfListParts: tile fastest, then kv head, then list
// entry li.
VK_HD void pf_list_part(uint32_t i, uint32_t n_seqs, uint32_t kvh, uint32_t qtiles, uint32_t& li,
                        uint32_t& kh, uint32_t& qt) {
  i = xcd_remap(i, n_seqs * qtiles * kvh);
  const uint32_t head = i / qtiles;
  qt = qtiles - 1 - (i - head * qtiles);
  li = head / kvh;
  kh = head - li * kvh;
}

// The most keys that an item walks, with at most max_q queries and max_k keys
// per sequence and the left window wl.
inline uint64_t prefill_keys(uint32_t max_q, uint32_t max_k, int32_t wl) {
  return wl >= 0 ? std::min<uint64_t>(max_k, (uint64_t)wl + max_q) : max_k;
}

// The order of a launch's tiles by classes of work (kPfByClass): classes, the
// longest context over kPfClasses each, from the longest down; in a class the
// sequences from the longest context down, each from its last tile to its first.
// A tile has `step` keys less than the one after it. Returns the tiles of a
// sequence of `key` keys and nt tiles in classes 0 .. c.
constexpr uint32_t kPfClasses = 16;
VK_HD uint32_t pf_tiles_to_class(uint32_t c, uint32_t longest, uint32_t key, uint32_t nt,
                                 float per_step) {
  if (c + 1 >= kPfClasses) return nt;
  const uint32_t t = longest / kPfClasses * (kPfClasses - 1 - c);
  if (key <= t) return 0;
  return pf_min(nt, (uint32_t)((float)(key - t) * per_step) + 1);
}
// Whether a sequence's first tile has less than half of the longest's work: if
// none has, the tiles are one class.
VK_HD bool pf_short_tile(uint32_t longest, uint32_t key, uint32_t nt, uint32_t step) {
  return nt > 0 && (uint64_t)(nt - 1) * step + longest / 2 > key;
}

// Bytes of one (item, split) partial block of a prefill key split: (m, l)
// f32 per row, then o / l per row in f32 (the split adds no rounding before
// the merge).
VK_HD constexpr uint64_t pf_part_bytes(uint32_t rows, uint32_t d) {
  return (uint64_t)rows * (8 + 4 * d);
}

// ---- balanced ranges of a prefill launch ------------------------------------
//
// A launch whose query tiles do not fill the GPU's workgroup slots evenly
// (fewer tiles than slots, or a last round that is nearly empty, or tiles of
// very different lengths) is cut into ranges of equal work instead, one
// workgroup each: a range may start and end inside a tile and cover whole
// tiles between. The tiles' order is kv head, then list order, then each
// sequence from its last tile to its first; XCD x runs a contiguous eighth of
// the ranges, so the tiles that run together on an XCD share a kv head's K/V.
// A tile's work is counted in sixteenths of a 32-key step and falls by a
// constant from a sequence's last tile to its first (the causal mask; not at
// all with a window), so sums over tiles have a closed form; a piece's share
// of that count is then its share of the tile's real steps.
//
// The first piece of range r that is not a whole tile goes to partial slot
// 2 r if it starts the range, else to 2 r + 1. The range that starts a tile
// without ending it describes the tile (PfSplitTile), and the merge joins its
// piece with the following ranges' first pieces.
constexpr uint32_t kPfMinSteps = 8;     // per range, in launches of few steps
constexpr uint32_t kPfMaxRanges = 256;  // one per CU
// Of all tiles' counts, S: products up to S (kPfMaxRanges + 1) stay in 32 bits
// (pf_range_last's is the largest).
constexpr uint64_t kPfMaxCount = 0xFFFFFFFFull / (kPfMaxRanges + 1);

struct PfSplitTile {
  uint32_t valid, seq, qt, kh;
  uint32_t first_slot, last;  // partial slot of the first piece, the last range
  uint32_t pad[2];
};

// The step of `steps` at count u of c: 0 at 0, all of them at c, never falling
// between, the same wherever it is computed.
VK_HD uint32_t pf_step_at(uint32_t u, uint32_t c, uint32_t steps) {
  return u >= c ? steps : pf_min(steps, (uint32_t)((float)u * ((float)steps / (float)c)));
}

VK_HD uint32_t pf_tiles_sum(uint32_t c, uint32_t f, uint32_t n) {
  return n * c - f * (n * (n - 1) / 2);
}

// The plan's entry for one sequence: its tiles, the last tile's count, what
// each earlier one has less. `cap` bounds a tile's count: kPfMaxCount over the
// launch's tiles, so that no lengths take the sum past kPfMaxCount. It only
// binds for lengths past the host's max_seqlen_k, whose pieces are then
// shares of fewer, larger counts.
struct PfEntry {
  uint32_t seq, q0, len_q, len_k;
  uint32_t nt, c_last, fall;
  uint32_t pad;
};
VK_HD uint32_t pf_count_cap(uint32_t tiles) {
  return (uint32_t)kPfMaxCount / pf_max(tiles, 1u);
}
VK_HD void pf_entry_tiles(PfEntry& e, uint32_t group, uint32_t qtiles, uint32_t rows, int32_t wl,
                          int32_t wr, uint32_t cap) {
  e.nt = (uint32_t)pf_min(((uint64_t)e.len_q * group + rows - 1) / rows, (uint64_t)qtiles);
  // Steps of the last tile, from its first row's window to its last key.
  const int32_t offset = (int32_t)(e.len_k - e.len_q);
  int32_t klo, khi, unused;
  key_range(offset + (int32_t)((e.nt - 1) * rows / group), (int32_t)e.len_k, wl, wr, klo, unused);
  key_range(offset + (int32_t)e.len_q - 1, (int32_t)e.len_k, wl, wr, unused, khi);
  const uint32_t steps = khi >= klo ? (uint32_t)((khi >> 5) - (klo >> 5) + 1) : 1u;
  e.c_last = pf_min(16u * steps, cap);
  e.fall = wl < 0 && wr >= 0 && e.nt > 1
               ? pf_min(rows / (2 * group), (e.c_last - 16) / (e.nt - 1))
               : 0u;
}

// The ranges of a launch of S counts, range r's first count, and the range
// that holds the count before `end`.
VK_HD uint32_t pf_range_count(uint32_t S, uint32_t ranges) {
  return pf_min(ranges, (S + 16 * kPfMinSteps - 1) / (16 * kPfMinSteps));
}
VK_HD uint32_t pf_range_at(uint32_t S, uint32_t nr, uint32_t r) { return S * r / nr; }
VK_HD uint32_t pf_range_last(uint32_t end, uint32_t S, uint32_t nr) {
  return pf_min((end * nr + S - 1) / S, nr) - 1;
}

// Range r of nr: piece(u0, u1, c, slot) for each of its pieces, counts
// [u0, u1) of the c of the walk's tile (slot: its partial, or ~0u for a whole
// tile), next() between two pieces to move the walk to the next tile, and
// opens(slot, last) after the piece that starts a tile and leaves the rest of
// it to the ranges up to `last`. False if no piece does. The walk counts
// `total` per kv head.
template <typename Walk, typename Piece, typename Next, typename Opens>
VK_HD bool pf_walk_pieces(Walk& w, uint32_t S, uint32_t nr, uint32_t r, uint32_t kvh,
                          uint32_t total, Piece piece, Next next, Opens opens) {
  uint32_t at = pf_range_at(S, nr, r);
  const uint32_t end = pf_range_at(S, nr, r + 1);
  const uint32_t kh0 = at / total;
  uint32_t u0 = w.seek(kh0, at - kh0 * total);
  uint32_t slot = 2 * r;
  bool open = false;
  while (at < end && w.kh < kvh) {
    const uint32_t c = w.count(), u1 = pf_min(c, u0 + (end - at));
    piece(u0, u1, c, u0 == 0 && u1 == c ? ~0u : slot);
    if (u0 == 0 && u1 < c) {  // starts here, ends in a later range
      open = true;
      opens(slot, pf_range_last(at + c, S, nr));
    }
    at += u1 - u0;
    if (at >= end) break;
    u0 = 0, slot = 2 * r + 1;
    next();
  }
  return open;
}

// The split tiles lead the workspace, the partials follow.
constexpr size_t kPfRangeHead = kPfMaxRanges * sizeof(PfSplitTile);
struct PfRangePlan {
  uint32_t ranges;  // 0: none, the launch runs its tiles as they are
  size_t bytes;     // of workspace
};

// ---- the 16-bit kernel (attn_prefill.hip) -------------------------------------

constexpr int kPfWaves = 8;
constexpr int kPfThreads = 64 * kPfWaves;
// Row tiles (16 rows each) per wave, and workgroups per CU at head_dim 128.
// At head_dim 256 a wave holds one row tile (its O and Q^T fragments, 64 +
// 32 registers, beside a 64-register K tile: two tiles would not fit the
// 256 registers of a wave at two waves per SIMD), and the ring's six
// buffers take 96 KiB of LDS.
constexpr int kPfRowTiles = 2;
constexpr int kPfRowTiles256 = 1;
constexpr int kPfOcc = 1;
// head_dim 64 fits in 128 registers: two workgroups per CU (four waves per
// SIMD) measured 1% faster than one on a config-3-shaped batch (676-678
// against 669-673 TFLOP/s), and four row tiles per wave at one workgroup
// per CU no faster (817-819 against 823-824).
constexpr int kPfOcc64 = 2;

// Query rows of one prefill workgroup.
inline uint32_t pf_rows(uint32_t head_dim) {
  return 16 * (head_dim == 256 ? kPfRowTiles256 : kPfRowTiles) * kPfWaves;
}

// Key splits for a launch of `base` workgroups (query tiles x kv heads x
// sequences) over at most max_k keys: enough to give every CU of a 256-CU
// GPU a workgroup (one workgroup per CU is the kernel's occupancy at
// head_dim 128), each split keeping at least 8 steps of 32 keys, at most 64.
inline uint32_t pf_splits(uint64_t base, uint32_t max_k) {
  constexpr uint64_t kTarget = 256;
  if (base == 0 || base >= kTarget) return 1;
  uint64_t n = (kTarget + base - 1) / base;
  n = std::min<uint64_t>(n, std::max<uint32_t>(1u, max_k / 256));
  return (uint32_t)std::min<uint64_t>(n, 64);
}

inline uint64_t pf_split_bytes(uint64_t base, uint32_t n, uint32_t head_dim,
                               uint32_t rows = 16 * kPfRowTiles * kPfWaves) {
  return n > 1 ? base * n * pf_part_bytes(rows, head_dim) : 0;
}

// At most this much workspace for the partials (fewer splits beyond).
constexpr uint64_t kPfSplitMaxBytes = 256ull << 20;

inline uint32_t pf_splits_within(uint64_t base, uint32_t max_k, uint32_t head_dim,
                                 uint64_t bytes, uint32_t rows = 16 * kPfRowTiles * kPfWaves) {
  uint32_t n = pf_splits(base, max_k);
  while (n > 1 && pf_split_bytes(base, n, head_dim, rows) > std::min(bytes, kPfSplitMaxBytes))
    --n;
  return n;
}

// Ranges of equal work instead of tiles or their n_split equal shares, where
// what those leave idle is more than the ranges' plan, partials and merge
// cost (a partial is written and read once; ~ranges + tiles of them against
// n_split per tile). A workspace smaller than asked for holds fewer ranges,
// which leave CUs without one: they are priced as they are, against the shares
// that the same workspace allows (16 MiB hold 62: 5 x 512 bf16 queries over
// 4,096 keys 626 us in ranges, 244 in tiles; 3 x 512 over 8,192 751 / 242).
// Measured
// (us, tiles or shares / ranges; bf16, 32 q / 8 kv heads): 3 x 512 queries
// over 4,096 keys (192 tiles in 384 shares) 150 / 126, 5 x 512 (320 tiles)
// 242 / 197, 10 chunks of 20-100 over ~1,000 keys 79 / 53; f32, 40 chunks of
// 16 over ~1,000 keys 378 / 168; and where it says no: 4 x 512 (256 tiles) 135
// / 154, 1 x 512 (256 shares) 57 / 63, 1 x 1,500 fresh 53 / 73.
inline PfRangePlan pf_range_plan(uint64_t items, uint32_t max_q, uint32_t max_k, uint32_t slots,
                          uint32_t n_split, float step_us, uint64_t part_bytes,
                          size_t ws_bytes) {
  constexpr float kMergeUs = 4.f, kPlanUs = 5.f, kMarginUs = 3.f, kBytesPerUs = 5e6f;
  PfRangePlan p{0, 0};
  if (items == 0 || items >= 4 * slots) return p;
  // The steps there can be, kPfMinSteps to a range; two partials each.
  const uint64_t steps = items * (max_k / 32 + 2);
  if (16 * steps > kPfMaxCount) return p;
  const uint64_t all = std::min<uint64_t>(kPfMaxRanges, (steps + kPfMinSteps - 1) / kPfMinSteps);
  const uint64_t bytes = std::min<uint64_t>(ws_bytes, kPfSplitMaxBytes);
  if (bytes <= kPfRangeHead) return p;
  const uint64_t n = std::min<uint64_t>(all, (bytes - kPfRangeHead) / (2 * part_bytes));
  if (n < 2) return p;
  const uint64_t wgs = items * n_split, rounds = (wgs + slots - 1) / slots;
  const float steps_now = (float)(max_k - std::min(max_q / 2, max_k)) / 32.f / (float)n_split;
  const float now_us = (float)rounds * steps_now * step_us;
  // Time in ranges: all of them divide what the rounds do not leave idle (5%
  // at least: the host knows the longest sequence only); fewer, for want of
  // workspace, walk the launch's steps without a share of that (two workgroups
  // on a CU take as long for a step each as one for two).
  const float idle = std::max(1.f - (float)wgs / (float)(rounds * slots), 0.05f);
  const float ranges_us =
      n == all ? now_us * (1.f - idle)
               : (float)wgs * steps_now * step_us / (float)n * (float)kPfMaxRanges / (float)slots;
  const float part_us = 2.f * (float)part_bytes / kBytesPerUs;
  const float cost = kPlanUs + kMergeUs + part_us * (float)(kPfMaxRanges + items) -
                     (n_split > 1 ? kMergeUs + part_us * (float)wgs : 0.f);
  if (now_us - ranges_us < cost + kMarginUs) return p;
  p.ranges = (uint32_t)n;
  p.bytes = kPfRangeHead + n * 2 * part_bytes;
  return p;
}

// Launches that may run as ranges: at head_dim 256 the walk over a range's
// pieces does not fit beside the kernel's registers, and longer lists do not
// fit the plan; those split every item equally where they split.
inline bool pf_ranges_ok(uint32_t n_seqs, uint32_t head_dim) {
  return n_seqs <= kPfSortSeqs && head_dim <= 128;
}

// A full workgroup's 32-key step (head_dim 128; less below).
constexpr float kPfStepUs = 1.15f;
// Workgroups of the tiled prefill that the GPU runs at once.
inline uint32_t pf_slots(uint32_t head_dim) { return 256u * (head_dim == 64 ? kPfOcc64 : kPfOcc); }

// How a 16-bit prefill launch over n_seqs listed sequences runs: its tiles
// whole, in n_split equal shares or, with ranges.ranges, as ranges of equal
// work. As many splits as the workspace given holds (none without one); a
// deterministic call does not split, so its output does not depend on the
// workspace it is given (`split_ok` false).
struct PfRoute {
  uint32_t rows, qtiles;
  uint64_t items;  // query tiles x kv heads x sequences
  uint32_t n_split;
  PfRangePlan ranges;
};
inline PfRoute pf_route(uint32_t n_seqs, uint32_t kvh, uint32_t group, uint32_t max_q,
                        uint32_t max_k, uint32_t head_dim, bool split_ok, uint64_t ws_bytes) {
  PfRoute r{pf_rows(head_dim), 0, 0, 1, {0, 0}};
  r.qtiles = (uint32_t)(((uint64_t)max_q * group + r.rows - 1) / r.rows);
  r.items = (uint64_t)r.qtiles * kvh * n_seqs;
  if (!split_ok) return r;
  r.n_split = pf_splits_within(r.items, max_k, head_dim, ws_bytes, r.rows);
  if (pf_ranges_ok(n_seqs, head_dim))
    r.ranges = pf_range_plan(r.items, max_q, max_k, pf_slots(head_dim), r.n_split, kPfStepUs,
                             pf_part_bytes(r.rows, head_dim), ws_bytes);
  return r;
}

// ---- the f32 kernels (attn_prefill_f32.hip) ------------------------------------

constexpr int kPf32Waves = 8;
constexpr int kPf32Threads = 64 * kPf32Waves;
constexpr uint32_t x3_rows(int row_tiles) { return 16u * (uint32_t)row_tiles * kPf32Waves; }
constexpr int kPfF32RowTiles = 2;
constexpr float kX3StepUs = 2.82f;  // a workgroup's 32-key step with one row tile per wave

// The kernel of a launch of n_seqs sequences: rows per item and the items
// that fill a 256-CU GPU.
struct F32Plan {
  bool x3;
  uint32_t row_tiles;  // per wave
  uint32_t rows;       // per item: a workgroup's (x3, one per CU) or a wave's
  uint32_t qtiles;
  uint64_t items, target;
};
inline F32Plan f32_plan(uint32_t n_seqs, uint32_t kvh, uint32_t group, uint32_t max_q) {
  F32Plan p;
  const uint64_t all = (uint64_t)max_q * group;
  // The split kernel from 128 rows per kv head (a full item), and below that
  // for few kv heads: an item with few rows leaves most of its waves without
  // MFMAs, so where items fill the GPU four f32 waves per CU go further. Per
  // call, contexts around 1,000 (x3 against f32 MFMAs): 320 items (40
  // sequences, 8 kv heads) of 128 rows 500 against 735 us, of 64 rows 492
  // against 379; 64 items of 12 rows 39 against 54 us, of 64 rows 54 against
  // 60; 128 items of 64 rows 93 against 90, of 96 rows 114 against 180; 192
  // items of 13 rows 120 against 102.
  const uint64_t heads = (uint64_t)kvh * n_seqs;
  p.x3 = all >= x3_rows(1) || heads <= 64 || (heads <= 128 && all > 64);
  // Two row tiles per wave halve the LDS reads per MFMA: with enough items
  // (8 x 512 rows over 4,096 keys, 512 items: 1,148 against 1,457 us with
  // one row tile); below that the smaller items balance better (4 ragged
  // chunks of 360-429 over ~2,100 keys, 16 q / 8 kv heads: 192 against 223).
  auto items = [&](uint64_t rows) { return (all + rows - 1) / rows * kvh * n_seqs; };
  p.row_tiles = !p.x3 || items(x3_rows(2)) >= 256 ? 2 : 1;
  p.rows = p.x3 ? x3_rows(p.row_tiles) : 16 * kPfF32RowTiles;
  p.qtiles = (uint32_t)((all + p.rows - 1) / p.rows);
  p.items = items(p.rows);
  p.target = p.x3 ? 256 : 1024;
  return p;
}

// The same launch in ranges: one row tile per wave (with two, the walk over a
// range's pieces does not fit the registers beside the kernel's).
inline F32Plan f32_range_plan(uint32_t n_seqs, uint32_t kvh, uint32_t group, uint32_t max_q) {
  F32Plan p = f32_plan(n_seqs, kvh, group, max_q);
  const uint64_t all = (uint64_t)max_q * group;
  // (Ranges balance the items that few rows would leave half idle: 40
  // sequences, 8 kv heads, 64 rows over ~1,000 keys: 378 us with f32 MFMAs.)
  p.x3 = p.x3 || all > 32;
  // Its items fill the GPU one per CU, whatever kernel the tiles would take: with
  // f32_plan's 1,024 here, ranges were priced against shares that nothing ran
  // and the workspace asked for held none (40 chunks of 10-60 over ~300 keys, 8 q
  // / 4 kv heads at head_dim 80: 81.7 us in f32 MFMAs, 44.3 in ranges).
  if (p.x3) p.target = 256;
  p.row_tiles = 1;
  p.rows = x3_rows(1);
  p.qtiles = (uint32_t)((all + p.rows - 1) / p.rows);
  p.items = (uint64_t)p.qtiles * kvh * n_seqs;
  return p;
}

// Key splits over at most max_k keys: enough to fill the GPU, each split
// keeping at least 8 steps of 32 keys, at most 64; fewer when the workspace
// given holds fewer partials (at most 256 MiB of them).
inline uint32_t pf32_splits(const F32Plan& p, uint32_t max_k, uint32_t head_dim, uint64_t bytes) {
  if (p.items == 0 || p.items >= p.target) return 1;
  uint64_t n = std::min<uint64_t>((p.target + p.items - 1) / p.items,
                                  std::max<uint32_t>(1u, max_k / 256));
  n = std::min<uint64_t>(n, 64);
  const uint64_t cap = std::min<uint64_t>(bytes, 256ull << 20);
  while (n > 1 && p.items * n * pf_part_bytes(p.rows, head_dim) > cap) --n;
  return (uint32_t)n;
}

inline PfRangePlan f32_ranges(const F32Plan& p, uint32_t n_seqs, uint32_t max_q, uint32_t max_k,
                              uint32_t head_dim, uint64_t bytes) {
  if (!p.x3 || n_seqs > kPfSortSeqs) return PfRangePlan{0, 0};
  return pf_range_plan(p.items, max_q, max_k, 256, pf32_splits(p, max_k, head_dim, bytes),
                       kX3StepUs, pf_part_bytes(p.rows, head_dim), bytes);
}

// How an f32 prefill launch runs (as PfRoute): `plan`'s kernel and items.
struct F32Route {
  F32Plan plan;
  uint32_t n_split;
  PfRangePlan ranges;
};
inline F32Route f32_route(uint32_t n_seqs, uint32_t kvh, uint32_t group, uint32_t max_q,
                          uint32_t max_k, uint32_t head_dim, bool split_ok, uint64_t ws_bytes) {
  F32Route r{f32_range_plan(n_seqs, kvh, group, max_q), 1, {0, 0}};
  if (split_ok) r.ranges = f32_ranges(r.plan, n_seqs, max_q, max_k, head_dim, ws_bytes);
  if (!r.ranges.ranges) {
    r.plan = f32_plan(n_seqs, kvh, group, max_q);
    if (split_ok) r.n_split = pf32_splits(r.plan, max_k, head_dim, ws_bytes);
  }
  return r;
}

}  // namespace vk
