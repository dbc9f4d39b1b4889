// vapi_amd/csrc/prefill_plan.hpp for the Python tests: the routes of prefill
// launches, and the walk over a launch's ranges run on the CPU for every
// range, checked in 64-bit arithmetic.
#include "prefill_plan.hpp"

#include <vector>

using namespace vk;

extern "C" {

// out: items, query tiles, n_split, ranges, workspace bytes of the ranges,
// the items' order (PfOrder).
void plan_route16(uint32_t n_seqs, uint32_t kvh, uint32_t group, uint32_t max_q, uint32_t max_k,
                  uint32_t head_dim, uint32_t row_bytes, int split_ok, uint64_t ws_bytes,
                  uint64_t* out) {
  const PfRoute r = pf_route(n_seqs, kvh, group, max_q, max_k, head_dim, split_ok, ws_bytes);
  out[0] = r.items, out[1] = r.qtiles, out[2] = r.n_split, out[3] = r.ranges.ranges;
  out[4] = r.ranges.bytes;
  out[5] = prefill_order(n_seqs, kvh, r.qtiles, r.items, r.n_split, max_k, row_bytes,
                         pf_slots(head_dim), false);
}

void plan_route_f32(uint32_t n_seqs, uint32_t kvh, uint32_t group, uint32_t max_q, uint32_t max_k,
                    uint32_t head_dim, uint32_t row_bytes, int split_ok, uint64_t ws_bytes,
                    uint64_t* out) {
  const F32Route r = f32_route(n_seqs, kvh, group, max_q, max_k, head_dim, split_ok, ws_bytes);
  out[0] = r.plan.items, out[1] = r.plan.qtiles, out[2] = r.n_split, out[3] = r.ranges.ranges;
  out[4] = r.ranges.bytes;
  out[5] = prefill_order(n_seqs, kvh, r.plan.qtiles, r.plan.items, r.n_split, max_k, row_bytes,
                         256, true);
}

// (list entry, kv head, tile) of every item of a launch in kPfListParts.
void plan_list_parts(uint32_t n_seqs, uint32_t kvh, uint32_t qtiles, uint32_t* out) {
  for (uint32_t i = 0; i < n_seqs * kvh * qtiles; ++i)
    pf_list_part(i, n_seqs, kvh, qtiles, out[3 * i], out[3 * i + 1], out[3 * i + 2]);
}

}  // extern "C"

namespace {

// PfWalk (attn_prefill.hpp) on the CPU.
struct Walk {
  std::vector<PfEntry> e;
  uint32_t li = 0, m = 0, kh = 0;
  uint32_t seek(uint32_t kh_, uint32_t at) {
    kh = kh_, m = 0;
    for (li = 0; li + 1 < e.size(); ++li) {
      const uint32_t all = pf_tiles_sum(e[li].c_last, e[li].fall, e[li].nt);
      if (at < all) break;
      at -= all;
    }
    while (m + 1 < e[li].nt && pf_tiles_sum(e[li].c_last, e[li].fall, m + 1) <= at) ++m;
    return at - pf_tiles_sum(e[li].c_last, e[li].fall, m);
  }
  uint32_t count() const { return e[li].c_last - e[li].fall * m; }
  void next() {
    if (++m < e[li].nt) return;
    m = 0;
    if (++li == e.size()) li = 0, ++kh;
  }
};

struct Piece {
  uint32_t r, u0, u1, c, slot;
};
struct Tile {
  std::vector<Piece> pieces;
  int opened = 0;
  uint32_t first_slot = 0, last = 0;
};

}  // namespace

// 0 if the ranges cover every tile's counts once, with each split tile's
// description naming exactly its pieces' slots; else the number of the check
// that failed.
extern "C" int plan_check_walk(uint32_t n_seqs, const uint32_t* lens_q, const uint32_t* lens_k,
                               uint32_t kvh, uint32_t group, uint32_t rows, uint32_t qtiles,
                               int32_t wl, int32_t wr, uint32_t ranges) {
  Walk w;
  uint64_t total = 0;
  std::vector<uint32_t> first;  // each entry's first tile of a kv head
  uint32_t tiles_per_head = 0;
  for (uint32_t s = 0; s < n_seqs; ++s) {
    PfEntry e{s, 0, lens_q[s], lens_k[s], 0, 16, 0, 0};
    if (lens_q[s] < 2) continue;
    pf_entry_tiles(e, group, qtiles, rows, wl, wr, pf_count_cap(qtiles * kvh * n_seqs));
    for (uint64_t m = 0; m < e.nt; ++m) {
      const int64_t c = (int64_t)e.c_last - (int64_t)e.fall * m;
      if (c < 16) return 1;
      total += c;
    }
    first.push_back(tiles_per_head);
    tiles_per_head += e.nt;
    w.e.push_back(e);
  }
  if (w.e.empty()) return 0;
  const uint64_t S = total * kvh;
  if (S > kPfMaxCount) return 2;
  const uint32_t nr = pf_range_count((uint32_t)S, ranges);
  if (nr == 0 || nr > ranges) return 3;
  std::vector<Tile> tiles((size_t)tiles_per_head * kvh);
  auto here = [&]() -> Tile& { return tiles[(size_t)w.kh * tiles_per_head + first[w.li] + w.m]; };
  for (uint32_t r = 0; r < nr; ++r) {
    if (pf_range_at((uint32_t)S, nr, r) != S * r / nr) return 4;
    int opens = 0;
    uint64_t counted = 0;
    const bool open = pf_walk_pieces(
        w, (uint32_t)S, nr, r, kvh, (uint32_t)total,
        [&](uint32_t u0, uint32_t u1, uint32_t c, uint32_t slot) {
          here().pieces.push_back({r, u0, u1, c, slot});
          counted += u1 - u0;
        },
        [&]() { w.next(); },
        [&](uint32_t slot, uint32_t last) {
          ++opens;
          Tile& t = here();
          ++t.opened;
          t.first_slot = slot, t.last = last;
        });
    if (opens != (open ? 1 : 0)) return 5;
    if (counted != S * (r + 1) / nr - S * r / nr) return 6;
  }
  std::vector<char> used(2 * (size_t)nr, 0);
  for (const Tile& t : tiles) {
    if (t.pieces.empty()) return 7;
    const uint32_t c = t.pieces[0].c, steps = (c + 15) / 16;
    uint32_t at = 0, step = 0;
    for (size_t i = 0; i < t.pieces.size(); ++i) {
      const Piece& p = t.pieces[i];
      if (p.c != c || p.u0 != at || p.u1 <= p.u0 || p.u1 > c) return 8;
      at = p.u1;
      if (pf_step_at(p.u0, c, steps) != step || pf_step_at(p.u1, c, steps) < step) return 9;
      step = pf_step_at(p.u1, c, steps);
      if (t.pieces.size() == 1) {
        if (p.slot != ~0u || t.opened) return 10;
        continue;
      }
      if (t.opened != 1 || t.last != t.pieces.back().r) return 11;
      if (p.r != t.pieces[0].r + i) return 12;
      if (p.slot != (i ? 2 * p.r : t.first_slot)) return 13;
      if (p.slot >= used.size() || used[p.slot]++) return 14;
    }
    if (at != c || step != steps) return 15;
  }
  return 0;
}

// The order of a sorted launch's tiles as prefill_item finds it, rank by rank:
// 0 if every tile comes once. `order` takes (sequence, tile) pairs.
extern "C" int plan_order(uint32_t n, const uint32_t* key, const uint32_t* nt, uint32_t step,
                          uint32_t* order) {
  uint32_t longest = 0, tiles = 0;
  bool classes = false;
  for (uint32_t s = 0; s < n; ++s)
    if (nt[s]) longest = pf_max(longest, key[s]), tiles += nt[s];
  for (uint32_t s = 0; s < n; ++s) classes = classes || pf_short_tile(longest, key[s], nt[s], step);
  std::vector<std::vector<char>> seen(n);
  for (uint32_t s = 0; s < n; ++s) seen[s].assign(nt[s], 0);
  auto to = [&](uint32_t c, uint32_t s) {
    return pf_tiles_to_class(c, longest, key[s], nt[s], 1.f / (float)step);
  };
  for (uint32_t rank = 0; rank < tiles; ++rank) {
    std::vector<uint32_t> first(n, 0), here(nt, nt + n);
    uint32_t before = 0;
    if (classes) {
      uint32_t c = 0;
      for (;; ++c) {
        uint32_t sum = 0;
        for (uint32_t s = 0; s < n; ++s) sum += to(c, s);
        if (rank < sum || c + 1 >= kPfClasses) break;
        before = sum;
        for (uint32_t s = 0; s < n; ++s) first[s] = to(c, s);
      }
      for (uint32_t s = 0; s < n; ++s) {
        if (to(c, s) < first[s] || to(c, s) > nt[s]) return 1;
        here[s] = to(c, s) - first[s];
      }
    }
    const uint32_t at = rank - before;
    int hits = 0;
    for (uint32_t s = 0; s < n; ++s) {
      uint32_t start = 0;
      for (uint32_t o = 0; o < n; ++o)
        start += key[o] > key[s] || (key[o] == key[s] && o < s) ? here[o] : 0u;
      if (at < start || at - start >= here[s]) continue;
      ++hits;
      const uint32_t m = first[s] + (at - start);
      if (seen[s][m]++) return 2;
      order[2 * rank] = s, order[2 * rank + 1] = nt[s] - 1 - m;
    }
    if (hits != 1) return 3;
  }
  return 0;
}
