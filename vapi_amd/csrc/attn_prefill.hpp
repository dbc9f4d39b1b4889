// Pieces shared by the prefill kernels that stage K and V in LDS by direct
// global-to-LDS loads (attn_prefill.hip, attn_prefill_f32.hip).
#pragma once

#include "attn_common.hpp"

namespace vk {

using LdsVoid = __attribute__((address_space(3))) void;


// The XOR swizzle of key row r's 16-byte chunks. D = 128 (16 chunks, a row
// is 256 bytes: every row starts at bank 0): the row index rotated left by
// one bit, a bijection on 0..15, so the 16 rows a K fragment read touches
// use 16 distinct chunk positions for any chunk, and the 8 rows of one
// half-wave of a transposing V read (rows 0..7 or 8..15, chunks 2t, 2t + 1)
// use 8 distinct chunk pairs (XOR with r alone puts rows 2m and 2m + 1 on
// the same pair). Measured 0.5-1% faster than XOR with r; the bank-conflict
// counter reads the same either way (2 cycles per transposing read).
// D = 256 (32 chunks, 512-byte rows): the same rotation, XORed into the
// low four bits of the chunk index (chunks p and p ^ 16 share banks).
// D = 64: r mod 8.
template <int D>
__device__ __forceinline__ uint32_t pf_swz(uint32_t r) {
  if constexpr (D >= 128) {
    const uint32_t x = r & 15;
    return ((x << 1) | (x >> 3)) & 15;
  } else {
    return r & (D / 8 - 1);
  }
}

// Element offset of 16-byte chunk p of key row r (0..31) in a step buffer.
template <int D>
__device__ __forceinline__ uint32_t pf_chunk(uint32_t r, uint32_t p) {
  constexpr uint32_t CPR = D / 8;  // chunks per row
  return (r * CPR + (p ^ pf_swz<D>(r))) * 8;
}

// Waits until at most n of this wave's vector memory loads are in flight
// (s_waitcnt: vmcnt in bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8). The
// ring's waits count only its own direct loads, which holds while the
// kernel uses no scratch (vapi_amd/build.py refuses a build where it does).
template <int n>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(n >= 0 && n < 16, "vmcnt immediate");
  __builtin_amdgcn_s_waitcnt(n | (0x7 << 4) | (0xF << 8));
}

// The workgroup barrier of the ring: this wave's loads of the next step
// have landed (the caller's wait_vmcnt), then s_barrier alone. A
// __syncthreads() would add a release fence, which waits for every load
// in flight into LDS, including the step issued two ahead.
__device__ __forceinline__ void ring_barrier() {
  __asm__ volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  __asm__ volatile("" ::: "memory");
}

// The LDS offset of p: the low half of its flat address. (A cast to the LDS
// address space would test for null first, inside the loops that use it.)
__device__ __forceinline__ uint32_t lds_addr(const uint16_t* p) { return (uint32_t)(uintptr_t)p; }

// ---- the walk over a range (prefill_plan.hpp says what ranges are) ------------

// A walk over the plan's tiles: tile m from the last of list entry li's.
struct PfWalk {
  // In LDS, one entry per sequence of the list (at most kPfSortSeqs, one per
  // lane while it is made). Every wave makes the same one and reads its own, so
  // no barrier stands between.
  PfEntry* plan;
  PfEntry mine;    // this lane's entry, until the first tile is found
  uint32_t sum;    // and the count of its tiles
  uint64_t some;   // entries with tiles
  uint32_t total;  // counts of one kv head
  uint32_t li, m, kh, c, f, n;  // (uniform) c: the count of the entry's last tile
  uint32_t seq, q0, len_q, len_k;

  __device__ __forceinline__ void init(const AttnArgs& a, const uint32_t* __restrict__ cu_q,
                                       const uint32_t* __restrict__ cu_k, uint32_t qtiles,
                                       uint32_t rows, PfEntry* entries) {
    const uint32_t lane = threadIdx.x & 63;
    PfEntry e{0, 0, 0, 0, 0, 16, 0, 0};
    if (lane < a.pf_seqs_n) {
      e.seq = a.pf_seqs ? a.pf_seqs[lane] : lane;
      if (e.seq < a.batch) {
        e.q0 = cu_q[e.seq], e.len_q = cu_q[e.seq + 1] - e.q0;
        e.len_k = cu_k[e.seq + 1] - cu_k[e.seq];
        if (e.len_q >= a.pf_min_q && e.len_q > 0)
          pf_entry_tiles(e, a.group, qtiles, rows, a.wl, a.wr,
                         pf_count_cap(qtiles * a.kvh * a.pf_seqs_n));
      }
    }
    mine = e;
    sum = pf_tiles_sum(e.c_last, e.fall, e.nt);
    some = __ballot(e.nt > 0);
    total = 0;
    for (uint64_t left = some; left; left &= left - 1)
      total += __builtin_amdgcn_readlane(sum, (uint32_t)__builtin_ctzll(left));
    plan = entries + 64 * (threadIdx.x >> 6);
    plan[lane] = e;  // for the pieces after the first
  }
  // To the tile holding count `at` of kv head kh_, as the walk's first (from
  // the lanes); returns its place in it.
  __device__ __forceinline__ uint32_t seek(uint32_t kh_, uint32_t at) {
    kh = kh_;
    uint64_t left = some;
    while (true) {
      li = (uint32_t)__builtin_ctzll(left);
      const uint32_t all = __builtin_amdgcn_readlane(sum, li);
      left &= left - 1;
      if (at < all || !left) break;
      at -= all;
    }
    c = __builtin_amdgcn_readlane(mine.c_last, li);
    f = __builtin_amdgcn_readlane(mine.fall, li);
    n = __builtin_amdgcn_readlane(mine.nt, li);
    uint32_t hi = n;
    m = 0;  // pf_tiles_sum(m) <= at < pf_tiles_sum(hi)
    while (hi - m > 1) {
      const uint32_t mid = (m + hi) >> 1;
      if (pf_tiles_sum(c, f, mid) <= at) m = mid;
      else hi = mid;
    }
    seq = __builtin_amdgcn_readlane(mine.seq, li);
    q0 = __builtin_amdgcn_readlane(mine.q0, li);
    len_q = __builtin_amdgcn_readlane(mine.len_q, li);
    len_k = __builtin_amdgcn_readlane(mine.len_k, li);
    return at - pf_tiles_sum(c, f, m);
  }
  __device__ __forceinline__ uint32_t count() const { return c - f * m; }
  __device__ __forceinline__ void next() {
    if (++m < n) return;
    m = 0;
    const uint64_t after = li < 63 ? some & (~0ull << (li + 1)) : 0ull;
    if (!after) ++kh;
    li = (uint32_t)__builtin_ctzll(after ? after : some);
    const PfEntry e = plan[li];
    c = __builtin_amdgcn_readfirstlane(e.c_last);
    f = __builtin_amdgcn_readfirstlane(e.fall);
    n = __builtin_amdgcn_readfirstlane(e.nt);
    seq = __builtin_amdgcn_readfirstlane(e.seq);
    q0 = __builtin_amdgcn_readfirstlane(e.q0);
    len_q = __builtin_amdgcn_readfirstlane(e.len_q);
    len_k = __builtin_amdgcn_readfirstlane(e.len_k);
  }
  __device__ __forceinline__ PfItem item() const {
    return PfItem{li, seq, n - 1 - m, kh, q0, len_q, (int32_t)len_k};
  }
};

// Workgroup `bid`'s range of at most `ranges`: piece(item, u0, u1, c, slot)
// for each of its pieces, counts [u0, u1) of the tile's c (slot: its partial,
// or ~0u for a whole tile), the workgroup's LDS free again between them.
template <int W, typename Piece>
__device__ __forceinline__ void pf_walk_range(const AttnArgs& a, const uint32_t* __restrict__ cu_q,
                                              const uint32_t* __restrict__ cu_k, uint32_t qtiles,
                                              uint32_t rows, uint32_t ranges,
                                              PfSplitTile* __restrict__ tiles, uint32_t bid,
                                              Piece piece) {
  __shared__ PfEntry entries[64 * W];
  PfWalk w;
  w.init(a, cu_q, cu_k, qtiles, rows, entries);
  const uint32_t S = w.total * a.kvh, nr = pf_range_count(S, ranges);
  if (bid >= nr || !w.some) {
    if (threadIdx.x == 0) tiles[bid].valid = 0;
    return;
  }
  const uint32_t x = bid % 8, r = x * (nr / 8) + min(x, nr % 8) + bid / 8;
  const bool open = pf_walk_pieces(
      w, S, nr, r, a.kvh, w.total,
      [&](uint32_t u0, uint32_t u1, uint32_t c, uint32_t slot) __attribute__((always_inline)) {
        piece(w.item(), u0, u1, c, slot);
      },
      [&]() __attribute__((always_inline)) {
        w.next();
        __syncthreads();
      },
      [&](uint32_t slot, uint32_t last) __attribute__((always_inline)) {
        if (threadIdx.x == 0) {
          const PfItem it = w.item();
          PfSplitTile t;
          t.valid = 1, t.seq = it.seq, t.qt = it.qt, t.kh = it.kh, t.first_slot = slot;
          t.last = last;
          t.pad[0] = t.pad[1] = 0;
          tiles[r] = t;
        }
      });
  if (threadIdx.x == 0 && !open) tiles[r].valid = 0;
}

void launch_prefill_range_merge(const AttnArgs& a, uint32_t ranges, uint32_t rows, uint32_t dtype,
                                uint32_t head_dim, const void* ws, hipStream_t s);

}  // namespace vk
