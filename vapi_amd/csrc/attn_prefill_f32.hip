// Chunked-prefill paged attention for f32 pools: two kernels.
//
// paged_prefill_f32x3: exact three-way bf16 splits on
// v_mfma_f32_16x16x32_bf16.
//
// gfx950 multiplies bf16 16 times as fast as f32. An f32 value is the sum of
// three bf16 ones, x = h + m + l with h = bf16(x), m = bf16(x - h), l =
// x - h - m, all three exact (round to nearest, 8 significant bits each), so
// a product x y is the six bf16 products hh', hm', mh', hl', mm', lh' up to
// the three dropped ones, about 2^-26 |x y| of either sign (2^-23 at most):
// the rounding of one f32 operation. All six are exact in the MFMA and added
// in f32, in an eighth as many steps as f32 MFMAs add them. Q, K, V and the
// probabilities are all split this way; nothing is held in fewer bits than
// before. Error against 64 bits (2-norm, relative), f32 MFMAs -> this: 4
// chunks of ~400 over ~2,100 keys 6.8e-7 -> 5.5e-7, head_dim 64 4.1e-7 ->
// 3.0e-7, head_dim 80 with a window 3.9e-7 -> 3.0e-7, head_dim 96 fresh
// 3.4e-7 -> 2.6e-7. Six bf16 MFMAs at 1/16 of an f32 MFMA's cost: 2.7 times
// the f32 rate. 8 chunks of 512 over 4,096 keys (32 q / 8 kv heads) 2,478 ->
// 1,165 us (105 -> 221 TFLOP/s), the 4 ragged chunks 442 -> 193 us.
//
// Values whose h would not be finite (infinities, NaN, |x| above the largest
// bf16) have no such split: their l is NaN, which reaches every sum that the
// value is part of, whatever it is multiplied with. And the low bits of m and l
// of a value below 2^-110 would lie outside bf16's range: the smallest nonzero
// magnitude is kept as values are split (a shift-add and half a min3 each). If
// a workgroup ends with a NaN, or met a value that is not zero and below
// 2^-100, it computes its item again with f32 MFMAs (f32_rows below) and stores
// that instead. (Probabilities are not checked: one below 2^-110 of its row's
// largest holds at most 17 good bits already, as the rounding of its exponent
// is 2^-18 or more.)
//
// Rows are the (query token, head) pairs of one kv head, r = j*G + h_local,
// as in the 16-bit prefill: a workgroup of 8 waves owns 128 RT rows and walks
// the keys they see in 32-key steps. A step's K and V (32 KiB at head_dim
// 128) go to LDS once as f32 by direct loads, issued a step ahead; each
// thread then splits the chunks that it loaded itself (so no barrier stands
// between) into the bf16 planes of the next step, 6 x 8 KiB, which every wave
// reads as MFMA operands: K rows as they are, V through transposing reads,
// chunks swizzled as in the 16-bit kernel. Planes are double buffered: one
// barrier per step. What bounds it: the matrix cores (96 MFMAs per 16 rows
// and step); splitting K and V costs 7 instructions per element, once per
// workgroup and step.
//
// paged_prefill_f32: f32 MFMAs (v_mfma_f32_16x16x4_f32) for launches of few
// rows per kv head. Each wave owns two tiles of 16 rows and walks its keys in
// 32-key steps, each as two 16-key halves in the f32 operand scheme of the
// decode (attend_half_f32), loaded straight into registers: a half is
// computed for both row tiles, then reloaded with the next step's half while
// the other half is computed. Four such waves per workgroup, one per SIMD,
// so a launch of one small tile per kv head keeps four items on each CU.
//
// Rows with len_q < a.pf_min_q are left to the decode stream (pf_min_q 1:
// every row here). kPad: a head_dim a.hd below D (a multiple of 4); chunks
// past it are filled with the row's first one, meet zeros of Q and reach only
// output columns that are not stored; output rows are a.hd apart. Numerical
// contract: paged_attention_cpu (vapi
// crates/vapi-backend-candle/src/attention.rs:90-163), f32 throughout.
#include <algorithm>
#include <type_traits>

#include "attn_common.hpp"
#include "attn_prefill.hpp"

namespace vk {

constexpr int kPfF32Waves = 4;

// Eight (or fewer) values split into three planes of packed bf16.
struct Split8 {
  uint4 h, m, l;
};

__device__ __forceinline__ void split2(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
  h = pack2<bf16_t>(a, b);
  a -= __uint_as_float(h << 16), b -= __uint_as_float(h & 0xffff0000u);
  m = pack2<bf16_t>(a, b);
  a -= __uint_as_float(m << 16), b -= __uint_as_float(m & 0xffff0000u);
  l = pack2<bf16_t>(a, b);
}
__device__ __forceinline__ Split8 split8(const float (&x)[8]) {
  Split8 s;
  split2(x[0], x[1], s.h.x, s.m.x, s.l.x);
  split2(x[2], x[3], s.h.y, s.m.y, s.l.y);
  split2(x[4], x[5], s.h.z, s.m.z, s.l.z);
  split2(x[6], x[7], s.h.w, s.m.w, s.l.w);
  return s;
}
// The smallest 2 |x| - 1 of the bits of the values noted (zeros wrap to the
// top).
__device__ __forceinline__ void note_small(uint32_t& small, const float (&x)[8]) {
#pragma unroll
  for (int i = 0; i < 8; i += 2)
    small = min(small, min((__float_as_uint(x[i]) << 1) - 1u, (__float_as_uint(x[i + 1]) << 1) - 1u));
}
constexpr uint32_t kSmallest = (0x0d800000u << 1) - 1u;  // 2^-100

// x y over 32 values of k in six MFMAs, the smallest products first.
__device__ __forceinline__ floatx4 mfma_split(const Split8& x, const Split8& y, floatx4 c) {
  c = mfma16x16x32<bf16_t>(x.l, y.h, c);
  c = mfma16x16x32<bf16_t>(x.h, y.l, c);
  c = mfma16x16x32<bf16_t>(x.m, y.m, c);
  c = mfma16x16x32<bf16_t>(x.m, y.h, c);
  c = mfma16x16x32<bf16_t>(x.h, y.m, c);
  return mfma16x16x32<bf16_t>(x.h, y.h, c);
}

// Six transposing LDS reads of one d tile, two 16-row halves of each plane
// (kHalf and kPlane bytes apart), issued without waiting.
template <int kHalf, int kPlane>
__device__ __forceinline__ void ds_read_tr16_issue6(uint2 (&r)[6], uint32_t addr) {
  __asm__ volatile(
      "ds_read_b64_tr_b16 %0, %6\n\t"
      "ds_read_b64_tr_b16 %1, %6 offset:%7\n\t"
      "ds_read_b64_tr_b16 %2, %6 offset:%8\n\t"
      "ds_read_b64_tr_b16 %3, %6 offset:%9\n\t"
      "ds_read_b64_tr_b16 %4, %6 offset:%10\n\t"
      "ds_read_b64_tr_b16 %5, %6 offset:%11"
      : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]), "=&v"(r[4]), "=&v"(r[5])
      : "v"(addr), "n"(kHalf), "n"(kPlane), "n"(kPlane + kHalf), "n"(2 * kPlane),
        "n"(2 * kPlane + kHalf)
      : "memory");
}
template <int N>
__device__ __forceinline__ void lgkm_wait(uint2 (&r)[6]) {
  __asm__ volatile("s_waitcnt lgkmcnt(%6)"
                   : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]), "+v"(r[4]), "+v"(r[5])
                   : "n"(N)
                   : "memory");
}

// RT row tiles of one wave in f32 MFMAs, straight from the pool over keys
// [klo, khi]: rows row0 .. of a sequence (its len_q * G rows are nrows). `pb`:
// the wave's item's partials of a key split ((m, l), then o / l per row,
// prow0 the wave's first row in the item's part_rows), or null for the output.
template <int D, int RT, bool kPad, int CL, bool kAhead>
__device__ __forceinline__ void f32_rows(const AttnArgs& a, const uint32_t* __restrict__ tab,
                                         uint32_t kh, uint32_t q0, uint32_t nrows, uint32_t row0,
                                         int32_t offset, int32_t len_k, int32_t klo, int32_t khi,
                                         char* pb, uint32_t prow0, uint32_t part_rows) {
  const uint32_t lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
  const uint32_t G = a.group;
  // This wave's rows: Q^T operands and visible key ranges.
  float4 qf[RT][D / 16];
  int32_t lo[RT];
  uint32_t cnt[RT];
  const uint32_t sg = a.q_sign ? 0x80000000u : 0u;
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const uint32_t r = row0 + 16 * t + col;
    const uint32_t rr = r < nrows ? r : 0;
    const uint32_t j = rr / G, hl = rr % G;
    int32_t hi;
    key_range(offset + (int32_t)j, len_k, a.wl, a.wr, lo[t], hi);
    cnt[t] = (uint32_t)max(hi - lo[t] + 1, 0);
    const float* qrow =
        (const float*)a.q + ((uint64_t)(q0 + j) * a.num_heads + kh * G + hl) * (kPad ? a.hd : D);
#pragma unroll
    for (int c = 0; c < D / 16; ++c) {
      uint4 x = make_uint4(0, 0, 0, 0);
      if (!kPad || 16 * c + 4 * g < a.hd) x = *(const uint4*)(qrow + 16 * c + 4 * g);
      x.x ^= sg, x.y ^= sg, x.z ^= sg, x.w ^= sg;
      qf[t][c] = make_float4(__uint_as_float(x.x), __uint_as_float(x.y), __uint_as_float(x.z),
                             __uint_as_float(x.w));
    }
  }
  float m_run[RT], l_run[RT];
  floatx4 o[RT][D / 16];
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    m_run[t] = kNegBig;
    l_run[t] = 0.f;
#pragma unroll
    for (int k = 0; k < D / 16; ++k) o[t][k] = floatx4{0.f, 0.f, 0.f, 0.f};
  }

  if (khi >= klo) {
    const float* kb = (const float*)a.k + kh * a.head_e;
    const float* vb = (const float*)a.v + kh * a.head_e;
    const int32_t s_last = khi & ~31;
    int32_t s0 = klo & ~31;
    if constexpr (!kAhead) {
      // One half at a time, nothing in flight beside it (few registers).
#pragma unroll 1
      for (int32_t h0 = s0; h0 <= khi; h0 += 16) {
        KHalfF32<D> kt;
        VHalfF32<D> vt;
        load_half_f32<D, false, kPad, CL>(kt, vt, tab, kb, vb, a, h0, 0, khi, col, g);
#pragma unroll
        for (int t = 0; t < RT; ++t) {
          const uint32_t base = (uint32_t)(h0 + 4 * (int32_t)g - lo[t]), n = cnt[t];
          attend_half_f32<D, CL>(kt, vt, qf[t], o[t], m_run[t], l_run[t], a.scale_log2,
                                 [&](int i) { return base + (uint32_t)i < n; });
        }
      }
    } else {
      KTileF32<D> kt;
      VTileF32<D> vt;
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
        load_half_f32<D, false, kPad, CL>(kt.h[tt], vt.h[tt], tab, kb, vb, a, s0, tt, khi, col, g);
      while (true) {
        // The next step's halves are loaded unconditionally (the last step
        // re-reads its own keys, from L2): a load inside a branch would make
        // the compiler wait for it before this step's MFMAs.
        const int32_t s_next = min(s0 + 32, s_last);
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
#pragma unroll
          for (int t = 0; t < RT; ++t) {
            const uint32_t base = (uint32_t)(s0 + 16 * tt + 4 * (int32_t)g - lo[t]);
            const uint32_t n = cnt[t];
            attend_half_f32<D, CL>(kt.h[tt], vt.h[tt], qf[t], o[t], m_run[t], l_run[t], a.scale_log2,
                               [&](int i) { return base + (uint32_t)i < n; });
          }
          load_half_f32<D, false, kPad, CL>(kt.h[tt], vt.h[tt], tab, kb, vb, a, s_next, tt, khi, col, g);
        }
        if (s0 >= s_last) break;
        s0 += 32;
      }
    }
  }

#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const float lt = wave_sum_g(l_run[t]);
    const float inv = lt > 0.f ? 1.f / lt : 0.f;
    const uint32_t r = row0 + 16 * t + col;
    if (pb) {
      const uint32_t pr = prow0 + 16 * t + col;
      if (g == 0) *(float2*)(pb + (uint64_t)pr * 8) = make_float2(m_run[t], lt);
      store_row_f32<D>((float*)(pb + (uint64_t)part_rows * 8) + (uint64_t)pr * D, o[t], inv, g);
    } else if (r < nrows) {
      const uint32_t j = r / G, hl = r % G;
      float* orow =
          (float*)a.out + ((uint64_t)(q0 + j) * a.num_heads + kh * G + hl) * (kPad ? a.hd : D);
      store_row_f32<D, kPad>(orow, o[t], inv, g, a.hd);
    }
  }
}

// One item: query tile it.qt of a sequence and kv head. kSplit, u0, u1, c,
// pb: as prefill_piece's. DL: the 16-column d tiles that hold head_dim (kPad;
// D / 16 otherwise): the MFMAs and reads of the tiles past them are left out.
template <int D, int RT, int kSplit, bool kPad, int DL>
__device__ __forceinline__ void x3_piece(const AttnArgs& a, const uint32_t* __restrict__ table,
                                         const PfItem& it, uint32_t u0, uint32_t u1, uint32_t c_all,
                                         char* pb) {
  constexpr uint32_t kPf32Rows = x3_rows(RT);
  constexpr int DT = D / 16, KCL = (DL + 1) / 2;
  constexpr uint32_t kPlane = 32 * D;       // elements of one plane of one tensor
  constexpr int kUnits = 8 * D / kPf32Threads;  // 8-element units a thread loads and splits a step
  constexpr int kHalfB = 16 * D * 2;        // bytes between rows r and r + 16 of a plane
  constexpr int kPlaneB = kPlane * 2;
  __shared__ __attribute__((aligned(16))) uint16_t kpl[2][3 * kPlane], vpl[2][3 * kPlane];
  __shared__ uint4 raw[kUnits][2][kPf32Threads];
  __shared__ uint32_t outside_lds;
  const uint32_t qt = it.qt, kh = it.kh, q0 = it.q0;
  const uint32_t G = a.group, nrows = it.len_q * G;
  const uint32_t row_base = qt * kPf32Rows;
  if (row_base >= nrows) return;
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t col = lane & 15, g = lane >> 4;
  const int32_t len_k = it.len_k, offset = len_k - (int32_t)it.len_q, last = len_k - 1;

  // The keys any row of the workgroup sees, and this split's share of them.
  const uint32_t wg_last = min(row_base + kPf32Rows, nrows) - 1;
  const int32_t pmin = offset + (int32_t)(row_base / G), pmax = offset + (int32_t)(wg_last / G);
  int32_t klo, khi, unused;
  key_range(pmin, len_k, a.wl, a.wr, klo, unused);
  key_range(pmax, len_k, a.wl, a.wr, unused, khi);
  if (kSplit) {
    const int32_t first = klo & ~31;
    const uint32_t steps = khi >= klo ? (uint32_t)(((khi & ~31) - first) / 32 + 1) : 0u;
    const uint32_t a0 = pf_step_at(u0, c_all, steps), a1 = pf_step_at(u1, c_all, steps);
    klo = max(klo, first + 32 * (int32_t)a0);
    khi = min(khi, first + 32 * (int32_t)a1 - 1);
  }
  // Steps inside [full_lo, full_hi] need no mask.
  int32_t full_lo, full_hi;
  key_range(pmax, len_k, a.wl, a.wr, full_lo, unused);
  key_range(pmin, len_k, a.wl, a.wr, unused, full_hi);

  const uint32_t* __restrict__ tab = table + (uint64_t)it.seq * a.max_blocks;
  const float* kb = (const float*)a.k + kh * a.head_e;
  const float* vb = (const float*)a.v + kh * a.head_e;
  // This thread's units of a step, tid + kPf32Threads j: K rows 0 .. 31, then
  // V's, D / 8 units each (a wave's units lie in one 16-key tile).
  constexpr uint32_t CPR = D / 8;
  constexpr uint32_t kRowsPerJ = kPf32Threads / CPR;  // key rows between units j and j + 1
  const uint32_t ur0 = tid / CPR, up = tid % CPR;
  const uint32_t wr0 = __builtin_amdgcn_readfirstlane(ur0);
  const uint32_t d0 = kPad && 8 * up >= a.hd ? 0 : 8 * up;
  const uint32_t d1 = kPad && 8 * up + 4 >= a.hd ? 0 : 8 * up + 4;
  auto dma = [&](int32_t s0) __attribute__((always_inline)) {
    using ConstU32 = const __attribute__((address_space(4))) uint32_t;
    uint32_t row0_ = ur0, c0 = d0, c1 = d1;  // opaque: see attend
    asm volatile("" : "+v"(row0_), "+v"(c0), "+v"(c1));
    uint64_t tile[2];
    int32_t ts[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      ts[h] = min(s0 + 16 * h, last & ~15);
      const uint32_t blk =
          min(((ConstU32*)tab)[min((uint32_t)ts[h] >> a.bs_shift, a.max_blocks - 1)], a.last_blk);
      tile[h] = (uint64_t)blk * a.blk_e + (uint64_t)((uint32_t)ts[h] & (a.block_size - 1)) * a.tok_e;
    }
#pragma unroll
    for (int j = 0; j < kUnits; ++j) {
      const uint32_t wr = wr0 + kRowsPerJ * j;  // the wave's first row of 64
      const bool is_v = wr >= 32, second = (wr & 16) != 0;
      const uint32_t r = (row0_ + kRowsPerJ * j) & 15;
      const float* row = (is_v ? vb : kb) + (second ? tile[1] : tile[0]) +
                         (uint32_t)min((int32_t)r, last - (second ? ts[1] : ts[0])) * a.tok_e;
      __builtin_amdgcn_global_load_lds((const void*)(row + c0), (LdsVoid*)&raw[j][0][64 * wave], 16, 0, 0);
      __builtin_amdgcn_global_load_lds((const void*)(row + c1), (LdsVoid*)&raw[j][1][64 * wave], 16, 0, 0);
    }
  };
  uint32_t small = ~0u;  // of what this thread split (note_small)
  // Splits this thread's loaded chunks into the planes of buffer b.
  float4 x0[kUnits], x1[kUnits];
  auto fetch = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < kUnits; ++j) {
      x0[j] = *(const float4*)&raw[j][0][tid];
      x1[j] = *(const float4*)&raw[j][1][tid];
    }
  };
  auto convert = [&](int b) __attribute__((always_inline)) {
    uint32_t row0_ = ur0, pos = up;  // opaque: see attend
    asm volatile("" : "+v"(row0_), "+v"(pos));
#pragma unroll
    for (int j = 0; j < kUnits; ++j) {
      const float x[8] = {x0[j].x, x0[j].y, x0[j].z, x0[j].w, x1[j].x, x1[j].y, x1[j].z, x1[j].w};
      const Split8 s = split8(x);
      const uint32_t wr = wr0 + kRowsPerJ * j;
      note_small(small, x);
      uint16_t* dst = (wr >= 32 ? vpl[b] : kpl[b]) + pf_chunk<D>((row0_ + kRowsPerJ * j) & 31, pos);
      *(uint4*)dst = s.h;
      *(uint4*)(dst + kPlane) = s.m;
      *(uint4*)(dst + 2 * kPlane) = s.l;
    }
  };

  const uint32_t wrow0 = wave * 16 * RT, row0 = row_base + wrow0;
  const bool active = row0 < nrows;  // waves without rows only load and split
  Split8 qf[RT][KCL];
  int32_t lo[RT], cnt[RT];
  const uint32_t sg = a.q_sign ? 0x80000000u : 0u;
  if (klo <= khi) dma(klo & ~31);
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const uint32_t r = row0 + 16 * t + col;
    const uint32_t rr = r < nrows ? r : 0;
    const uint32_t j = rr / G, hl = rr % G;
    int32_t hi;
    key_range(offset + (int32_t)j, len_k, a.wl, a.wr, lo[t], hi);
    cnt[t] = max(hi - lo[t] + 1, 0);
    const float* qrow =
        (const float*)a.q + ((uint64_t)(q0 + j) * a.num_heads + kh * G + hl) * (kPad ? a.hd : D);
#pragma unroll
    for (int c = 0; c < KCL; ++c) {
      uint4 u = make_uint4(0, 0, 0, 0), v = u;
      if (!kPad || 32 * c + 8 * g < a.hd) u = *(const uint4*)(qrow + 32 * c + 8 * g);
      if (!kPad || 32 * c + 8 * g + 4 < a.hd) v = *(const uint4*)(qrow + 32 * c + 8 * g + 4);
      const float x[8] = {__uint_as_float(u.x ^ sg), __uint_as_float(u.y ^ sg),
                          __uint_as_float(u.z ^ sg), __uint_as_float(u.w ^ sg),
                          __uint_as_float(v.x ^ sg), __uint_as_float(v.y ^ sg),
                          __uint_as_float(v.z ^ sg), __uint_as_float(v.w ^ sg)};
      qf[t][c] = split8(x);
      note_small(small, x);
    }
  }
  float m_run[RT], l_run[RT];
  floatx4 o[RT][DT];
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    m_run[t] = kNegBig;
    l_run[t] = 0.f;
#pragma unroll
    for (int k = 0; k < DT; ++k) o[t][k] = floatx4{0.f, 0.f, 0.f, 0.f};
  }

  // Fragment offsets (bytes) within a plane at chunk 0 / d tile 0. Rows 16
  // apart differ by a constant, as the swizzle repeats after 16 rows; chunk
  // and tile indices are XORed in, as the swizzle is.
  const uint32_t k_off = 2 * pf_chunk<D>(col, g);
  const uint32_t vj = col >> 2, vq = col & 3;
  const uint32_t v_off = 2 * (pf_chunk<D>(4 * g + vj, vq >> 1) + 4 * (vq & 1));

  int32_t s0_ = klo & ~31;
  const int32_t s_last = khi & ~31;
  if (klo <= khi) {
    wait_vmcnt<0>();
    fetch();
    convert(0);
    dma(min(s0_ + 32, s_last));
    lds_barrier();
  }
  // Scores, softmax and O^T += V^T P^T of the step at s0, planes in buffer B.
  auto attend = [&](int32_t s0, auto cur) __attribute__((always_inline)) {
    constexpr int B = decltype(cur)::value;
    // Opaque copies: the addresses derived from them are computed in the
    // step (one XOR each) instead of being held in registers across it.
    uint32_t ko = k_off, vo = v_off;
    asm volatile("" : "+v"(ko), "+v"(vo));
    const bool masked = !(s0 >= full_lo && s0 + 31 <= full_hi);
    floatx4 acc[RT][2];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
#pragma unroll
      for (int t = 0; t < RT; ++t) acc[t][tt] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < KCL; ++c) {
        const uint16_t* p = kpl[B] + ((ko ^ (64u * c)) >> 1) + tt * (kHalfB / 2);
        Split8 kf;
        kf.h = *(const uint4*)p;
        kf.m = *(const uint4*)(p + kPlane);
        kf.l = *(const uint4*)(p + 2 * kPlane);
#pragma unroll
        for (int t = 0; t < RT; ++t) acc[t][tt] = mfma_split(kf, qf[t][c], acc[t][tt]);
      }
    }
    const uint32_t vbase = lds_addr(vpl[B]);
    uint2 vr[2][6];
    ds_read_tr16_issue6<kHalfB, kPlaneB>(vr[0], vbase + vo);
    Split8 pf[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      float s[8];
      const uint32_t base = (uint32_t)(s0 + 4 * (int32_t)g - lo[t]), n = (uint32_t)cnt[t];
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int i = 0; i < 4; ++i) s[4 * tt + i] = acc[t][tt][i];
      if (masked) {
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (!(base + 16 * tt + i < n)) s[4 * tt + i] = -INFINITY;
      }
      const float mx = max3_nc(max3_nc(s[0], s[1], s[2]), max3_nc(s[3], s[4], s[5]),
                               max_nc(s[6], s[7])) * a.scale_log2;
      rescale_rows<D, DL>(mx, o[t], m_run[t], l_run[t]);
      float p[8], ps = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        p[j] = fast_exp2(__builtin_fmaf(s[j], a.scale_log2, -m_run[t]));
        ps += p[j];
      }
      l_run[t] += ps;
      pf[t] = split8(p);
    }
#pragma unroll
    for (int k = 0; k < DL; ++k) {
      uint2(&r)[6] = vr[k & 1];
      if (k + 1 < DL) {
        ds_read_tr16_issue6<kHalfB, kPlaneB>(vr[(k + 1) & 1], vbase + (vo ^ (32u * (k + 1))));
        lgkm_wait<6>(r);
      } else {
        lgkm_wait<0>(r);
      }
      Split8 vf;
      vf.h = make_uint4(r[0].x, r[0].y, r[1].x, r[1].y);
      vf.m = make_uint4(r[2].x, r[2].y, r[3].x, r[3].y);
      vf.l = make_uint4(r[4].x, r[4].y, r[5].x, r[5].y);
#pragma unroll
      for (int t = 0; t < RT; ++t) o[t][k] = mfma_split(vf, pf[t], o[t][k]);
    }
  };
  auto step = [&](auto cur) __attribute__((always_inline)) {
    constexpr int B = decltype(cur)::value;
    const int32_t s0 = __builtin_amdgcn_readfirstlane(s0_);
    // The next step: its f32 chunks (loaded since the last step) into
    // registers, the one after it on its way, its planes written.
    wait_vmcnt<0>();
    fetch();
    wait_lds();
    dma(min(s0 + 64, s_last));
    convert(1 - B);
    if (active) attend(s0, std::integral_constant<int, B>{});
    lds_barrier();
    s0_ += 32;
  };
  while (true) {
    if (s0_ > khi) break;
    step(std::integral_constant<int, 0>{});
    if (s0_ > khi) break;
    step(std::integral_constant<int, 1>{});
  }
  wait_vmcnt<0>();  // no load may land in LDS after the workgroup ends

  // Values without a split anywhere in the workgroup's share: f32 MFMAs. (NaN
  // is looked for in the bits: the build's float compares assume there is none.)
  if (tid == 0) outside_lds = 0;
  __syncthreads();
  {
    uint32_t top = 0;
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      top = max(top, __float_as_uint(l_run[t]) << 1);
#pragma unroll
      for (int k = 0; k < DL; ++k)
#pragma unroll
        for (int i = 0; i < 4; ++i) top = max(top, __float_as_uint(o[t][k][i]) << 1);
    }
    if (__any(small < kSmallest || top > (0x7f800000u << 1)) && lane == 0) outside_lds = 1;
  }
  __syncthreads();
  if (__builtin_amdgcn_readfirstlane(outside_lds)) {
#pragma unroll 1
    for (uint32_t t = 0; t < (uint32_t)RT; ++t)
      f32_rows<D, 1, kPad, D / 16, false>(a, tab, kh, q0, nrows, row0 + 16 * t, offset, len_k, klo,
                                          khi, kSplit ? pb : nullptr, wrow0 + 16 * t, kPf32Rows);
    return;
  }
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const float lt = wave_sum_g(l_run[t]);
    const float inv = lt > 0.f ? 1.f / lt : 0.f;
    const uint32_t r = row0 + 16 * t + col;
    float* dst;
    const bool partial = kSplit == 1 || (kSplit == 2 && pb);
    if (partial) {
      const uint32_t pr = wrow0 + 16 * t + col;
      if (g == 0) *(float2*)(pb + (uint64_t)pr * 8) = make_float2(m_run[t], lt);
      dst = (float*)(pb + (uint64_t)kPf32Rows * 8) + (uint64_t)pr * D;
    } else {
      if (r >= nrows) continue;
      const uint32_t j = r / G, hl = r % G;
      dst = (float*)a.out + ((uint64_t)(q0 + j) * a.num_heads + kh * G + hl) * (kPad ? a.hd : D);
    }
#pragma unroll
    for (int k = 0; k < DL; ++k)
      if (!kPad || partial || 16 * k + 4 * g < a.hd)
        *(float4*)(dst + 16 * k + 4 * g) = make_float4(o[t][k][0] * inv, o[t][k][1] * inv,
                                                       o[t][k][2] * inv, o[t][k][3] * inv);
  }
}
// Workgroups of a launch: an item each, or (kSplit) one of n_split equal
// shares of each item's steps, to be merged (a batch too small to fill the
// GPU with query tiles alone).
template <int D, int RT, bool kSplit, bool kPad, int DL = D / 16>
__global__ __launch_bounds__(kPf32Threads, 1) void paged_prefill_f32x3(
    AttnArgs a, const uint32_t* __restrict__ cu_q, const uint32_t* __restrict__ cu_k,
    const uint32_t* __restrict__ table, uint32_t qtiles, uint32_t n_split_arg,
    float* __restrict__ part) {
  constexpr uint32_t kRows = x3_rows(RT);
  const uint32_t n_split = kSplit ? n_split_arg : 1u;
  __shared__ uint32_t order[64 * kPf32Waves];
  const uint32_t hr = blockIdx.x / a.kvh, split = hr % n_split;
  PfItem it;
  if (!prefill_item<kPf32Waves>(a, cu_q, cu_k, (hr / n_split) * a.kvh + blockIdx.x % a.kvh, qtiles,
                                kRows, order, it))
    return;
  char* pb = nullptr;
  if (kSplit)
    pb = (char*)part + ((uint64_t)((it.li * a.kvh + it.kh) * qtiles + it.qt) * n_split + split) *
                           pf_part_bytes(kRows, D);
  x3_piece<D, RT, kSplit ? 1 : 0, kPad, DL>(a, table, it, split, split + 1, n_split, pb);
}

// The same over ranges of equal work (see attn_prefill.hpp).
template <int D, int RT, bool kPad, int DL = D / 16>
__global__ __launch_bounds__(kPf32Threads, 1) void paged_prefill_f32x3_ranges(
    AttnArgs a, const uint32_t* __restrict__ cu_q, const uint32_t* __restrict__ cu_k,
    const uint32_t* __restrict__ table, uint32_t qtiles, uint32_t ranges,
    PfSplitTile* __restrict__ tiles, char* __restrict__ part) {
  constexpr uint32_t kRows = x3_rows(RT);
  pf_walk_range<kPf32Waves>(a, cu_q, cu_k, qtiles, kRows, ranges, tiles, blockIdx.x,
                            [&](const PfItem& it, uint32_t u0, uint32_t u1, uint32_t c,
                                uint32_t slot) __attribute__((always_inline)) {
                              x3_piece<D, RT, 2, kPad, DL>(
                                  a, table, it, u0, u1, c,
                                  slot == ~0u ? nullptr
                                              : part + (uint64_t)slot * pf_part_bytes(kRows, D));
                            });
}

// kSplit: the keys a wave would walk are cut into n_split contiguous runs
// of steps, one wave each (a batch too small to fill the GPU with query
// tiles alone); each writes its rows' (m, l, o / l) to `part`
// (pf_part_bytes of 16 * RT rows per (item, split)) for the merge.
// CL: the 16-column chunks of d that hold head_dim (kPad; D / 16
// otherwise): K chunks past them are neither loaded nor multiplied.
template <int D, int RT, bool kSplit, bool kPad, int CL = D / 16>
__global__ __launch_bounds__(64 * kPfF32Waves, 1) void paged_prefill_f32(
    AttnArgs a, uint32_t qtiles, uint32_t n_items, uint32_t n_split_arg,
    float* __restrict__ part) {
  const uint32_t n_split = kSplit ? n_split_arg : 1u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t item = xcd_remap(blockIdx.x, gridDim.x) * kPfF32Waves + wave;
  if (item >= n_items) return;
  // Item order: query tile fastest, then key split, kv head, sequence.
  const uint32_t qt = item % qtiles, rest_s = item / qtiles;
  const uint32_t split = rest_s % n_split, rest = rest_s / n_split;
  const uint32_t kh = rest % a.kvh;
  const uint32_t seq = a.pf_seqs ? a.pf_seqs[rest / a.kvh] : rest / a.kvh;
  if (seq >= a.batch) return;
  const uint32_t q0 = a.cu_q[seq];
  const uint32_t len_q = a.cu_q[seq + 1] - q0;
  if (len_q < a.pf_min_q || len_q == 0) return;
  const uint32_t G = a.group;
  const uint32_t nrows = len_q * G;
  const uint32_t row0 = qt * 16 * RT;
  if (row0 >= nrows) return;
  const int32_t len_k = (int32_t)(a.cu_k[seq + 1] - a.cu_k[seq]);
  const int32_t offset = len_k - (int32_t)len_q;

  // The keys any row of the wave sees: from the first row's window start to
  // the last row's last key.
  const uint32_t r_last = min(row0 + 16 * RT, nrows) - 1;
  int32_t klo, khi, unused;
  key_range(offset + (int32_t)(row0 / G), len_k, a.wl, a.wr, klo, unused);
  key_range(offset + (int32_t)(r_last / G), len_k, a.wl, a.wr, unused, khi);
  if (kSplit) {
    // This split's share of the wave's 32-key steps (empty: khi < klo).
    const int32_t first = klo & ~31;
    const uint32_t steps = khi >= klo ? (uint32_t)(((khi & ~31) - first) / 32 + 1) : 0u;
    const uint32_t a0 = split * steps / n_split, a1 = (split + 1) * steps / n_split;
    klo = max(klo, first + 32 * (int32_t)a0);
    khi = min(khi, first + 32 * (int32_t)a1 - 1);
  }

  char* const pb = kSplit ? (char*)part + ((uint64_t)(rest * qtiles + qt) * n_split + split) *
                                              pf_part_bytes(16 * RT, D)
                          : nullptr;
  f32_rows<D, RT, kPad, CL, true>(a, a.table + (uint64_t)seq * a.max_blocks, kh, q0, nrows, row0, offset,
                            len_k, klo, khi, pb, 0, 16 * RT);
}


uint64_t prefill_f32_items(uint32_t n_seqs, uint32_t kvh, uint32_t group, uint32_t max_q) {
  return f32_plan(n_seqs, kvh, group, max_q).items;
}

size_t prefill_f32_split_bytes(uint32_t batch, uint32_t kvh, uint32_t group, uint32_t head_dim,
                               uint32_t max_q, uint32_t max_k) {
  if (max_q <= 1) return 0;
  const F32Plan p = f32_plan(batch, kvh, group, max_q);
  const uint32_t n = pf32_splits(p, max_k, head_dim, ~0ull);
  const size_t split = n > 1 ? (size_t)(p.items * n * pf_part_bytes(p.rows, head_dim)) : 0;
  return std::max(split,
                  f32_route(batch, kvh, group, max_q, max_k, head_dim, true, ~0ull).ranges.bytes);
}

void launch_prefill_f32(const AttnArgs& a_in, uint32_t max_q, uint32_t max_k, uint32_t head_dim,
                        void* split_ws, size_t split_ws_bytes, hipStream_t s) {
  AttnArgs a = a_in;
  // No split without a workspace, nor for a deterministic call (its output
  // must not depend on the workspace it is given).
  const F32Route route = f32_route(a.pf_seqs_n, a.kvh, a.group, max_q, max_k, head_dim,
                                   split_ws && !a.deterministic, split_ws_bytes);
  const F32Plan& p = route.plan;
  const PfRangePlan rp = route.ranges;
  const uint32_t qtiles = p.qtiles, n_split = route.n_split;
  const uint64_t items = p.items * n_split;
  a.pf_order = prefill_order(a.pf_seqs_n, a.kvh, qtiles, p.items, n_split,
                             prefill_keys(max_q, max_k, a.wl), a.hd * sizeof(float), 256,
                             true);
  const uint32_t wgs = (uint32_t)((items + kPfF32Waves - 1) / kPfF32Waves);
  float* part = n_split > 1 ? (float*)split_ws : nullptr;
#define VK_X3(DD, RT, SPLIT, PAD, CL)                                                            \
  hipLaunchKernelGGL((paged_prefill_f32x3<DD, RT, SPLIT, PAD, CL>), dim3((uint32_t)items),       \
                     dim3(kPf32Threads), 0, s, a, a.cu_q, a.cu_k, a.table, qtiles, n_split, part)
#define VK_X3R(DD, PAD, CL)                                                                      \
  hipLaunchKernelGGL((paged_prefill_f32x3_ranges<DD, 1, PAD, CL>), dim3(rp.ranges),              \
                     dim3(kPf32Threads), 0, s, a, a.cu_q, a.cu_k, a.table, qtiles, rp.ranges,    \
                     (PfSplitTile*)split_ws, (char*)split_ws + kPfRangeHead)
#define VK_PF32(DD, PAD, CL)                                                                     \
  do {                                                                                           \
    if (rp.ranges) {                                                                             \
      VK_X3R(DD, PAD, CL);                                                                       \
      launch_prefill_range_merge(a, rp.ranges, p.rows, VAPI_KV_F32, DD, split_ws, s);            \
    } else if (p.x3) {                                                                                  \
      if (p.row_tiles == 2) {                                                                    \
        VK_X3(DD, 2, false, PAD, CL); /* enough items: never split */                            \
      } else if (n_split > 1) {                                                                  \
        VK_X3(DD, 1, true, PAD, CL);                                                             \
      } else {                                                                                   \
        VK_X3(DD, 1, false, PAD, CL);                                                            \
      }                                                                                          \
    } else if (n_split > 1) {                                                                    \
      hipLaunchKernelGGL((paged_prefill_f32<DD, kPfF32RowTiles, true, PAD, CL>), dim3(wgs),      \
                         dim3(64 * kPfF32Waves), 0, s, a, qtiles, (uint32_t)items, n_split,      \
                         part);                                                                  \
    } else {                                                                                     \
      hipLaunchKernelGGL((paged_prefill_f32<DD, kPfF32RowTiles, false, PAD, CL>), dim3(wgs),     \
                         dim3(64 * kPfF32Waves), 0, s, a, qtiles, (uint32_t)items, 1u, nullptr); \
    }                                                                                            \
    if (n_split > 1)                                                                             \
      launch_prefill_merge_f32(a, qtiles, p.rows, n_split, part, p.items, DD, s);                \
  } while (0)
  // A head_dim below the kernel's D runs the padded variant, which skips
  // what lies wholly past it where the launch has a variant that stops there
  // (64: 32 columns; 128: 80 or 96).
  const uint32_t live = (a.hd + 15) / 16;
  if (head_dim == 128) {
    if (a.hd == 128) VK_PF32(128, false, 8);
    else if (live <= 5) VK_PF32(128, true, 5);
    else if (live <= 6) VK_PF32(128, true, 6);
    else VK_PF32(128, true, 8);
  } else {
    if (a.hd == 64) VK_PF32(64, false, 4);
    else if (live <= 2) VK_PF32(64, true, 2);
    else VK_PF32(64, true, 4);
  }
#undef VK_PF32
#undef VK_X3R
#undef VK_X3
}

}  // namespace vk
