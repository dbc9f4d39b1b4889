// Decode (len_q == 1) of short contexts: a workgroup per (sequence, kv head),
// or a few of them.
//
// A workgroup walks all of the row's keys (or one of n_split equal shares of
// its 32-key steps): its waves take the steps in turn (the decode stream's
// step: K and V straight from the pool into MFMA operands, each reloaded for
// the next step as soon as the MFMAs have read it), then combine their (m, l,
// o) through LDS in wave order. Unsplit, nothing goes through memory and
// nothing is planned: one launch of a workgroup's latency (lengths, table,
// K/V: three dependent round trips), where the stream plans, writes a partial
// per wave and merges. A split row's shares write one partial per workgroup,
// merged by a second launch. decode_small_plan holds the line. Fixed work
// split: the same result on every call.
//
// V of keys outside [lo, len_k) in a row's first and last step is zeroed
// before it meets their zero probabilities, so what those rows of the pool
// hold (infinities included) does not reach the output.
//
// Fused append: workgroups past the rows' copy the new rows to their slots;
// the rows read their new key from the new rows, so no read of the launch
// depends on a write of it.
#include <algorithm>

#include "attn_decode.hpp"

namespace vk {

constexpr int kSmallWaves = 8;
constexpr uint32_t kSmallPad = 4;  // floats between rows of O in LDS (bank conflicts)

// One 16-key tile for two query heads on the VALU: lane (col, g) dots key
// col's d = 16c + 4g .. +3 with both heads (the groups' sums added with lane
// swaps), then adds p of keys 4g + i, fetched from their lanes, times its V
// values to both heads' sums.
template <int D>
struct V2State {
  float m[2] = {kNegBig, kNegBig}, l[2] = {0.f, 0.f};
  float4 o[2][D / 64] = {};
};
template <int D>
__device__ __forceinline__ void attend_half_v2(const KHalfF32<D>& kt, const VHalfF32<D>& vt,
                                               const float4 (&q)[2][D / 4], V2State<D>& st,
                                               float scale_log2, bool visible, uint32_t col,
                                               uint32_t g) {
  uint32_t gq = g;  // opaque: Q is read from LDS for every tile, not kept
  asm volatile("" : "+v"(gq));
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
#pragma unroll
    for (int c = 0; c < D / 16; ++c) {
      const float4 qc = q[h][4 * c + gq];  // (LDS, the same for a key's 16 lanes)
      s0 = __builtin_fmaf(kt.k[c].x, qc.x, s0);
      s1 = __builtin_fmaf(kt.k[c].y, qc.y, s1);
      s2 = __builtin_fmaf(kt.k[c].z, qc.z, s2);
      s3 = __builtin_fmaf(kt.k[c].w, qc.w, s3);
    }
    float s = wave_sum_g((s0 + s1) + (s2 + s3));
    if (!visible) s = -INFINITY;
    const float mx = s * scale_log2;
    if (__any(mx > st.m[h] + kRescaleSlack)) {
      float mr = mx;
#pragma unroll
      for (int x = 1; x < 16; x <<= 1) mr = fmaxf(mr, __shfl_xor(mr, x));
      const float mn = fmaxf(st.m[h], mr), f = fast_exp2(st.m[h] - mn);
      st.m[h] = mn;
      st.l[h] *= f;
#pragma unroll
      for (int b = 0; b < D / 64; ++b)
        st.o[h][b].x *= f, st.o[h][b].y *= f, st.o[h][b].z *= f, st.o[h][b].w *= f;
    }
    const float p = fast_exp2(__builtin_fmaf(s, scale_log2, -st.m[h]));
    st.l[h] += p;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float pi = __shfl(p, (int)(16 * g + 4 * g) + i);
#pragma unroll
      for (int b = 0; b < D / 64; ++b) {
        const float4& v = vt.v[i][b];
        st.o[h][b].x = __builtin_fmaf(pi, v.x, st.o[h][b].x);
        st.o[h][b].y = __builtin_fmaf(pi, v.y, st.o[h][b].y);
        st.o[h][b].z = __builtin_fmaf(pi, v.z, st.o[h][b].z);
        st.o[h][b].w = __builtin_fmaf(pi, v.w, st.o[h][b].w);
      }
    }
  }
}

// kV2 (f32, at most two query heads per kv head): the products on the VALU,
// where f32 MFMAs would spend 14 of their 16 columns on padding (4,096 cycles
// a step against ~1,300): 8 sequences of 82-401 keys, 16 q / 8 kv heads, with
// their cache write 16.8 -> 13.5 us.
template <typename T, int D, bool kFuse, bool kPad, bool kSplit, bool kV2 = false>
__global__ __launch_bounds__(64 * kSmallWaves, 1) void paged_decode_small(
    AttnArgs a, const uint32_t* __restrict__ cu_q, const uint32_t* __restrict__ cu_k,
    const uint32_t* __restrict__ table, uint32_t n_wg, uint32_t n_split_arg) {
  const uint32_t n_split = kSplit ? n_split_arg : 1u;
  constexpr int W = kSmallWaves, DPL = D / 16;
  constexpr bool kF32 = sizeof(T) == 4;
  static_assert(!kV2 || kF32, "the VALU variant is f32's");
  extern __shared__ __attribute__((aligned(16))) float o_lds[];  // [W][group][D + kSmallPad]
  __shared__ float2 ml_lds[W][16];
  if constexpr (kFuse) {
    if (blockIdx.x >= n_wg) {
      copy_new_rows<T, D>(a, blockIdx.x - n_wg, gridDim.x - n_wg);
      return;
    }
  }
  const uint32_t tid = threadIdx.x, lane = tid & 63, col = lane & 15, g = lane >> 4;
  const int32_t wave = (int32_t)__builtin_amdgcn_readfirstlane(tid >> 6);
  DecodePos p;
  const uint32_t seg = blockIdx.x / n_split, split = blockIdx.x - seg * n_split;
  p.seq = seg / a.kvh;
  p.kh = seg - p.seq * a.kvh;
  p.q0 = cu_q[p.seq];
  p.len_k = (int32_t)(cu_k[p.seq + 1] - cu_k[p.seq]);
  if (cu_q[p.seq + 1] - p.q0 != 1 || p.len_k <= 0) return;
  const int32_t lo = a.wl >= 0 ? max(0, p.len_k - 1 - a.wl) : 0, len_k = p.len_k;
  p.lo = lo;
  // This workgroup's keys: all of the row's, or its split's whole steps.
  const int32_t first = lo & ~31;
  int32_t key_end = len_k;
  p.key0 = first;
  if constexpr (kSplit) {
    const uint32_t steps = (uint32_t)(len_k - first + 31) >> 5;
    p.key0 = first + 32 * (int32_t)(split * steps / n_split);
    key_end = min(len_k, first + 32 * (int32_t)((split + 1) * steps / n_split));
  }
  p.key0 += 32 * wave;
  p.fuse = 0;
  if constexpr (kFuse) {
    p.fuse = fused_row(a, cu_q, cu_k, table, p.seq);
  }

  float m_run = kNegBig, l_run = 0.f;
  V2State<D> v2;
  floatx4 o[DPL];
#pragma unroll
  for (int k = 0; k < DPL; ++k) o[k] = floatx4{0.f, 0.f, 0.f, 0.f};
  const uint32_t count = vhead_count(a, p.kh), h0 = vhead_base(a, p.kh);
  const uint32_t hd = kPad ? a.hd : (uint32_t)D;
  const T* qrow0 = (const T*)a.q + ((uint64_t)p.q0 * a.num_heads + h0) * hd;
  const T* qrow = qrow0 + (col < count ? col : 0) * hd;

  const uint32_t sg = a.q_sign ? 0x80000000u : 0u;
  __shared__ float4 q_lds[kV2 ? 2 : 1][kV2 ? D / 4 : 1];
  if constexpr (kV2) {
    if (tid < 2 * (D / 4)) {
      const uint32_t h = tid / (D / 4), d = 4 * (tid % (D / 4));
      uint4 x = make_uint4(0u, 0u, 0u, 0u);
      if (d < hd) x = *(const uint4*)(qrow0 + (h < count ? h : 0) * hd + d);
      q_lds[h][d / 4] = make_float4(__uint_as_float(x.x ^ sg), __uint_as_float(x.y ^ sg),
                                    __uint_as_float(x.z ^ sg), __uint_as_float(x.w ^ sg));
    }
    __syncthreads();
  }
  if (p.key0 < key_end) {
    auto visible = [&](int32_t key) { return key >= lo && key < len_k; };
    if constexpr (kF32) {
      const float* kb = (const float*)a.k + a.kv_parts.div(p.kh) * a.head_e;
      const float* vb = (const float*)a.v + a.kv_parts.div(p.kh) * a.head_e;
      const uint32_t* tab = table + (uint64_t)p.seq * a.max_blocks;
      KTileF32<D> kt;
      VTileF32<D> vt;
      auto load = [&](int tt, int32_t s0) __attribute__((always_inline)) {
        load_half_f32<D, true, kPad>(kt.h[tt], vt.h[tt], tab, kb, vb, a, s0, tt, len_k - 1, col, g);
      };
      load(0, p.key0);
      load(1, p.key0);
      float4 qf[D / 16];
      if constexpr (!kV2) {
#pragma unroll
        for (int c = 0; c < D / 16; ++c) {
          uint4 x = make_uint4(0u, 0u, 0u, 0u);
          if (!kPad || 16 * c + 4 * g < hd) x = *(const uint4*)(qrow + 16 * c + 4 * g);
          qf[c] = make_float4(__uint_as_float(x.x ^ sg), __uint_as_float(x.y ^ sg),
                              __uint_as_float(x.z ^ sg), __uint_as_float(x.w ^ sg));
        }
      }
      auto attend = [&](int tt, int32_t s0) __attribute__((always_inline)) {
        const int32_t k0 = s0 + 16 * tt + 4 * (int32_t)g;
        if (s0 < lo || s0 + 32 > len_k) {  // (uniform)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (!visible(k0 + i))
#pragma unroll
              for (int h = 0; h < D / 64; ++h) vt.h[tt].v[i][h] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
        if constexpr (kV2)
          attend_half_v2<D>(kt.h[tt], vt.h[tt], q_lds, v2, a.scale_log2,
                            visible(s0 + 16 * tt + (int32_t)col), col, g);
        else
          attend_half_f32<D>(kt.h[tt], vt.h[tt], qf, o, m_run, l_run, a.scale_log2,
                             [&](int i) { return visible(k0 + i); });
      };
      int32_t s0 = p.key0;
      for (; s0 + 32 * W < key_end; s0 += 32 * W) {
        attend(0, s0);
        load(0, s0 + 32 * W);
        attend(1, s0);
        load(1, s0 + 32 * W);
      }
      attend(0, s0);
      attend(1, s0);
    } else {
      KTile<D> kt;
      VTile<D> vt;
      auto load_kt = [&]() __attribute__((always_inline)) {
        load_step_k<T, D, kPad>(kt, a, table, p, col, g);
      };
      auto load_vt = [&]() __attribute__((always_inline)) {
        load_step_v<T, D, kPad>(vt, a, table, p, col, g);
      };
      load_kt();
      load_vt();
      uint4 qf[D / 32];
#pragma unroll
      for (int c = 0; c < D / 32; ++c) {
        uint4 x = make_uint4(0u, 0u, 0u, 0u);
        if (!kPad || 32 * c + 8 * g < hd) x = *(const uint4*)(qrow + 32 * c + 8 * g);
        qf[c] = make_uint4(x.x ^ a.q_sign, x.y ^ a.q_sign, x.z ^ a.q_sign, x.w ^ a.q_sign);
      }
      auto scores = [&](int32_t s0) __attribute__((always_inline)) {
        const int32_t k0 = s0 + 4 * (int32_t)g;
        return attend_qk<T, D>(kt, qf, o, m_run, l_run, a.scale_log2, g,
                               [&](int tt, int i) { return visible(k0 + 16 * tt + i); });
      };
      auto values = [&](uint4 pf, int32_t s0) __attribute__((always_inline)) {
        if (s0 < lo || s0 + 32 > len_k) {  // (uniform)
          const int32_t k0 = s0 + 4 * (int32_t)g;
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (!visible(k0 + 16 * (j >> 2) + (j & 3)))
#pragma unroll
              for (int w = 0; w < DPL / 2; ++w) vt.v[j].w[w] = 0u;
        }
        attend_pv<T, D>(vt, pf, o);
      };
      // K and V are reloaded for the next step as soon as this one's MFMAs
      // have read them; the last step of a wave loads nothing.
      while (true) {
        const int32_t s0 = p.key0;
        if (s0 + 32 * W >= key_end) break;
        p.key0 += 32 * W;
        const uint4 pf = scores(s0);
        load_kt();
        values(pf, s0);
        load_vt();
      }
      const int32_t s0 = p.key0;
      values(scores(s0), s0);
    }
  }

  constexpr uint32_t S = D + kSmallPad;
  if constexpr (kV2) {
    // Lane (g, col) holds the sums of its keys at d = 64 b + 4 col + j.
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float l = v2.l[h];  // a lane per key, the same in the four groups
#pragma unroll
      for (int x = 1; x < 16; x <<= 1) l += __shfl_xor(l, x);
      if (lane == 0) ml_lds[wave][h] = make_float2(v2.m[h], l);
#pragma unroll
      for (int b = 0; b < D / 64; ++b) {
        float4 y = v2.o[h][b];
        y.x = wave_sum_g(y.x), y.y = wave_sum_g(y.y), y.z = wave_sum_g(y.z), y.w = wave_sum_g(y.w);
        if (g == 0 && h < (int)count)
          *(float4*)(o_lds + ((uint32_t)wave * a.group + h) * S + 64 * b + 4 * col) = y;
      }
    }
  } else {
    const float l_tot = wave_sum_g(l_run);
    if (g == 0) ml_lds[wave][col] = make_float2(m_run, l_tot);
    if (col < count) {
      float* row = o_lds + ((uint32_t)wave * a.group + col) * S;
      if constexpr (kF32) {
        store_row_f32<D>(row, o, 1.f, g);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int k = 0; k < DPL; k += 4)
            *(float4*)(row + v_d<D>(4 * g + i, k)) =
                make_float4(o[k][i], o[k + 1][i], o[k + 2][i], o[k + 3][i]);
      }
    }
  }
  __syncthreads();
  for (uint32_t e = 4 * tid; e < count * D; e += 4 * 64 * W) {
    const uint32_t c = e / D, d = e % D;
    if (kPad && d >= hd) continue;
    float m[W], l[W], M = kNegBig, L = 0.f;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const float2 x = ml_lds[w][c];
      m[w] = x.x, l[w] = x.y;
      M = fmaxf(M, m[w]);
    }
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const float f = fast_exp2(m[w] - M);
      const float4 y = *(const float4*)(o_lds + ((uint32_t)w * a.group + c) * S + d);
      L += l[w] * f;
      x.x += y.x * f, x.y += y.y * f, x.z += y.z * f, x.w += y.w * f;
    }
    if constexpr (kSplit) {
      const uint64_t slot = (uint64_t)blockIdx.x * a.group + c;
      *(float4*)(a.ws_o + slot * D + d) = x;
      if (d == 0) *(float2*)(a.ws_ml + slot * 2) = make_float2(M, L);
      continue;
    }
    const float inv = L > 0.f ? 1.f / L : 0.f;
    T* dst = (T*)a.out + ((uint64_t)p.q0 * a.num_heads + h0 + c) * hd + d;
    if constexpr (kF32)
      *(float4*)dst = make_float4(x.x * inv, x.y * inv, x.z * inv, x.w * inv);
    else
      *(uint2*)dst = make_uint2(pack2<T>(x.x * inv, x.y * inv), pack2<T>(x.z * inv, x.w * inv));
  }
}

// Combines a split row's partials, a workgroup per (sequence, kv head):
// thread (part of the splits, four outputs), the parts through LDS in order.
template <typename T, int D, bool kPad>
__global__ __launch_bounds__(64 * kSmallWaves) void paged_decode_small_merge(
    AttnArgs a, const uint32_t* __restrict__ cu_q, const uint32_t* __restrict__ cu_k,
    uint32_t n_split) {
  constexpr uint32_t NT = 64 * kSmallWaves;
  __shared__ float4 o_s[NT];
  __shared__ float2 ml_s[NT];
  const uint32_t seq = blockIdx.x / a.kvh, kh = blockIdx.x - seq * a.kvh;
  const uint32_t q0 = cu_q[seq], q1 = cu_q[seq + 1], k0 = cu_k[seq], k1 = cu_k[seq + 1];
  if ((q1 - q0 != 1) | ((int32_t)(k1 - k0) <= 0)) return;
  const uint32_t count = vhead_count(a, kh), h0 = vhead_base(a, kh), tid = threadIdx.x;
  const uint32_t hd = kPad ? a.hd : (uint32_t)D;
  const uint32_t per = min(a.group * (D / 4), NT);  // threads side by side
  const uint32_t parts = min(NT / per, n_split), part = tid / per;
  for (uint32_t e0 = 0; e0 < a.group * D; e0 += 4 * per) {
    const uint32_t e = e0 + 4 * (tid - part * per), c = e / D, d = e % D;
    float M = kNegBig, L = 0.f;
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
    if (part < parts && c < a.group) {
      constexpr uint32_t kB = 8;  // splits per round trip
      for (uint32_t s0 = part; s0 < n_split; s0 += kB * parts) {
        float2 ml[kB];
        float4 y[kB];
#pragma unroll
        for (uint32_t u = 0; u < kB; ++u) {
          const uint32_t s = s0 + u * parts;
          const bool in = s < n_split;
          const uint64_t slot = ((uint64_t)blockIdx.x * n_split + (in ? s : part)) * a.group + c;
          ml[u] = *(const float2*)(a.ws_ml + slot * 2);
          y[u] = *(const float4*)(a.ws_o + slot * D + d);
          if (!in) ml[u].y = 0.f;
        }
        float Mn = M;
#pragma unroll
        for (uint32_t u = 0; u < kB; ++u) Mn = fmaxf(Mn, ml[u].y > 0.f ? ml[u].x : kNegBig);
        const float f = fast_exp2(M - Mn);
        L *= f, x.x *= f, x.y *= f, x.z *= f, x.w *= f;
#pragma unroll
        for (uint32_t u = 0; u < kB; ++u) {
          if (!(ml[u].y > 0.f)) continue;  // a share without keys, or past the last
          const float w = fast_exp2(ml[u].x - Mn);
          L += ml[u].y * w;
          x.x += y[u].x * w, x.y += y[u].y * w, x.z += y[u].z * w, x.w += y[u].w * w;
        }
        M = Mn;
      }
    }
    if (parts > 1) {
      o_s[tid] = x;
      ml_s[tid] = make_float2(M, L);
      __syncthreads();
      if (part == 0) {
        float Mn = M;
        for (uint32_t p = 1; p < parts; ++p) Mn = fmaxf(Mn, ml_s[p * per + tid].x);
        const float f = fast_exp2(M - Mn);
        L *= f, x.x *= f, x.y *= f, x.z *= f, x.w *= f;
        for (uint32_t p = 1; p < parts; ++p) {
          const float2 ml = ml_s[p * per + tid];
          const float4 y = o_s[p * per + tid];
          const float w = fast_exp2(ml.x - Mn);
          L += ml.y * w;
          x.x += y.x * w, x.y += y.y * w, x.z += y.z * w, x.w += y.w * w;
        }
      }
      __syncthreads();  // the LDS is reused by the next outputs
    }
    if (part == 0 && c < count && d < hd) {
      const float inv = L > 0.f ? 1.f / L : 0.f;
      T* dst = (T*)a.out + ((uint64_t)q0 * a.num_heads + h0 + c) * hd + d;
      if constexpr (sizeof(T) == 4)
        *(float4*)dst = make_float4(x.x * inv, x.y * inv, x.z * inv, x.w * inv);
      else
        *(uint2*)dst = make_uint2(pack2<T>(x.x * inv, x.y * inv), pack2<T>(x.z * inv, x.w * inv));
    }
  }
}

static size_t small_lds(uint32_t group, uint32_t head_dim) {
  return (size_t)kSmallWaves * group * (head_dim + kSmallPad) * sizeof(float);
}

static size_t small_part_bytes(uint64_t wgs, uint32_t group, uint32_t head_dim) {
  return (size_t)(wgs * group * (head_dim + 2) * sizeof(float));
}

// The line against the decode stream, in bytes of K per row (`bytes`: the
// host's bound on a row's keys): a workgroup streams its share at ~25 KB/us
// after ~4.5 us, and a split's merge adds ~3.5 us; the stream and its merge
// take 12-16 us for any small batch. Measured (32 q / 8 kv heads, bf16, us,
// stream / this): 1 x 100 keys 15.4 / 4.7, 1 x 300 15.3 / 6.7 (split 8.3),
// 1 x 700 15.4 / 8.7 (unsplit 10.1), 1 x 8,191 20.1 / 13.1, 4 x 2,000 16.8 /
// 12.4, 16 x 700 19.4 / 13.8, 32 x 300 19.6 / 10.1, 32 x 700 26.6 / 18.4; f32
// (the VALU kernel or the stream / this): 8 x 200 (16 q / 8 kv heads) 12.2 /
// 10.6, 8 x 500 16.0 / 12.8, 32 x 300 26.5 / 16.2, 2 x 300 (32 q / 8 kv
// heads) 11.7 / 10.4. Batches of equal contexts gain far
// past this line (16 x 3,000: 43.6 / 37.9), but a share of a long row beside
// short ones ends after the balanced stream does (16 rows of 700 to 8,007
// keys: 44.5 / 79.4), and the host knows only the longest: so a workgroup
// gets at most kSmallMaxBytes, where a batch of one such row and any others
// still wins.
constexpr uint64_t kSmallWgs = 256;            // workgroups at once, one per CU
constexpr uint64_t kSmallUnsplit = 120 << 10;  // rows up to this are not split,
constexpr uint64_t kSmallUnsplitF32 = 72 << 10;  // (on f32 MFMAs, which bound a share)
constexpr uint64_t kSmallShare = 32 << 10;     // else into shares of at least this
constexpr uint64_t kSmallMaxBytes = 160 << 10;
SmallPlan decode_small_plan(uint32_t batch, uint32_t kvh, uint32_t group, uint32_t head_dim,
                            uint32_t dtype, uint32_t max_k, int32_t wl, size_t part_bytes) {
  const uint64_t seg = (uint64_t)batch * kvh;
  // O of every wave in LDS, within what a launch gets without asking.
  if (seg > kSmallWgs || small_lds(group, head_dim) > 56 * 1024) return {false, 1};
  const bool f32 = dtype == VAPI_KV_F32;
  const uint64_t span = wl >= 0 ? std::min<uint64_t>(max_k, (uint64_t)wl + 32) : max_k;
  const uint64_t bytes = span * head_dim * (f32 ? 4 : 2);
  uint64_t n = 1;
  if (bytes > (f32 && group > 2 ? kSmallUnsplitF32 : kSmallUnsplit))
    n = std::max<uint64_t>(std::min<uint64_t>(kSmallWgs / seg, (bytes + kSmallShare - 1) / kSmallShare), 1);
  n = std::min<uint64_t>(n, 32);
  while (n > 1 && small_part_bytes(seg * n, group, head_dim) > part_bytes) --n;
  return {bytes <= n * kSmallMaxBytes, (uint32_t)n};
}

void launch_decode_small(const AttnArgs& a_in, uint32_t head_dim, uint32_t dtype, SmallPlan plan,
                         void* part, hipStream_t s) {
  AttnArgs a = a_in;
  const uint32_t n_seg = a.batch * a.kvh, n_split = plan.n_split, n_wg = n_seg * n_split;
  const bool fuse = a.k_new != nullptr, pad = a.hd != head_dim;
  a.ws_o = (float*)part;
  a.ws_ml = (float*)part + (uint64_t)n_wg * a.group * head_dim;
  uint32_t copy_wgs = 0;
  if (fuse) {
    const uint64_t chunks = 2ull * a.n_new * a.kvh * (head_dim / 8);
    copy_wgs = (uint32_t)std::min<uint64_t>((chunks + 64 * kMergeWaves - 1) / (64 * kMergeWaves), 1024);
  }
  const size_t lds = small_lds(a.group, head_dim);
  const dim3 grid(n_wg + copy_wgs), block(64 * kSmallWaves);
#define VK_SM(T, DD, F, PAD) VK_SM2(T, DD, F, PAD, false)
#define VK_SM2(T, DD, F, PAD, V2)                                                                 \
  do {                                                                                            \
    if (n_split > 1) {                                                                            \
      hipLaunchKernelGGL((paged_decode_small<T, DD, F, PAD, true, V2>), grid, block, lds, s, a,   \
                         a.cu_q, a.cu_k, a.table, n_wg, n_split);                                 \
      hipLaunchKernelGGL((paged_decode_small_merge<T, DD, PAD>), dim3(n_seg), block, 0, s, a,     \
                         a.cu_q, a.cu_k, n_split);                                                \
    } else {                                                                                      \
      hipLaunchKernelGGL((paged_decode_small<T, DD, F, PAD, false, V2>), grid, block, lds, s, a,  \
                         a.cu_q, a.cu_k, a.table, n_wg, 1u);                                      \
    }                                                                                             \
  } while (0)
  // Fused appends run on a kernel's own head dims only.
#define VK_SM_D(T, DD)                        \
  do {                                        \
    if (pad) VK_SM(T, DD, false, true);       \
    else if (fuse) VK_SM(T, DD, true, false); \
    else VK_SM(T, DD, false, false);          \
  } while (0)
#define VK_SM_F(DD, PAD)                                        \
  do {                                                          \
    if (a.group <= 2) VK_SM2(float, DD, false, PAD, true);      \
    else VK_SM(float, DD, false, PAD);                          \
  } while (0)
  if (dtype == VAPI_KV_F32) {  // no fused append
    if (head_dim == 128 && pad) VK_SM_F(128, true);
    else if (head_dim == 128) VK_SM_F(128, false);
    else if (pad) VK_SM_F(64, true);
    else VK_SM_F(64, false);
  } else if (dtype == VAPI_KV_BF16) {
    if (head_dim == 256) VK_SM_D(bf16_t, 256);
    else if (head_dim == 128) VK_SM_D(bf16_t, 128);
    else VK_SM_D(bf16_t, 64);
  } else {
    if (head_dim == 256) VK_SM_D(f16_t, 256);
    else if (head_dim == 128) VK_SM_D(f16_t, 128);
    else VK_SM_D(f16_t, 64);
  }
#undef VK_SM_F
#undef VK_SM_D
#undef VK_SM2
#undef VK_SM
}

}  // namespace vk
