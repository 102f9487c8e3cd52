// Query rows straight from qkv into the MFMA B-operand registers (norm, rotate-half RoPE, softmax scale), shared by
// the dense and the tiled band kernels.
//
// Lane (lr, lh) of a wave holds the 16-byte chunks 2 kk + lh (dims 16 kk + 8 lh .. + 8) of query lr of a column
// tile, which is what the B operand of S^T = K Q^T wants: lanes exchange only what the row's sum of squares needs,
// and with one column tile per wave no row is prepared twice. A rotary pair (chunks c and c + half / 8) lies in one
// lane whenever half is a multiple of 16; otherwise the partner chunk belongs to the other lane half and each lane
// loads and normalises it a second time (B = 2, L = 2584, 4 x 64, one workgroup per CU: 52.1 us at half 24 against 48.5
// at 16; 49.6 at 24 when a lane held the whole row).
//
// The prologue is bound by latency (nothing else runs on the SIMD yet), so every load of it is issued before the
// first use. Before, each lane prepared a whole row and v_permlane32_swap redistributed it; with one column tile the
// two lane halves did the same row, and at head_dim 128 the tables were loaded chunk by chunk. Prologue with the
// softmax plan, median of the workgroups' timestamps: head_dim 128 with 8 waves 12.8 -> 6.5 us, head_dim 64 with 64
// queries 5.4 -> 3.5; the self-attention calls of B = 2, L = 1292, 12 x 128 (fp16) 109.5 -> 101.5 us and of B = 1,
// L = 1422, 24 x 64 (bf16) 48.2 -> 46.1.
#pragma once

#include <type_traits>

#include "common.h"

namespace hb {

// RMSNorm (dit.py:45-57) with the dense path's cast points: the compute dtype IO after the gain and after the
// rotation (dense_attention.py:66, 69).
template <class IO, int D>
struct RmsQuery {
  struct Par {
    f32x4 w[2];
  };
  const float* __restrict__ qw;
  float eps;

  __device__ __forceinline__ Par par(int chunk) const {
    const f32x4_align4* p = reinterpret_cast<const f32x4_align4*>(qw + 8 * chunk);
    return Par{{p[0], p[1]}};
  }
  // 1 / rms of every row, in both lane halves. A row's squares are added in the order of its dims, as by a lane that
  // holds the whole row, so that a seed renders the same bits as with such lanes: the sum of the two halves' own sums
  // rounds otherwise, which moves 2e-4 of an attention's results by one bf16 step and, over the 24 blocks of a
  // denoiser, its output by 2e-2. Two rows are added by one lane half each, which gets the other's chunks (one chain of
  // D additions for both); for a single row the sum goes from half to half. Against the halves' own sums:
  // cross-attention B = 2, L = 2584 x 257, 24 x 64 33.4 -> 33.5 us, L = 8192 x 33 26.4 -> 27.5, 12 x 128 37.1 -> 37.7;
  // self-attention B = 2, L = 1292, 12 x 128 97.6 -> 98.3, 24 x 64 unchanged.
  template <int NCT>
  __device__ __forceinline__ void stats(const u32x4 (&raw)[NCT][1][D / 16], float (&st)[NCT][1]) const {
    static_assert(NCT == 1 || NCT == 2, "one row, or one per lane half");
    float ss = 0.f;
    auto add = [&](u32x4 chunk) {
      float x[8];
      IO::unpack8(chunk, x);
#pragma unroll
      for (int j = 0; j < 8; ++j) ss = __fmaf_rn(x[j], x[j], ss);
    };
    auto halves = [](float v, float (&h)[2]) {  // lanes 0-31's value and lanes 32-63's, each in both
      const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
      h[0] = __uint_as_float(r[0]);
      h[1] = __uint_as_float(r[1]);
    };
    float h[2];
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk) {
      if constexpr (NCT == 1) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {  // chunk 2 kk + i, this lane's in half i
          add(raw[0][0][kk]);
          halves(ss, h);
          ss = h[i];
        }
      } else {
        u32x4 c[2];  // chunks 2 kk and 2 kk + 1 of the first row in lanes 0-31, of the second in lanes 32-63
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const auto r = __builtin_amdgcn_permlane32_swap(raw[0][0][kk][e], raw[1][0][kk][e], false, false);
          c[0][e] = r[0];
          c[1][e] = r[1];
        }
        add(c[0]);
        add(c[1]);
      }
    }
    const float inv = rsqrtf(ss / static_cast<float>(D) + eps);
    halves(inv, h);
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) st[ct][0] = h[ct];
  }
  __device__ __forceinline__ void apply(u32x4 raw, const Par& p, float inv, float (&y)[8]) const {
    IO::unpack8(raw, y);
#pragma unroll
    for (int j = 0; j < 8; ++j) y[j] = IO::round((y[j] * inv) * p.w[j >> 2][j & 3]);
  }
  // rotate_half (dit.py:96-98): d < half takes -x[d + half], d >= half takes x[d - half]
  __device__ static __forceinline__ float rot1(float y1, float y2, float c, float s) {
    return IO::round(y1 * c + (-y2) * s);
  }
  __device__ static __forceinline__ float rot2(float y1, float y2, float c, float s) {
    return IO::round(y2 * c + y1 * s);
  }
};

// DyT (same_l.py:58-69) in fp32 with the one bf16 rounding at the end (band_attention.py:82-85, 104).
template <class IO, int D>
struct DytQuery {
  struct Par {
    f32x4 g[2], b[2];
  };
  const float* __restrict__ dyt;  // [alpha, gamma[D], beta[D]]

  __device__ __forceinline__ Par par(int chunk) const {
    const f32x4_align4* g = reinterpret_cast<const f32x4_align4*>(dyt + 1 + 8 * chunk);
    const f32x4_align4* b = reinterpret_cast<const f32x4_align4*>(dyt + 1 + D + 8 * chunk);
    return Par{{g[0], g[1]}, {b[0], b[1]}};
  }
  template <int NCT, int NB>
  __device__ __forceinline__ void stats(const u32x4 (&)[NCT][NB][D / 16], float (&st)[NCT][NB]) const {
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
      for (int b = 0; b < NB; ++b) st[ct][b] = 2.f * kLog2e * dyt[0];
  }
  __device__ __forceinline__ void apply(u32x4 raw, const Par& p, float a2, float (&y)[8]) const {
    IO::unpack8(raw, y);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float g = p.g[j >> 2][j & 3], b = p.b[j >> 2][j & 3];
      y[j] = dyt_tanh(y[j], a2, -2.f * g, g + b);
    }
  }
  __device__ static __forceinline__ float rot1(float y1, float y2, float c, float s) {
    return __fmaf_rn(y1, c, -(y2 * s));
  }
  __device__ static __forceinline__ float rot2(float y1, float y2, float c, float s) {
    return __fmaf_rn(y2, c, y1 * s);
  }
};

__device__ __forceinline__ u32x4 pack_scaled(const float (&y)[8], float qscale) {
  float o[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) o[j] = y[j] * qscale;
  return pack8(o);  // the packing conversion is the final bf16 rounding
}

// One column tile's rows of NB branches, half = 16 E: chunks kk and kk + E of a lane are a rotary pair.
template <int E, int D, int NB, int NCT, class Q>
__device__ __forceinline__ void rotate_even(const Q& q, const u32x4 (&raw)[NB][D / 16],
                                            const typename Q::Par (&par)[D / 16], const float (&st)[NB],
                                            const float* __restrict__ cs, const float* __restrict__ sn, int lh,
                                            float qscale, u32x4 (&out)[NB][NCT][D / 16], int ct) {
  f32x4 cv[E + 1][2], sv[E + 1][2];
#pragma unroll
  for (int kk = 0; kk < E; ++kk)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      cv[kk][u] = *reinterpret_cast<const f32x4*>(cs + 16 * kk + 8 * lh + 4 * u);
      sv[kk][u] = *reinterpret_cast<const f32x4*>(sn + 16 * kk + 8 * lh + 4 * u);
    }
#pragma unroll
  for (int b = 0; b < NB; ++b) {
#pragma unroll
    for (int kk = 0; kk < E; ++kk) {
      float y1[8], y2[8], o1[8], o2[8];
      q.apply(raw[b][kk], par[kk], st[b], y1);
      q.apply(raw[b][kk + E], par[kk + E], st[b], y2);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float c = cv[kk][j >> 2][j & 3], s = sv[kk][j >> 2][j & 3];
        o1[j] = Q::rot1(y1[j], y2[j], c, s);
        o2[j] = Q::rot2(y1[j], y2[j], c, s);
      }
      out[b][ct][kk] = pack_scaled(o1, qscale);
      out[b][ct][kk + E] = pack_scaled(o2, qscale);
    }
#pragma unroll
    for (int kk = 2 * E; kk < D / 16; ++kk) {
      float y[8];
      q.apply(raw[b][kk], par[kk], st[b], y);
      out[b][ct][kk] = pack_scaled(y, qscale);
    }
  }
}

// half = 8 h8 with h8 odd: the partner chunk is the other lane half's, loaded again.
template <int D, int NB, int NCT, class Q>
__device__ __forceinline__ void rotate_odd(const Q& q, const uint16_t* const (&row)[NB],
                                           const u32x4 (&raw)[NB][D / 16], const float (&st)[NB],
                                           const float* __restrict__ cs,
                                           const float* __restrict__ sn, int h8, int lh, float qscale,
                                           u32x4 (&out)[NB][NCT][D / 16], int ct) {
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk) {
    const int c = 2 * kk + lh;
    const bool first = c < h8, rot = kk < h8;  // chunks 0 .. 2 h8 - 1 rotate: kk < h8 in both lane halves
    const int p = !rot ? c : first ? c + h8 : c - h8;
    f32x4 cv[2] = {}, sv[2] = {};
    const typename Q::Par own = q.par(c), other = q.par(p);
    if (rot) {
      const int t = 8 * (first ? c : p);
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        cv[u] = *reinterpret_cast<const f32x4*>(cs + t + 4 * u);
        sv[u] = *reinterpret_cast<const f32x4*>(sn + t + 4 * u);
      }
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      float y[8];
      q.apply(raw[b][kk], own, st[b], y);
      if (rot) {
        float z[8];
        q.apply(ld16(row[b] + 8 * p), other, st[b], z);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float co = cv[j >> 2][j & 3], si = sv[j >> 2][j & 3];
          y[j] = first ? Q::rot1(y[j], z[j], co, si) : Q::rot2(z[j], y[j], co, si);
        }
      }
      out[b][ct][kk] = pack_scaled(y, qscale);
    }
  }
}

// Raw chunks of every row a wave prepares: branch b of column tile ct is `row[ct][b]` (D elements in qkv). Issue the
// loads with `load`, then finish with `prep` once the softmax plan is known.
template <class Q, int D, int NB, int NCT>
struct QueryRows {
  const uint16_t* row[NCT][NB];
  u32x4 raw[NCT][NB][D / 16];
  typename Q::Par par[D / 16];

  __device__ __forceinline__ void load(const Q& q, int lh) {
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk) raw[ct][b][kk] = ld16(row[ct][b] + 16 * kk + 8 * lh);
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk) par[kk] = q.par(2 * kk + lh);
  }

  // `cs[ct]`, `sn[ct]`: the (half) columns of the tables of this lane's row of column tile ct (unused when half is 0;
  // ROPE false: half is known to be 0).
  template <bool ROPE = true>
  __device__ __forceinline__ void prep(const Q& q, const float* const (&cs)[NCT], const float* const (&sn)[NCT],
                                       int half, int lh, float qscale, u32x4 (&qf)[NB][NCT][D / 16]) const {
    float st[NCT][NB];
    q.stats(raw, st);
    const int h8 = half / 8;  // half % 8 == 0 and half <= D / 2 are checked on the host
    if constexpr (!ROPE) {
      even<0>(q, st, cs, sn, lh, qscale, qf);
      return;
    }
    if (h8 & 1) {
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct)
        rotate_odd<D, NB, NCT>(q, row[ct], raw[ct], st[ct], cs[ct], sn[ct], h8, lh, qscale, qf, ct);
    } else if (h8 == 0) {
      even<0>(q, st, cs, sn, lh, qscale, qf);
    } else if (h8 == 2) {
      even<1>(q, st, cs, sn, lh, qscale, qf);
    } else if (D == 64 || h8 == 4) {
      even<2>(q, st, cs, sn, lh, qscale, qf);
    } else if constexpr (D == 128) {
      if (h8 == 6) even<3>(q, st, cs, sn, lh, qscale, qf);
      else even<4>(q, st, cs, sn, lh, qscale, qf);
    }
  }

 private:
  template <int E>
  __device__ __forceinline__ void even(const Q& q, const float (&st)[NCT][NB], const float* const (&cs)[NCT],
                                       const float* const (&sn)[NCT], int lh, float qscale,
                                       u32x4 (&qf)[NB][NCT][D / 16]) const {
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct)
      rotate_even<E, D, NB, NCT>(q, raw[ct], par, st[ct], cs[ct], sn[ct], lh, qscale, qf, ct);
  }
};

}  // namespace hb
