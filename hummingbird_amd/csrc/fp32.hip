// fp32 inputs: the dense and band differential attentions at fp32 accuracy.
//
// This is the parity path of the reference's FP32_PARITY preset (sa3jax/dtypes.py:41-49), under which every
// cast of the XLA chain is a no-op: RMSNorm or DyT, RoPE, the logits, the softmax, P V and the subtraction all
// stay fp32 (sa3jax/dit.py:45-57, 90-98, 113-119, 146; sa3jax/same_l.py:58-69, 92-100, 134-148, 168-169).
// Norms, RoPE, softmax, row sums, accumulators and the subtraction are fp32. The two products run on the half
// matrix cores (v_mfma_f32_32x32x16_f16, 16 times the rate of the fp32 ones) on operands split exactly enough not to
// lose fp32 accuracy: x = hi + lo, hi = half(x), lo = half(x - hi), which leaves at most 2^-23 of x, and three products
// lo hi + hi lo + hi hi (the lo lo one left out is below 2^-22 of the product at its largest, 2^-25 rms) accumulated in
// fp32. An fp32 MFMA chain rounds its accumulator once per two dims and key tile after key tile; these round it three
// times per sixteen, and a tile's P V is added up apart, so the results are nearer to the 64-bit ones than the fp32
// chain's were: relative error (2-norm) 3.4e-7 against 8.9e-7 on dense B = 2, L = 1292, 2.8e-7 against 6.9e-7 on the
// band at S = 16384, w = 128. Times, whole calls against the fp32 matrix cores fed through registers: dense (2, 1292,
// 24 heads) 529 -> 186 us, L = 2584 1570 -> 594, head_dim 128 (2, 1292, 12 heads) 684 -> 166, cross (2, 2584 x 257) 204
// -> 75, band S = 16384, w = 128 467 -> 141. Three bf16 terms and six products, which need no scaling, were measured
// too: 290 us for the first of these. The matrix cores slow down on such operands (about 27 ns per 32x32x16 product and
// SIMD), so the number of products sets the time.
//
//   S^T[key][query] = K Q^T   A = K rows from LDS, B = q in registers
//   P = exp2(S^T c - m)       m the max of the tile's S^T c, one FMA per score; masked scores are -inf and give 0
//   acc = V^T P^T             A = V^T rows from LDS, B = P straight from the S^T accumulators
//   O^T[d][query] += acc      online softmax: one factor per query takes the tile's share to the running max
//
// Ranges. A half holds 2^-24 .. 65504, so every operand is scaled by powers of two (exact, undone in c and at the end):
//   - dim d of the keys by 2^k[d] and of the queries by 2^q[d], from the norm parameters (ScaleTable), so that gains
//     of many magnitudes leave no dim out; then each key tile and each query row by a power of two from its own largest
//     value, so that neither tables that are no rotation nor norms far below their bounds leave the half range. What a
//     half cannot hold is below 2^-37 of a tile's largest key value and 2^-39 of a row's largest query value, so
//     scaled.
//   - V by a power of two per key tile, from the tile's largest magnitude and stored with the tile. A tile whose keys
//     or dims differ too much for that (VTile), or that holds an infinity or NaN, keeps its fp32 bits, and its P V runs
//     on the fp32 matrix cores: every dim and every query has fp32 accuracy relative to its own size, whatever other
//     values V holds.
//   - P by 2^14, relative to the tile's own largest.
//
// Work split: a workgroup (4 waves) owns 64 queries of one (batch, head); waves 0-1 run branch 1 on 32 queries
// each, waves 2-3 branch 2, and the branch-2 waves hand lam * O2 / l2 to the branch-1 waves through LDS. Keys
// stream through LDS in 32-key tiles, prepared once per call into the workspace as the bytes the tile has in LDS
// (K, K_diff and V^T, each a plane of hi and a plane of lo halves: the 4 bytes per value of the fp32 rows) and copied
// there by DMA. The band call without a workspace prepares the tiles of each query block's window itself.
#include "api.h"
#include "attn_tile.h"
#include "common.h"
#include "tiles.h"

namespace hb {

__device__ __forceinline__ f32x4 ld4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ void st4(float* p, f32x4 v) { *reinterpret_cast<f32x4*>(p) = v; }

// One key tile, the same bytes in LDS and in the workspace: K, K_diff and V, each a hi and a lo plane of KT x D halves.
// K planes are [key][d], V planes V^T [d][position] in v_tile_key order; the 16-byte chunks of a row are XOR-swizzled,
// so that the 16 rows that a pass of the operand reads takes fall in distinct banks.
// D = 64: two stages (48 KB), three workgroups per CU (161 VGPRs). D = 128: one (48 KB), two workgroups per CU by
// registers (256 VGPRs).
template <int D>
struct SplitTile {
  static constexpr int KT = 32;
  static constexpr int PLANE = KT * D;       // halves per plane
  static constexpr int TENSOR = 2 * PLANE;   // hi and lo
  static constexpr int STAGE = 3 * TENSOR;   // K, K_diff, V
  static constexpr int STAGES = D == 64 ? 2 : 1;
  static constexpr int OCC = D == 64 ? 3 : 2;  // workgroups per CU
  static constexpr int ELEMS = STAGES * STAGE;
  static constexpr int VN = PLANE / 8 / 256;   // (dim, 8 positions) chunks of V per thread
  static constexpr int XBUF_BYTES = 2 * (D / 32) * 16 * 64 * 4;  // epilogue hand-over, aliases the stages
  static_assert(XBUF_BYTES <= 2 * ELEMS, "epilogue buffer must fit in the stages");
  __device__ static __forceinline__ int k_at(int row, int chunk) { return swz<D>(row, chunk); }
  __device__ static __forceinline__ int v_at(int d, int chunk) { return d * KT + 8 * (chunk ^ ((d >> 2) & 3)); }
};

// x - h for the low (hi false) or high half h of a pair, in one instruction (the compiler converts, then subtracts).
template <bool HI>
__device__ __forceinline__ float minus_half(float x, uint32_t pair) {
  float r;
  if constexpr (HI)
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(pair), "v"(x));
  else
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(pair), "v"(x));
  return r;
}

// 8 values as hi + lo halves: per pair, two packed conversions (v_cvt_pk_f16_f32) and two mixed subtractions. Written
// value by value the pair took ten instructions, six of them at half rate; the splits of P are a fifth of a tile's
// vector work. With the key tile's fragments read ahead of the products (attend_tile_f32): dense (2, 1292, 24 heads)
// 181 -> 171 us, cross (2, 2584 x 257) 74 -> 70, band S = 16384, w = 128 137 -> 133; the same bits.
__device__ __forceinline__ void split8(const float (&x)[8], u32x4& hi, u32x4& lo) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f32x2 v = {x[2 * i], x[2 * i + 1]};
    const uint32_t h = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2));
    const f32x2 r = {minus_half<false>(v[0], h), minus_half<true>(v[1], h)};
    hi[i] = h;
    lo[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, f16x2));
  }
}

// Exponent of the leading bit of a bound, within [-100, 100] (zero, subnormal, infinite and NaN bounds included).
__device__ __forceinline__ int bound_exp(float b) {
  const int e = static_cast<int>((__float_as_uint(b) >> 23) & 255u) - 127;
  return e < -100 ? -100 : e > 100 ? 100 : e;
}

// Powers of two for the operand dims, from the norm parameters: a key's dim d is taken times 2^k[d], a query's times
// 2^q[d], and the logit is the product sum times 2^logit; the products of no dim exceed those of another because of its
// gains then. `kb(d)`, `qb(d)`: bounds of dim d before RoPE, which mixes dims d and d +- half.
struct ScaleTable {
  int k[128], q[128], logit;
};
// Exponent of the key bound of dim d.
template <class KBound>
__device__ __forceinline__ int key_exp(int d, int half, KBound kb) {
  const int p = d < half ? d + half : d < 2 * half ? d - half : d;
  return bound_exp(fmaxf(kb(d), kb(p)));
}
// The keys' part, before a barrier.
template <int D, class KBound>
__device__ __forceinline__ void key_scales(ScaleTable& t, int half, KBound kb) {
  for (int d = threadIdx.x; d < D; d += 256) t.k[d] = -key_exp(d, half, kb);
}
// The queries' part, by the first wave, before a barrier: `ek(d)` is -k[d], the exponent of the key bound of dim d.
template <int D, class KExp, class QBound>
__device__ __forceinline__ void query_scales(ScaleTable& t, int half, KExp ek, QBound qb) {
  const int lane = threadIdx.x & 63;
  if (threadIdx.x >= 64) return;
  int k[D / 64], emax = -1000;
#pragma unroll
  for (int i = 0; i < D / 64; ++i) {
    const int d = lane + 64 * i, p = d < half ? d + half : d < 2 * half ? d - half : d;
    k[i] = ek(d);
    const int e = bound_exp(fmaxf(qb(d), qb(p))) + k[i];
    emax = e > emax ? e : emax;
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const int other = __shfl_xor(emax, off, kWave);
    emax = other > emax ? other : emax;
  }
#pragma unroll
  for (int i = 0; i < D / 64; ++i) t.q[lane + 64 * i] = k[i] - emax;
  if (lane == 0) t.logit = emax;
}
// After RMSNorm |x_d| <= sqrt(D) |w_d|; |DyT(x)_d| <= |gamma_d| + |beta_d| (`dyt` = [alpha, gamma, beta]).
template <int D>
__device__ __forceinline__ auto rms_bound(const float* __restrict__ w) {
  return [w](int d) { return sqrtf(static_cast<float>(D)) * fabsf(w[d]); };
}
template <int D>
__device__ __forceinline__ auto dyt_bound(const float* __restrict__ dyt) {
  return [dyt](int d) { return fabsf(dyt[1 + d]) + fabsf(dyt[1 + D + d]); };
}

// Exponent of the leading bit of the largest magnitude `amax` (its bits) of operands scaled by a ScaleTable, at least
// -100. An infinite one (gains or tables) must not cost the finite ones beside it their place: they are about 1 or
// less.
__device__ __forceinline__ int lead_exp(uint32_t amax) {
  const int e = static_cast<int>(amax >> 23) - 127;
  return e < -100 ? -100 : e > 127 ? 1 : e;
}
__device__ __forceinline__ uint32_t amax8(const float (&x)[8]) {
  float a = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) a = fmaxf(a, fabsf(x[j]));  // passes over NaN
  return __float_as_uint(a);
}

// 8 values times 2^up, split, into a hi chunk and the lo chunk `plane` halves on; `edit(l)` may change the lo ones
// first.
template <class Edit>
__device__ __forceinline__ void st_split(uint16_t* __restrict__ hi, int plane, const float (&x)[8], int up, Edit edit) {
  float y[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) y[j] = ldexpf(x[j], up);
  u32x4 h, l;
  split8(y, h, l);
  edit(l);
  *reinterpret_cast<u32x4*>(hi) = h;
  *reinterpret_cast<u32x4*>(hi + plane) = l;
}
__device__ __forceinline__ void st_split(uint16_t* __restrict__ hi, int plane, const float (&x)[8], int up) {
  st_split(hi, plane, x, up, [](u32x4&) {});
}

// Reductions over 8 neighbouring lanes and over the wave without LDS (DPP and lane swaps); every lane gets the result.
template <class Op>
__device__ __forceinline__ uint32_t reduce8(uint32_t v, Op op) {
  v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, false));   // row_half_mirror: lanes i and 7 - i
  v = op(v, __builtin_amdgcn_update_dpp(0, v, 0xb1, 0xf, 0xf, false));    // quad_perm [1, 0, 3, 2]
  return op(v, __builtin_amdgcn_update_dpp(0, v, 0x4e, 0xf, 0xf, false));  // quad_perm [2, 3, 0, 1]
}
template <class Op>
__device__ __forceinline__ uint32_t reduce64(uint32_t v, Op op) {
  v = reduce8(v, op);
  v = op(v, __builtin_amdgcn_update_dpp(0, v, 0x128, 0xf, 0xf, false));  // row_ror:8
  const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  v = op(r[0], r[1]);
  const auto h = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return op(h[0], h[1]);
}
struct MaxU32 {
  __device__ uint32_t operator()(uint32_t a, uint32_t b) const { return a > b ? a : b; }
};
struct MinU32 {
  __device__ uint32_t operator()(uint32_t a, uint32_t b) const { return a < b ? a : b; }
};

// The largest and smallest magnitudes of a V tile, as the bits of non-negative floats (which order as the floats do,
// with infinities and then NaN last), collected in LDS by VTile::stats: of every key's row (over D / 64 waves), and the
// smallest nonzero one of the 8-key pieces of dims.
template <int D>
struct VStats {
  uint32_t rows[D / 64][SplitTile<D>::KT];
  uint32_t cells[SplitTile<D>::VN * 4];
};

// V of one key tile in registers: a lane per dim, so that a wave's loads are whole rows and the transpose costs no
// shuffle. A tile is stored in one of two forms, told apart by the 8-bit code in it (read_code):
//   - split: v 2^-e as hi + lo halves, the largest in [2^11, 2^12); code e + 128. What a half cannot hold costs up to
//     2^-37 of the tile's largest value, so a tile takes this form only if every key and every 8-key piece of a dim has
//     a value of at least 2^-12 of it (keys past the sequence aside, which no query weighs, and zero pieces): the error
//     is then at most 2^-25 of any key's and any dim's own largest. A tile of zeros is exact.
//   - wide: the fp32 bits, upper and lower halves in the two planes, for the fp32 matrix cores; code 0. Tiles with a
//     key of zeros among others are wide too: a query may give that key nearly all of its weight, and then needs its
//     small probabilities to fp32 accuracy, which P's halves have only near the tile's largest. A call of wide tiles
//     only (dense (2, 1292, 24 heads), every tenth key masked) takes 291 us against 180, and 527 with both products on
//     the fp32 matrix cores.
// The code lies in the first 8 lo values (dim 0, positions 0-7), at bit 14 of each: a lo half is at most 1 there (half
// a unit of a hi below 2^12), so that bit is free in a split tile; in a wide one it changes places with bit 0, which is
// lost (those 8 values keep 23 bits).
constexpr float kWideRange = 0x1p-12f;
constexpr uint32_t kCodeBits = 0x40004000u;
constexpr int kCodeKey = 16;  // the row of a K tile that holds its code (KeyRows)
// The bits of `code` for values 2 w and 2 w + 1.
__device__ __forceinline__ uint32_t code_bits(int code, int w) {
  return (((code >> (2 * w)) & 1u) << 14) | (((code >> (2 * w + 1)) & 1u) << 30);
}
template <int D>
struct VTile {
  using T = SplitTile<D>;
  float v[T::VN][8];
  // Rows k0 .. of `V`, `pitch` floats apart, times `mask` (null: 1); rows at or past `end` are zeros.
  __device__ __forceinline__ void fetch(const float* __restrict__ V, int64_t pitch, int k0, int end,
                                        const float* __restrict__ mask) {
#pragma unroll
    for (int i = 0; i < T::VN; ++i) {
      const int at = threadIdx.x + 256 * i, d = at % D;
      const int key0 = k0 + v_tile_key(8 * (at / D));  // position p0 + j holds key key0 + 8 (j / 4) + j % 4
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int key = key0 + 8 * (j >> 2) + (j & 3);
        v[i][j] = key < end ? V[key * pitch + d] : 0.f;
        if (mask && key < end) v[i][j] *= mask[key];
      }
    }
  }
  // This thread's share of `st`, which the workgroup may read after a barrier.
  __device__ __forceinline__ void stats(VStats<D>& st) const {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < T::VN; ++i) {
      uint32_t m[8], cell = 0;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        m[j] = __float_as_uint(v[i][j]) & 0x7fffffffu;
        cell = m[j] > cell ? m[j] : cell;
      }
      // Over the wave's 64 dims: the first three steps halve the keys that a lane holds, the last three the dims.
      const MaxU32 max;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const auto r = __builtin_amdgcn_permlane32_swap(m[j], m[j + 4], false, false);
        m[j] = max(r[0], r[1]);
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const auto r = __builtin_amdgcn_permlane16_swap(m[j], m[j + 2], false, false);
        m[j] = max(r[0], r[1]);
      }
      const bool up = lane & 8;
      m[0] = max(up ? m[1] : m[0], __builtin_amdgcn_update_dpp(0, up ? m[0] : m[1], 0x128, 0xf, 0xf, false));
      m[0] = reduce8(m[0], max);
      cell = reduce64(cell ? cell : ~0u, MinU32());
      const int at = threadIdx.x + 256 * i;  // lane l holds position 8 (at / D) + l / 8 of the wave's dims
      if (lane % 8 == 0) st.rows[at % D / 64][8 * (at / D) + lane / 8] = m[0];
      if (lane == 0) st.cells[4 * i + wave_id()] = cell;
    }
  }
  // The tile's code from `st`; `valid`: its keys before the end of the sequence. The same in every lane.
  __device__ static __forceinline__ int code(const VStats<D>& st, int valid) {
    const int lane = threadIdx.x & 63, pos = lane % T::KT;
    uint32_t row = 0;
#pragma unroll
    for (int i = 0; i < D / 64; ++i) row = st.rows[i][pos] > row ? st.rows[i][pos] : row;
    uint32_t least = st.cells[lane % (4 * T::VN)];
    if (v_tile_key(pos) < valid && row < least) least = row;
    const uint32_t amax = __builtin_amdgcn_readfirstlane(reduce64(row, MaxU32()));
    const uint32_t amin = __builtin_amdgcn_readfirstlane(reduce64(least, MinU32()));
    if (amax == 0) return 128;
    const int lead = static_cast<int>(amax >> 23) - 127;
    if (lead < -100 || lead > 127 || __uint_as_float(amin) < kWideRange * __uint_as_float(amax)) return 0;
    return lead - 11 + 128;  // 17 .. 244
  }
  __device__ __forceinline__ void store(uint16_t* __restrict__ hi, int code) const {
#pragma unroll
    for (int i = 0; i < T::VN; ++i) {
      const int at = threadIdx.x + 256 * i;
      u32x4 h, l;
      if (code) {
        float y[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) y[j] = ldexpf(v[i][j], 128 - code);
        split8(y, h, l);
      } else {
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          // a NaN whose payload lies in the bits that may be lost must stay one
          const uint32_t x0 = __float_as_uint(v[i][2 * w] == v[i][2 * w] ? v[i][2 * w] : __uint_as_float(0x7fc00000u));
          const uint32_t x1 =
              __float_as_uint(v[i][2 * w + 1] == v[i][2 * w + 1] ? v[i][2 * w + 1] : __uint_as_float(0x7fc00000u));
          h[w] = (x0 >> 16) | (x1 & 0xffff0000u);
          l[w] = (x0 & 0xffffu) | (x1 << 16);
        }
      }
      if (i == 0 && threadIdx.x == 0) {
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          if (!code) l[w] = (l[w] & ~0x00010001u) | ((l[w] & kCodeBits) >> 14);
          l[w] = (l[w] & ~kCodeBits) | code_bits(code, w);
        }
      }
      uint16_t* dst = hi + T::v_at(at % D, at / D);
      *reinterpret_cast<u32x4*>(dst) = h;
      *reinterpret_cast<u32x4*>(dst + T::PLANE) = l;
    }
  }
};

// The 8-bit code in bit 14 of the 8 halves at `p` in LDS, wave-uniform.
__device__ __forceinline__ int read_code(const uint16_t* __restrict__ p) {
  const u32x4 l = lds16(p);
  uint32_t code = 0;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const uint32_t x = __builtin_amdgcn_readfirstlane(l[w]);
    code |= (((x >> 14) & 1u) | ((x >> 29) & 2u)) << (2 * w);
  }
  return static_cast<int>(code);
}

// Copies tile t from the workspace into an LDS stage (byte address), 1 KB blocks by DMA, no registers.
template <int D>
struct SplitCopy {
  const uint16_t* src[3];
  uint32_t voff;
  __device__ __forceinline__ SplitCopy(const float* ws, int64_t region, int64_t row0) {
#pragma unroll
    for (int s = 0; s < 3; ++s) src[s] = reinterpret_cast<const uint16_t*>(ws + s * region + row0 * D);
    voff = wave_id() * 1024 + (threadIdx.x & 63) * 16;
  }
  __device__ __forceinline__ void operator()(int t, uint32_t stage) const {
    using T = SplitTile<D>;
#pragma unroll
    for (int s = 0; s < 3; ++s)
#pragma unroll
      for (int u = 0; u < 2 * T::TENSOR / 4096; ++u)
        lds_dma16(src[s] + static_cast<int64_t>(t) * T::TENSOR, voff + 4096 * u,
                  stage + 2 * s * T::TENSOR + 4096 * u + wave_id() * 1024);
  }
};

// Online-softmax state of one wave: 32 queries (lane % 32) of one branch.
template <int D>
struct Branch {
  f32x16 o[D / 32];
  float l, m;
  __device__ __forceinline__ Branch() : l(0.f), m(-INFINITY) {
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt) o[dt] = f32x16{};
  }
};

// One key tile for one wave. `sK`, `sV`: the hi planes of the branch's K and of V. `q`: this lane's query, hi and lo,
// in MFMA B operand order (dims 16 kk + 8 lh .. +8); the logit is the product sum times 2^(n + the K tile's code).
// `masked` (wave-uniform): `valid(k)` says whether key k of the tile
// takes part for this lane's query.
// The tile's probabilities are relative to its own largest logit (at most 1, and 1 somewhere), its products go into
// accumulators of their own, and one factor per query then takes both to the state: so neither the halves of P nor the
// power of two of V depends on what other tiles hold. That costs 16 FMAs per 32 dims: dense (2, 1292, 24 heads) 175 ->
// 187 us against products straight into O, and halves the error (6.2e-7 -> 3.3e-7); adding straight into O while a
// tile's maximum and power of two are near the state's is 3 % faster and has neither that accuracy nor one path. The
// state is rescaled only when some lane's maximum moves (it would multiply by exactly 1).
template <int D, class Valid>
__device__ __forceinline__ void attend_tile_f32(const uint16_t* __restrict__ sK, const uint16_t* __restrict__ sV,
                                                const u32x4 (&q)[2][D / 16], Branch<D>& b, int n, bool masked,
                                                Valid valid) {
  using T = SplitTile<D>;
  const int lane = threadIdx.x & 63, lr = lane & 31, lh = lane >> 5;
  const int code = read_code(sV + T::PLANE + T::v_at(0, 0));
  const float c =
      ldexpf(kLog2e / sqrtf(static_cast<float>(D)), n + read_code(sK + T::PLANE + T::k_at(kCodeKey, 0)) - 128);
  f32x16 s = f32x16{};
  u32x4 kf[2][D / 16];  // all in flight before the first product: one wait for LDS instead of one per product pair
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk)
#pragma unroll
    for (int i = 0; i < 2; ++i) kf[i][kk] = lds16(sK + i * T::PLANE + T::k_at(lr, 2 * kk + lh));
  if constexpr (D == 64) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk) {
    const u32x4 hi = kf[0][kk];
    u32x4 lo = kf[1][kk];
    if (kk == 0) lo &= ~kCodeBits;
    s = mfma_f16_32x32x16(lo, q[0][kk], s);
    s = mfma_f16_32x32x16(hi, q[1][kk], s);
    s = mfma_f16_32x32x16(hi, q[0][kk], s);
  }
  if (masked) {
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = valid(acc_key(0, r, lh)) ? s[r] : -INFINITY;
  }
  float mx = s[0];
#pragma unroll
  for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
  const float mt = fmaxf(mx, __shfl_xor(mx, 32, kWave)) * c;
  const float mnew = fmaxf(b.m, mt);
  const float muse = mnew == -INFINITY ? 0.f : mnew;  // a query with no valid key so far keeps O = l = 0
  if (__any(mnew != b.m)) {
    const float alpha = fast_exp2(b.m - muse);
    b.l *= alpha;
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt) b.o[dt] *= alpha;
    b.m = mnew;
  }
  const float beta = fast_exp2(mt - muse);        // 0 for a query with no valid key in the tile
  const float mtile = mt == -INFINITY ? 0.f : mt;
  float l = 0.f;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    s[r] = fast_exp2(__fmaf_rn(s[r], c, -mtile));
    l += s[r];
  }
  b.l = __fmaf_rn(l, beta, b.l);
  auto add = [&](int dt, const f32x16& acc, float up) {
#pragma unroll
    for (int r = 0; r < 16; ++r) b.o[dt][r] = __fmaf_rn(acc[r], up, b.o[dt][r]);
  };
  if (code) {
    u32x4 ph[2], pl[2];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      float p[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) p[j] = s[8 * g + j] * 0x1p14f;  // in the exponent it would cost 4 bits of argument
      split8(p, ph[g], pl[g]);
    }
    const float up = ldexpf(beta, code - 128 - 14);
#pragma unroll
    for (int d0 = 0; d0 < D / 32; d0 += 2) {
      if constexpr (D == 128) __builtin_amdgcn_sched_barrier(0);  // no registers for the next pair's operands
      f32x16 acc[2] = {};
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int at = T::v_at(32 * (d0 + i) + lr, 2 * g + lh);
          const u32x4 hi = lds16(sV + at);
          u32x4 lo = lds16(sV + T::PLANE + at);
          if (g == 0 && d0 + i == 0) lo &= ~kCodeBits;  // the code's bit, clear in all other values
          acc[i] = mfma_f16_32x32x16(lo, ph[g], acc[i]);
          acc[i] = mfma_f16_32x32x16(hi, pl[g], acc[i]);
          acc[i] = mfma_f16_32x32x16(hi, ph[g], acc[i]);
        }
#pragma unroll
      for (int i = 0; i < 2; ++i) add(d0 + i, acc[i], up);
    }
  } else {
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt) {
      f32x16 acc = {};
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const int at = T::v_at(32 * dt + lr, 2 * g + lh);
        const u32x4 hi = lds16(sV + at);
        u32x4 lo = lds16(sV + T::PLANE + at);
        if (g == 0 && dt == 0 && lane == 0) {
#pragma unroll
          for (int w = 0; w < 4; ++w) lo[w] = (lo[w] & ~(kCodeBits | 0x00010001u)) | ((lo[w] & 0x00010001u) << 14);
        }
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          acc = mfma_f32_32x32x2(__uint_as_float((hi[w] << 16) | (lo[w] & 0xffffu)), s[8 * g + 2 * w], acc);
          acc = mfma_f32_32x32x2(__uint_as_float((hi[w] & 0xffff0000u) | (lo[w] >> 16)), s[8 * g + 2 * w + 1], acc);
        }
      }
      add(dt, acc, beta);
    }
  }
}

// Epilogue shared by the kernels: out[q] = O1 / l1 - lam * O2 / l2 in fp32, each product rounded on its own so
// that identical branches cancel exactly. Must follow a barrier after the last use of the tiles.
template <int D>
__device__ __forceinline__ void store_diff_f32(uint16_t* __restrict__ stages, const Branch<D>& b, int br, float lamh,
                                               float* __restrict__ orow) {
  float* smem = reinterpret_cast<float*>(stages);
  const int lane = threadIdx.x & 63, lh = lane >> 5, wave = wave_id();
  const int slot0 = (wave & 1) * (D / 32) * 16;
  const float inv = __frcp_rn(b.l + __shfl_xor(b.l, 32, kWave));
  if (br == 1) {
    const float i1 = __fmul_rn(lamh, inv);
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) smem[(slot0 + dt * 16 + r) * 64 + lane] = __fmul_rn(b.o[dt][r], i1);
  }
  __syncthreads();
  if (br == 0 && orow) {
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        f32x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int r = 4 * g + j;
          v[j] = __fsub_rn(__fmul_rn(b.o[dt][r], inv), smem[(slot0 + dt * 16 + r) * 64 + lane]);
        }
        st4(orow + 32 * dt + 8 * g + 4 * lh, v);
      }
  }
}

// The split forms of k and k_diff of ROWS keys (32-key tiles), a (row, RoPE group pair) per thread and pass as
// rms_rows_f32 and band_rows_f32 hand them out: scaled by the ScaleTable as they come (`take`), then, when the
// workgroup has found each tile's largest magnitude (`stats`, a barrier), by the tile's own power of two, so that the
// largest lies in [2^11, 2^12) whatever the norms, the tables and the inputs made of it. What a half cannot hold is
// below 2^-37 of it. The tile's code (its power of two + 128) lies in bit 14 of the first 8 lo values of key kCodeKey,
// which is free there as in a split V tile. So do the powers of two of the dims (128 - k), for the calls that attend to
// keys which another call prepared: bit r of dim d's in key r < 8 of the first tile of k (`scales` not null).
template <int D, int ROWS>
struct KeyRows {
  using T = SplitTile<D>;
  static constexpr int PAIRS = D / 16, TASKS = (ROWS * PAIRS + 255) / 256, PARTS = 4 * TASKS;
  static constexpr int PER_TILE = PAIRS / 2;  // waves (and passes) that share a tile's rows
  struct Stats {
    uint32_t part[2][PARTS];
  };
  float y[TASKS][2][2][8] = {};
  int m1 = 0, m2 = 0;
  __device__ __forceinline__ void take(const ScaleTable& scale, int tsr, int i, int g1, const float (&x1)[8], int g2,
                                       const float (&x2)[8]) {
    m1 = g1;
    m2 = g2;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      y[i][tsr][0][j] = ldexpf(x1[j], scale.k[8 * g1 + j]);
      y[i][tsr][1][j] = ldexpf(x2[j], scale.k[8 * g2 + j]);
    }
  }
  __device__ __forceinline__ void stats(Stats& st) const {
    const MaxU32 max;
#pragma unroll
    for (int i = 0; i < TASKS; ++i)
#pragma unroll
      for (int tsr = 0; tsr < 2; ++tsr) {
        const uint32_t a = reduce64(max(amax8(y[i][tsr][0]), amax8(y[i][tsr][1])), max);
        if ((threadIdx.x & 63) == 0) st.part[tsr][4 * i + wave_id()] = a;
      }
  }
  // `planes(tensor, tile)`: the hi plane of a tile.
  template <class Planes>
  __device__ __forceinline__ void store(const Stats& st, const ScaleTable* scales, Planes planes) const {
    if (ROWS * PAIRS < 256 && threadIdx.x >= ROWS * PAIRS) return;
#pragma unroll
    for (int i = 0; i < TASKS; ++i) {
      const int row = (threadIdx.x + 256 * i) / PAIRS, tile = row / T::KT, r = row % T::KT;
#pragma unroll
      for (int tsr = 0; tsr < 2; ++tsr) {
        uint32_t amax = 0;
#pragma unroll
        for (int w = 0; w < PER_TILE; ++w) amax = MaxU32()(amax, st.part[tsr][PER_TILE * tile + w]);
        const int up = 11 - lead_exp(amax);
        uint16_t* hi = planes(tsr, tile);
        const bool dims = scales && tsr == 0 && row < 8;
        st_split(hi + T::k_at(r, m1), T::PLANE, y[i][tsr][0], up, [&](u32x4& l) {
          if (r == kCodeKey && m1 == 0) add_code(l, 128 - up);
          if (dims) add_code(l, scale_bits(*scales, m1, row));
        });
        st_split(hi + T::k_at(r, m2), T::PLANE, y[i][tsr][1], up, [&](u32x4& l) {
          if (dims) add_code(l, scale_bits(*scales, m2, row));
        });
      }
    }
  }
  // Bit r of the codes of group g's dims.
  __device__ static __forceinline__ int scale_bits(const ScaleTable& scales, int g, int r) {
    int bits = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) bits |= (((128 - scales.k[8 * g + j]) >> r) & 1) << j;
    return bits;
  }
  // Puts a code into 8 split values. Only the lo halves of infinities and NaNs may have the bit set; they may lose it.
  __device__ static __forceinline__ void add_code(u32x4& l, int code) {
#pragma unroll
    for (int w = 0; w < 4; ++w) l[w] = (l[w] & ~kCodeBits) | code_bits(code, w);
  }
};

// The workspace's K, K_diff and V^T tiles of the 64 keys from l0, by the whole workgroup; V^T through LDS, so that the
// stores are whole lines. `ws`: the first of the 64 rows in the K region.
template <int D>
__device__ __forceinline__ void store_tiles(const KeyRows<D, 64>& keys, const ScaleTable* scales,
                                            const float* __restrict__ V, int64_t pitch, int l0, int end,
                                            const float* __restrict__ mask, float* __restrict__ ws, int64_t region) {
  using T = SplitTile<D>;
  constexpr int NT = 64 / T::KT;
  __shared__ __attribute__((aligned(16))) uint16_t image[NT * T::TENSOR];
  __shared__ VStats<D> st[NT];
  __shared__ typename KeyRows<D, 64>::Stats kst;
  keys.stats(kst);
  __syncthreads();
  keys.store(kst, scales, [&](int tsr, int tile) {
    return reinterpret_cast<uint16_t*>(ws + tsr * region) + tile * T::TENSOR;
  });
  VTile<D> v[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) v[i].fetch(V, pitch, l0 + T::KT * i, end, mask);
#pragma unroll
  for (int i = 0; i < NT; ++i) v[i].stats(st[i]);
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NT; ++i) v[i].store(image + i * T::TENSOR, VTile<D>::code(st[i], end - (l0 + T::KT * i)));
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NT * T::TENSOR / 8 / 256; ++i) {
    const int at = 8 * (threadIdx.x + 256 * i);
    st16(reinterpret_cast<uint16_t*>(ws + 2 * region) + at, lds16(image + at));
  }
}

// RMSNorm (dit.py:45-57) and rotate-half RoPE (dit.py:90-98) in fp32 of two tensors (row offsets offA, offB) for the
// ROWS positions from pos0 (of the batch whose rows start at `xb`): `sink(tensor, pass, row, group, values, group,
// values)` takes the two 8-dim groups; positions at or past L give zeros. One (row, RoPE group pair) per thread and
// pass: the rotation partner of every dim is in the thread's own registers; the mean of squares is reduced over the D /
// 16 lanes of a row, neighbours in one wave.
template <int D, int ROWS, class Sink>
__device__ __forceinline__ void rms_rows_f32(const float* __restrict__ xb, int64_t rs, int64_t offA, int64_t offB,
                                             int pos0, int L, int half, const float* __restrict__ w, float eps,
                                             const float* __restrict__ cosT, const float* __restrict__ sinT,
                                             Sink sink) {
  constexpr int PAIRS = D / 16, TASKS = ROWS * PAIRS / 256;
  static_assert(ROWS * PAIRS % 256 == 0, "whole passes of the workgroup");
  const int p = threadIdx.x % PAIRS;
  int m1, m2;
  pair_groups(p, half / 8, m1, m2);
  const bool rot = p < half / 8;
#pragma unroll
  for (int i = 0; i < TASKS; ++i) {
    const int r = (threadIdx.x + 256 * i) / PAIRS, pos = pos0 + r;
    const bool in = pos < L;
    const float* row = xb + static_cast<int64_t>(in ? pos : 0) * rs;
    f32x4 x[2][2][2], cs[2], sn[2];
#pragma unroll
    for (int tsr = 0; tsr < 2; ++tsr)
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        x[tsr][0][hf] = ld4(row + (tsr ? offB : offA) + 8 * m1 + 4 * hf);
        x[tsr][1][hf] = ld4(row + (tsr ? offB : offA) + 8 * m2 + 4 * hf);
      }
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      cs[hf] = f32x4{1.f, 1.f, 1.f, 1.f};
      sn[hf] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (rot) {
        const int64_t at = static_cast<int64_t>(in ? pos : 0) * half + 8 * m1 + 4 * hf;
        cs[hf] = ld4(cosT + at);
        sn[hf] = ld4(sinT + at);
      }
    }
#pragma unroll
    for (int tsr = 0; tsr < 2; ++tsr) {
      float ss = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        ss = __fmaf_rn(x[tsr][1][j >> 2][j & 3], x[tsr][1][j >> 2][j & 3],
                       __fmaf_rn(x[tsr][0][j >> 2][j & 3], x[tsr][0][j >> 2][j & 3], ss));
#pragma unroll
      for (int off = 1; off < PAIRS; off <<= 1) ss += __shfl_xor(ss, off, kWave);
      const float inv = rsqrtf(ss / static_cast<float>(D) + eps);
      float o1[8], o2[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float y1 = __fmul_rn(__fmul_rn(x[tsr][0][j >> 2][j & 3], inv), w[8 * m1 + j]);
        const float y2 = __fmul_rn(__fmul_rn(x[tsr][1][j >> 2][j & 3], inv), w[8 * m2 + j]);
        const float c = cs[j >> 2][j & 3], s = sn[j >> 2][j & 3];
        const float r1 = rot ? __fadd_rn(__fmul_rn(y1, c), __fmul_rn(-y2, s)) : y1;
        const float r2 = rot ? __fadd_rn(__fmul_rn(y2, c), __fmul_rn(y1, s)) : y2;
        o1[j] = in ? r1 : 0.f;
        o2[j] = in ? r2 : 0.f;
      }
      sink(tsr, i, r, m1, o1, m2, o2);
    }
  }
}

// The split q and q_diff of the workgroup's 64 queries, through LDS in passes of 64 rows (32 at head_dim 128):
// `rows(r0, sink)` prepares the pass that starts at row r0. Besides the ScaleTable's, each row of each branch has a
// power of two of its own, from its largest magnitude (then in [2^13, 2^14)). Returns the power of two of this lane's
// logits but for the key tile's. Ends with a barrier, the stages free.
template <int D>
constexpr int kQueryRows = 4096 / D;
template <int D, class Rows>
__device__ __forceinline__ int queries_f32(const ScaleTable& scale, uint16_t* __restrict__ smem,
                                           u32x4 (&qf)[2][D / 16], Rows rows) {
  constexpr int ROWS = kQueryRows<D>, PLANE = 4096, PAIRS = D / 16;
  __shared__ int lead[2][64];
  static_assert(4 * PLANE <= SplitTile<D>::ELEMS, "q and q_diff of one pass must fit in the stages");
  const int lane = threadIdx.x & 63, wave = wave_id(), lr = lane & 31, lh = lane >> 5;
  const int row = (wave & 1) * 32 + lr;
#pragma unroll 1
  for (int r0 = 0; r0 < 64; r0 += ROWS) {
    rows(r0, [&](int tsr, int, int r, int g1, const float (&x1)[8], int g2, const float (&x2)[8]) {
      float y1[8], y2[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        y1[j] = ldexpf(x1[j], scale.q[8 * g1 + j]);
        y2[j] = ldexpf(x2[j], scale.q[8 * g2 + j]);
      }
      const MaxU32 max;
      uint32_t a = max(amax8(y1), amax8(y2));
#pragma unroll
      for (int off = 1; off < PAIRS; off <<= 1) a = max(a, __shfl_xor(a, off, kWave));
      const int e = lead_exp(a);
      if (threadIdx.x % PAIRS == 0) lead[tsr][r0 + r] = e;
      st_split(smem + 2 * tsr * PLANE + swz<D>(r, g1), PLANE, y1, 13 - e);
      st_split(smem + 2 * tsr * PLANE + swz<D>(r, g2), PLANE, y2, 13 - e);
    });
    __syncthreads();
    if (row / ROWS == r0 / ROWS) {  // wave-uniform
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk)
          qf[i][kk] = lds16(smem + (2 * (wave >> 1) + i) * PLANE + swz<D>(row % ROWS, 2 * kk + lh));
    }
    __syncthreads();
  }
  return scale.logit + lead[wave >> 1][row] - 13;
}

// k and k_diff after RMSNorm and RoPE and V * mask for 64 tokens of one head into the workspace's tiles.
template <int D>
__global__ __launch_bounds__(256) void dense_prep_f32(const float* __restrict__ qkv, int64_t rs, int sk, int skd,
                                                      int sv, const float* __restrict__ kw,
                                                      const float* __restrict__ cosT,
                                                      const float* __restrict__ sinT,
                                                      int half, const float* __restrict__ vmask, int L, int Lp, int H,
                                                      float eps, int64_t region, float* __restrict__ ws) {
  __shared__ ScaleTable scale;
  const int l0 = blockIdx.x * 64, h = blockIdx.y, b = blockIdx.z;
  const int64_t HD = static_cast<int64_t>(H) * D, bh = static_cast<int64_t>(b) * H + h;
  const float* xb = qkv + static_cast<int64_t>(b) * L * rs + h * D;
  float* block = ws + (bh * Lp + l0) * D;
  key_scales<D>(scale, half, rms_bound<D>(kw));
  __syncthreads();
  KeyRows<D, 64> keys;
  rms_rows_f32<D, 64>(xb, rs, sk * HD, skd * HD, l0, L, half, kw, eps, cosT, sinT,
                      [&](int tsr, int i, int, int g1, const float (&x1)[8], int g2, const float (&x2)[8]) {
                        keys.take(scale, tsr, i, g1, x1, g2, x2);
                      });
  store_tiles<D>(keys, l0 == 0 ? &scale : nullptr, xb + sv * HD, rs, l0, L,
                 vmask ? vmask + static_cast<int64_t>(b) * L : nullptr, block, region);
}

// The key tiles [t_lo, t_hi) through the stages: `attend(stage, t)` for each, after `first(stage)` for the first one.
template <int D, class First, class Attend>
__device__ __forceinline__ void stream_tiles(const SplitCopy<D>& copy, int t_lo, int t_hi,
                                             uint16_t* __restrict__ smem, First first, Attend attend) {
  using T = SplitTile<D>;
  const uint32_t ldsA = lds_addr(smem);
  if constexpr (T::STAGES == 2) {
    // The next tile is copied into the other stage while the current one is attended; unrolled over the two stages so
    // that both have fixed addresses.
    const uint32_t ldsB = ldsA + 2 * T::STAGE;
    copy(t_lo, ldsA);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    first(smem);
    for (int t = t_lo; t < t_hi; t += 2) {
      if (t + 1 < t_hi) copy(t + 1, ldsB);
      attend(smem, t);
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
      if (t + 1 >= t_hi) break;
      if (t + 2 < t_hi) copy(t + 2, ldsA);
      attend(smem + T::STAGE, t + 1);
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
    }
  } else {  // the other workgroup on the CU works while this one's copy is under way
    for (int t = t_lo; t < t_hi; ++t) {
      copy(t, ldsA);
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
      if (t == t_lo) first(smem);
      attend(smem, t);
      __syncthreads();
    }
  }
}

template <int D>
__global__ __launch_bounds__(256, SplitTile<D>::OCC) void dense_attend_f32(
    const float* __restrict__ qkv, int64_t rs, int sqd, const float* __restrict__ qw,
    const float* __restrict__ cosT, const float* __restrict__ sinT, int half, float eps, const float* __restrict__ ws,
    int64_t region, int B, int L, int Lk, int Lkp, int H, const float* __restrict__ lam, float* __restrict__ out) {
  using T = SplitTile<D>;
  __shared__ __attribute__((aligned(16))) uint16_t smem[T::ELEMS];
  __shared__ ScaleTable scale;
  const int nqb = (L + 63) / 64;
  const int tile = xcd_remap(blockIdx.x, B * H * nqb);
  const int qb = tile % nqb, bh = tile / nqb, h = bh % H, b = bh / H;
  const int wave = wave_id(), br = wave >> 1, q = qb * 64 + (wave & 1) * 32 + (threadIdx.x & 31);
  // The powers of two that the preparation gave the keys' dims, from its own k_weight (KeyRows).
  const uint16_t* lo = reinterpret_cast<const uint16_t*>(ws + static_cast<int64_t>(bh) * Lkp * D) + T::PLANE;
  query_scales<D>(scale, half, [&](int d) {
    int code = 0;
#pragma unroll
    for (int r = 0; r < 8; ++r) code |= ((lo[T::k_at(r, d / 8) + d % 8] >> 14) & 1) << r;
    return code - 128;
  }, rms_bound<D>(qw));
  __syncthreads();

  u32x4 qf[2][D / 16];
  const float* xb = qkv + static_cast<int64_t>(b) * L * rs + h * D;
  const int n = queries_f32<D>(scale, smem, qf, [&](int r0, auto sink) {
    rms_rows_f32<D, kQueryRows<D>>(xb, rs, 0, static_cast<int64_t>(sqd) * H * D, qb * 64 + r0, L, half, qw, eps, cosT,
                                   sinT, sink);
  });
  Branch<D> state;
  // Keys past Lk are zeros in the workspace (Lkp is a multiple of 128).
  const SplitCopy<D> copy(ws, region, static_cast<int64_t>(bh) * Lkp);
  auto clear = [&](uint16_t* s) {  // the dims' powers of two leave the first tile
    const int d = 4 * (threadIdx.x % (D / 4)), step = 256 / (D / 4);
    for (int r = threadIdx.x / (D / 4); r < 8; r += step)
      *reinterpret_cast<u32x2*>(s + T::PLANE + T::k_at(r, d / 8) + d % 8) &= ~kCodeBits;
    __syncthreads();
  };
  stream_tiles<D>(copy, 0, (Lk + T::KT - 1) / T::KT, smem, clear, [&](const uint16_t* s, int t) {
    attend_tile_f32<D>(s + br * T::TENSOR, s + 2 * T::TENSOR, qf, state, n, (t + 1) * T::KT > Lk,
                       [&](int k) { return t * T::KT + k < Lk; });
  });
  float* orow = q < L ? out + (static_cast<int64_t>(b) * L + q) * (static_cast<int64_t>(H) * D) + h * D : nullptr;
  store_diff_f32<D>(smem, state, br, lam ? lam[h] : 1.f, orow);
}

// tanh in fp32. Below 0.625: y + y^3 Q(y^2), Q a degree-5 least-maximum fit of (tanh(y)/y - 1)/y^2 (made for this
// kernel; its fp32 coefficients are within 2^-28.5 of tanh before rounding). Above: 1 - 2 / (1 + 2^(2 log2(e) |y|))
// with the rounding error of the exponent carried into the exponential and one Newton step on the reciprocal; 2 / (1 +
// e) is below 0.45 there, so the hardware exponential's error is at least halved. Both sides are computed and one is
// selected: 22 instructions without a branch, where the library's tanhf branches per element (both sides run in most
// waves).
__device__ __forceinline__ float tanh_f32(float y) {
  const float z = __fmul_rn(y, y);
  float q = 0.0021429606713354588f;
  q = __fmaf_rn(q, z, -0.008177396841347218f);
  q = __fmaf_rn(q, z, 0.021700702607631683f);
  q = __fmaf_rn(q, z, -0.05394676327705383f);
  q = __fmaf_rn(q, z, 0.1333320587873459f);
  q = __fmaf_rn(q, z, -0.3333333134651184f);
  const float small = __fmaf_rn(__fmul_rn(y, z), q, y);
  float a = fabsf(y);
  a = a > 10.f ? 10.f : a;  // tanh rounds to 1 there; NaN stays NaN
  constexpr float kTwoLog2e = 2.8853900432586670f, kTwoLog2eLo = 3.851926e-08f, kLn2 = 0.6931471824645996f;
  const float t = __fmul_rn(a, kTwoLog2e);
  const float lo = __fmaf_rn(a, kTwoLog2eLo, __fmaf_rn(a, kTwoLog2e, -t));
  float e = fast_exp2(t);
  e = __fmaf_rn(e, __fmul_rn(lo, kLn2), e);
  const float d = __fadd_rn(e, 1.f);
  float r = __builtin_amdgcn_rcpf(d);
  r = __fmaf_rn(r, __fmaf_rn(-d, r, 1.f), r);
  const float big = copysignf(__fmaf_rn(-2.f, r, 1.f), y);
  return fabsf(y) < 0.625f ? small : big;
}

// The DyT parameters of one RoPE group pair (8-dim groups m1 and m2 of a head), held by the thread that prepares that
// pair: `dyt` = [alpha, gamma[0..D), beta[0..D)]. A thread's pair is the same for every row it prepares.
template <int D>
struct DytPair {
  int m1, m2;
  bool rot;
  float alpha, g1[8], b1[8], g2[8], b2[8];
  __device__ __forceinline__ DytPair(const float* __restrict__ dyt, int half) {
    const int p = threadIdx.x % (D / 16);
    pair_groups(p, half / 8, m1, m2);
    rot = p < half / 8;
    alpha = dyt[0];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      g1[j] = dyt[1 + 8 * m1 + j];
      b1[j] = dyt[1 + D + 8 * m1 + j];
      g2[j] = dyt[1 + 8 * m2 + j];
      b2[j] = dyt[1 + D + 8 * m2 + j];
    }
  }
};

// DyT (same_l.py:58-69) and RoPE (same_l.py:92-100) in fp32 of two tensors (row offsets offA, offB) for the ROWS
// positions from pos0: `sink` as in rms_rows_f32; positions outside [0, S) give zeros. One (row, RoPE group pair) per
// thread and pass: the rotation partner of every dim is in the thread's own registers, and the pass's 16-byte loads are
// all issued before its arithmetic. Measured at S = 16384, 8 heads of 64: the key kernel 199.6 -> 42.0 us (201 MB at
// the rate of a large copy) against the library tanhf with the parameters read per element.
template <int D, int ROWS, class Sink>
__device__ __forceinline__ void band_rows_f32(const float* __restrict__ xb, int64_t rs, int64_t offA, int64_t offB,
                                              int pos0, int S, int half, const DytPair<D>& dp,
                                              const float* __restrict__ cosT, const float* __restrict__ sinT,
                                              Sink sink) {
  constexpr int PAIRS = D / 16, TASKS = (ROWS * PAIRS + 255) / 256;
  static_assert(ROWS * PAIRS % 256 == 0 || ROWS * PAIRS < 256, "whole passes of the workgroup, or part of one");
  if (ROWS * PAIRS < 256 && threadIdx.x >= ROWS * PAIRS) return;
#pragma unroll
  for (int i = 0; i < TASKS; ++i) {
    const int r = (threadIdx.x + 256 * i) / PAIRS, pos = pos0 + r;
    const bool in = pos >= 0 && pos < S;
    const float* row = xb + static_cast<int64_t>(in ? pos : 0) * rs;
    f32x4 x[2][2][2], cs[2], sn[2];
#pragma unroll
    for (int tsr = 0; tsr < 2; ++tsr)
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        x[tsr][0][hf] = ld4(row + (tsr ? offB : offA) + 8 * dp.m1 + 4 * hf);
        x[tsr][1][hf] = ld4(row + (tsr ? offB : offA) + 8 * dp.m2 + 4 * hf);
      }
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      cs[hf] = f32x4{1.f, 1.f, 1.f, 1.f};
      sn[hf] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (dp.rot) {
        const int64_t at = static_cast<int64_t>(in ? pos : 0) * half + 8 * dp.m1 + 4 * hf;
        cs[hf] = ld4(cosT + at);
        sn[hf] = ld4(sinT + at);
      }
    }
#pragma unroll
    for (int tsr = 0; tsr < 2; ++tsr) {
      float o1[8], o2[8];
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int j = 4 * hf + e;
          const float y1 = __fadd_rn(__fmul_rn(dp.g1[j], tanh_f32(__fmul_rn(dp.alpha, x[tsr][0][hf][e]))), dp.b1[j]);
          const float y2 = __fadd_rn(__fmul_rn(dp.g2[j], tanh_f32(__fmul_rn(dp.alpha, x[tsr][1][hf][e]))), dp.b2[j]);
          const float r1 = dp.rot ? __fadd_rn(__fmul_rn(y1, cs[hf][e]), __fmul_rn(-y2, sn[hf][e])) : y1;
          const float r2 = dp.rot ? __fadd_rn(__fmul_rn(y2, cs[hf][e]), __fmul_rn(y1, sn[hf][e])) : y2;
          o1[j] = in ? r1 : 0.f;
          o2[j] = in ? r2 : 0.f;
        }
      sink(tsr, i, r, dp.m1, o1, dp.m2, o2);
    }
  }
}

// The keys of the band prepared once: DyT and RoPE of k and k_diff (the same steps as inside band_attend_f32 without
// a workspace) and V as it is, for 64-key block blockIdx.x of (batch blockIdx.z, head blockIdx.y), into the workspace's
// tiles (Sp rows per (batch, head), zeros past S).
template <int D>
__global__ __launch_bounds__(256) void band_keys_f32(const float* __restrict__ qkv, int64_t rs, int S, int Sp, int H,
                                                     const float* __restrict__ kdyt, const float* __restrict__ cosT,
                                                     const float* __restrict__ sinT, int half, int64_t region,
                                                     float* __restrict__ ws) {
  __shared__ ScaleTable scale;
  const int t = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int64_t HD = static_cast<int64_t>(H) * D, bh = static_cast<int64_t>(b) * H + h;
  const float* xb = qkv + static_cast<int64_t>(b) * S * rs + h * D;
  float* block = ws + (bh * Sp + 64 * t) * D;
  key_scales<D>(scale, half, dyt_bound<D>(kdyt));
  __syncthreads();
  KeyRows<D, 64> keys;
  band_rows_f32<D, 64>(xb, rs, HD, 4 * HD, 64 * t, S, half, DytPair<D>(kdyt, half), cosT, sinT,
                       [&](int tsr, int i, int, int g1, const float (&x1)[8], int g2, const float (&x2)[8]) {
                         keys.take(scale, tsr, i, g1, x1, g2, x2);
                       });
  store_tiles<D>(keys, nullptr, xb + 2 * HD, rs, 64 * t, S, nullptr, block, region);
}

// WS: the key tiles that meet the block's band come from the workspace of band_keys_f32; otherwise each query block
// prepares its own from qkv, with one workgroup less per CU, for the registers of the preparation: three at head_dim 64
// spill 110 and take 322 us where two take 286 (S = 16384, w = 128, 8 x 64); two at 128 spill 223 and take 614 where one
// takes 627 without (4 x 128, w = 300). With each key tile's own power of two found there: 314 and 676.
template <int D, bool WS>
__global__ __launch_bounds__(256, WS ? SplitTile<D>::OCC : SplitTile<D>::OCC - 1) void band_attend_f32(
    const float* __restrict__ qkv, int64_t rs, int B, int S, int Sp, int H, int w, const float* __restrict__ qdyt,
    const float* __restrict__ kdyt, const float* __restrict__ cosT, const float* __restrict__ sinT, int half,
    const float* __restrict__ ws, int64_t region, const float* __restrict__ lam, float* __restrict__ out) {
  using T = SplitTile<D>;
  __shared__ __attribute__((aligned(16))) uint16_t smem[T::ELEMS];
  __shared__ ScaleTable scale;
  // query-block-major order: the heads of one query block run together and share key rows in L2
  const int qb = blockIdx.x / (B * H), bh = blockIdx.x % (B * H), h = bh % H, b = bh / H;
  const int lane = threadIdx.x & 63, wave = wave_id(), lr = lane & 31;
  const int br = wave >> 1, q0 = qb * 64, qw0 = q0 + (wave & 1) * 32, q = qw0 + lr;
  const int64_t HD = static_cast<int64_t>(H) * D;
  const float* xb = qkv + static_cast<int64_t>(b) * S * rs + h * D;

  if constexpr (!WS) key_scales<D>(scale, half, dyt_bound<D>(kdyt));
  query_scales<D>(scale, half, [&](int d) { return key_exp(d, half, dyt_bound<D>(kdyt)); }, dyt_bound<D>(qdyt));
  __syncthreads();
  u32x4 qf[2][D / 16];
  int n;
  {
    const DytPair<D> dp(qdyt, half);
    n = queries_f32<D>(scale, smem, qf, [&](int r0, auto sink) {
      band_rows_f32<D, kQueryRows<D>>(xb, rs, 0, 3 * HD, q0 + r0, S, half, dp, cosT, sinT, sink);
    });
  }

  Branch<D> state;
  const int t_lo = (q0 - w > 0 ? q0 - w : 0) / T::KT;
  const int t_hi = ((q0 + 64 + w < S ? q0 + 64 + w : S) + T::KT - 1) / T::KT;
  auto attend = [&](const uint16_t* s, int t) {
    const int k0 = t * T::KT, k1 = k0 + T::KT - 1;
    // the tile reaches this wave's band, and lies inside the band of every one of its queries
    if (k0 > qw0 + 31 + w || k1 < qw0 - w) return;
    const bool inside = k1 <= qw0 + w && k0 >= qw0 + 31 - w && k1 < S;
    attend_tile_f32<D>(s + br * T::TENSOR, s + 2 * T::TENSOR, qf, state, n, !inside, [&](int k) {
      const int kk = k0 + k, dist = kk - q;
      return kk < S && dist <= w && -dist <= w;
    });
  };
  if constexpr (WS) {  // every tile's rows lie below Sp: Sp is a multiple of 128 and k0 < S
    const SplitCopy<D> copy(ws, region, static_cast<int64_t>(bh) * Sp);
    stream_tiles<D>(copy, t_lo, t_hi, smem, [](uint16_t*) {}, attend);
  } else {
    __shared__ VStats<D> st;
    __shared__ typename KeyRows<D, T::KT>::Stats kst;
    const DytPair<D> kp(kdyt, half);
    for (int t = t_lo; t < t_hi; ++t) {
      VTile<D> v;
      v.fetch(xb + 2 * HD, rs, t * T::KT, S, nullptr);
      v.stats(st);
      KeyRows<D, T::KT> keys;
      band_rows_f32<D, T::KT>(xb, rs, HD, 4 * HD, t * T::KT, S, half, kp, cosT, sinT,
                              [&](int tsr, int i, int, int g1, const float (&x1)[8], int g2, const float (&x2)[8]) {
                                keys.take(scale, tsr, i, g1, x1, g2, x2);
                              });
      keys.stats(kst);
      __syncthreads();
      keys.store(kst, nullptr, [&](int tsr, int) { return smem + tsr * T::TENSOR; });
      v.store(smem + 2 * T::TENSOR, VTile<D>::code(st, S - t * T::KT));
      __syncthreads();
      attend(smem, t);
      __syncthreads();
    }
  }
  float* orow = q < S ? out + (static_cast<int64_t>(b) * S + q) * HD + h * D : nullptr;
  store_diff_f32<D>(smem, state, br, lam ? lam[h] : 1.f, orow);
}

static int launched(const char* what) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(HB_ERR_LAUNCH, "%s launch failed: %s", what, hipGetErrorString(e));
  return HB_OK;
}

int launch_dense_prep_f32(hipStream_t stream, const void* qkv, int64_t rs, int sk, int skd, int sv, const float* kw,
                          const float* cosT, const float* sinT, int half, const float* vmask, int B, int L, int H, int D,
                          float eps, const DenseLayout& lay, void* ws) {
  const dim3 grid(static_cast<unsigned>(lay.Lp / 64), static_cast<unsigned>(H), static_cast<unsigned>(B));
  const float* x = static_cast<const float*>(qkv);
  float* w = static_cast<float*>(ws);
  const int Lp = static_cast<int>(lay.Lp);
  if (D == 64)
    hipLaunchKernelGGL(dense_prep_f32<64>, grid, dim3(256), 0, stream, x, rs, sk, skd, sv, kw, cosT, sinT, half, vmask,
                       L, Lp, H, eps, lay.region_elems, w);
  else
    hipLaunchKernelGGL(dense_prep_f32<128>, grid, dim3(256), 0, stream, x, rs, sk, skd, sv, kw, cosT, sinT, half,
                       vmask, L, Lp, H, eps, lay.region_elems, w);
  return launched("dense_prep_f32");
}

int launch_dense_attend_f32(hipStream_t stream, const void* qkv, int64_t rs, int sqd, const float* qw,
                            const float* cosT, const float* sinT, int half, float eps, const void* ws, const float* lam,
                            void* out, int B, int L, int Lk, int H, int D, const DenseLayout& lay) {
  const int nblocks = B * H * ((L + 63) / 64);
  const float* x = static_cast<const float*>(qkv);
  const float* w = static_cast<const float*>(ws);
  float* o = static_cast<float*>(out);
  const int Lkp = static_cast<int>(lay.Lp);
  auto attend = D == 64 ? dense_attend_f32<64> : dense_attend_f32<128>;
  hipLaunchKernelGGL(attend, dim3(nblocks), dim3(256), 0, stream, x, rs, sqd, qw, cosT, sinT, half, eps, w,
                     lay.region_elems, B, L, Lk, Lkp, H, lam, o);
  return launched("dense_attend_f32");
}

int launch_band_f32_ws(hipStream_t stream, const void* qkv, int64_t rs, const float* qdyt, const float* kdyt,
                       const float* cosT, const float* sinT, int half, int window, const float* lam, void* out, int B,
                       int S, int H, int D, void* workspace) {
  const DenseLayout lay = dense_layout(HB_F32, B, S, H, D);
  const int Sp = static_cast<int>(lay.Lp);
  const float* x = static_cast<const float*>(qkv);
  float* ws = static_cast<float*>(workspace);
  float* o = static_cast<float*>(out);
  const dim3 kgrid(static_cast<unsigned>(Sp / 64), static_cast<unsigned>(H), static_cast<unsigned>(B));
  const int nblocks = B * H * ((S + 63) / 64);
  auto keys = D == 64 ? band_keys_f32<64> : band_keys_f32<128>;
  auto attend = D == 64 ? band_attend_f32<64, true> : band_attend_f32<128, true>;
  hipLaunchKernelGGL(keys, kgrid, dim3(256), 0, stream, x, rs, S, Sp, H, kdyt, cosT, sinT, half, lay.region_elems, ws);
  hipLaunchKernelGGL(attend, dim3(nblocks), dim3(256), 0, stream, x, rs, B, S, Sp, H, window, qdyt, kdyt, cosT, sinT,
                     half, ws, lay.region_elems, lam, o);
  return launched("band_attend_f32");
}

int launch_band_f32(hipStream_t stream, const void* qkv, int64_t rs, const float* qdyt, const float* kdyt,
                    const float* cosT, const float* sinT, int half, int window, const float* lam, void* out, int B,
                    int S, int H, int D) {
  const int nblocks = B * H * ((S + 63) / 64);
  const float* x = static_cast<const float*>(qkv);
  float* o = static_cast<float*>(out);
  auto attend = D == 64 ? band_attend_f32<64, false> : band_attend_f32<128, false>;
  hipLaunchKernelGGL(attend, dim3(nblocks), dim3(256), 0, stream, x, rs, B, S, S, H, window, qdyt, kdyt, cosT, sinT,
                     half, static_cast<const float*>(nullptr), int64_t(0), lam, o);
  return launched("band_attend_f32");
}

}  // namespace hb
