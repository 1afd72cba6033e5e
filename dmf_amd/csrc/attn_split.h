// Attention kernel bodies for fp32 and fp16 operands on the 16-bit matrix pipes.
//
// What bounds the fp32 mode is the matrix pipe: v_mfma_f32_32x32x2_f32 runs at 1/16 of the bf16 rate (157 TFLOP/s nominal,
// 137 reached by a large library product).  A product of fp32 operands is formed here from bf16 MFMAs instead, without giving
// up fp32 precision: every operand is the sum of three bf16 numbers (8 + 8 + 8 significant bits, each the rounded remainder
// of the one before: x = x0 + x1 + x2 up to 2^-27 |x|), and of the nine plane products the six with i + j <= 2 are
// accumulated in fp32, smallest first; the three left out are below 2^-26 of the product, a quarter of the rounding of an
// fp32 multiplication.  Six MFMAs of 32x32x16 take 192 cycles where eight of 32x32x2 take 512.
//
// fp16 operands are exact in one f16 plane, so the score-like products are single f16 MFMAs; the probability-like operand
// W (P, P*dS, dS: fp32 values) is split into two f16 planes (21 significant bits of P, 23 of the others) so that nothing is rounded to
// 11 bits before the final store.  f16 has no digits below 2^-24, so P is formed times a power of two that puts its largest value near the
// top of the range (kFwdBias, kBwdBias: part of the exponent, hence free): formed as it is, a weight of e^-10 kept 10 bits and one of e^-14
// four, which the rows of a key with nearly all of the weight and a zero value are made of (N1024: results 6.8e-4 and 3.6e-2 off where
// fp16 rounds to 2e-4).  Operands that carry a tangent or gradient factor have no bound and are kept in range by a power of two per row
// (RowScale), raised lazily like the running maximum.
//
// Layouts are those of attn_common.h (transposed scores, per-lane softmax state, accumulator tile = next B operand).
// A work-group of NW waves owns 32 NW rows of one (batch, head); tiles of 32 streamed rows travel HBM -> registers -> planes
// -> LDS, each element being split once per work-group, and every plane chunk read from LDS feeds up to three MFMAs.
#pragma once
#include "attn_common.h"
#include "attn_kernels.h"

namespace dmf {

typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;

// NI planes of a loaded operand, NWT of a probability-like one.
template <typename T> struct SplitType;
template <> struct SplitType<float> { static constexpr int NI = 3, NWT = 3; static constexpr bool F16 = false; };
template <> struct SplitType<_Float16> { static constexpr int NI = 1, NWT = 2; static constexpr bool F16 = true; };

// log2 of the factor on P in the f16 kernels: P reaches 2^6 in the forward (kSplitLazyLog2), the range 2^16; in the backward P reaches 1, and
// more by what lse is rounded (2^5.8 at scores of 10^8).  Scores from 2^24 on (log2 units), whose last digit is a whole number, go without
// the factor: it would be rounded to a larger one.
template <typename T> constexpr float kFwdBias = SplitType<T>::F16 ? 9.f : 0.f;
template <typename T> constexpr float kBwdBias = SplitType<T>::F16 ? 10.f : 0.f;
// What an accumulator of P (its planes' sum: split8) is multiplied by at the end.
template <typename T> constexpr float kWeightUnit = SplitType<T>::F16 ? 1.f / (1.f + 1.f / 1024.f) : 1.f;
constexpr float kBiasedScores = 0x1p24f;
template <typename T>
__device__ __forceinline__ float running_max(float mx) {   // what is kept of it: a whole number in the f16 kernels, less kFwdBias
  if constexpr (!SplitType<T>::F16) return mx;
  return ceilf(mx) - (fabsf(mx) < kBiasedScores ? kFwdBias<T> : 0.f);
}
constexpr uint32_t kRowScaleBias = 9;   // and of RowScale's largest value before it is raised: 2^5 times that

template <>
__device__ __forceinline__ void store4<_Float16>(_Float16* dst, float a, float b, float c, float d) {
  typedef __attribute__((ext_vector_type(4))) _Float16 f16x4;
  *reinterpret_cast<f16x4*>(dst) = f16x4{(_Float16)a, (_Float16)b, (_Float16)c, (_Float16)d};
}

template <typename T>
__device__ __forceinline__ void mma_one(f32x16& acc, const u32x4& a, const u32x4& b) {
  if constexpr (SplitType<T>::F16)
    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), acc, 0, 0, 0);
  else
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
}
template <typename T>
__device__ __forceinline__ void mma_one16(f32x4& acc, const u32x4& a, const u32x4& b) {
  if constexpr (SplitType<T>::F16)
    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), acc, 0, 0, 0);
  else
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
}

// acc += sum of a_i b_j over i + j < max(NA, NB), smallest products first.
template <int NA, int NB, typename F>
__device__ __forceinline__ void for_plane_pairs(F&& f) {
  constexpr int MX = (NA > NB ? NA : NB) - 1;
#pragma unroll
  for (int s = MX; s >= 0; --s)
#pragma unroll
    for (int i = 0; i < NA; ++i)
      if (s - i >= 0 && s - i < NB) f(i, s - i);
}
template <typename T, int NA, int NB>
__device__ __forceinline__ void mma_planes(f32x16& acc, const u32x4 (&a)[NA], const u32x4 (&b)[NB]) {
  for_plane_pairs<NA, NB>([&](int i, int j) { mma_one<T>(acc, a[i], b[j]); });
}
template <typename T, int NA, int NB>
__device__ __forceinline__ void mma_planes16(f32x4& acc, const u32x4 (&a)[NA], const u32x4 (&b)[NB]) {
  for_plane_pairs<NA, NB>([&](int i, int j) { mma_one16<T>(acc, a[i], b[j]); });
}

// x minus the low (0) / high (1) f16 half of w: one mixed-precision instruction where conversion and subtraction take two
// (exact either way: the difference is).  WEIGHT: minus 1 - 2^-10 times it.
template <int HALF, bool WEIGHT = false>
__device__ __forceinline__ float sub_half(float x, uint32_t w) {
  float r;
  if constexpr (WEIGHT) {
    const float m = -1.f + 1.f / 1024.f;
    if constexpr (HALF == 0) asm("v_fma_mix_f32 %0, %1, %3, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(w), "v"(x), "s"(m));
    else asm("v_fma_mix_f32 %0, %1, %3, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(w), "v"(x), "s"(m));
  } else if constexpr (HALF == 0) asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(w), "v"(x));
  else asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(w), "v"(x));
  return r;
}

// two fp32 values to f16, rounded to nearest
__device__ __forceinline__ uint32_t pack_f16x2(float a, float b) {
  typedef __attribute__((ext_vector_type(2))) float f32x2;
  typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{a, b}), f16x2));
}

// Eight fp32 values as NP planes of eight 16-bit ones.  ANY (operands as the caller gave them, in bf16 planes): all but the last
// plane are held within the finite range, so that a value above the largest bf16 number does not round to infinity and an
// infinity or NaN ends up in the last plane alone -- it then meets only the first plane of the other operand, whose sign is the
// value's.  WEIGHT (probabilities, in f16 planes): the second plane is the remainder plus 2^-10 of the first, which is at least twice the
// rounding and makes it positive wherever the value is, so that an infinity among the elements it weighs stays one (next to an exact first
// plane it met a zero).  The planes' sum is then 1 + 2^-10 times the value, up to 2^-21 of it: kWeightUnit takes that off the accumulator.
template <typename T, bool ANY = false, bool WEIGHT = false, int NP>
__device__ __forceinline__ void split8(const float (&x)[8], u32x4 (&pl)[NP]) {
  constexpr float kMax = 3.38953139e38f;   // the largest bf16 number
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = x[2 * i], b = x[2 * i + 1];
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      if constexpr (SplitType<T>::F16) {
        pl[k][i] = pack_f16x2(a, b);
        if (k + 1 < NP) {
          a = sub_half<0, WEIGHT>(a, pl[k][i]);
          b = sub_half<1, WEIGHT>(b, pl[k][i]);
        }
      } else {
        const bool hold = ANY && k + 1 < NP;
        const uint32_t h = hold ? pack_bf16x2(__builtin_amdgcn_fmed3f(a, -kMax, kMax), __builtin_amdgcn_fmed3f(b, -kMax, kMax)) : pack_bf16x2(a, b);
        pl[k][i] = h;
        if (k + 1 < NP) {
          a -= __uint_as_float(h << 16);
          b -= __uint_as_float(h & 0xffff0000u);
        }
      }
    }
  }
}

// Odd, and rows 0 .. 3 apart modulo 16 vectors: free of bank conflicts for row and for transposed reads.
constexpr int split_pitch(int min_vectors) {
  for (int p = min_vectors | 1;; p += 2) {
    const int m = p % 16;
    if (m == 3 || m == 7 || m == 9 || m == 13) return p;
  }
}

template <typename T, int D, int NW>
struct SplitCfg {
  using S = SplitType<T>;
  static constexpr int VPR = D / 8, NCHUNK = (D + 15) / 16;          // 8-element vectors per row; contraction chunks over the head dim
  static constexpr int P = split_pitch(2 * NCHUNK), STR = P * 8;     // tile row pitch in vectors / elements
  static constexpr int PLANE = 32 * P * 16, TILE = S::NI * PLANE;    // bytes
  static constexpr bool TAIL = (D % 32) != 0 && (D % 32) <= 16;      // 16-wide remainder by 16x16x32 MFMAs (72, 80)
  static constexpr int NMT = TAIL ? D / 32 : (D + 31) / 32;
  static constexpr int RAW = sizeof(T) / 2;                          // 16-byte registers quads per vector
  static constexpr int STAGE_ROWS_BYTES = 32 * NW * Cfg<T, D>::OROWV * 16;
};

// One streamed tensor tile of 32 rows: load() requests this thread's vectors (rows at or past nrows read as zero), commit()
// splits them and writes the planes.  FAST: full tiles are read through a buffer descriptor and 32-bit offsets kept from tile to
// tile (the per-lane 64-bit addresses and row checks are a tenth of the vector instructions of an fp16 tile); the ragged last one,
// and rows 2^26 bytes or more apart, take the general addresses.  In kernels of one wave per SIMD the branch between the two costs
// more than it saves (it ends the block in which loads are scheduled among the products).
template <typename T, int D, int NW, bool FAST = false>
struct TileLoad {
  using C = SplitCfg<T, D, NW>;
  static constexpr int NVEC = 32 * C::VPR, ITERS = (NVEC + 64 * NW - 1) / (64 * NW);   // vectors of a tile; per thread
  u32x4 r[ITERS][C::RAW];
  uint32_t off[FAST ? ITERS : 1];
  bool near;
  __device__ __forceinline__ void init(int64_t row_stride, int tid) {
    if constexpr (FAST) {
      near = row_stride < (int64_t)(1 << 26) / (int64_t)sizeof(T);
#pragma unroll
      for (int it = 0; it < ITERS; ++it) {
        const int v = tid + it * 64 * NW, row = v / C::VPR, cv = v % C::VPR;
        // (threads without a vector in the last round read the tile's first one)
        off[it] = v < NVEC ? static_cast<uint32_t>(row) * static_cast<uint32_t>(row_stride * (int64_t)sizeof(T)) + cv * (uint32_t)sizeof(T) * 8 : 0u;
      }
    }
  }
  __device__ __forceinline__ void load(const T* src, int64_t row_stride, int row0, int nrows, int tid) {
    if constexpr (FAST) {
      if (near && row0 + 32 <= nrows) {
        const __amdgpu_buffer_rsrc_t rsrc = make_rows_rsrc(src + (int64_t)row0 * row_stride, (uint32_t)row_stride * (uint32_t)sizeof(T), 32, D * (int)sizeof(T));
#pragma unroll
        for (int it = 0; it < ITERS; ++it)
#pragma unroll
          for (int k = 0; k < C::RAW; ++k) r[it][k] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off[it] + 16 * k, 0, 0));
        return;
      }
    }
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int v = tid + it * 64 * NW, row = v / C::VPR, cv = v % C::VPR;
      const bool ok = v < NVEC && row0 + row < nrows;
      const u32x4* g = reinterpret_cast<const u32x4*>(src + (int64_t)(row0 + row) * row_stride + cv * 8);
#pragma unroll
      for (int k = 0; k < C::RAW; ++k) r[it][k] = ok ? g[k] : u32x4{0, 0, 0, 0};
    }
  }
  __device__ __forceinline__ void commit(char* tile, int tid) const {
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int v = tid + it * 64 * NW, row = v / C::VPR, cv = v % C::VPR;
      if (v < NVEC) {
        char* dst = tile + (row * C::P + cv) * 16;
        if constexpr (sizeof(T) == 2) {   // one plane, as it is
          *reinterpret_cast<u32x4*>(dst) = r[it][0];
        } else {
          float x[8];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            x[e] = __uint_as_float(r[it][0][e]);
            x[4 + e] = __uint_as_float(r[it][C::RAW - 1][e]);
          }
          u32x4 pl[SplitType<T>::NI];
          split8<T, true>(x, pl);
#pragma unroll
          for (int k = 0; k < SplitType<T>::NI; ++k) *reinterpret_cast<u32x4*>(dst + k * C::PLANE) = pl[k];
        }
      }
    }
  }
};

// Operand planes of this lane's own row (register resident): chunk c = elements 16c + 8g .. +7; zero past the head dim or the end.
template <typename T, int D, int NW>
__device__ __forceinline__ void load_own_row(const T* base, int64_t row_stride, int row, int nrows, int g,
                                             u32x4 (&out)[SplitCfg<T, D, NW>::NCHUNK][SplitType<T>::NI]) {
  using C = SplitCfg<T, D, NW>;
#pragma unroll
  for (int c = 0; c < C::NCHUNK; ++c) {
    const bool in = row < nrows && 2 * c + g < C::VPR;
    const u32x4* p = reinterpret_cast<const u32x4*>(base + (int64_t)row * row_stride + 16 * c + 8 * g);
    const u32x4 a = in ? p[0] : u32x4{0, 0, 0, 0};
    if constexpr (sizeof(T) == 2) {   // one plane, as it is (16 bytes of the row per chunk and half)
      out[c][0] = a;
    } else {
      const u32x4 b = in ? p[1] : u32x4{0, 0, 0, 0};
      float x[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[e] = __uint_as_float(a[e]);
        x[4 + e] = __uint_as_float(b[e]);
      }
      split8<T, true>(x, out[c]);
    }
  }
}

// Planes of operand chunk c of row `row` of a tile (contraction along the row) ...
template <typename T, int D, int NW>
__device__ __forceinline__ void row_planes(const char* tile, int row, int c, int g, u32x4 (&out)[SplitType<T>::NI]) {
  using C = SplitCfg<T, D, NW>;
#pragma unroll
  for (int k = 0; k < SplitType<T>::NI; ++k)
    out[k] = *reinterpret_cast<const u32x4*>(tile + k * C::PLANE + (row * C::P + 2 * c + g) * 16);
}
// ... and of the transposed one: 16 tile rows (step s) at columns col0 .. col0 + 31,
template <typename T, int D, int NW>
__device__ __forceinline__ void col_planes(const char* tile, int col0, int s, int lane, u32x4 (&out)[SplitType<T>::NI]) {
  using C = SplitCfg<T, D, NW>;
#pragma unroll
  for (int k = 0; k < SplitType<T>::NI; ++k)
    out[k] = lds_col_operand<__bf16, C::STR>(reinterpret_cast<const __bf16*>(tile + k * C::PLANE), 0, col0, s, lane).v;
}
// or all 32 tile rows at the 16 remainder columns.
template <typename T, int D, int NW>
__device__ __forceinline__ void tail_planes(const char* tile, int lane, u32x4 (&out)[SplitType<T>::NI]) {
  using C = SplitCfg<T, D, NW>;
#pragma unroll
  for (int k = 0; k < SplitType<T>::NI; ++k) {
    const __bf16* p = reinterpret_cast<const __bf16*>(tile + k * C::PLANE) + tail_lane_offset(lane, C::STR, 32 * C::NMT);
    const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(s16x4, p)));
    const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(s16x4, p + 8 * C::STR)));
    out[k] = u32x4{lo[0], lo[1], hi[0], hi[1]};
  }
}

// Transposed accumulators of 32 output rows: NMT full 32-wide tiles and, with a remainder, two 16x16 ones (one per half of the
// wave's 32 rows).
template <typename T, int D, int NW>
struct OutAcc {
  using C = SplitCfg<T, D, NW>;
  f32x16 t[C::NMT];
  f32x4 tail[2];
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int i = 0; i < C::NMT; ++i) t[i] = f32x16{0};
    tail[0] = tail[1] = f32x4{0, 0, 0, 0};
  }
  // by a factor per row (= lane % 32)
  __device__ __forceinline__ void scale(float f) {
#pragma unroll
    for (int i = 0; i < C::NMT; ++i) t[i] *= f;
    if constexpr (C::TAIL) {
      float f0, f1;
      swap16f(f, f0, f1);
      tail[0] *= f0;
      tail[1] *= f1;
    }
  }
};

// W operand of a 32x32 tile: planes of steps 0 and 1, and their re-distribution for the remainder products.
template <typename T>
struct WOperand {
  u32x4 s[2][SplitType<T>::NWT];
  template <bool WEIGHT = false>
  __device__ __forceinline__ void form(const f32x16& e) {
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      float x[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = e[8 * st + i];
      split8<T, false, WEIGHT>(x, s[st]);
    }
  }
  __device__ __forceinline__ void tail(u32x4 (&h0)[SplitType<T>::NWT], u32x4 (&h1)[SplitType<T>::NWT]) const {
#pragma unroll
    for (int k = 0; k < SplitType<T>::NWT; ++k) {
      ColOperand a, b, x, y;
      a.v = s[0][k];
      b.v = s[1][k];
      tail_operands(a, b, x, y);
      h0[k] = x.v;
      h1[k] = y.v;
    }
  }
};

// acc^T += tile^T W over the 32 rows of a tile, for one or two (acc, W) pairs that share the tile.
template <typename T, int D, int NW>
__device__ __forceinline__ void contract_rows(const char* tile, int lane, OutAcc<T, D, NW>& a0, const WOperand<T>& w0) {
  using C = SplitCfg<T, D, NW>;
  constexpr int NI = SplitType<T>::NI, NWT = SplitType<T>::NWT;
#pragma unroll
  for (int st = 0; st < 2; ++st)
#pragma unroll
    for (int t = 0; t < C::NMT; ++t) {
      u32x4 v[NI];
      col_planes<T, D, NW>(tile, 32 * t, st, lane, v);
      mma_planes<T>(a0.t[t], v, w0.s[st]);
    }
  if constexpr (C::TAIL) {
    u32x4 v[NI], h0[NWT], h1[NWT];
    tail_planes<T, D, NW>(tile, lane, v);
    w0.tail(h0, h1);
    mma_planes16<T>(a0.tail[0], v, h0);
    mma_planes16<T>(a0.tail[1], v, h1);
  }
}
template <typename T, int D, int NW>
__device__ __forceinline__ void contract_rows(const char* tile, int lane, OutAcc<T, D, NW>& a0, const WOperand<T>& w0,
                                              OutAcc<T, D, NW>& a1, const WOperand<T>& w1) {
  using C = SplitCfg<T, D, NW>;
  constexpr int NI = SplitType<T>::NI, NWT = SplitType<T>::NWT;
#pragma unroll
  for (int st = 0; st < 2; ++st)
#pragma unroll
    for (int t = 0; t < C::NMT; ++t) {
      u32x4 v[NI];
      col_planes<T, D, NW>(tile, 32 * t, st, lane, v);
      mma_planes<T>(a0.t[t], v, w0.s[st]);
      mma_planes<T>(a1.t[t], v, w1.s[st]);
    }
  if constexpr (C::TAIL) {
    u32x4 v[NI], h0[NWT], h1[NWT];
    tail_planes<T, D, NW>(tile, lane, v);
    w0.tail(h0, h1);
    mma_planes16<T>(a0.tail[0], v, h0);
    mma_planes16<T>(a0.tail[1], v, h1);
    w1.tail(h0, h1);
    mma_planes16<T>(a1.tail[0], v, h0);
    mma_planes16<T>(a1.tail[1], v, h1);
  }
}

// Power of two per output row that keeps an unbounded W operand inside the f16 range (fp16 operands only): W is multiplied by
// `mul` before it is split and the accumulator it feeds carries the same factor until the epilogue divides it out.  mul = 2^(9-e)
// for the largest magnitude 2^e seen when it was last set (2^14 is the most that W then reaches, and its small elements lie as
// far above the end of the f16 range as they can); raised when a magnitude exceeds 32 times that, and lowered together
// with the accumulator where a larger maximum scales what was summed so far away.
template <typename T>
struct RowScale {
  float mul = 1.f, limit = 0.f;
  // The accumulator's factor where its row is to be scaled by alpha = 2^-drop, drop >= 0.  The reference magnitude shrinks with the row:
  // left where an early tile put it, the f16 steps of later, smaller W would be as coarse as that tile's (dO behind a step of the scores
  // by 30 nats, tangent scores 10^5 times larger in front of it: 2.6e-2 off; fp16 rounding 5e-4).
  __device__ __forceinline__ float decay(float alpha, float drop) {
    if constexpr (!SplitType<T>::F16) return alpha;
    const uint32_t k = static_cast<uint32_t>(fminf(drop, 120.f));
    const float m2 = mul * __uint_as_float((127u + k) << 23);
    const bool ok = k < 120u && m2 < 0x1p120f;   // beyond: back to the start, with what is left of the row in its own units
    const float f = alpha * (ok ? __uint_as_float((127u + k) << 23) : 1.f / mul);
    limit = ok ? limit * __uint_as_float((127u - k) << 23) : 0.f;
    mul = ok ? m2 : 1.f;
    return f;
  }
  template <typename A>
  __device__ __forceinline__ void update(const f32x16& w, A& acc) {
    if constexpr (SplitType<T>::F16) {
      float mx = fmaxf(fabsf(w[0]), fabsf(w[1]));
#pragma unroll
      for (int i = 2; i < 16; ++i) mx = fmaxf(mx, fabsf(w[i]));
      mx = xhalf_max(mx);
      if (__builtin_amdgcn_ballot_w64(mx > limit) != 0) {
        const uint32_t e = __float_as_uint(mx) & 0x7f800000u;
        const bool up = mx > limit && e > 0 && e < 0x7f000000u;
        const uint32_t scaled = 0x7f000000u + (kRowScaleBias << 23) - e;
        const float m2 = up ? __uint_as_float(scaled < 0x7e800000u ? scaled : 0x7e800000u) : mul;
        limit = up ? 32.f * __uint_as_float(e) : limit;
        acc.scale(m2 / mul);
        mul = m2;
      }
    }
  }
  __device__ __forceinline__ float inverse() const { return SplitType<T>::F16 ? 1.f / mul : 1.f; }
};

// Zero the vectors past the head dim of NT tile planes once; commits never touch them.
template <typename T, int D, int NW>
__device__ __forceinline__ void zero_plane_pads(char* planes, int nplanes, int tid) {
  using C = SplitCfg<T, D, NW>;
  constexpr int PADV = C::P - C::VPR;
  for (int i = tid; i < nplanes * 32 * PADV; i += 64 * NW)
    *reinterpret_cast<u32x4*>(planes + (i / PADV) * C::P * 16 + (C::VPR + i % PADV) * 16) = u32x4{0, 0, 0, 0};
}

// Epilogue: rows of a transposed accumulator, times a factor per row, staged through LDS and stored.
template <typename T, int D, int NW>
__device__ __forceinline__ void store_out(char* smem, T* dst, int64_t row_stride, int row0, int nrows, int tid, const OutAcc<T, D, NW>& a,
                                          float f) {
  using C = SplitCfg<T, D, NW>;
  float f16[2] = {f, f};
  if constexpr (C::TAIL) swap16f(f, f16[0], f16[1]);
  store_rows_transposed<T, D, NW, C::NMT>(reinterpret_cast<T*>(smem), dst, row_stride, row0, nrows, tid,
                                          [&](int t, int i) { return a.t[t][i] * f; },
                                          [&](void* ws) {
                                            if constexpr (C::TAIL)
                                              store_tail16<T, D, C::NMT>(ws, tid & 63, [&](int hq, int e) { return a.tail[hq][e] * f16[hq]; });
                                          });
}

// ------------------------------------------------------------------------------------------------- forward (+ JVP)
// Start of the running maximum (log2 units).  Finite, and above what keys masked by the lowest number of their type give, so that
// a tile of nothing but such keys or of -inf scores weighs nothing: with its own maximum m subtracted, fma(S, c2, -m) would be the
// rounding error of m, which is large where m is.
constexpr float kLowestMax = -1e30f;
constexpr float kSplitLazyLog2 = 6.0f;   // the running maximum is raised when exceeded by more than 2^6 (exact: normalised once at the end)

// Two forms of the forward.  NW = 4 (128 rows): the tiles of the next step are requested before a step's products and committed
// after them, into the other of two LDS stages where two fit (one barrier per step).  NW = 8 (256 rows): what bounds the 4-wave
// form with tangents is that a wave has a SIMD's register file to itself (422 of 512 registers at fp16 D72, 352 at fp32 D64), so
// nothing runs beside its softmax and its splitting (matrix pipe 37 % busy).  Here a wave stays within 256: one LDS stage, K and V
// requested and committed a phase apart (half as many loads in flight), the planes of dQ in LDS; and with twice as many rows to a
// tile the splitting of fp32 elements, a third of the vector instructions, is shared by twice as many waves -- with tangents four
// of them bring the primal tile of a pair and four the tangent's.  us (4 -> 8 waves): fp16 + tangents B8 H16 N1024 D72 311 -> 188,
// fp32 + tangents B4 H16 N1024 D64 267 -> 233, fp16 B8 H16 N1024 D72 97 -> 78 (four waves per SIMD instead of three).  Without tangents two stages fit
// beside one another even so, and K and V come together, one barrier a step instead of two; with products ahead of the other waves' vector
// instructions (s_setprio) 72.3 -> 69.7 (of which 1 the barrier), B64 N256 50.4 -> 47.3, B4 N2048 137 -> 133, two thirds of a round B12 N1024 115 -> 116;
// with tangents the priority changes nothing (fp32 B16 H12 N256 D64 153 -> 153).
template <typename T, int D, bool JVP, int NW>
struct SplitFwdPlan {
  using C = SplitCfg<T, D, NW>;
  static constexpr bool WIDE = NW == 8, PAIR = JVP && WIDE, PHASED = PAIR;   // PHASED: one stage, K and V a phase apart
  static constexpr int NT = JVP ? 4 : 2, STAGE = NT * C::TILE;
  static constexpr int STAGES = !PHASED && 2 * STAGE <= (WIDE ? 80 : 160) * 1024 ? 2 : 1;
  static constexpr bool DQ_LDS = PAIR && (sizeof(T) == 4 || D > 64);
  static constexpr int DQ_OFF = STAGES * STAGE, DQ_BYTES = DQ_LDS ? NW * C::NCHUNK * SplitType<T>::NI * 64 * 16 : 0;
  static constexpr int BYTES = DQ_OFF + DQ_BYTES > C::STAGE_ROWS_BYTES ? DQ_OFF + DQ_BYTES : C::STAGE_ROWS_BYTES;
  static_assert(BYTES <= 160 * 1024, "LDS budget");
};

template <typename T, int D, bool JVP, int NW>
__device__ __forceinline__ void split_fwd_body(const FwdParams& p) {
  using C = SplitCfg<T, D, NW>;
  using Plan = SplitFwdPlan<T, D, JVP, NW>;
  constexpr int NI = SplitType<T>::NI, NCHUNK = C::NCHUNK, BQ = 32 * NW;
  constexpr bool F16 = SplitType<T>::F16;
  extern __shared__ __attribute__((aligned(16))) char smem[];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c32 = lane & 31, g = lane >> 5;
  const uint32_t nqb = (p.Lq + BQ - 1) / BQ;
  const uint32_t wg = xcd_remap(blockIdx.x, gridDim.x);
  const int bh = wg / nqb, q0 = (wg % nqb) * BQ, b = bh / p.H, h = bh % p.H;
  auto base = [&](int t) { return (int64_t)b * p.st[t][0] + (int64_t)h * p.st[t][2]; };
  const int qrow = q0 + wave * 32 + c32;

  zero_plane_pads<T, D, NW>(smem, Plan::STAGES * Plan::NT * NI, tid);

  // K [, dK] and V [, dV] tiles
  constexpr int LW = Plan::PAIR ? NW / 2 : NW;
  const bool second = Plan::PAIR && wave >= LW;
  const int ltid = Plan::PAIR ? tid & (64 * LW - 1) : tid;
  const int tk = second ? 4 : 1, tv = second ? 5 : 2;
  const T *gk = static_cast<const T*>(second ? p.tk : p.k) + base(tk), *gv = static_cast<const T*>(second ? p.tv : p.v) + base(tv);
  auto tile = [&](int it, int t) { return smem + (Plan::STAGES == 2 ? (it & 1) * Plan::STAGE : 0) + t * C::TILE; };
  TileLoad<T, D, LW, Plan::WIDE> lk, lv, ldk, ldv;
  lk.init(p.st[tk][1], ltid);
  lv.init(p.st[tv][1], ltid);
  auto load_k = [&](int it) {
    lk.load(gk, p.st[tk][1], it * 32, p.Lkv, ltid);
    if constexpr (JVP && !Plan::PAIR) ldk.load(static_cast<const T*>(p.tk) + base(4), p.st[4][1], it * 32, p.Lkv, tid);
  };
  auto load_v = [&](int it) {
    lv.load(gv, p.st[tv][1], it * 32, p.Lkv, ltid);
    if constexpr (JVP && !Plan::PAIR) ldv.load(static_cast<const T*>(p.tv) + base(5), p.st[5][1], it * 32, p.Lkv, tid);
  };
  auto commit_k = [&](int it) {
    lk.commit(tile(it, second ? 2 : 0), ltid);
    if constexpr (JVP && !Plan::PAIR) ldk.commit(tile(it, 2), tid);
  };
  auto commit_v = [&](int it) {
    lv.commit(tile(it, second ? 3 : 1), ltid);
    if constexpr (JVP && !Plan::PAIR) ldv.commit(tile(it, 3), tid);
  };
  load_k(0);
  load_v(0);

  // dQ planes beside Q's in registers, or where that would spill in LDS, in the order in which this wave reads them back
  u32x4 Q[NCHUNK][NI], dQ[JVP && !Plan::DQ_LDS ? NCHUNK : 1][NI];
  u32x4* const dQl = reinterpret_cast<u32x4*>(smem + Plan::DQ_OFF) + wave * (NCHUNK * NI * 64) + lane;
  // The sign of the softmax scale goes into Q and dQ, and one of zero makes them zero, so that the scores keep their order: keys are masked and
  // the maximum is taken of the unscaled ones.
  const uint32_t keep = p.scale_log2 == 0.f ? 0u : ~0u, flip = p.scale_log2 < 0.f ? 0x80008000u : 0u;
  auto signed_rows = [&](u32x4 (&x)[NCHUNK][NI]) {
#pragma unroll
    for (int c = 0; c < NCHUNK; ++c)
#pragma unroll
      for (int k = 0; k < NI; ++k) x[c][k] = (x[c][k] & keep) ^ flip;
  };
  load_own_row<T, D, NW>(static_cast<const T*>(p.q) + base(0), p.st[0][1], qrow, p.Lq, g, Q);
  signed_rows(Q);
  if constexpr (Plan::DQ_LDS) {
    u32x4 x[NCHUNK][NI];
    load_own_row<T, D, NW>(static_cast<const T*>(p.tq) + base(3), p.st[3][1], qrow, p.Lq, g, x);
    signed_rows(x);
#pragma unroll
    for (int c = 0; c < NCHUNK; ++c)
#pragma unroll
      for (int k = 0; k < NI; ++k) dQl[(c * NI + k) * 64] = x[c][k];
  } else if constexpr (JVP) {
    load_own_row<T, D, NW>(static_cast<const T*>(p.tq) + base(3), p.st[3][1], qrow, p.Lq, g, dQ);
    signed_rows(dQ);
  }

  OutAcc<T, D, NW> O, dO, dOv;   // dOv (fp16 tangents only): dV^T P, apart because dO carries the row scale of P*dS
  O.zero();
  if constexpr (JVP) {
    dO.zero();
    if constexpr (F16) dOv.zero();
  }
  RowScale<T> gs;
  float m_run = kLowestMax, l_run = 0.f, mu_run = 0.f;   // m_run: the running maximum less kFwdBias
  auto uniform = [](float x) { return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(x))); };   // (else in a vector register)
  const float c2 = uniform(p.scale_log2 == 0.f ? 1.f : fabsf(p.scale_log2)), scale = uniform(fabsf(p.scale));

  // The fused product less m leaves m's own rounding error in the exponent, the same for every key of a row: harmless until it leaves the f16
  // range.  From kBiasedScores on (a wave with such rows takes the branch below for every tile) the scores are rounded like m.
  uint64_t large = 0;
  float c2_fma = c2;

  const int ntiles = (p.Lkv + 31) / 32;
  commit_k(0);
  if constexpr (!Plan::PHASED) commit_v(0);
  for (int it = 0; it < ntiles; ++it) {
    __syncthreads();   // the tile (wide: its K half) is in LDS; wide: every wave is done with V of the tile before
    if constexpr (Plan::PHASED) commit_v(it);
    if (it + 1 < ntiles) {   // in flight during the math
      load_k(it + 1);
      if constexpr (!Plan::PHASED) load_v(it + 1);
    }
    const char *Kt = tile(it, 0), *Vt = tile(it, 1), *dKt = tile(it, 2), *dVt = tile(it, 3);
    if constexpr (Plan::WIDE && !JVP) __builtin_amdgcn_s_setprio(1);
    f32x16 S = {0}, dS = {0};
#pragma unroll
    for (int c = 0; c < NCHUNK; ++c) {
      u32x4 k[NI];
      row_planes<T, D, NW>(Kt, c32, c, g, k);
      mma_planes<T>(S, k, Q[c]);
      if constexpr (JVP) {
        u32x4 dk[NI];
        row_planes<T, D, NW>(dKt, c32, c, g, dk);
        if constexpr (Plan::DQ_LDS) {
          mma_planes<T>(dS, dk, Q[c]);
          u32x4 dq[NI];
#pragma unroll
          for (int i = 0; i < NI; ++i) dq[i] = dQl[(c * NI + i) * 64];
          mma_planes<T>(dS, k, dq);
        } else {
          mma_planes<T>(dS, k, dQ[c]);
          mma_planes<T>(dS, dk, Q[c]);
        }
      }
    }
    if constexpr (Plan::WIDE && !JVP) __builtin_amdgcn_s_setprio(0);
    if ((it + 1) * 32 > p.Lkv) {
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (it * 32 + acc_row(i, g) >= p.Lkv) S[i] = -INFINITY;
    }
    float mx = fmaxf(S[0], S[1]);
#pragma unroll
    for (int i = 2; i < 16; ++i) mx = fmaxf(mx, S[i]);
    mx = xhalf_max(mx) * c2;
    if ((__builtin_amdgcn_ballot_w64(mx - m_run > kSplitLazyLog2 + kFwdBias<T>) | large) != 0) {
      // (whole numbers in the f16 kernels: alpha is a power of two, and nothing is rounded when kFwdBias is taken off)
      const float m_new = fmaxf(m_run, running_max<T>(mx)), drop = m_new - m_run, alpha = fast_exp2(-drop);
      m_run = m_new;
      l_run *= alpha;
      O.scale(alpha);
      if constexpr (JVP) {
        mu_run *= alpha;
        dO.scale(gs.decay(alpha, drop));
        if constexpr (F16) dOv.scale(alpha);
      }
      if constexpr (F16) {
        large = __builtin_amdgcn_ballot_w64(fabsf(m_run) >= kBiasedScores);
        c2_fma = uniform(large != 0 ? 1.f : c2);
        if (large != 0) S *= c2;
      }
    }
    f32x16 E, G;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      E[i] = fast_exp2(fmaf(S[i], c2_fma, -m_run));
      l_run += E[i];
      if constexpr (JVP) {
        G[i] = E[i] * (dS[i] * scale);
        mu_run += G[i];
      }
    }
    WOperand<T> we;
    we.template form<true>(E);
    if constexpr (Plan::PHASED) {
      __syncthreads();   // V is in LDS; every wave is done with K
      if (it + 1 < ntiles) {
        commit_k(it + 1);
        load_v(it + 1);
      }
    }
    if constexpr (Plan::WIDE && !JVP) __builtin_amdgcn_s_setprio(1);
    if constexpr (JVP) {
      gs.update(G, dO);
      if constexpr (F16) G *= gs.mul;
      WOperand<T> wg_;
      wg_.form(G);
      contract_rows<T, D, NW>(Vt, lane, O, we, dO, wg_);
      if constexpr (F16) contract_rows<T, D, NW>(dVt, lane, dOv, we);
      else contract_rows<T, D, NW>(dVt, lane, dO, we);
    } else {
      contract_rows<T, D, NW>(Vt, lane, O, we);
    }
    if constexpr (Plan::WIDE && !JVP) __builtin_amdgcn_s_setprio(0);
    if constexpr (!Plan::PHASED) {
      if constexpr (Plan::STAGES == 1) __syncthreads();   // every wave is done with the stage
      if (it + 1 < ntiles) {
        commit_k(it + 1);
        commit_v(it + 1);
      }
    }
  }

  const float l_tot = xhalf_sum(l_run), inv_l = 1.0f / l_tot;
  const float mu_n = JVP ? xhalf_sum(mu_run) * inv_l : 0.f;
  if (g == 0 && qrow < p.Lq) {
    if (p.lse != nullptr) p.lse[(int64_t)bh * p.Lq + qrow] = (m_run + log2f(l_tot)) * kLn2;
    if constexpr (JVP)
      if (p.dlse != nullptr) p.dlse[(int64_t)bh * p.Lq + qrow] = mu_n;
  }
  store_out<T, D, NW>(smem, static_cast<T*>(p.o) + base(6), p.st[6][1], q0, p.Lq, tid, O, inv_l * kWeightUnit<T>);
  if constexpr (JVP) {
    // dO/l - (mu/l) O, in place
    const float gi = gs.inverse(), mu_o = mu_n * kWeightUnit<T>;
#pragma unroll
    for (int t = 0; t < C::NMT; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float d = F16 ? fmaf(dO.t[t][i], gi, dOv.t[t][i] * kWeightUnit<T>) : dO.t[t][i];
        dO.t[t][i] = fmaf(-mu_o, O.t[t][i], d);
      }
    if constexpr (C::TAIL) {
      float mu16[2], gi16[2];
      swap16f(mu_o, mu16[0], mu16[1]);
      swap16f(gi, gi16[0], gi16[1]);
#pragma unroll
      for (int hq = 0; hq < 2; ++hq)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float d = F16 ? fmaf(dO.tail[hq][e], gi16[hq], dOv.tail[hq][e] * kWeightUnit<T>) : dO.tail[hq][e];
          dO.tail[hq][e] = fmaf(-mu16[hq], O.tail[hq][e], d);
        }
    }
    store_out<T, D, NW>(smem, static_cast<T*>(p.to) + base(7), p.st[7][1], q0, p.Lq, tid, dO, inv_l);
  }
}

// --------------------------------------------------------------------------------------------------------- backward
// Stages of the backward's two tensors in LDS: two when they fit beside each other (one barrier per tile), else one.
template <typename T, int D, int NW, int NT>
struct SplitStages {
  static constexpr int STAGE = NT * SplitCfg<T, D, NW>::TILE;
  static constexpr int N = 2 * STAGE <= 160 * 1024 ? 2 : 1;
  static constexpr int BYTES = N * STAGE > SplitCfg<T, D, NW>::STAGE_ROWS_BYTES ? N * STAGE : SplitCfg<T, D, NW>::STAGE_ROWS_BYTES;
  static_assert(STAGE <= 160 * 1024 && BYTES <= 160 * 1024, "LDS budget");
};

template <typename T, int D, int NW>
__device__ __forceinline__ void split_bwd_dq_body(const BwdParams& p) {
  using C = SplitCfg<T, D, NW>;
  constexpr int NI = SplitType<T>::NI, NCHUNK = C::NCHUNK, BQ = 32 * NW;
  using ST = SplitStages<T, D, NW, 2>;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c32 = lane & 31, g = lane >> 5;
  const uint32_t nqb = (p.Lq + BQ - 1) / BQ;
  const uint32_t wg = xcd_remap(blockIdx.x, gridDim.x);
  const int bh = wg / nqb, q0 = (wg % nqb) * BQ, b = bh / p.H, h = bh % p.H;
  auto base = [&](int t) { return (int64_t)b * p.st[t][0] + (int64_t)h * p.st[t][2]; };
  const int qrow = q0 + wave * 32 + c32;
  const bool qok = qrow < p.Lq;

  zero_plane_pads<T, D, NW>(smem, ST::N * 2 * NI, tid);
  TileLoad<T, D, NW> lk, lv;
  auto load = [&](int it) {
    lk.load(static_cast<const T*>(p.k) + base(2), p.st[2][1], it * 32, p.Lkv, tid);
    lv.load(static_cast<const T*>(p.v) + base(3), p.st[3][1], it * 32, p.Lkv, tid);
  };
  auto tile = [&](int it) { return smem + (ST::N == 2 ? (it & 1) * ST::STAGE : 0); };
  auto commit = [&](int it) {
    lk.commit(tile(it), tid);
    lv.commit(tile(it) + C::TILE, tid);
  };
  load(0);

  u32x4 Q[NCHUNK][NI], dO[NCHUNK][NI];
  load_own_row<T, D, NW>(static_cast<const T*>(p.q) + base(1), p.st[1][1], qrow, p.Lq, g, Q);
  load_own_row<T, D, NW>(static_cast<const T*>(p.dout) + base(0), p.st[0][1], qrow, p.Lq, g, dO);
  float dpart = 0.f;   // delta = rowsum(dout * o)
  if (qok) {
    const T* gdo = static_cast<const T*>(p.dout) + base(0) + (int64_t)qrow * p.st[0][1] + 8 * g;
    const T* go = static_cast<const T*>(p.o) + base(4) + (int64_t)qrow * p.st[4][1] + 8 * g;
#pragma unroll
    for (int c = 0; c < NCHUNK; ++c)
      if (2 * c + g < C::VPR)
#pragma unroll
        for (int e = 0; e < 8; ++e) dpart = fmaf((float)gdo[16 * c + e], (float)go[16 * c + e], dpart);
  }
  const float delta = xhalf_sum(dpart);
  float lse2 = INFINITY;   // +inf switches padded rows off
  if (qok) {
    lse2 = p.lse[(int64_t)bh * p.Lq + qrow] * kLog2e;
    if (g == 0) p.delta[(int64_t)bh * p.Lq + qrow] = delta;
  }
  OutAcc<T, D, NW> acc;
  acc.zero();
  RowScale<T> gs;
  const float c2 = p.scale_log2;
  const int ntiles = (p.Lkv + 31) / 32;
  commit(0);
  for (int it = 0; it < ntiles; ++it) {
    __syncthreads();
    if (it + 1 < ntiles) load(it + 1);
    const char *Kt = tile(it), *Vt = Kt + C::TILE;
    f32x16 S = {0}, dP = {0}, dS;
#pragma unroll
    for (int c = 0; c < NCHUNK; ++c) {
      u32x4 x[NI];
      row_planes<T, D, NW>(Kt, c32, c, g, x);
      mma_planes<T>(S, x, Q[c]);
      row_planes<T, D, NW>(Vt, c32, c, g, x);
      mma_planes<T>(dP, x, dO[c]);
    }
    const bool last = (it + 1) * 32 > p.Lkv;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float pr = fast_exp2(fmaf(S[i], c2, -lse2));
      if (last && it * 32 + acc_row(i, g) >= p.Lkv) pr = 0.f;
      dS[i] = pr * (dP[i] - delta);
    }
    gs.update(dS, acc);
    if constexpr (SplitType<T>::F16) dS *= gs.mul;
    WOperand<T> w;
    w.form(dS);
    contract_rows<T, D, NW>(Kt, lane, acc, w);
    if constexpr (ST::N == 1) __syncthreads();
    if (it + 1 < ntiles) commit(it + 1);
  }
  store_out<T, D, NW>(smem, static_cast<T*>(p.dq) + base(5), p.st[5][1], q0, p.Lq, tid, acc, p.scale * gs.inverse());
}

template <typename T, int D, int NW>
__device__ __forceinline__ void split_bwd_dkv_body(const BwdParams& p) {
  using C = SplitCfg<T, D, NW>;
  constexpr int NI = SplitType<T>::NI, NCHUNK = C::NCHUNK, BK = 32 * NW;
  using ST = SplitStages<T, D, NW, 2>;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c32 = lane & 31, g = lane >> 5;
  const uint32_t nkb = (p.Lkv + BK - 1) / BK;
  const uint32_t wg = xcd_remap(blockIdx.x, gridDim.x);
  const int bh = wg / nkb, k0 = (wg % nkb) * BK, b = bh / p.H, h = bh % p.H;
  auto base = [&](int t) { return (int64_t)b * p.st[t][0] + (int64_t)h * p.st[t][2]; };
  const int krow = k0 + wave * 32 + c32;

  zero_plane_pads<T, D, NW>(smem, ST::N * 2 * NI, tid);
  TileLoad<T, D, NW> lq, lo;
  // lse (log2 units; +inf for rows past the end: P = 0) and delta of the tile's 32 queries, one per lane: rows acc_row order
  // is read back with bpermute-free broadcasts from LDS
  float* stat = reinterpret_cast<float*>(smem + ST::BYTES);   // [stage][2][32]
  float st_pre = 0.f;
  auto load = [&](int it) {
    lq.load(static_cast<const T*>(p.q) + base(1), p.st[1][1], it * 32, p.Lq, tid);
    lo.load(static_cast<const T*>(p.dout) + base(0), p.st[0][1], it * 32, p.Lq, tid);
    if (tid < 64) {
      const int r = it * 32 + (tid & 31);
      const bool ok = r < p.Lq;
      if (tid < 32) st_pre = ok ? fmaf(p.lse[(int64_t)bh * p.Lq + r], kLog2e, -kBwdBias<T>) : INFINITY;   // P, and dS with it, times 2^kBwdBias
      else st_pre = ok ? p.delta[(int64_t)bh * p.Lq + r] : 0.f;
    }
  };
  auto tile = [&](int it) { return smem + (ST::N == 2 ? (it & 1) * ST::STAGE : 0); };
  auto commit = [&](int it) {
    lq.commit(tile(it), tid);
    lo.commit(tile(it) + C::TILE, tid);
    if (tid < 64) stat[(it & 1) * 64 + tid] = st_pre;
  };
  load(0);
  u32x4 K[NCHUNK][NI], V[NCHUNK][NI];
  load_own_row<T, D, NW>(static_cast<const T*>(p.k) + base(2), p.st[2][1], krow, p.Lkv, g, K);
  load_own_row<T, D, NW>(static_cast<const T*>(p.v) + base(3), p.st[3][1], krow, p.Lkv, g, V);
  OutAcc<T, D, NW> dK, dV;
  dK.zero();
  dV.zero();
  RowScale<T> gs;
  const float c2 = p.scale_log2;
  const int ntiles = (p.Lq + 31) / 32;
  commit(0);
  for (int it = 0; it < ntiles; ++it) {
    __syncthreads();
    if (it + 1 < ntiles) load(it + 1);
    const char *Qt = tile(it), *dOt = Qt + C::TILE;
    const float* ls = stat + (it & 1) * 64 + 4 * g;
    f32x16 S = {0}, dP = {0}, Pm, dS;
#pragma unroll
    for (int c = 0; c < NCHUNK; ++c) {
      u32x4 x[NI];
      row_planes<T, D, NW>(Qt, c32, c, g, x);
      mma_planes<T>(S, x, K[c]);
      row_planes<T, D, NW>(dOt, c32, c, g, x);
      mma_planes<T>(dP, x, V[c]);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f32x4 l4 = *reinterpret_cast<const f32x4*>(ls + 8 * j), d4 = *reinterpret_cast<const f32x4*>(ls + 32 + 8 * j);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 4 * j + e;
        Pm[i] = fast_exp2(fmaf(S[i], c2, -l4[e]));
        dS[i] = Pm[i] * (dP[i] - d4[e]);
      }
    }
    WOperand<T> wp;
    wp.template form<true>(Pm);
    contract_rows<T, D, NW>(dOt, lane, dV, wp);
    gs.update(dS, dK);
    if constexpr (SplitType<T>::F16) dS *= gs.mul;
    WOperand<T> ws;
    ws.form(dS);
    contract_rows<T, D, NW>(Qt, lane, dK, ws);
    if constexpr (ST::N == 1) __syncthreads();
    if (it + 1 < ntiles) commit(it + 1);
  }
  constexpr float kUnbias = SplitType<T>::F16 ? 1.f / 1024.f : 1.f;   // 2^-kBwdBias
  store_out<T, D, NW>(smem, static_cast<T*>(p.dk) + base(6), p.st[6][1], k0, p.Lkv, tid, dK, p.scale * kUnbias * gs.inverse());
  store_out<T, D, NW>(smem, static_cast<T*>(p.dv) + base(7), p.st[7][1], k0, p.Lkv, tid, dV, kUnbias * kWeightUnit<T>);
}

}  // namespace dmf
