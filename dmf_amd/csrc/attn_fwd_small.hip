// Attention forward (+ JVP) for grids that leave most of the device idle.
//
// The tuned kernel gives a work-group 256 (128) query rows and all of the keys: a sampling call of two images has 32 such
// work-groups for 256 CUs, and each of them walks through every key tile with its waves waiting for one another.  Here a work-group
// owns 32 query rows of one (batch, head) and its four waves take every fourth key tile each -- eight times as many
// work-groups, a quarter of the tiles in a row, and no barrier in the loop, because nothing is shared: a wave reads its K
// rows straight into operand registers (a lane's 16-byte chunks are the MFMA operand as they are) and only V, whose operand
// is transposed, goes through a tile of LDS of its own.  The four partial softmax states are merged once at the end.
// What it gives up is reuse: every 32 query rows stream the keys from L2 again, so it is the right choice only while the
// grid is small (fwd_small_grid, with both sides measured).
//
// Arithmetic: that of attn_split.h with one plane (bf16) or with its fp16 operands; the scale is applied to the fp32 scores.
#include "attn_split.h"

#include <cstdio>

namespace dmf {

template <> struct SplitType<__bf16> { static constexpr int NI = 1, NWT = 1; static constexpr bool F16 = false; };

constexpr int kSmallWaves = 4;   // waves per work-group = ways the keys are split

template <typename T, int D, bool JVP>
struct SmallCfg {
  using C = SplitCfg<T, D, 1>;
  static constexpr int VTILES = JVP ? 2 : 1;
  static constexpr int WAVE_BYTES = VTILES * C::TILE;
  static constexpr int ROWS_BYTES = 32 * kSmallWaves * Cfg<float, D>::OROWV * 16;   // the fp32 rows of the four waves, over the tiles
  static constexpr int TILES_BYTES = kSmallWaves * WAVE_BYTES;
  static constexpr int STAT_OFF = ROWS_BYTES > TILES_BYTES ? ROWS_BYTES : TILES_BYTES;   // m, l, mu of every wave and row
  static constexpr int LDS_BYTES = STAT_OFF + 3 * kSmallWaves * 32 * 4;
};

// 1/rms of this lane's row in the summation order of rmsnorm_fwd_kernel (which adds the 16 vectors of a row in a butterfly over
// distances 8, 4, 2, 1), so that normalised rows come out with that kernel's bits; likewise the product with the tangent.
template <int NCHUNK>
__device__ __forceinline__ float row_tree_sum(const float (&s)[NCHUNK]) {   // s[c] = sum over vector 2c + g
  float v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = i < NCHUNK ? s[i] : 0.f;
  const float a0 = v[0] + v[4], a1 = v[1] + v[5], a2 = v[2] + v[6], a3 = v[3] + v[7];   // distance 8
  return xhalf_sum((a0 + a2) + (a1 + a3));                                              // distances 4, 2, 1
}

__device__ __forceinline__ float bf_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

// x -> x r gain (and t -> (t r + x dr) gain) on a lane's chunks of a bf16 row; element for element rmsnorm_fwd_kernel.  `valid`:
// rows past the end stay zero.
template <int D, bool JVP>
__device__ __forceinline__ void normalise_row(u32x4 (*x)[1], u32x4 (*t)[1], const float* gain, float eps, int g, bool valid) {
  constexpr int NCHUNK = (D + 15) / 16, VPR = D / 8;
  float ss[NCHUNK], st[NCHUNK];
#pragma unroll
  for (int c = 0; c < NCHUNK; ++c) {
    ss[c] = st[c] = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float a = bf_lo(x[c][0][e]), b = bf_hi(x[c][0][e]);
      ss[c] = fmaf(b, b, fmaf(a, a, ss[c]));
      if (JVP) st[c] = fmaf(b, bf_hi(t[c][0][e]), fmaf(a, bf_lo(t[c][0][e]), st[c]));
    }
  }
  const float inv_d = 1.f / static_cast<float>(D);
  const float r = valid ? 1.f / sqrtf(row_tree_sum<NCHUNK>(ss) * inv_d + eps) : 0.f;
  const float dr = JVP ? -r * r * r * row_tree_sum<NCHUNK>(st) * inv_d : 0.f;
#pragma unroll
  for (int c = 0; c < NCHUNK; ++c) {
    const bool in = 2 * c + g < VPR;
    const f32x4* gp = reinterpret_cast<const f32x4*>(gain + (in ? 16 * c + 8 * g : 0));
    const f32x4 g0 = gp[0], g1 = gp[1];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float ga = e < 2 ? g0[2 * e] : g1[2 * e - 4], gb = e < 2 ? g0[2 * e + 1] : g1[2 * e - 3];
      const float a = bf_lo(x[c][0][e]), b = bf_hi(x[c][0][e]);
      if (JVP) {
        const uint32_t w = pack_bf16x2(fmaf(bf_lo(t[c][0][e]), r, a * dr) * ga, fmaf(bf_hi(t[c][0][e]), r, b * dr) * gb);
        t[c][0][e] = in ? w : 0u;
      }
      x[c][0][e] = in ? pack_bf16x2(a * r * ga, b * r * gb) : 0u;
    }
  }
}

// NORM: per-head RMS norm of q and, where p.k_gain is given, of k (and of their tangents).
template <typename T, int D, bool JVP, bool NORM>
__global__ __launch_bounds__(64 * kSmallWaves, 1) void attn_fwd_small_kernel(const FwdParams p) {
  static_assert(!NORM || std::is_same<T, __bf16>::value, "the in-kernel norms take bf16");
  using C = SplitCfg<T, D, 1>;
  using S = SmallCfg<T, D, JVP>;
  constexpr int NI = SplitType<T>::NI, NCHUNK = C::NCHUNK, NW = kSmallWaves;
  constexpr bool F16 = SplitType<T>::F16;
  extern __shared__ __attribute__((aligned(16))) char smem[];

  const int tid = threadIdx.x, lane = tid & 63, c32 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t nqb = (p.Lq + 31) / 32;
  const uint32_t wg = xcd_remap(blockIdx.x, gridDim.x);
  const int bh = wg / nqb, qb = wg % nqb, q0 = qb * 32, b = bh / p.H, h = bh % p.H;
  auto base = [&](int t) { return (int64_t)b * p.st[t][0] + (int64_t)h * p.st[t][2]; };
  const int qrow = q0 + c32;
  const T *gk = static_cast<const T*>(p.k) + base(1), *gv = static_cast<const T*>(p.v) + base(2);
  const T *gtk = JVP ? static_cast<const T*>(p.tk) + base(4) : nullptr, *gtv = JVP ? static_cast<const T*>(p.tv) + base(5) : nullptr;

  char* Vt = smem + wave * S::WAVE_BYTES;
  char* dVt = Vt + C::TILE;
  zero_plane_pads<T, D, 1>(Vt, S::VTILES * NI, lane);

  TileLoad<T, D, 1> lv, ldv;
  u32x4 K[NCHUNK][NI], dK[JVP ? NCHUNK : 1][NI];
  auto request = [&](int it) {
    load_own_row<T, D, 1>(gk, p.st[1][1], it * 32 + c32, p.Lkv, g, K);
    if constexpr (JVP) load_own_row<T, D, 1>(gtk, p.st[4][1], it * 32 + c32, p.Lkv, g, dK);
    lv.load(gv, p.st[2][1], it * 32, p.Lkv, lane);
    if constexpr (JVP) ldv.load(gtv, p.st[5][1], it * 32, p.Lkv, lane);
  };
  u32x4 Q[NCHUNK][NI], dQ[JVP ? NCHUNK : 1][NI];
  load_own_row<T, D, 1>(static_cast<const T*>(p.q) + base(0), p.st[0][1], qrow, p.Lq, g, Q);
  if constexpr (JVP) load_own_row<T, D, 1>(static_cast<const T*>(p.tq) + base(3), p.st[3][1], qrow, p.Lq, g, dQ);
  const int ntiles = (p.Lkv + 31) / 32;
  request(wave);   // (a wave without a tile reads zeros)
  if constexpr (NORM) {
    normalise_row<D, JVP>(Q, dQ, p.q_gain, p.q_eps, g, qrow < p.Lq);
    if (p.q_hat != nullptr && wave == 0 && qrow < p.Lq) {
      T* dst = static_cast<T*>(p.q_hat) + (((int64_t)b * p.Lq + qrow) * p.H + h) * D + 8 * g;
#pragma unroll
      for (int c = 0; c < NCHUNK; ++c)
        if (2 * c + g < C::VPR) *reinterpret_cast<u32x4*>(dst + 16 * c) = Q[c][0];
    }
  }

  OutAcc<T, D, 1> O, dO, dOv;
  O.zero();
  if constexpr (JVP) {
    dO.zero();
    if constexpr (F16) dOv.zero();
  }
  RowScale<T> gs;
  // Start of the running maximum (log2 units; less kFwdBias, as in split_fwd_body): finite, so that a tile of nothing but keys masked by -inf weighs nothing, and no higher
  // than any score, so that a row whose keys all carry the lowest number still has its maximum (which is subtracted exactly: weights of one).
  float m_run = -3.40282347e38f, l_run = 0.f, mu_run = 0.f;
  const float c2 = p.scale_log2;
  for (int it = wave; it < ntiles; it += NW) {
    if constexpr (NORM) {
      if (p.k_gain != nullptr) {
        const int key = it * 32 + c32;
        normalise_row<D, JVP>(K, dK, p.k_gain, p.q_eps, g, key < p.Lkv);
        if (p.k_hat != nullptr && qb == 0 && key < p.Lkv) {   // the first query block of the head hands the rows to the backward pass
          T* dst = static_cast<T*>(p.k_hat) + (((int64_t)b * p.Lkv + key) * p.H + h) * D + 8 * g;
#pragma unroll
          for (int c = 0; c < NCHUNK; ++c)
            if (2 * c + g < C::VPR) *reinterpret_cast<u32x4*>(dst + 16 * c) = K[c][0];
        }
      }
    }
    f32x16 Sc = {0}, dS = {0};
#pragma unroll
    for (int c = 0; c < NCHUNK; ++c) {
      mma_planes<T>(Sc, K[c], Q[c]);
      if constexpr (JVP) {
        mma_planes<T>(dS, K[c], dQ[c]);
        mma_planes<T>(dS, dK[c], Q[c]);
      }
    }
    lv.commit(Vt, lane);
    if constexpr (JVP) ldv.commit(dVt, lane);
    if (it + NW < ntiles) request(it + NW);   // in flight during the softmax and the output products
    // Scaled before anything is masked or compared: c2 may be negative (the order of the scores is reversed) or zero.
    Sc *= c2;
    if ((it + 1) * 32 > p.Lkv) {
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (it * 32 + acc_row(i, g) >= p.Lkv) Sc[i] = -INFINITY;
    }
    float mx = fmaxf(Sc[0], Sc[1]);
#pragma unroll
    for (int i = 2; i < 16; ++i) mx = fmaxf(mx, Sc[i]);
    mx = xhalf_max(mx);
    if (__builtin_amdgcn_ballot_w64(mx - m_run > kSplitLazyLog2 + kFwdBias<T>) != 0) {
      const float m_new = fmaxf(m_run, running_max<T>(mx)), drop = m_new - m_run, alpha = fast_exp2(-drop);
      m_run = m_new;
      l_run *= alpha;
      O.scale(alpha);
      if constexpr (JVP) {
        mu_run *= alpha;
        dO.scale(gs.decay(alpha, drop));
        if constexpr (F16) dOv.scale(alpha);
      }
    }
    f32x16 E, G;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      E[i] = fast_exp2(Sc[i] - m_run);
      l_run += E[i];
      if constexpr (JVP) {
        G[i] = E[i] * (dS[i] * p.scale);
        mu_run += G[i];
      }
    }
    WOperand<T> we;
    we.template form<true>(E);
    if constexpr (JVP) {
      gs.update(G, dO);
      if constexpr (F16) G *= gs.mul;
      WOperand<T> wg_;
      wg_.form(G);
      contract_rows<T, D, 1>(Vt, lane, O, we, dO, wg_);
      if constexpr (F16) contract_rows<T, D, 1>(dVt, lane, dOv, we);
      else contract_rows<T, D, 1>(dVt, lane, dO, we);
    } else {
      contract_rows<T, D, 1>(Vt, lane, O, we);
    }
  }

  // ---- merge: every wave's state is brought to the largest maximum of the row (a wave without keys has l = 0)
  float* stat = reinterpret_cast<float*>(smem + S::STAT_OFF);   // [m | l | mu][wave][row]
  const float l_w = xhalf_sum(l_run), mu_w = JVP ? xhalf_sum(mu_run) : 0.f;
  if (g == 0) stat[wave * 32 + c32] = m_run;
  __syncthreads();   // (also: every wave is done with its tiles)
  float m = stat[c32];
#pragma unroll
  for (int w = 1; w < NW; ++w) m = fmaxf(m, stat[w * 32 + c32]);
  const float f = fast_exp2(m_run - m); 
  if (g == 0) {
    stat[(NW + wave) * 32 + c32] = l_w * f;
    stat[(2 * NW + wave) * 32 + c32] = mu_w * f;
  }
  float* rows = reinterpret_cast<float*>(smem);
  constexpr int OSTR = Cfg<float, D>::OSTRIDE;
  auto stage = [&](const OutAcc<T, D, 1>& a, float s) {
    float s16[2] = {s, s};
    if constexpr (C::TAIL) swap16f(s, s16[0], s16[1]);
    stage_rows<float, D, C::NMT>(rows, tid, [&](int t, int i) { return a.t[t][i] * s; },
                                 [&](void* ws) {
                                   if constexpr (C::TAIL)
                                     store_tail16<float, D, C::NMT>(ws, lane, [&](int hq, int e) { return a.tail[hq][e] * s16[hq]; });
                                 });
  };
  stage(O, f * kWeightUnit<T>);
  __syncthreads();
  float inv_l, mu_n = 0.f;
  auto row_stats = [&](int r) {
    float l = stat[NW * 32 + r], mu = stat[2 * NW * 32 + r];
#pragma unroll
    for (int w = 1; w < NW; ++w) {
      l += stat[(NW + w) * 32 + r];
      mu += stat[(2 * NW + w) * 32 + r];
    }
    inv_l = 1.f / l;
    mu_n = mu * inv_l;
    return l;
  };
  if (tid < 32) {
    const float l = row_stats(tid);
    const int row = q0 + tid;
    if (row < p.Lq) {
      if (p.lse != nullptr) p.lse[(int64_t)bh * p.Lq + row] = (m + log2f(l)) * kLn2;
      if constexpr (JVP)
        if (p.dlse != nullptr) p.dlse[(int64_t)bh * p.Lq + row] = mu_n;
    }
  }
  constexpr int NV = 32 * D / 8, PER = (NV + 255) / 256;   // 8-element vectors of the 32 rows; per thread
  float o[PER][8];
  auto gather = [&](int v, float (&x)[8]) {
    const float* src = rows + (v / C::VPR) * OSTR + (v % C::VPR) * 8;
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = src[e];
#pragma unroll
    for (int w = 1; w < NW; ++w)
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] += src[w * 32 * OSTR + e];
  };
  auto put = [&](T* dst, int64_t stride, int v, const float (&x)[8]) {
    T* d = dst + (int64_t)(q0 + v / C::VPR) * stride + (v % C::VPR) * 8;
    store4<T>(d, x[0], x[1], x[2], x[3]);
    store4<T>(d + 4, x[4], x[5], x[6], x[7]);
  };
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int v = tid + 256 * k;
    if (v < NV && q0 + v / C::VPR < p.Lq) {
      row_stats(v / C::VPR);
      gather(v, o[k]);
#pragma unroll
      for (int e = 0; e < 8; ++e) o[k][e] *= inv_l;
      put(static_cast<T*>(p.o) + base(6), p.st[6][1], v, o[k]);
    }
  }
  if constexpr (JVP) {
    __syncthreads();
    if constexpr (F16) {   // dO carries the row scale of P*dS
      const float gi = gs.inverse();
      float gi16[2] = {gi, gi};
      if constexpr (C::TAIL) swap16f(gi, gi16[0], gi16[1]);
#pragma unroll
      for (int t = 0; t < C::NMT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) dO.t[t][i] = fmaf(dO.t[t][i], gi, dOv.t[t][i] * kWeightUnit<T>);
#pragma unroll
      for (int hq = 0; hq < 2; ++hq)
#pragma unroll
        for (int e = 0; e < 4; ++e) dO.tail[hq][e] = fmaf(dO.tail[hq][e], gi16[hq], dOv.tail[hq][e] * kWeightUnit<T>);
    }
    stage(dO, f);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int v = tid + 256 * k;
      if (v < NV && q0 + v / C::VPR < p.Lq) {
        float x[8];
        row_stats(v / C::VPR);
        gather(v, x);
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = fmaf(-mu_n, o[k][e], x[e] * inv_l);
        put(static_cast<T*>(p.to) + base(7), p.st[7][1], v, x);
      }
    }
  }
}

template <typename T, int D, bool JVP, bool NORM>
static int launch_small_t(const FwdParams& p, int BH, hipStream_t stream) {
  constexpr int smem = SmallCfg<T, D, JVP>::LDS_BYTES;
  static_assert(smem <= 160 * 1024, "LDS budget");
  auto kern = attn_fwd_small_kernel<T, D, JVP, NORM>;
  static bool lds_ok[64] = {};
  if (!ensure_dynamic_lds(kern, smem, lds_ok)) return -7;
  return launch_kernel(kern, dim3((uint32_t)((p.Lq + 31) / 32) * (uint32_t)BH), dim3(64 * kSmallWaves), smem, stream, p);
}

// With tangents a wave keeps K, dK, Q, dQ and two accumulator sets: 336 .. 492 registers up to head dim 80, and beyond that
// more than there are (head dim 128: 86 .. 534 spilled), so those stay with the tuned kernel.
constexpr int kSmallMaxDimJvp = 80;

template <typename T, int D, bool NORM>
static int launch_small_n(const FwdParams& p, int BH, bool jvp, hipStream_t stream) {
  if constexpr (D <= kSmallMaxDimJvp) {
    if (jvp) return launch_small_t<T, D, true, NORM>(p, BH, stream);
  }
  return launch_small_t<T, D, false, NORM>(p, BH, stream);
}

template <int D>
static int launch_small_d(const FwdParams& p, int BH, ElemType type, bool jvp, hipStream_t stream) {
  if (type == ElemType::f16) return launch_small_n<_Float16, D, false>(p, BH, jvp, stream);
  if (p.q_gain != nullptr) return launch_small_n<__bf16, D, true>(p, BH, jvp, stream);
  return launch_small_n<__bf16, D, false>(p, BH, jvp, stream);
}

// Policy.  Measured on MI355X, small kernel against the tuned one (bf16, us; "blocks" = 32-row work-groups of the small kernel):
//   * up to one block per CU it wins from four key tiles on, forward / with tangents:
//       D64: N128 5.7 -> 4.7 / 8.6 -> 7.2, N256 8.6 -> 5.6 / 13.8 -> 9.1, N512 13.4 -> 7.5 / 21.9 -> 12.5 (256 blocks each),
//            N1024 22.4 -> 10.7 / 37.6 -> 18.8 (192 blocks); D72: N128 6.1 -> 5.6 / 10.0 -> 9.2, N256 8.7 -> 6.6 / 15.1 -> 11.5,
//            N512 13.4 -> 8.9 / 23.4 -> 16.3, N1024 22.2 -> 12.0 / 40.0 -> 22.3;
//     with two tiles it is at best equal (N64 4.2 -> 4.2), with one it loses (N32 3.6 -> 4.0);
//   * with two blocks per CU only the forward without tangents (two work-groups fit a CU) still wins, on long sequences:
//       512 blocks: D64 N512 13.6 -> 10.4, N1024 23.4 -> 15.1; D72 N512 13.6 -> 12.9, N1024 23.1 -> 19.3, but N256 8.9 -> 9.2;
//   * at four per CU it loses everywhere (N512 14.2 -> 17.6 / 23.9 -> 41.6).
bool fwd_small_grid(int Lq, int Lkv, int D, int BH, ElemType type, bool jvp) {
  if (type == ElemType::f32 || (D != 64 && D != 72 && D != 80 && D != 96 && D != 128) || (jvp && D > kSmallMaxDimJvp)) return false;
  const int64_t blocks = (int64_t)BH * ((Lq + 31) / 32), cus = compute_units();
  if (blocks <= cus) return Lkv > 96;
  return !jvp && blocks <= 2 * cus && Lkv >= 320;
}

int launch_fwd_small(const FwdParams& p, int BH, int D, ElemType type, bool jvp, hipStream_t stream) {
  switch (D) {
    case 64: return launch_small_d<64>(p, BH, type, jvp, stream);
    case 72: return launch_small_d<72>(p, BH, type, jvp, stream);
    case 80: return launch_small_d<80>(p, BH, type, jvp, stream);
    case 96: return launch_small_d<96>(p, BH, type, jvp, stream);
    case 128: return launch_small_d<128>(p, BH, type, jvp, stream);
    default: return 1;
  }
}

void plan_fwd_small(int D, bool jvp, bool norm, ElemType type, char* buf, size_t n) {
  snprintf(buf, n, "dmf::attn_fwd_small_kernel<%s, %d, %s, %s>", type == ElemType::f16 ? "_Float16" : "__bf16", D, jvp ? "true" : "false",
           norm ? "true" : "false");
}

}  // namespace dmf
