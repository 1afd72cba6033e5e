// The adaLN modulations of a whole stack of blocks in one launch: out_g = S_{c(g)} W_g^T + b_g for every group g (one block's
// 6 C x C projection, or the final layer's 2 C x C), S = silu of one of at most two conditioning vectors, B rows of it, and with
// tangents T_g = dS_{c(g)} W_g^T.
//
// What bounds it is reading the weights once: 12 blocks of C = 768 are 85 MB against 3 to 24 MFLOP per MB, and a library product
// per block spends 7 to 9 us on 7 MB, twice with tangents.  A wave owns 32 output columns and all rows: its 32 weight rows are MFMA
// operands as they lie in memory (16 bytes of a row per lane), each is loaded once and used for every 32-row tile of S and dS,
// which the waves of a work-group share through the first-level cache.  No LDS, no barrier: with all groups in one grid some 1700
// waves are resident, four weight steps in flight each.
// us, both silu launches included, against a library product per group (and stream): C = 768, 12 blocks, B = 16 33 (the kernel 29, 3.0 TB/s)
// against 89, B = 64 with tangents 85 against 201, B = 128 with tangents 144 against 227; C = 1152, 28 blocks, B = 16 125 (3.6 TB/s) against
// 251, B = 32 with tangents 221 against 404.  From 64 rows up the operand reads of S and dS, not the weights, take the time.
#include "attn_common.h"
#include "attn_kernels.h"
#include "../../include/dmf_fused.h"

namespace dmf {

constexpr int kModMaxGroups = 64, kModStep = 32, kModAhead = 4;   // k elements per step; steps of weights in flight

struct ModulationParams {
  const __bf16* s[2];    // silu of the conditioning vectors: B primal rows, with tangents followed by B tangent rows
  const __bf16 *w[kModMaxGroups], *bias[kModMaxGroups];
  __bf16* out[kModMaxGroups];   // B primal rows of n columns, with tangents followed by B tangent rows
  uint64_t cond_bits;    // bit g: which conditioning vector
  int groups, B, K, n, n_last, tiles, tiles_last;   // columns and 128-column tiles of a group, of the last one
};

// NT 32-row tiles: the first half primal, the second tangents (JVP), or all primal.
template <int NT, bool JVP>
__global__ __launch_bounds__(256) void modulation_kernel(const ModulationParams p) {
  const int lane = threadIdx.x & 63, c32 = lane & 31, g = lane >> 5, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int last = p.groups - 1, in_blocks = last * p.tiles, wg = blockIdx.x;
  const int grp = wg < in_blocks ? wg / p.tiles : last, tile = wg < in_blocks ? wg % p.tiles : wg - in_blocks;
  const int N = grp == last ? p.n_last : p.n, n0 = tile * 128 + wave * 32;
  if (n0 >= N) return;
  constexpr int PT = JVP ? NT / 2 : NT;   // primal tiles
  const __bf16* s = p.s[(p.cond_bits >> grp) & 1];
  const __bf16* w = p.w[grp] + (int64_t)(n0 + c32) * p.K + 8 * g;
  const __bf16* srow[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {   // (rows past the end repeat the last one: those columns of the result are not stored)
    const int row = min((t % PT) * 32 + c32, p.B - 1) + (t >= PT ? p.B : 0);
    srow[t] = s + (int64_t)row * p.K + 8 * g;
  }
  const int steps = p.K / kModStep;
  u32x4 W[kModAhead][2];
  auto request = [&](int i, int step) {
    W[i][0] = *reinterpret_cast<const u32x4*>(w + step * kModStep);
    W[i][1] = *reinterpret_cast<const u32x4*>(w + step * kModStep + 16);
  };
#pragma unroll
  for (int i = 0; i < kModAhead; ++i) request(i, i);   // (K is a multiple of 128)
  f32x16 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f32x16{0};
  for (int s0 = 0; s0 < steps; s0 += kModAhead) {
#pragma unroll
    for (int i = 0; i < kModAhead; ++i) {
      u32x4 S[NT][2];
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h) S[t][h] = *reinterpret_cast<const u32x4*>(srow[t] + (s0 + i) * kModStep + 16 * h);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int t = 0; t < NT; ++t)
          acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, W[i][h]), __builtin_bit_cast(bf16x8, S[t][h]), acc[t], 0, 0, 0);
      if (s0 + kModAhead < steps) request(i, s0 + kModAhead + i);
    }
  }
  // lane: batch row c32 of each tile; four consecutive columns per accumulator quad
  const __bf16* bias = p.bias[grp];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int col = n0 + 8 * q + 4 * g;
    float b[4] = {0.f, 0.f, 0.f, 0.f};
    if (bias != nullptr) {
      const u32x2 raw = *reinterpret_cast<const u32x2*>(bias + col);
      b[0] = __uint_as_float(raw[0] << 16);
      b[1] = __uint_as_float(raw[0] & 0xffff0000u);
      b[2] = __uint_as_float(raw[1] << 16);
      b[3] = __uint_as_float(raw[1] & 0xffff0000u);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int row = (t % PT) * 32 + c32;
      const bool primal = t < PT;
      if (row < p.B) {
        const f32x16& a = acc[t];
        const u32x2 v{pack_bf16x2(a[4 * q] + (primal ? b[0] : 0.f), a[4 * q + 1] + (primal ? b[1] : 0.f)),
                      pack_bf16x2(a[4 * q + 2] + (primal ? b[2] : 0.f), a[4 * q + 3] + (primal ? b[3] : 0.f))};
        *reinterpret_cast<u32x2*>(p.out[grp] + (int64_t)(row + (primal ? 0 : p.B)) * N + col) = v;
      }
    }
  }
}

}  // namespace dmf

extern "C" int dmf_modulation_fwd(const void* const* s, const void* const* w, const void* const* bias, void* const* out, const int* cond, int groups, int B,
                                  int K, int n, int n_last, int jvp, void* stream) {
  if (s == nullptr || w == nullptr || bias == nullptr || out == nullptr || cond == nullptr) return DMF_ATTN_ENULL;
  if (groups < 1 || groups > dmf::kModMaxGroups || B < 1 || B > 128 || K < 128 || K % 128 || n < 32 || n % 32 || n_last < 32 || n_last % 32)
    return DMF_ATTN_ESHAPE;
  dmf::ModulationParams p{};
  for (int g = 0; g < groups; ++g) {
    if (w[g] == nullptr || out[g] == nullptr || cond[g] < 0 || cond[g] > 1 || s[cond[g]] == nullptr) return DMF_ATTN_ENULL;
    if (reinterpret_cast<uintptr_t>(w[g]) % 16 || reinterpret_cast<uintptr_t>(out[g]) % 8 || reinterpret_cast<uintptr_t>(bias[g]) % 8 ||
        reinterpret_cast<uintptr_t>(s[cond[g]]) % 16)
      return DMF_ATTN_EALIGN;
    p.w[g] = static_cast<const __bf16*>(w[g]);
    p.bias[g] = static_cast<const __bf16*>(bias[g]);
    p.out[g] = static_cast<__bf16*>(out[g]);
    p.cond_bits |= (uint64_t)cond[g] << g;
  }
  p.s[0] = static_cast<const __bf16*>(s[0]);
  p.s[1] = static_cast<const __bf16*>(s[1]);
  p.groups = groups; p.B = B; p.K = K; p.n = n; p.n_last = n_last;
  p.tiles = (n + 127) / 128;
  p.tiles_last = (n_last + 127) / 128;
  const dim3 grid((groups - 1) * p.tiles + p.tiles_last), block(256);
  auto stm = static_cast<hipStream_t>(stream);
  const int rt = B <= 32 ? 1 : B <= 64 ? 2 : 4;
  if (jvp) {
    if (rt == 1) return dmf::launch_kernel(dmf::modulation_kernel<2, true>, grid, block, 0, stm, p);
    if (rt == 2) return dmf::launch_kernel(dmf::modulation_kernel<4, true>, grid, block, 0, stm, p);
    return dmf::launch_kernel(dmf::modulation_kernel<8, true>, grid, block, 0, stm, p);
  }
  if (rt == 1) return dmf::launch_kernel(dmf::modulation_kernel<1, false>, grid, block, 0, stm, p);
  if (rt == 2) return dmf::launch_kernel(dmf::modulation_kernel<2, false>, grid, block, 0, stm, p);
  return dmf::launch_kernel(dmf::modulation_kernel<4, false>, grid, block, 0, stm, p);
}
