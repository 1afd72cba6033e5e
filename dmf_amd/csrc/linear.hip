// y = x W^T + b and, with tangents, ty = tx W^T: the linear layers' forward, bf16 with fp32 accumulation.  With GELU (tanh form) the
// activation is applied in the epilogue, to the primal and, through its derivative, to the tangent, so that neither pre-activation
// travels to HBM and back.
//
// The library ran the two products of a layer one after the other (two partly empty last rounds), in tiles that fit these widths
// badly, and spent 18 us of host time on each.  Here both are one grid; 192 columns divide most layer widths of the models.
#include <algorithm>
#include <cstdio>
#include <type_traits>
#include <utility>
#include "attn_common.h"
#include "attn_kernels.h"
#include "../../include/dmf_fused.h"

namespace dmf {

struct LinearParams {
  const __bf16 *x[2], *w, *bias;   // x[1]: the tangent's rows (second half of the grid), no bias
  __bf16 *y[2], *pre;              // pre: the pre-activation x w^T + bias as well (kLinGeluJvpPre)
  int M, N, K, mtiles, ntiles;
};

constexpr int kLinK = 64;   // contraction elements per step: one 128-byte line of every row

// A work-group of 2 x 2 waves owns BM rows of x against BN rows of W.  Both tiles travel HBM -> LDS by DMA, whole 128-byte lines, one
// step ahead, into the other of two stages; slot v of row r holds vector v ^ (r / 2) % 8, so that sixteen rows read at one
// vector meet all sixteen 16-byte bank groups.  A wave takes its operands of a step into registers before the next step's DMA is
// issued: the matrix products then run against loads in flight and nothing in LDS is waited for twice.  Two work-groups per CU
// cover each other's reads.
// MODE: plain; gelu; or gelu with its tangent, where the BM rows of a work-group are BM / 2 of x and the same ones of tx, so that a wave
// holds both sums of an element.
// kLinGeluJvpPre (walking kernel): that, and the pre-activation for a backward pass.
enum LinMode { kLinPlain, kLinGelu, kLinGeluJvp, kLinGeluJvpPre };

// sigma = 1 / (1 + exp(-2 u)), u = sqrt(2 / pi) (v + 0.044715 v^3): gelu(v) = 0.5 v (1 + tanh u) = v sigma.  The epilogues' arithmetic is not covered by
// products (a quarter of a gelu pair's time): the constants are multiplied out, sigma is four operations, an exp2 and a reciprocal
// (with the bias in LDS, pairs N 4C: C768 M16384 165 -> 155 us, C1152 M8192 167 -> 157; the errors against fp64 stay the same to seven digits).
constexpr double kGelu2u = 1.5957691216057308, kGeluCubic = 0.044715;   // 2 u = kGelu2u v (1 + kGeluCubic v^2)
__device__ __forceinline__ float gelu_sigma(float v) {
  constexpr double log2e = 1.4426950408889634;
  return __builtin_amdgcn_rcpf(1.f + fast_exp2(v * fmaf((float)(-log2e * kGelu2u * kGeluCubic), v * v, (float)(-log2e * kGelu2u))));
}
// d gelu = sigma (1 + v (1 - sigma) d(2 u))
__device__ __forceinline__ float gelu_slope(float v, float sigma) {
  return sigma * fmaf(fmaf(-v, sigma, v), fmaf((float)(3 * kGelu2u * kGeluCubic), v * v, (float)kGelu2u), 1.f);
}

template <int BM, int BN, int NST, int MODE>
__global__ __launch_bounds__(256, 2) void linear_kernel(const LinearParams p) {
  constexpr int MT = BM / 64, NT = BN / 64, STAGE = (BM + BN) * 128, OPITCH = BN * 2 + 16;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, c32 = lane & 31, g = lane >> 5, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  constexpr bool BOTH = MODE == kLinGeluJvp;
  constexpr int ROWS = BOTH ? BM / 2 : BM, WROWS = BOTH ? 32 : BM / 2, MROWS = BOTH ? BM / 2 : 32;   // of y; of a wave; between its row tiles
  static_assert(!BOTH || MT == 2, "one row tile of x and one of tx per wave");
  // order: groups of eight row blocks, column blocks within, so that the work-groups of one XCD share tiles in its L2
  const uint32_t per = (uint32_t)p.mtiles * p.ntiles;
  uint32_t id = xcd_remap(blockIdx.x, gridDim.x);
  const int second = id >= per;
  if (second) id -= per;
  const uint32_t grp = id / (8 * p.ntiles), first = grp * 8, rows_in = min((uint32_t)p.mtiles - first, 8u), in = id - grp * 8 * p.ntiles;
  const int m0 = (first + in % rows_in) * ROWS, n0 = (in / rows_in) * BN;

  const uint32_t kb = (uint32_t)p.K * 2;
  const __amdgpu_buffer_rsrc_t rx = make_rows_rsrc(p.x[second] + (int64_t)m0 * p.K, kb, min(ROWS, p.M - m0), (int)kb);
  const __amdgpu_buffer_rsrc_t rtx = BOTH ? make_rows_rsrc(p.x[1] + (int64_t)m0 * p.K, kb, min(ROWS, p.M - m0), (int)kb) : rx;
  const __amdgpu_buffer_rsrc_t rw = make_rows_rsrc(p.w + (int64_t)n0 * p.K, kb, min(BN, p.N - n0), (int)kb);
  const uint32_t voff = (lane >> 3) * kb + (((lane & 7) ^ ((4 * (wave & 1) + (lane >> 4)) & 7)) * 16);
  auto issue = [&](int step) {
    char* st = smem + (step % NST) * STAGE;
#pragma unroll
    for (int j = 0; j < BM / 32; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(BOTH && j >= BM / 64 ? rtx : rx, (__attribute__((address_space(3))) void*)(st + (4 * j + wave) * 1024), 16,
                                               voff, (4 * (j % (ROWS / 32)) + wave) * 8 * kb + step * 128, 0, 0);
#pragma unroll
    for (int j = 0; j < BN / 32; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (__attribute__((address_space(3))) void*)(st + BM * 128 + (4 * j + wave) * 1024), 16, voff,
                                               (4 * j + wave) * 8 * kb + step * 128, 0, 0);
  };

  f32x16 acc[NT][MT];
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[n][m] = f32x16{0};
  uint32_t xaddr[4], waddr[4];   // this lane's vector of chunk c in its row of either tile
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const uint32_t k = ((2 * c + g) ^ ((c32 >> 1) & 7)) * 16;
    xaddr[c] = lds_addr(smem) + (wm * WROWS + c32) * 128 + k;
    waddr[c] = lds_addr(smem) + BM * 128 + (wn * (BN / 2) + c32) * 128 + k;
  }
  constexpr int IN_FLIGHT = (NST - 2) * (BM + BN) / 32;   // DMA instructions of a wave behind those of the step it waits for
  static_assert(NST >= 2 && IN_FLIGHT <= 63, "vmcnt immediate");
  const int steps = p.K / kLinK;
  // (steps past the end are requested like the others -- bytes of other rows, or zeros past the last -- so that the number in flight
  //  is constant; nothing reads them, and the epilogue waits for them)
#pragma unroll
  for (int s = 0; s < NST - 1; ++s) issue(s);
  for (int s = 0; s < steps; ++s) {
    __builtin_amdgcn_s_waitcnt(0x0F70 | (IN_FLIGHT & 15) | ((IN_FLIGHT >> 4) << 14));   // this wave's share of step s is in LDS
    asm volatile("s_barrier" ::: "memory");   // everybody's is, and everybody has its operands of step s - 1
    const uint32_t st = (s % NST) * STAGE;
    u32x4 X[4][MT], W[4][NT];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const uint32_t xa = xaddr[c] + st, wa = waddr[c] + st;
      X[c][0] = lds_read128_issue<0>(xa);
      if constexpr (MT > 1) X[c][1] = lds_read128_issue<MROWS * 128>(xa);
      W[c][0] = lds_read128_issue<0>(wa);
      if constexpr (NT > 1) W[c][1] = lds_read128_issue<4096>(wa);
      if constexpr (NT > 2) W[c][2] = lds_read128_issue<8192>(wa);
    }
    issue(s + NST - 1);
    auto chunk = [&](auto cc) {
      constexpr int c = decltype(cc)::value, LATER = (3 - c) * (MT + NT) < 15 ? (3 - c) * (MT + NT) : 15;   // reads issued after this chunk's
      if constexpr (MT == 2) lds_read128_wait<LATER>(X[c][0], X[c][1]);
      else lds_read128_wait<LATER>(X[c][0]);
      if constexpr (NT >= 2) lds_read128_wait<LATER>(W[c][0], W[c][1]);
      else lds_read128_wait<LATER>(W[c][0]);
      if constexpr (NT == 3) lds_read128_wait<LATER>(W[c][2]);
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m)
          acc[n][m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, W[c][n]), __builtin_bit_cast(bf16x8, X[c][m]), acc[n][m], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    };
    chunk(std::integral_constant<int, 0>{});
    chunk(std::integral_constant<int, 1>{});
    chunk(std::integral_constant<int, 2>{});
    chunk(std::integral_constant<int, 3>{});
  }

  // the bias of this lane's columns: quad q of column tile n holds four consecutive ones
  u32x2 braw[NT][4];
  const bool biased = p.bias != nullptr && !second;
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int col = n0 + wn * (BN / 2) + 32 * n + 8 * q + 4 * g;
      braw[n][q] = biased ? *reinterpret_cast<const u32x2*>(p.bias + min(col, p.N - 4)) : u32x2{0, 0};
    }
  // rows of y through LDS: whole 16-byte vectors, BN * 2 contiguous bytes per row
  __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
  __syncthreads();
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int col = wn * (BN / 2) + 32 * n + 8 * q + 4 * g;
      const u32x2 raw = braw[n][q];
      const float b[4] = {__uint_as_float(raw[0] << 16), __uint_as_float(raw[0] & 0xffff0000u), __uint_as_float(raw[1] << 16),
                          __uint_as_float(raw[1] & 0xffff0000u)};
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] = acc[n][m][4 * q + e] + (BOTH && m == 1 ? 0.f : b[e]);
          if constexpr (MODE == kLinGelu) v[e] *= gelu_sigma(v[e]);
          if constexpr (BOTH) {
            const float x = acc[n][0][4 * q + e] + b[e], sg = gelu_sigma(x);
            if (m == 0) v[e] = x * sg;
            else v[e] *= gelu_slope(x, sg);
          }
        }
        const int row = wm * WROWS + MROWS * m + c32;
        *reinterpret_cast<u32x2*>(smem + row * OPITCH + col * 2) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
      }
    }
  __syncthreads();
  constexpr int VPRW = BN / 8, ROUNDS = BM * VPRW / 256;
  __bf16* y = p.y[second];
  u32x4 out[ROUNDS];
#pragma unroll
  for (int i = 0; i < ROUNDS; ++i) {
    const int v = tid + 256 * i;
    out[i] = *reinterpret_cast<const u32x4*>(smem + (v / VPRW) * OPITCH + (v % VPRW) * 16);
  }
#pragma unroll
  for (int i = 0; i < ROUNDS; ++i) {
    const int v = tid + 256 * i, row = v / VPRW % ROWS, cv = v % VPRW;
    __bf16* dst = BOTH && v / VPRW >= ROWS ? p.y[1] : y;
    if (m0 + row < p.M && n0 + cv * 8 < p.N) *reinterpret_cast<u32x4*>(dst + (int64_t)(m0 + row) * p.N + n0 + cv * 8) = out[i];
  }
}

template <int BM, int BN, int NST, int MODE>
static int launch_linear(LinearParams& p, bool jvp, hipStream_t stream) {
  constexpr int stages = NST * (BM + BN) * 128, out_rows = BM * (BN * 2 + 16), smem = stages > out_rows ? stages : out_rows;
  constexpr int rows = MODE == kLinGeluJvp ? BM / 2 : BM;
  auto kern = linear_kernel<BM, BN, NST, MODE>;
  static bool lds_ok[64] = {};
  if (!ensure_dynamic_lds(kern, smem, lds_ok)) return -7;
  p.mtiles = (p.M + rows - 1) / rows;
  p.ntiles = (p.N + BN - 1) / BN;
  return launch_kernel(kern, dim3((uint32_t)p.mtiles * p.ntiles * (jvp && MODE == kLinPlain ? 2 : 1)), dim3(256), smem, stream, p);
}

// ---- products with many tiles ------------------------------------------------------------------------------------------------
//
// linear_kernel's 128 x 192 tile needs 29 bytes per clock and CU from the L2 at the matrix pipes' pace, which is what it gets: C768 M16384 N 3C
// (pair) 145 us, 800 TFLOP/s.  Here one work-group of four waves has the CU to itself, one wave per SIMD with 512 registers and MT x NT accumulator
// tiles: 256 x 192 takes 30 % fewer bytes and a third fewer LDS reads per product.  The work-groups stay and walk through the tiles, so that a
// tile's first stages arrive during the last ones of the tile before and its stores drain behind the next one's products: 113 us, 1026 TFLOP/s; C768
// M16384 K 4C 153 -> 125, gelu pair N 4C 195 -> 162; C1152 M8192 N 3C 126 -> 115, K 4C 170 -> 148, gelu pair 176 -> 163.  Without its DMA the loop runs at
// 1560 TFLOP/s: what is left is the waves' wait at the CU's one address unit, four requests at a time (letting the waves take turns by branches cost
// more than it gave: 8192 cubed 819 -> 927 us), and a tile's end (3 us of 19 at 12 steps; the 6 us a tile of the estimate below are what it takes
// beyond its steps at the pace of deep products).
// Stages are 64 contraction elements, whole 128-byte lines (stages of 32 with twice the depth: 8192 x 3 unchanged, but 12 % more time in light
// grids, where each half line is a request of its own); three of x and two of w fill the LDS, x being the operand that comes from HBM.  Slot v of
// row r holds vector v ^ r / 2 % 8: 16 rows read at one vector meet all sixteen 16-byte bank groups.  While the products of one 16-deep chunk issue,
// the operands of the next are read, one LDS read behind each product.
// 128 x 96, one row tile per wave: products of at most 256 such tiles, deep or flat, filled half of the CUs or took the 64 x 64 kernel's bytes.  Five stages
// of both operands; its LDS is what bounds it (a step writes 28 KB and reads 64, W once per wave: 736 clocks of 768 with few work-groups, 920 with 256):
// C768 M4096 K 4C library 26.5 -> 24.0 us, K C 10.7 -> 9.5; C1152 M2048 K 4C 31.9 -> 28.6, K C 13.1 -> 10.9; C768 M1024 N 3C 10.2 -> 9.0.
// Results are stored past the caches (nt): C768 M16384 N 3C 122 -> 117, 256 x 128 tiles 140 -> 116.
template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N <= 63, "vmcnt immediate");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

template <int OFF>
__device__ __forceinline__ u32x2 lds_read64_issue(uint32_t lane_addr) {
  u32x2 r;
  asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(r) : "v"(lane_addr), "n"(OFF));
  return r;
}

// one element of a product's sums
__device__ __forceinline__ float sum(float a) {
  float v;
  asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(a));
  return v;
}
__device__ __forceinline__ void lds_write64(uint32_t addr, u32x2 v) { asm volatile("ds_write_b64 %0, %1" ::"v"(addr), "v"(v) : "memory"); }

// (after a wait: keeps uses of what has been read behind it)
__device__ __forceinline__ void landed_in(u32x4& v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void landed_in(u32x2& v) { asm volatile("" : "+v"(v)); }

__device__ __forceinline__ void landed_in(TrPair& v) { asm volatile("" : "+v"(v.lo), "+v"(v.hi)); }
__device__ __forceinline__ bf16x8 as_operand(const u32x4& v) { return __builtin_bit_cast(bf16x8, v); }
__device__ __forceinline__ bf16x8 as_operand(const TrPair& v) { return __builtin_bit_cast(bf16x8, tr_operand(v).v); }

template <class F, int... I>
__device__ __forceinline__ void for_each(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}

template <int MT_, int NT_, int WM_, int NSX_, int NSW_>
struct WalkTile {
  static constexpr int MT = MT_, NT = NT_, WM = WM_, WN = 4 / WM, NSX = NSX_, NSW = NSW_, BM = 32 * MT * WM, BN = 32 * NT * WN;
  static constexpr int XS = BM * 128, WS = BN * 128;
  // results pass through 4 KB of LDS per wave, its own or, where the stages take everything, the KBs of the next emptied slot of x that the wave
  // itself will request into
  static constexpr bool IN_SLOT = NSX * XS + NSW * WS + 4 * 4096 > 160 * 1024;
  static constexpr int LDS = NSX * XS + NSW * WS + (IN_SLOT ? 0 : 4 * 4096);
  static constexpr int PX = XS / 4096, PW = WS / 4096, STORES = (MT * NT + 1) / 2 * 4;
  // chunks whose operands are read ahead: with one row tile the products of one chunk are too short to hide its reads
  static constexpr int AHEAD = MT == 1 ? 2 : 1, LAST = 3 - AHEAD;   // LAST: the chunk before the one that changes stages
  // requests of a wave that may be in flight behind the stage that is waited for
  static constexpr int BEHIND = NSX > NSW ? (NSW - 2) * (PX + PW) + PX : (NSW - 2) * (PX + PW);
  static constexpr int BEFORE = NSX > NSW ? NSW - 2 : NSW - 3;   // last stage of a tile whose last chunk waits for requests from before the stores
  static_assert(!IN_SLOT || NSX > NSW && XS >= 16 * 1024);   // (the slot is requested into behind the tile's end)
  static_assert(NSW >= 2 && (NSX == NSW || NSX == NSW + 1) && LDS <= 160 * 1024 && (MT % 2 == 0 || MT == 1 && NT == 3) && BEHIND + STORES + 1 <= 63);
  // two accumulator tiles leave together, side by side where the row allows: a pass' tile h (0, 1)
  static constexpr int row_of(int pass, int h) { return MT == 1 ? 0 : NT == 3 ? 2 * (pass / 3) + (pass % 3 == 2 ? h : pass % 3) : pass / (NT / 2); }
  static constexpr int col_of(int pass, int h) { return MT == 1 ? 2 * pass + h : NT == 3 ? (pass % 3 == 2 ? 2 : h) : 2 * (pass % (NT / 2)) + h; }
};

constexpr int kNonTemporal = 2;   // (buffer instructions' aux bits)

template <class T, int MODE, bool COLS = false>
__device__ __forceinline__ void linear_walk(const LinearParams& p) {
  constexpr int MT = T::MT, NT = T::NT, BM = T::BM, BN = T::BN;
  constexpr bool BOTH = MODE >= kLinGeluJvp, BIAS = !COLS;
  constexpr int KINDS = MODE == kLinGeluJvpPre ? 3 : BOTH ? 2 : 1, STORES = BOTH ? T::STORES / 2 * KINDS : T::STORES;   // of results of an element of x
  static_assert(T::BEHIND + STORES + 1 <= 63, "vmcnt immediate");
  static_assert(!BOTH || MT % 2 == 0, "as many row tiles of x as of tx");
  constexpr int ROWS = BOTH ? BM / 2 : BM, MX = BOTH ? MT / 2 : MT;   // of y: a tile's rows, a wave's row tiles (WM * 32 rows apart)
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int lane = threadIdx.x & 63, c32 = lane & 31, g = lane >> 5, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / T::WN, wn = wave % T::WN;
  const uint32_t per = (uint32_t)p.mtiles * p.ntiles, total = MODE == kLinPlain && p.x[1] != nullptr ? 2 * per : per, G = gridDim.x;
  // The n-th tile of this work-group.  The work-groups of an XCD take neighbours; where the last round has tiles for half of them at most,
  // every tile of it is two of half the rows.
  constexpr bool HALVES = !BOTH && MT % 2 == 0;
  constexpr uint32_t END = ~0u;
  struct Place { int second, m0, n0, rows; };   // rows: of the tile (ROWS, or half of it, or what is left of M; none is possible in the second half)
  auto nth_tile = [&](uint32_t n) -> uint32_t {   // 4 * tile + (0: whole; 1, 2: a half)
    if (n * G >= total) return END;
    const uint32_t left = total - n * G, halves = HALVES && 2 * left <= G, take = left >= G ? G : left << halves;
    if (blockIdx.x >= take) return END;
    const uint32_t i = xcd_remap(blockIdx.x, take);
    return halves ? 4 * (n * G + i / 2) + 1 + i % 2 : 4 * (n * G + i);
  };
  // groups of eight row blocks, column blocks within (as linear_kernel)
  auto place = [&](uint32_t tile) {
    Place t;
    uint32_t id = tile >> 2;
    t.second = id >= per;
    if (t.second) id -= per;
    const uint32_t grp = id / (8 * p.ntiles), first = grp * 8, rows_in = min((uint32_t)p.mtiles - first, 8u), in = id - grp * 8 * p.ntiles;
    t.m0 = (int)(first + in % rows_in) * ROWS + (tile % 4 == 2 ? ROWS / 2 : 0);
    t.n0 = (int)(in / rows_in) * BN;
    t.rows = max(0, min(tile % 4 ? ROWS / 2 : ROWS, p.M - t.m0));
    t.second = __builtin_amdgcn_readfirstlane(t.second);
    t.m0 = __builtin_amdgcn_readfirstlane(t.m0);
    t.n0 = __builtin_amdgcn_readfirstlane(t.n0);
    t.rows = __builtin_amdgcn_readfirstlane(t.rows);
    return t;
  };

  const uint32_t kb = (uint32_t)p.K * 2;
  const int steps = p.K / kLinK;
  const uint32_t drow = lane >> 3;
  uint32_t voff[T::PX > T::PW ? T::PX : T::PW];   // rows 32 j + 8 wave on
#pragma unroll
  for (int j = 0; j < (T::PX > T::PW ? T::PX : T::PW); ++j)
    voff[j] = (32 * j + 8 * wave + drow) * kb + (((lane & 7) ^ ((4 * (wave & 1) + (drow >> 1)) & 7)) * 16);
  // the stages being requested, of x (with tx) and of w: tile, step, slot
  // COLS: w is (K, N) and a stage 64 of its rows, in panels of 64 columns (128-byte lines) of 8 KB each; a request is 8 rows of one panel.  The 64-byte
  // halves of rows 4 i + 2 and 4 i + 3 are exchanged: 32 lanes of a transposed read take 64 bytes of four consecutive rows, and meet all 64 banks.
  const uint32_t nb = (uint32_t)p.N * 2;
  uint32_t wvoff[COLS ? T::PW : 1];
  if constexpr (COLS) {
#pragma unroll
    for (int j = 0; j < T::PW; ++j) {
      const int b = 4 * j + wave;
      wvoff[j] = (8 * (b & 7) + drow) * nb + (b >> 3) * 128 + (((lane & 7) ^ ((drow >> 1 & 1) * 4)) * 16);
    }
  }
  struct Cursor { uint32_t nth, slot; int step; };
  Cursor cx{0, 0, 0}, cw{0, 0, 0};
  __amdgpu_buffer_rsrc_t rx, rtx, rw;
  auto aim_x = [&](uint32_t id) {
    const Place t = place(id);
    rx = make_rows_rsrc(p.x[t.second] + (int64_t)t.m0 * p.K, kb, t.rows, (int)kb);
    rtx = BOTH ? make_rows_rsrc(p.x[1] + (int64_t)t.m0 * p.K, kb, t.rows, (int)kb) : rx;
  };
  auto aim_w = [&](uint32_t id) {
    const Place t = place(id);
    // (COLS: columns past the last are those of the next row, or zeros behind the last one, and their results are not stored)
    if constexpr (COLS) rw = make_rows_rsrc(p.w + t.n0, nb, p.K, (int)(nb - t.n0 * 2));
    else rw = make_rows_rsrc(p.w + (int64_t)t.n0 * p.K, kb, min(BN, p.N - t.n0), (int)kb);
  };
  auto request_x = [&](int j) {   // a wave's j-th KB of the stage
    char* dst = smem + cx.slot * T::XS + (4 * j + wave) * 1024;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(BOTH && j >= ROWS / 32 ? rtx : rx, (__attribute__((address_space(3))) void*)dst, 16, voff[j % (ROWS / 32)],
                                             cx.step * 128, 0, 0);
  };
  auto request_w = [&](int j) {
    char* dst = smem + T::NSX * T::XS + cw.slot * T::WS + (4 * j + wave) * 1024;
    if constexpr (COLS) __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (__attribute__((address_space(3))) void*)dst, 16, wvoff[j], cw.step * 64 * nb, 0, 0);
    else __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (__attribute__((address_space(3))) void*)dst, 16, voff[j], cw.step * 128, 0, 0);
  };
  // (past the last tile's last step the requests go on -- bytes of other rows, or zeros -- so that the number in flight is constant; nothing
  //  reads them, and the kernel's end waits for them)
  auto advance = [&](Cursor& c, uint32_t ring, auto&& aim) {
    c.slot = c.slot + 1 == ring ? 0 : c.slot + 1;
    if (++c.step == steps) {
      const uint32_t next = nth_tile(c.nth + 1);
      if (next != END) {
        ++c.nth;
        c.step = 0;
        aim(next);
      } else if constexpr (COLS) {
        --c.step;   // (rows of w past its last one would be addressed: the last step's again)
      }
    }
  };

  // this lane's vector of chunk c in its row of either tile
  uint32_t xaddr[4], waddr[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const uint32_t k = ((2 * c + g) ^ ((c32 >> 1) & 7)) * 16;
    xaddr[c] = lds_addr(smem) + (wm * 32 + c32) * 128 + k;
    waddr[c] = lds_addr(smem) + T::NSX * T::XS + (wn * 32 * NT + c32) * 128 + k;
  }
  // COLS: of column group i, rows 8 g .. + 3 of a chunk's 16 (the other four: + 512), so that a lane's slots are those of its rows of x
  static_assert(NT <= 4);   // (of the bias too: two columns per lane)
  if constexpr (COLS) {
    const uint32_t i16 = lane & 15, in_panel = (8 * g + (i16 >> 2)) * 128 + ((lane >> 4) & 1) * 32 + (i16 & 3) * 8, swap = (i16 >> 3) & 1;
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const uint32_t c = wn * NT + i;
      waddr[i] = lds_addr(smem) + T::NSX * T::XS + (c >> 1) * 8192 + in_panel + ((c & 1) ^ swap) * 64;
    }
  }
  constexpr int WREADS = COLS ? 2 : 1;   // LDS reads of an operand of w
  constexpr int AHEAD = T::AHEAD, BUFS = 2 * AHEAD;
  u32x4 X[BUFS][MT];
  std::conditional_t<COLS, TrPair, u32x4> W[BUFS][NT];
  uint32_t xslot = 0, wslot = 0;   // of the stage being read
  auto read = [&](auto cc, auto ii) {   // operand ii of chunk cc
    constexpr int c = decltype(cc)::value, i = decltype(ii)::value, b = c % BUFS;
    if constexpr (i < NT && COLS) W[b][i] = lds_tr16_issue<c * 2048, c * 2048 + 512>(waddr[i] + wslot * T::WS);
    else if constexpr (i < NT) W[b][i] = lds_read128_issue<i * 4096>(waddr[c] + wslot * T::WS);
    else X[b][i - NT] = lds_read128_issue<((i - NT) % MX * 32 * T::WM + (i - NT) / MX * ROWS) * 128>(xaddr[c] + xslot * T::XS);
  };
  auto landed = [&](auto cc, auto rows) {   // chunk cc's operands; where stages change, all that are read
    constexpr int c = decltype(cc)::value, b = c % BUFS;
    if constexpr (AHEAD == 1 || c == T::LAST + 1) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    else asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(MT + NT * WREADS) : "memory");
#pragma unroll
    for (int i = 0; i < NT; ++i) landed_in(W[b][i]);
#pragma unroll
    for (int i = 0; i < decltype(rows)::value; ++i) landed_in(X[b][i]);
  };
  // The operands that are read ahead of a tile's first chunk.  The compiler takes what an assembly read returns for there and may copy it
  // before it is: at the branch into a half tile it did.  So nothing is under way where the control flow is more than the loop over a tile's
  // steps; across that loop's back edge the reads stay in flight, and that no instruction touches their registers before the wait is
  // checked on the built code.
  auto settle = [&] {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int b = 0; b < AHEAD; ++b) {
#pragma unroll
      for (int i = 0; i < NT; ++i) landed_in(W[b][i]);
#pragma unroll
      for (int i = 0; i < MT; ++i) landed_in(X[b][i]);
    }
  };
  f32x16 acc[NT][MT];

  // One stage's products.  Between the last chunk's and the next stage's, the emptied slots are requested again: w's at once, x's over the three
  // chunks that follow (all together the requests queue up in the CU's one address unit, and the waves with them).  `stores`: those of the
  // tile before may be in flight behind the stage that the last chunk waits for.
  auto stage = [&](auto first_, auto rows_, bool stores) {
    constexpr bool FIRST = decltype(first_)::value;
    constexpr int MA = decltype(rows_)::value;   // row tiles: all, or in half a tile the first half
    for_each(std::make_integer_sequence<int, 4>{}, [&](auto cc) {
      constexpr int c = decltype(cc)::value, NEXT = (c + AHEAD) % 4, NM = MA * NT, R = MA + NT, CHANGE = T::LAST + 1;
      landed(cc, rows_);
      if constexpr (c == CHANGE) {
        if (stores) wait_vm<T::BEHIND + STORES + BIAS>();
        else wait_vm<T::BEHIND>();
        asm volatile("s_barrier" ::: "memory");   // the next stage is in LDS and everybody has taken its operands of this one
        xslot = xslot + 1 == T::NSX ? 0 : xslot + 1;
        wslot = wslot + 1 == T::NSW ? 0 : wslot + 1;
      }
      for_each(std::make_integer_sequence<int, NM>{}, [&](auto ii) {
        constexpr int i = decltype(ii)::value, n = i / MA, m = i % MA;
        acc[n][m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_operand(W[c % BUFS][n]), as_operand(X[c % BUFS][m]),
                                                            FIRST && c == 0 ? f32x16{0} : acc[n][m], 0, 0, 0);
        constexpr int SLOTS = NM < R ? NM : R, r0 = i < SLOTS ? i * R / SLOTS : R, r1 = i < SLOTS ? (i + 1) * R / SLOTS : R;
        for_each(std::make_integer_sequence<int, r1 - r0>{}, [&](auto rr) {
          read(std::integral_constant<int, NEXT>{}, std::integral_constant<int, r0 + decltype(rr)::value>{});
        });
        if constexpr (c == CHANGE) {
#pragma unroll
          for (int j = i * T::PW / NM; j < (i + 1) * T::PW / NM; ++j) request_w(j);
        } else {
          constexpr int at = (c + 3 - CHANGE) % 4 * NM + i;
#pragma unroll
          for (int j = at * T::PX / (3 * NM); j < (at + 1) * T::PX / (3 * NM); ++j) request_x(j);
        }
        __builtin_amdgcn_sched_barrier(0);
      });
      if constexpr (c == CHANGE) advance(cw, T::NSW, aim_w);
      if constexpr (c == T::LAST) advance(cx, T::NSX, aim_x);
    });
  };

  aim_x(nth_tile(0));
  aim_w(nth_tile(0));
#pragma unroll
  for (int s = 0; s < T::NSW; ++s) {
#pragma unroll
    for (int j = 0; j < T::PW; ++j) request_w(j);
    advance(cw, T::NSW, aim_w);
    if (s < T::NSX - 1) {
#pragma unroll
      for (int j = 0; j < T::PX; ++j) request_x(j);
      advance(cx, T::NSX, aim_x);
    }
  }
  wait_vm<(T::NSW - 1) * T::PW + (T::NSX - 2) * T::PX>();
  asm volatile("s_barrier" ::: "memory");
  for_each(std::make_integer_sequence<int, MT + NT>{}, [&](auto ii) { read(std::integral_constant<int, 0>{}, ii); });
  if constexpr (AHEAD == 2) {   // (what the chunk before would have read and requested)
    for_each(std::make_integer_sequence<int, MT + NT>{}, [&](auto ii) { read(std::integral_constant<int, 1>{}, ii); });
#pragma unroll
    for (int j = 0; j < T::PX / 3; ++j) request_x(j);
  }
  settle();

  // Output rows leave two accumulator tiles at a time through this wave's 4 KB of LDS (32 rows of 128 bytes, slot v of row r holding vector
  // v ^ r / 2 % 8), in whole 16-byte vectors; while one pass is on its way through LDS the next one is computed.
  constexpr int GROUP = T::IN_SLOT ? 4096 : 1024;   // between groups of eight rows
  uint32_t own, put, get;   // get: rows + 8 i: slot ^ 4 i % 8
  auto pass_through = [&](uint32_t base) {
    own = base;
    put = own + (c32 >> 3) * GROUP + (c32 & 7) * 128 + ((c32 >> 1) & 7) * 16 + g * 8;
    get = own + (lane >> 3) * 128 + (((lane & 7) ^ (lane >> 4)) * 16);
  };
  if constexpr (!T::IN_SLOT) pass_through(lds_addr(smem) + T::NSX * T::XS + T::NSW * T::WS + wave * 4096);
  uint32_t bias2 = 0;
  const int half = (lane >> 2) & 1;
  auto finish = [&](uint32_t id, auto rows_) {
    constexpr int MA = decltype(rows_)::value;
    settle();
    if constexpr (T::IN_SLOT) pass_through(lds_addr(smem) + cx.slot * T::XS + wave * 1024);
    const Place at = place(id);
    u32x2 braw[BIAS ? NT * 4 : 1];   // bias of columns 8 v + 4 g .. + 3
    if constexpr (BIAS) {
      if constexpr (T::IN_SLOT) {
        wait_vm<T::PX + T::PW>();   // (as many requests are behind it at least, and no more in flight here)
        asm volatile("ds_write_b32 %0, %1" ::"v"(own + lane * 4), "v"(bias2) : "memory");
      } else if (steps < T::BEFORE + 2) {
        wait_vm<T::PX + T::PW>();   // (else the tile's last stage has waited for it)
      }
      for_each(std::make_integer_sequence<int, NT * 4>{}, [&](auto vv) {
        braw[decltype(vv)::value] = lds_read64_issue<decltype(vv)::value * 16>(own + g * 8);
      });
    }
    // (sums are taken out of their registers one quad at a time: left to itself the compiler copies all of them at once, and spills; the wait
    //  states between the last product and the first of these reads are written out, as it does not look into assembly)
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 15\n\ts_nop 7" ::: "memory");
    if constexpr (BIAS) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
      for (int v = 0; v < NT * 4; ++v) landed_in(braw[v]);
    }
    const int ncols = min(BN, p.N - at.n0);
    __amdgpu_buffer_rsrc_t ry[KINDS];
#pragma unroll
    for (int h = 0; h < KINDS; ++h) {
      __bf16* y = MODE == kLinGeluJvpPre && h == 0 ? p.pre : p.y[BOTH ? h - (KINDS - 2) : at.second];
      ry[h] = make_rows_rsrc(y + (int64_t)at.m0 * p.N + at.n0, nb, at.rows, at.rows > 0 ? ncols * 2 : (int)nb);
    }
    // with tangents: of x (first as it is, with kLinGeluJvpPre), then of tx, by turns
    constexpr int PASSES = (MA * NT + 1) / 2 * KINDS / (BOTH ? 2 : 1);
    u32x4 out[2][4];
    auto pass_row = [](int pass, int h) constexpr { return T::row_of(pass / KINDS, h) + (BOTH && pass % KINDS == KINDS - 1 ? MX : 0); };
    auto pass_col = [](int pass, int h) constexpr { return T::col_of(pass / KINDS, h); };
    auto store = [&](auto pp) {
      constexpr int pass = decltype(pp)::value, m0 = pass_row(pass, 0), m1 = pass_row(pass, 1), n0 = pass_col(pass, 0), n1 = pass_col(pass, 1);
      static_assert(m0 / MX == m1 / MX, "both of x, or both of tx");
      constexpr int kind = BOTH ? pass % KINDS : 0;
      const int tile = half ? n1 : n0, col = (wn * NT + tile) * 32 + (lane & 3) * 8, row = ((half ? m1 % MX : m0 % MX) * T::WM + wm) * 32 + (lane >> 3);
      const uint32_t off = (row * nb + col * 2) | (col < ncols && tile < NT ? 0u : 0x80000000u);   // (past the end: dropped)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        landed_in(out[pass & 1][i]);
        __builtin_amdgcn_raw_buffer_store_b128(out[pass & 1][i], ry[kind], off, 8 * i * nb, kNonTemporal);
      }
    };
    float slope[BOTH ? 2 : 1][16];   // d gelu of the pass' elements, for their tangents; before that, with kLinGeluJvpPre, the elements
    for_each(std::make_integer_sequence<int, PASSES>{}, [&](auto pp) {
      constexpr int pass = decltype(pp)::value;
      for_each(std::make_integer_sequence<int, pass_col(pass, 1) < NT ? 8 : 4>{}, [&](auto vv) {   // (a last tile by itself: half the rows' bytes)
        constexpr int v = decltype(vv)::value, h = v / 4, m = pass_row(pass, h), n = pass_col(pass, h), q = v % 4;
        const u32x2 raw = braw[BIAS ? 4 * n + q : 0];
        const float bb[4] = {__uint_as_float(raw[0] << 16), __uint_as_float(raw[0] & 0xffff0000u), __uint_as_float(raw[1] << 16),
                             __uint_as_float(raw[1] & 0xffff0000u)};
        float o[4];
        for_each(std::make_integer_sequence<int, 4>{}, [&](auto ee) {
          constexpr int e = decltype(ee)::value;
          constexpr int kind = pass % KINDS;
          if constexpr (MODE == kLinGeluJvpPre && kind == 1) o[e] = slope[h][4 * q + e];
          else o[e] = sum(acc[n][m][4 * q + e]);
          if constexpr (BOTH && kind == KINDS - 1) {
            o[e] *= slope[h][4 * q + e];
          } else {
            if constexpr (BIAS && kind == 0) o[e] += bb[e];
            if constexpr (MODE == kLinGeluJvpPre && kind == 0) {
              slope[h][4 * q + e] = o[e];
            } else if constexpr (MODE != kLinPlain) {
              const float x = o[e], sg = gelu_sigma(x);
              o[e] = x * sg;
              if constexpr (BOTH) slope[h][4 * q + e] = gelu_slope(x, sg);
            }
          }
        });
        lds_write64(put ^ (v * 16), u32x2{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])});
        __builtin_amdgcn_sched_barrier(0);
      });
      if constexpr (pass > 0) {
        asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(pass_col(pass, 1) < NT ? 8 : 4) : "memory");   // (what was read before these writes)
        store(std::integral_constant<int, pass - 1>{});
      }
      for_each(std::make_integer_sequence<int, 4>{}, [&](auto ii) {
        constexpr int i = decltype(ii)::value;
        out[pass & 1][i] = lds_read128_issue<i * GROUP>(i & 1 ? get ^ 64 : get);
      });
      __builtin_amdgcn_sched_barrier(0);
    });
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    store(std::integral_constant<int, PASSES - 1>{});
    asm volatile("s_nop 1" ::: "memory");   // (before assembly may write these registers again)
  };

  // A tile's bias is requested before its first stage (scalar loads at the tile's end left everything waiting for them: pairs C768 M16384 N 3C 119 ->
  // 113 us, C1152 M8192 N 4C 154 -> 149; 128 x 96 tiles, C768 M4096 N C 10.1 -> 9.4): this wave's columns, two per lane (by dwords, as a bias is 8-byte
  // aligned), zeros past the last one and for tangents, to where the results will pass through.  Without LDS for it, into a register; in assembly,
  // as the compiler would wait for all requests in flight at its use, and that nothing touches it before its wait is checked on the built code.
  auto request_bias = [&](uint32_t id) {
    const Place t = place(id);
    const int bytes = p.bias != nullptr && !t.second ? (p.N - t.n0) * 2 : 0;
    if constexpr (T::IN_SLOT) {
      const u32x4 rb = rows_rsrc_words(p.bias + t.n0, 0, 1, bytes);
      asm volatile("s_nop 4\n\tbuffer_load_dword %0, %1, %2, 0 offen" : "=v"(bias2) : "v"((wn * 32 * NT + 2 * lane) * 2), "s"(rb) : "memory");
    } else {
      const __amdgpu_buffer_rsrc_t rb = make_rows_rsrc(p.bias + t.n0, 0, 1, bytes);
      char* dst = smem + T::NSX * T::XS + T::NSW * T::WS + wave * 4096;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (__attribute__((address_space(3))) void*)dst, 4, (wn * 32 * NT + 2 * lane) * 2, 0, 0, 0);
    }
  };

  using Whole = std::integral_constant<int, MT>;
  using Half = std::integral_constant<int, HALVES ? MT / 2 : MT>;
  for (uint32_t n = 0;; ++n) {
    const uint32_t id = nth_tile(n);
    if (id == END) break;
    const bool stores = n > 0 && T::BEFORE >= 0;
    if constexpr (BIAS) request_bias(id);
    if (!HALVES || id % 4 == 0) {
      stage(std::true_type{}, Whole{}, stores);
      for (int t = 1; t < steps; ++t) stage(std::false_type{}, Whole{}, stores && t <= T::BEFORE);
      finish(id, Whole{});
    } else {
      if constexpr (HALVES) {
        stage(std::true_type{}, Half{}, stores);
        for (int t = 1; t < steps; ++t) stage(std::false_type{}, Half{}, stores && t <= T::BEFORE);
        finish(id, Half{});
      }
    }
  }
  wait_vm<0>();   // (no DMA may outlive the work-group's LDS)
}

template <class T, int MODE>
__global__ __launch_bounds__(256, 1) void linear_walk_kernel(const LinearParams p) {
  linear_walk<T, MODE>(p);
}

// 256 x 256: a seventh fewer bytes and LDS reads per product than 256 x 192, all of the accumulation registers and of the LDS (results pass through
// the slot that is to be requested into next).  Where the rounds are as full: pairs C768 M16384 N 3C 114 -> 107 us, N 4C with gelu 162 -> 149; C1152 M8192
// N 4C 148 -> 143; C1024 M8192 N 4C with gelu 140 -> 123; single C1152 M12288 K 4C 124 -> 105; 8192 cubed 867 -> 798 (1378 TFLOP/s).
using WalkWide = WalkTile<4, 4, 2, 3, 2>;
template <int MODE>
__global__ __launch_bounds__(256, 1) void linear_walk_wide_kernel(const LinearParams p) {
  linear_walk<WalkWide, MODE>(p);
}

// The MLP's first half where a backward pass follows: pre-activation, activation and its tangent from one product pair, where an activation kernel (50 us at
// 8192 x 4608) read the pre-activations of both back.  XL/2-width training step, four blocks, 6.74 -> 6.64 ms.
template <class T>
__global__ __launch_bounds__(256, 1) void linear_walk_pre_kernel(const LinearParams p) {
  linear_walk<T, kLinGeluJvpPre>(p);
}

template <class T, int MODE>
static int launch_walk(LinearParams& p, bool jvp, hipStream_t stream) {
  constexpr int rows = MODE >= kLinGeluJvp ? T::BM / 2 : T::BM;
  void (*kern)(LinearParams);
  if constexpr (MODE == kLinGeluJvpPre) kern = linear_walk_pre_kernel<T>;
  else if constexpr (std::is_same_v<T, WalkWide>) kern = linear_walk_wide_kernel<MODE>;
  else kern = linear_walk_kernel<T, MODE>;
  static bool lds_ok[64] = {};
  if (!ensure_dynamic_lds(kern, T::LDS, lds_ok)) return -7;
  p.mtiles = (p.M + rows - 1) / rows;
  p.ntiles = (p.N + T::BN - 1) / T::BN;
  const int64_t tiles = (int64_t)p.mtiles * p.ntiles * (jvp && MODE == kLinPlain ? 2 : 1);
  const int64_t cus = compute_units(), grid = tiles >= cus ? cus : MODE < kLinGeluJvp && T::MT % 2 == 0 && 2 * tiles <= cus ? 2 * tiles : tiles;
  return launch_kernel(kern, dim3((uint32_t)grid), dim3(256), T::LDS, stream, p);
}

// The input gradient gx = g W: the same walk with w read by columns, contracted over its rows as they lie in memory.  The library's products ran at
// 560 to 910 TFLOP/s here (C1152 M8192: 3C -> C 84.6 us, C -> C 38.7, 4C -> C 108, C -> 4C 97.5); these at 800 to 1170 (57 to 63, 24 to 27, 74 to 84, 78 to 81, by the card), bounded like
// the forward's by the address unit and the tiles' ends: transposed reads of w take as many bytes out of LDS as rows of it.
template <class T>
__global__ __launch_bounds__(256, 1) void linear_dgrad_kernel(const LinearParams p) {
  linear_walk<T, kLinPlain, true>(p);
}

template <class T>
static int launch_dgrad(LinearParams& p, hipStream_t stream) {
  auto kern = linear_dgrad_kernel<T>;
  static bool lds_ok[64] = {};
  if (!ensure_dynamic_lds(kern, T::LDS, lds_ok)) return -7;
  p.mtiles = (p.M + T::BM - 1) / T::BM;
  p.ntiles = (p.N + T::BN - 1) / T::BN;
  const int64_t tiles = (int64_t)p.mtiles * p.ntiles, cus = compute_units();
  const int64_t grid = tiles >= cus ? cus : T::MT % 2 == 0 && 2 * tiles <= cus ? 2 * tiles : tiles;
  return launch_kernel(kern, dim3((uint32_t)grid), dim3(256), T::LDS, stream, p);
}

// Tile policy: the shortest of the estimates, in 10 ns, of seven kernels.  linear_kernel: a K step (64) and a work-group's start and end with one,
// two, three work-groups on a CU, more of them never taking less; linear_walk_kernel: a step and what a tile takes beyond its steps at that
// pace, of whole and of half a tile, and the launch's.  Fitted to 1440 products of
// widths 384 to 1280, 64 to 32768 rows, single and in pairs, with and without gelu, seven tenths of them, before there was 256 x 256 and before the walking
// kernels' tiles ended as they do now; all of them, measured since, and the fit's aim are in profiles/linear_tiles.txt.  Tiles within 1.3 of the fastest
// one are met to 5 (128 x 96) to 9 % (64 x 64); the tile taken is 0.87 % slower than the fastest in the mean, 15 % in one of a hundred.  128 x 192 is all but
// never that tile; it is here for the rows of more than 65536 elements that the walking kernel does not take.  The estimate of 256 x 256 was set by hand on
// 175 products of up to 16384 rows; where it takes a product from another tile (710 of 2110) it needs 0.94 of that one's time, 1.06 at most.
struct LinTile { int bm, bn, per_cu, a[3], b[3]; };
constexpr LinTile kLinTiles[3] = {{128, 192, 2, {82, 113, 0}, {541, 761, 0}}, {128, 64, 3, {48, 68, 80}, {262, 364, 466}}, {64, 64, 2, {23, 39, 0}, {279, 263, 0}}};
constexpr bool never_shorter_with_more(const LinTile& t) {
  for (int o = 1; o < t.per_cu; ++o)
    if (t.a[o] < t.a[o - 1] || t.a[o] + t.b[o] < t.a[o - 1] + t.b[o - 1]) return false;
  return true;
}
static_assert(never_shorter_with_more(kLinTiles[0]) && never_shorter_with_more(kLinTiles[1]) && never_shorter_with_more(kLinTiles[2]));
struct LinWalk { int bm, bn, a, b, a_half, b_half, launch; };
constexpr LinWalk kLinWalks[3] = {{256, 192, 94, 607, 59, 433, 136}, {256, 128, 73, 386, 45, 413, 135}, {256, 256, 116, 800, 64, 640, 136}};

static int64_t walk_cost(const LinWalk& c, int64_t M, int64_t N, int64_t steps, int products, bool halves) {
  const int64_t cus = compute_units(), tiles = ((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn) * products, rest = tiles % cus;
  return c.launch + tiles / cus * (c.a * steps + c.b) + (rest == 0 ? 0 : halves && 2 * rest <= cus ? c.a_half * steps + c.b_half : c.a * steps + c.b);
}

// A gelu pair holds an element of x and its tangent in one wave, half of the rows of each: it has as many work-groups as a single product of twice
// the rows, takes the tiles with two row tiles per wave, and whole ones.
static int linear_tile(int64_t M, int N, int K, bool jvp, bool gelu) {
  const int64_t cus = compute_units(), steps = K / kLinK;
  const bool both = jvp && gelu;
  if (both) {
    M *= 2;
    jvp = false;
  }
  int best = 0;
  int64_t cost_best = INT64_MAX;
  auto take = [&](int tile, int64_t cost) {
    if (cost < cost_best) {
      cost_best = cost;
      best = tile;
    }
  };
  for (int t = 0; t < (both ? 2 : 3); ++t) {
    const LinTile& c = kLinTiles[t];
    const int64_t wgs = ((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn) * (jvp ? 2 : 1), slots = cus * c.per_cu, rest = wgs % slots;
    auto full = [&](int64_t occ) { return c.a[occ] * steps + c.b[occ]; };
    auto round = [&](int64_t n) {   // some CUs with one work-group more than the others: the step up, and the rest by their share
      const int64_t o = (n + cus - 1) / cus - 1, over = n - o * cus;
      return o == 0 || over == cus ? full(o) : full(o - 1) + (full(o) - full(o - 1)) * (35 * cus + 65 * over) / (100 * cus);
    };
    take(t, wgs / slots * round(slots) + (rest ? round(rest) : 0));
  }
  // 128 x 96, where all tiles run at once: an L2 shared by more than half of the CUs lengthens the step
  if (!both && N <= 65536 && K <= 65536) {
    const int64_t tiles = ((M + 127) / 128) * ((N + 95) / 96) * (jvp ? 2 : 1);
    if (tiles <= cus) take(5, 534 + (31 * cus + 14 * std::max<int64_t>(0, tiles - cus / 2)) * steps / cus);
  }
  // (the walking kernel's row offsets within a tile are 32-bit)
  for (int t = 0; t < 2 && N <= 65536 && K <= 65536; ++t) take(3 + t, walk_cost(kLinWalks[t], M, N, steps, jvp ? 2 : 1, !both));
  // 256 x 256 from nearly a round on (M12288 C1152 K 4C, 240 tiles, 131 -> 106 us; half tiles alone are no use: M3072 pair 67 against 74)
  if (N <= 65536 && K <= 65536 && 8 * ((M + 255) / 256) * ((N + 255) / 256) * (jvp ? 2 : 1) >= 7 * cus)
    take(6, walk_cost(kLinWalks[2], M, N, steps, jvp ? 2 : 1, !both));
  return best;
}

template <int MODE>
static int launch_linear_tile(int tile, LinearParams& p, bool jvp, hipStream_t stream) {
  switch (tile) {
    case 0: return launch_linear<128, 192, 2, MODE>(p, jvp, stream);
    case 1: return launch_linear<128, 64, 2, MODE>(p, jvp, stream);
    case 3: return launch_walk<WalkTile<4, 3, 2, 3, 2>, MODE>(p, jvp, stream);
    case 4: return launch_walk<WalkTile<4, 2, 2, 3, 3>, MODE>(p, jvp, stream);
    case 5:
      if constexpr (MODE != kLinGeluJvp) return launch_walk<WalkTile<1, 3, 4, 5, 5>, MODE>(p, jvp, stream);
      break;
    case 6: return launch_walk<WalkWide, MODE>(p, jvp, stream);
    default: break;
  }
  if constexpr (MODE == kLinGeluJvp) return DMF_ATTN_ESHAPE;   // (linear_tile does not answer this)
  else return launch_linear<64, 64, 4, MODE>(p, jvp, stream);
}

}  // namespace dmf

// Which calls these kernels are the faster ones for (us on the GPU, library -> here, all in profiles/linear_tiles.txt; C: model width, M rows; called from
// the host a library product takes 18 us at least, one of these 5):
//   pairs: C768 M16384 N 3C 139 -> 107, N C 48 -> 42, K 4C 134 -> 131; C1152 M8192 160 -> 112, 64 -> 44, N 4C 174 -> 143, K 4C 169 -> 149;
//     M4096 83 -> 60, 40 -> 25, K 4C 93 -> 75;
//   single: C768 M1024 N 3C 11.6 -> 9.0, M2048 16.4 -> 12.7, M4096 19.7 -> 19.0, N C 12.0 -> 10.7; C1152 M8192 N 3C 80 -> 61, K 4C 80 -> 73;
//     K 4C: M1024 C768 15.2 -> 13.4, M2048 C384 9.9 -> 8.6, C1152 32.5 -> 28.2, M3000 C768 24.0 -> 20.8, M4096 26.8 -> 25.0, M8192 38.2 -> 37.7.
// The library's time moves by a fifth to either side with its own choice of tile, so that no line is sharp.  It keeps
//   single products deeper than they are wide (K 4C) whose 128 x 96 tiles need up to a third of a second round (M4500 C768 28.0 against 29.8, M3072 C1024 30.0
//     against 32.1, M3000 C1152 37.1 against 38.5; one round, M4096 C768, 26.8 against 25.0; from four thirds on even in the mean);
//   those that spread a short K over a large result (N 4C: C768 M16384 pairs 135 against 136, M32768 single 132 against 137), rows of 2 or 8 KB on
//     large results (C1024: M16384 K 4C 94 against 105, N C 29.9 against 32.2, M8192 N 4C 56 against 60);
//   and outputs narrower than a tile.
// These lines were drawn before 256 x 256 tiles: the 287 products that they leave to the library would take 0.95 of its time here, in the mean.
// Deep products of few rows are a trade: on the GPU alone, as replayed from a graph, the library's are faster (K 4C: M64 C768 10.2 against 12.5, M256
// 9.3 against 13.1, M512 12.9 against 12.8, M2048 18.9 against 20.5), called from the host slower where that is what bounds the calls (18.3
// against 12.1 up to M512; the library taken for M2197 C768, two blocks sampled by a host that does not run ahead: 1.68 -> 1.73 ms).  They are taken.
//   pairs with gelu (library pair and activation kernel; this kernel's pair and the activation kernel -> here), N 4C, wins from one row up:
//     M16 C384 10.4; 7.7 -> 5.3, C768 11.3; 8.1 -> 7.1, C1152 12.7; 9.2 -> 8.9;  M512 C768 23.4; 15.5 -> 12.0, C1152 34.0; 24.1 -> 18.2;
//     M4096 C768 61.7; 58.2 -> 40.7, C1152 131; 104 -> 82;  M8192 C384 63.8; 43.6 -> 28.6, C1024 152; 182 -> 138, C1152 212; 212 -> 159.
extern "C" int dmf_linear_plan(int64_t M, int N, int K, int jvp, int gelu) {
  if (M < 1 || N < 64 || N % 8 || K < 64 || K % 64 || M * K > (int64_t)1 << 30 || (int64_t)N * K > (int64_t)1 << 30 || M * N > (int64_t)1 << 30) return 0;
  if (jvp && gelu) return 1;
  if (!jvp && K > 2048 && K >= 2 * N) {
    const int64_t cus = dmf::compute_units(), tiles = ((M + 127) / 128) * ((N + 95) / 96);
    if (tiles > cus && 3 * tiles <= 4 * cus) return 0;
  }
  if (K >= 1024 && (K & (K - 1)) == 0 && (M >= 16384 || (N >= 4 * K && M >= 4096))) return 0;
  if (M * N > 40000000 && N > 3 * K && N > 2048 && (jvp || K < 1024)) return 0;
  return 1;
}

extern "C" int dmf_linear_gelu_plan(int64_t M, int N, int K) {
  if (!dmf_linear_plan(M, N, K, 1, 1) || N > 65536 || K > 65536) return 0;
  const int tile = dmf::linear_tile(M, N, K, true, true);
  return tile == 3 || tile == 4 || tile == 6;
}

extern "C" int dmf_linear_gelu_fwd(const void* x, const void* tx, const void* w, const void* bias, void* pre, void* y, void* ty, int M, int N, int K, void* stream) {
  if (x == nullptr || tx == nullptr || w == nullptr || pre == nullptr || y == nullptr || ty == nullptr) return DMF_ATTN_ENULL;
  if (!dmf_linear_gelu_plan(M, N, K)) return DMF_ATTN_ESHAPE;
  for (const void* q : {x, tx, w, bias, (const void*)pre, (const void*)y, (const void*)ty})
    if (reinterpret_cast<uintptr_t>(q) % (q == bias ? 8 : 16)) return DMF_ATTN_EALIGN;
  dmf::LinearParams p{};
  p.x[0] = static_cast<const __bf16*>(x);
  p.x[1] = static_cast<const __bf16*>(tx);
  p.w = static_cast<const __bf16*>(w);
  p.bias = static_cast<const __bf16*>(bias);
  p.y[0] = static_cast<__bf16*>(y);
  p.y[1] = static_cast<__bf16*>(ty);
  p.pre = static_cast<__bf16*>(pre);
  p.M = M; p.N = N; p.K = K;
  auto stm = static_cast<hipStream_t>(stream);
  const int tile = dmf::linear_tile(M, N, K, true, true);
  return tile == 3   ? dmf::launch_walk<dmf::WalkTile<4, 3, 2, 3, 2>, dmf::kLinGeluJvpPre>(p, true, stm)
         : tile == 4 ? dmf::launch_walk<dmf::WalkTile<4, 2, 2, 3, 3>, dmf::kLinGeluJvpPre>(p, true, stm)
                     : dmf::launch_walk<dmf::WalkWide, dmf::kLinGeluJvpPre>(p, true, stm);
}

extern "C" int dmf_linear_fwd_plan(int64_t M, int N, int K, int jvp, int gelu, char* buf, int buflen) {
  if (M < 1 || M > INT32_MAX || N < 8 || N % 8 || K < 64 || K % 64 || M * K > (int64_t)1 << 30 || (int64_t)N * K > (int64_t)1 << 30 || M * N > (int64_t)1 << 30)
    return DMF_ATTN_ESHAPE;
  if (buf == nullptr || buflen < 1) return DMF_ATTN_ENULL;
  const int mode = !gelu ? dmf::kLinPlain : jvp ? dmf::kLinGeluJvp : dmf::kLinGelu;
  const char* form[7] = {"linear_kernel<128, 192, 2, %d>", "linear_kernel<128, 64, 2, %d>", "linear_kernel<64, 64, 4, %d>",
                         "linear_walk_kernel<dmf::WalkTile<4, 3, 2, 3, 2>, %d>", "linear_walk_kernel<dmf::WalkTile<4, 2, 2, 3, 3>, %d>",
                         "linear_walk_kernel<dmf::WalkTile<1, 3, 4, 5, 5>, %d>", "linear_walk_wide_kernel<%d>"};
  const int n = snprintf(buf, (size_t)buflen, "dmf::");
  if (n < buflen) snprintf(buf + n, (size_t)(buflen - n), form[dmf::linear_tile(M, N, K, jvp != 0, gelu != 0)], mode);
  return DMF_ATTN_OK;
}

extern "C" int dmf_linear_fwd(const void* x, const void* tx, const void* w, const void* bias, void* y, void* ty, int M, int N, int K, int gelu, void* stream) {
  if (x == nullptr || w == nullptr || y == nullptr || (tx == nullptr) != (ty == nullptr)) return DMF_ATTN_ENULL;
  if (M < 1 || N < 8 || N % 8 || K < 64 || K % 64 || (int64_t)M * K > (int64_t)1 << 30 || (int64_t)N * K > (int64_t)1 << 30 || (int64_t)M * N > (int64_t)1 << 30)
    return DMF_ATTN_ESHAPE;
  for (const void* q : {x, tx, w, (const void*)y, (const void*)ty})
    if (reinterpret_cast<uintptr_t>(q) % 16) return DMF_ATTN_EALIGN;
  if (reinterpret_cast<uintptr_t>(bias) % 8) return DMF_ATTN_EALIGN;
  dmf::LinearParams p{};
  p.x[0] = static_cast<const __bf16*>(x);
  p.x[1] = static_cast<const __bf16*>(tx);
  p.w = static_cast<const __bf16*>(w);
  p.bias = static_cast<const __bf16*>(bias);
  p.y[0] = static_cast<__bf16*>(y);
  p.y[1] = static_cast<__bf16*>(ty);
  p.M = M; p.N = N; p.K = K;
  auto stm = static_cast<hipStream_t>(stream);
  const bool jvp = tx != nullptr;
  const int tile = dmf::linear_tile(M, N, K, jvp, gelu != 0);
  if (jvp && gelu) return dmf::launch_linear_tile<dmf::kLinGeluJvp>(tile, p, true, stm);
  return gelu ? dmf::launch_linear_tile<dmf::kLinGelu>(tile, p, false, stm) : dmf::launch_linear_tile<dmf::kLinPlain>(tile, p, jvp, stm);
}

static bool dgrad_shape_ok(int64_t M, int64_t N, int64_t K) {
  constexpr int64_t most = (int64_t)1 << 30;   // (and rows within a tile are addressed in 32 bits)
  return M >= 1 && M <= INT32_MAX && N >= 64 && N % 64 == 0 && K >= 8 && K % 8 == 0 && N <= 65536 && K <= 65536 && M * N <= most && N * K <= most && M * K <= most;
}

// Which input gradients the walking kernel is the faster one for, N -> K (us on the GPU, library -> here, of the 389 products of
// profiles/linear_train_products.txt, widths 384 to 1152, 64 to 46080 rows; the 250 it takes need 0.84 of the library's time in the mean, and 5 us of
// host time where that takes 18):
//   from 3072 rows on (2048 where a row of tiles is not mostly idle or cut): C768 M4096 3C -> C 26.8 -> 21.5, M16384 53.9 -> 48.8; C1152 M16384 150 -> 114;
//     C384 M16384 22.9 -> 19.5; but C384 M2048 10.6 against 13.0, C1024 M2048 25.3 against 27.5, C768 M1536 17.5 against 20.5;
//   C -> 4C from 768 rows on: C768 M1024 13.8 -> 11.4, C1152 23.7 -> 15.1; not with one to 4/3 rounds of 256 x 192 tiles: C768 M5120 28.2 against 30.6,
//     C1024 M3072 28.5 against 32.6, on another card 28.1 against 27.1 and 28.9 against 28.6;
//   deep ones of a width that 256 columns divide lose with one to 4/3 rounds: C768 M19200 3C -> C 62.0 against 64.1, 4C -> C 77.7 against 80.9, M21120
//     63.7 against 65.8 (C1152 M13482 170 -> 95, C384 M38400 45 -> 38; C768 M22080 83 -> 71);
//   widths that 192 columns do not divide lose in many rows: C1024 M12288 3C -> C 64.8 against 70.4, M16384 80.7 against 85.9 (M8192 49.9 -> 44.7);
//   outputs narrower than a tile lose, M8192 1152 -> 64 9.1 against 11.5, and up to 6144 rows narrow ones that fill none: M3072 3072 -> 320 18.5 against 25.5.
extern "C" int dmf_linear_dgrad_plan(int64_t M, int N, int K) {
  if (!dgrad_shape_ok(M, N, K) || M < 768 || K < 192) return 0;
  if (K >= 3 * (int64_t)N) {
    const int64_t cus = dmf::compute_units(), tiles = ((M + 255) / 256) * ((K + 191) / 192);
    return tiles <= cus || 3 * tiles > 4 * cus;
  }
  if (K % 256 == 0 && N >= 3 * (int64_t)K) {
    const int64_t cus = dmf::compute_units(), tiles = ((M + 255) / 256) * ((K + 191) / 192);
    if (tiles > cus && 3 * tiles <= 4 * cus) return 0;
  }
  if (M < 3072 && (M < 2048 || K < 512 || K % 192 != 0)) return 0;
  if (M < 6144 && K < 512 && K % 192 != 0) return 0;
  return K % 192 == 0 || M < 10240;
}

// (the forward's estimates, by linear_tile's numbers: on the products above the tile they choose takes 0.4 % more than the faster of the two in the mean)
static int dgrad_tile(int64_t M, int N, int K) {
  return dmf::walk_cost(dmf::kLinWalks[0], M, K, N / dmf::kLinK, 1, true) <= dmf::walk_cost(dmf::kLinWalks[1], M, K, N / dmf::kLinK, 1, true) ? 3 : 4;
}

extern "C" int dmf_linear_dgrad(const void* g, const void* w, void* gx, int M, int N, int K, void* stream) {
  if (g == nullptr || w == nullptr || gx == nullptr) return DMF_ATTN_ENULL;
  if (!dgrad_shape_ok(M, N, K)) return DMF_ATTN_ESHAPE;
  for (const void* q : {g, w, (const void*)gx})
    if (reinterpret_cast<uintptr_t>(q) % 16) return DMF_ATTN_EALIGN;
  dmf::LinearParams p{};
  p.x[0] = static_cast<const __bf16*>(g);
  p.w = static_cast<const __bf16*>(w);
  p.y[0] = static_cast<__bf16*>(gx);
  p.M = M; p.N = K; p.K = N;   // (of the product: columns of the result, depth)
  auto stm = static_cast<hipStream_t>(stream);
  return dgrad_tile(M, N, K) == 3 ? dmf::launch_dgrad<dmf::WalkTile<4, 3, 2, 3, 2>>(p, stm) : dmf::launch_dgrad<dmf::WalkTile<4, 2, 2, 3, 3>>(p, stm);
}

namespace dmf {

// ---- weight gradient: gw = g^T x, contracted over the rows of both ----------------------------------------------------------
//
// The result is small (4608 x 1152 at most in the models) and the contraction thousands of rows deep, so that output tiles alone leave
// most CUs idle: the library's products reached 160 to 400 TFLOP/s here.  The rows are split over work-groups until the grid fills the
// chip; each writes its fp32 sums to the workspace and a second kernel adds them in a fixed order.
// Both tiles lie in LDS as they lie in memory, 64 rows of 64-column panels (128-byte lines); the transposed reads give operands that
// contract over rows.  The 64-byte halves of rows 4 i + 2 and 4 i + 3 are exchanged, so that the 32 lanes of a pass, which read 64 bytes
// of four consecutive rows, meet all 64 banks.  Step, stages and register plan are linear_kernel's.
// Relative error against fp64, library and separate column sum -> here: weights 5.7e-7 -> 1.6e-7, bias 6.7e-8 -> 6.0e-8 (8192 rows), 7.8e-7 ->
// 2.5e-7, 1.6e-7 -> 9.1e-8 (32768): the splits shorten the chains.
struct WgradParams {
  const __bf16 *g, *x;   // (M, N), (M, K)
  float* out;            // gw, or with splits the partial sums, N * K apart
  float* bias;           // the column sums of g (partial ones: N apart), or null
  int M, N, K, ntiles, ktiles, splits, per;   // per: steps of 64 rows per split
};
constexpr int kWgN = 128, kWgK = 192, kWgStage = (kWgN + kWgK) * 128;

// 32 x 32 sums out of a wave's registers through 4 KB of LDS of its own, in whole lines of 128 bytes per row; vector v of row r lies in slot v ^ r % 8.
// Stored from the registers as they are, 32 bytes of each row at a time, a tile's end took 2 to 3 us more (wide kernel with the partial sums', M 8192:
// 4608 x 1152 100.4 -> 97.0 us, 1152 x 1152 40.3 -> 38.0, 3072 x 768 53.4 -> 50.9, past the caches 97.3, 39.2, 51.5; linear_wgrad_kernel: 6912 x 1152 M 32 12.9
// -> 9.8, 3456 x 1152 M 512 15.6 -> 14.6, 768 x 768 M 4096 24.4 -> 23.9).
__device__ __forceinline__ void store_sums(char* own, const f32x16& a, float* out, int row0, int col0, int N, int K, int lane) {
  const int c32 = lane & 31, g = lane >> 5, col = col0 + (lane & 7) * 4;
#pragma unroll
  for (int q = 0; q < 4; ++q)
    *reinterpret_cast<f32x4*>(own + c32 * 128 + (((2 * q + g) ^ (c32 & 7)) * 16)) = f32x4{a[4 * q], a[4 * q + 1], a[4 * q + 2], a[4 * q + 3]};
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (no other wave is waited for)
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 8 * i + (lane >> 3), row = row0 + r;
    const f32x4 v = *reinterpret_cast<const f32x4*>(own + r * 128 + (((lane & 7) ^ (lane >> 3)) * 16));
    if (row < N && col < K) *reinterpret_cast<f32x4*>(out + (int64_t)row * K + col) = v;
  }
}

__global__ __launch_bounds__(256, 2) void linear_wgrad_kernel(const WgradParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int lane = threadIdx.x & 63, c32 = lane & 31, g = lane >> 5, i16 = lane & 15, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  // the tiles of one split are neighbours, in bands of six k tiles: the work-groups of an XCD share few columns of either operand in its L2
  const uint32_t per = (uint32_t)p.ntiles * p.ktiles, id = xcd_remap(blockIdx.x, gridDim.x), split = id / per, tile = id - split * per;
  const uint32_t band = tile / (6 * p.ntiles), in = tile - band * 6 * p.ntiles, wide = min((uint32_t)p.ktiles - 6 * band, 6u);
  const int n0 = (int)(in / wide) * kWgN, k0 = (int)(6 * band + in % wide) * kWgK;
  const int first = (int)split * p.per, steps = max(0, min(p.per, (p.M + 63) / 64 - first));

  // the whole operands from the tile's first column on: rows past the last read as zeros, columns past the last are not stored
  const uint32_t gb = (uint32_t)p.N * 2, xb = (uint32_t)p.K * 2;
  const __amdgpu_buffer_rsrc_t rg = make_rows_rsrc(p.g + n0, gb, p.M, (int)(gb - n0 * 2));
  const __amdgpu_buffer_rsrc_t rx = make_rows_rsrc(p.x + k0, xb, p.M, (int)(xb - k0 * 2));
  const uint32_t vec = ((lane & 7) ^ (((lane >> 4) & 1) * 4)) * 16, gvoff = (lane >> 3) * gb + vec, xvoff = (lane >> 3) * xb + vec;
  auto issue = [&](int step) {
    char* st = smem + (step & 1) * kWgStage;
    const uint32_t row0 = (uint32_t)(first + step) * 64;
#pragma unroll
    for (int j = 0; j < kWgN / 32; ++j) {   // block b: rows 8 (b % 8) .. + 7 of panel b / 8
      const int b = 4 * j + wave;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rg, (__attribute__((address_space(3))) void*)(st + b * 1024), 16, gvoff,
                                               (row0 + (b & 7) * 8) * gb + (b >> 3) * 128, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < kWgK / 32; ++j) {
      const int b = 4 * j + wave;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (__attribute__((address_space(3))) void*)(st + kWgN * 128 + b * 1024), 16, xvoff,
                                               (row0 + (b & 7) * 8) * xb + (b >> 3) * 128, 0, 0);
    }
  };

  // lane address of 32-column group c of either tile (see lds_col_operand); rows 16 s + 8 h on: + 2048 s + 1024 h
  const uint32_t in_panel = (4 * g + (i16 >> 2)) * 128 + ((lane >> 4) & 1) * 32 + (i16 & 3) * 8, swap = (i16 >> 3) & 1;
  auto group = [&](uint32_t base, int c) { return base + (c >> 1) * 8192 + in_panel + (((uint32_t)c & 1) ^ swap) * 64; };
  uint32_t gaddr[2], xaddr[3];
#pragma unroll
  for (int m = 0; m < 2; ++m) gaddr[m] = group(lds_addr(smem), 2 * wm + m);
#pragma unroll
  for (int n = 0; n < 3; ++n) xaddr[n] = group(lds_addr(smem) + kWgN * 128, 3 * wn + n);

  f32x16 acc[3][2];
#pragma unroll
  for (int n = 0; n < 3; ++n)
#pragma unroll
    for (int m = 0; m < 2; ++m) acc[n][m] = f32x16{0};
  // column sums of g, the bias gradient: the first k tile's work-groups have every element in registers; a step's 64 rows are summed by
  // themselves, then added to the others' (a separate column sum read g again, 11 us and a 4 us reduction a layer: four-block XL/2-width
  // training step 8.59 -> 8.42 ms)
  const bool sums = p.bias != nullptr && k0 == 0 && wn == 0;
  float total[2] = {0.f, 0.f};
  issue(0);
  for (int s = 0; s < steps; ++s) {
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): this wave's share of step s is in LDS
    asm volatile("s_barrier" ::: "memory");   // everybody's is, and everybody has its operands of step s - 1
    const uint32_t st = (s & 1) * kWgStage;
    TrPair G[4][2], X[4][3];
    auto read = [&](auto cc) {
      constexpr int c = decltype(cc)::value;
#pragma unroll
      for (int m = 0; m < 2; ++m) G[c][m] = lds_tr16_issue<c * 2048, c * 2048 + 1024>(gaddr[m] + st);
#pragma unroll
      for (int n = 0; n < 3; ++n) X[c][n] = lds_tr16_issue<c * 2048, c * 2048 + 1024>(xaddr[n] + st);
    };
    read(std::integral_constant<int, 0>{});
    read(std::integral_constant<int, 1>{});
    read(std::integral_constant<int, 2>{});
    read(std::integral_constant<int, 3>{});
    issue(s + 1);   // (past the last step too: rows of the next split, or zeros; nothing reads them, the end waits for them)
    auto chunk = [&](auto cc) {
      constexpr int c = decltype(cc)::value, LATER = (3 - c) * 10 < 15 ? (3 - c) * 10 : 15;
      lds_tr16_wait<LATER>(G[c][0], G[c][1]);
      lds_tr16_wait<LATER>(X[c][0], X[c][1]);
      lds_tr16_wait<LATER>(X[c][2]);
#pragma unroll
      for (int n = 0; n < 3; ++n)
#pragma unroll
        for (int m = 0; m < 2; ++m)
          acc[n][m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, tr_operand(X[c][n]).v),
                                                              __builtin_bit_cast(bf16x8, tr_operand(G[c][m]).v), acc[n][m], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    };
    chunk(std::integral_constant<int, 0>{});
    chunk(std::integral_constant<int, 1>{});
    chunk(std::integral_constant<int, 2>{});
    chunk(std::integral_constant<int, 3>{});
    if (sums) {
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        float t = 0.f;
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const uint32_t pair = tr_operand(G[c][m]).v[e];
            t += __uint_as_float(pair << 16) + __uint_as_float(pair & 0xffff0000u);
          }
        total[m] += t;
      }
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);   // (no DMA may be on its way into what follows)
  __syncthreads();
  float* out = p.out + (int64_t)split * p.N * p.K;
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    const int row = n0 + 64 * wm + 32 * m + c32;
    if (sums) {
      const float both = total[m] + __shfl_xor(total[m], 32);   // the halves of a wave hold different rows
      if (g == 0 && row < p.N) p.bias[(int64_t)split * p.N + row] = both;
    }
#pragma unroll
    for (int n = 0; n < 3; ++n) store_sums(smem + wave * 8192 + ((3 * m + n) & 1) * 4096, acc[n][m], out, n0 + 64 * wm + 32 * m, k0 + 96 * wn + 32 * n, p.N, p.K, lane);
  }
}

// Much work: the walking forward kernel's tile, stages and order of reads, products and requests (see linear_walk), of 256 columns of g against 192 of x,
// a work-group per CU.  Both operands lie in 64-column panels of 64 rows and are read by columns.  A step of 6.3 MFLOP takes 0.8 to 1.2 us, by how many
// CUs take part (two of linear_wgrad_kernel's, the same work, 1.25); start, end and launch 12 us where that takes 9 (both 2 less since the
// sums leave by store_sums).  With column sums and the partial sums' kernel, M 8192: 4608 x 1152 109 -> 93 us, 3456 x 1152 81 -> 74, 3072 x 768 52.7 -> 50.6,
// 3072 x 1024 78 -> 67, 1152 x 1152 39.1 -> 37.6; M 16384: 4608 x 1152 191 -> 168.
// The two waves that hold the same columns of g sum two chunks of a step each for the bias (two thirds of the room between a chunk's products).
struct WgradWide : WalkTile<4, 3, 2, 3, 2> { static constexpr int STAGES = NSX * XS + NSW * WS; };

__global__ __launch_bounds__(256, 1) void linear_wgrad_wide_kernel(const WgradParams p) {
  using T = WgradWide;
  constexpr int MT = T::MT, NT = T::NT;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int lane = threadIdx.x & 63, c32 = lane & 31, g = lane >> 5, i16 = lane & 15, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / T::WN, wn = wave % T::WN;
  // as in linear_wgrad_kernel: the tiles of one split are neighbours, in bands of six k tiles
  // (a contiguous range of them to each XCD, also where eight do not divide the grid: dealt in turn, every XCD read all of g and x.  M 8192 3456 x 1152,
  // 252 work-groups, 81.5 -> 74 us; M 32768 768 x 768 59.4 -> 54.3, where linear_wgrad_kernel takes 56.8)
  const uint32_t xcd = blockIdx.x % 8, id = xcd * (gridDim.x / 8) + min(xcd, gridDim.x % 8) + blockIdx.x / 8;
  const uint32_t per = (uint32_t)p.ntiles * p.ktiles, split = id / per, tile = id - split * per;
  const uint32_t band = tile / (6 * p.ntiles), in = tile - band * 6 * p.ntiles, wide = min((uint32_t)p.ktiles - 6 * band, 6u);
  const int n0 = (int)(in / wide) * T::BM, k0 = (int)(6 * band + in % wide) * T::BN;
  const int first = (int)split * p.per, steps = min(p.per, (p.M + 63) / 64 - first);   // (at least one: no split is empty)

  const uint32_t gb = (uint32_t)p.N * 2, xb = (uint32_t)p.K * 2;
  const __amdgpu_buffer_rsrc_t rg = make_rows_rsrc(p.g + n0, gb, p.M, (int)(gb - n0 * 2));
  const __amdgpu_buffer_rsrc_t rx = make_rows_rsrc(p.x + k0, xb, p.M, (int)(xb - k0 * 2));
  uint32_t gvoff[T::PX], xvoff[T::PW];   // a wave's j-th KB of a stage: 8 rows of a panel
#pragma unroll
  for (int j = 0; j < T::PX; ++j) {
    const int b = 4 * j + wave;
    const uint32_t row = 8 * (b & 7) + (lane >> 3), col = (b >> 3) * 128 + ((lane & 7) ^ (((lane >> 4) & 1) * 4)) * 16;
    gvoff[j] = row * gb + col;
    if (j < T::PW) xvoff[j] = row * xb + col;
  }
  // steps being requested, and the slots they go to (past the last step: that one again; nothing reads it)
  int sg = 0, sx = 0;
  uint32_t gto = 0, xto = 0;
  auto request_g = [&](int j) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rg, (__attribute__((address_space(3))) void*)(smem + gto * T::XS + (4 * j + wave) * 1024), 16, gvoff[j],
                                             (uint32_t)(first + sg) * 64 * gb, 0, 0);
  };
  auto request_x = [&](int j) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (__attribute__((address_space(3))) void*)(smem + T::NSX * T::XS + xto * T::WS + (4 * j + wave) * 1024), 16,
                                             xvoff[j], (uint32_t)(first + sx) * 64 * xb, 0, 0);
  };
  auto advance_g = [&] { gto = gto + 1 == T::NSX ? 0 : gto + 1; sg = min(sg + 1, steps - 1); };
  auto advance_x = [&] { xto = xto + 1 == T::NSW ? 0 : xto + 1; sx = min(sx + 1, steps - 1); };

  const uint32_t in_panel = (8 * g + (i16 >> 2)) * 128 + ((lane >> 4) & 1) * 32 + (i16 & 3) * 8, swap = (i16 >> 3) & 1;
  const uint32_t gaddr = lds_addr(smem) + in_panel + (wm ^ swap) * 64;   // column group 2 m + wm: half wm of panel m
  uint32_t xaddr[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) xaddr[n] = lds_addr(smem) + T::NSX * T::XS + ((wn * NT + n) >> 1) * 8192 + in_panel + (((wn * NT + n) & 1) ^ swap) * 64;
  TrPair G[2][MT], X[2][NT];
  uint32_t gslot = 0, xslot = 0;   // of the stage being read
  auto read = [&](auto cc, auto ii) {   // operand ii of chunk cc
    constexpr int c = decltype(cc)::value, i = decltype(ii)::value, b = c % 2;
    if constexpr (i < NT) X[b][i] = lds_tr16_issue<c * 2048, c * 2048 + 512>(xaddr[i] + xslot * T::WS);
    else G[b][i - NT] = lds_tr16_issue<(i - NT) * 8192 + c * 2048, (i - NT) * 8192 + c * 2048 + 512>(gaddr + gslot * T::XS);
  };
  auto landed = [&](auto bb) {
    constexpr int b = decltype(bb)::value;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int i = 0; i < NT; ++i) landed_in(X[b][i]);
#pragma unroll
    for (int i = 0; i < MT; ++i) landed_in(G[b][i]);
  };
  f32x16 acc[NT][MT];
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[n][m] = f32x16{0};
  float total[MT] = {};
  auto stage = [&](auto sums_) {   // sums_: 0, 1: of chunks 0 and 1, or 2 and 3; 2: none
    float part[MT] = {};
    for_each(std::make_integer_sequence<int, 4>{}, [&](auto cc) {
      constexpr int c = decltype(cc)::value, NM = MT * NT, R = MT + NT;
      landed(std::integral_constant<int, c % 2>{});
      if constexpr (c == 3) {
        wait_vm<T::BEHIND>();
        asm volatile("s_barrier" ::: "memory");   // the next stage is in LDS and everybody has taken its operands of this one
        gslot = gslot + 1 == T::NSX ? 0 : gslot + 1;
        xslot = xslot + 1 == T::NSW ? 0 : xslot + 1;
      }
      for_each(std::make_integer_sequence<int, NM>{}, [&](auto ii) {
        constexpr int i = decltype(ii)::value, n = i / MT, m = i % MT;
        acc[n][m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_operand(X[c % 2][n]), as_operand(G[c % 2][m]), acc[n][m], 0, 0, 0);
        if constexpr (i < R) read(std::integral_constant<int, (c + 1) % 4>{}, ii);
        if constexpr (c == 3) {
#pragma unroll
          for (int j = i * T::PW / NM; j < (i + 1) * T::PW / NM; ++j) request_x(j);
        } else {
          constexpr int at = c * NM + i;
#pragma unroll
          for (int j = at * T::PX / (3 * NM); j < (at + 1) * T::PX / (3 * NM); ++j) request_g(j);
        }
        if constexpr (decltype(sums_)::value == c / 2 && i >= NM - MT) {
          constexpr int k = i - (NM - MT);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const uint32_t pair = tr_operand(G[c % 2][k]).v[e];
            part[k] += __uint_as_float(pair << 16) + __uint_as_float(pair & 0xffff0000u);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      });
      if constexpr (c == 3) advance_x();
      if constexpr (c == 2) advance_g();
    });
    if constexpr (decltype(sums_)::value < 2) {
#pragma unroll
      for (int m = 0; m < MT; ++m) total[m] += part[m];
    }
  };

#pragma unroll
  for (int s = 0; s < T::NSW; ++s) {
#pragma unroll
    for (int j = 0; j < T::PW; ++j) request_x(j);
    advance_x();
    if (s < T::NSX - 1) {
#pragma unroll
      for (int j = 0; j < T::PX; ++j) request_g(j);
      advance_g();
    }
  }
  wait_vm<(T::NSW - 1) * T::PW + (T::NSX - 2) * T::PX>();
  asm volatile("s_barrier" ::: "memory");
  const bool sums = p.bias != nullptr && k0 == 0;
  auto run = [&](auto sums_) {
    for_each(std::make_integer_sequence<int, MT + NT>{}, [&](auto ii) { read(std::integral_constant<int, 0>{}, ii); });
    for (int s = 0; s < steps; ++s) stage(sums_);
    landed(std::integral_constant<int, 0>{});   // (of a stage past the last: nothing may be under way where control flow meets)
  };
  if (!sums) run(std::integral_constant<int, 2>{});
  else if (wn == 0) run(std::integral_constant<int, 0>{});
  else run(std::integral_constant<int, 1>{});
  wait_vm<0>();   // (no DMA may outlive the work-group's LDS)

  if (sums) {   // of both waves, and of the halves of a wave, which hold different rows
    asm volatile("s_barrier" ::: "memory");
    float* both = reinterpret_cast<float*>(smem) + wm * MT * 64;
#pragma unroll
    for (int m = 0; m < MT; ++m)
      if (wn == 1) both[m * 64 + lane] = total[m];
    __syncthreads();
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int row = n0 + 64 * m + 32 * wm + c32;
      float t = total[m] + both[m * 64 + lane];
      t += __shfl_xor(t, 32);
      if (wn == 0 && g == 0 && row < p.N) p.bias[(int64_t)split * p.N + row] = t;
    }
  }
  __syncthreads();
  float* out = p.out + (int64_t)split * p.N * p.K;
#pragma unroll
  for (int m = 0; m < MT; ++m) {
#pragma unroll
    for (int n = 0; n < NT; ++n) store_sums(smem + wave * 8192 + ((m * NT + n) & 1) * 4096, acc[n][m], out, n0 + 64 * m + 32 * wm, k0 + 96 * wn + 32 * n, p.N, p.K, lane);
  }
}

// out = the sum of `splits` arrays of 4 n4 floats, in order; behind them, arrays of 4 b4 floats into bias
struct SumSplitsParams { const f32x4* part; f32x4 *out, *bias; int64_t n4, b4; int splits; };
__global__ __launch_bounds__(256) void sum_splits_kernel(const SumSplitsParams p) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= p.n4 + p.b4) return;
  const bool weight = i < p.n4;
  const int64_t stride = weight ? p.n4 : p.b4;
  const f32x4* part = weight ? p.part + i : p.part + p.splits * p.n4 + (i - p.n4);
  f32x4 s = part[0];
  for (int j = 1; j < p.splits; j += 4) {
    f32x4 v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = j + k < p.splits ? part[(j + k) * stride] : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < 4; ++k) s += v[k];
  }
  if (weight) p.out[i] = s;
  else p.bias[i - p.n4] = s;
}

// Splits of the rows: the least of the estimated times, a step and a work-group's start and end fitted to M = 8192 .. 32768, plus the
// partial sums' way through memory (written once, read once, at some 5 TB/s) and a launch.
static int wgrad_splits(int64_t M, int64_t N, int64_t K) {
  const int64_t cus = compute_units(), tiles = ((N + kWgN - 1) / kWgN) * ((K + kWgK - 1) / kWgK), total = (M + 63) / 64;
  int best = 1;
  int64_t cost_best = INT64_MAX;
  for (int s = 1; s <= 64 && s <= total; ++s) {
    const int64_t per = (total + s - 1) / s, wgs = tiles * s, rounds = wgs / (2 * cus), rest = wgs % (2 * cus);
    const int64_t one = 95 * per + 350, two = 125 * per + 450;   // one, two work-groups on a CU, in 10 ns
    int64_t cost = rounds * two + (rest == 0 ? 0 : rest <= cus ? one : one + (two - one) * (35 * cus + 65 * (rest - cus)) / (100 * cus));
    if (s > 1) cost += N * K * 4 * (2 * s + 1) / 50000 + 300;
    if (cost < cost_best) {
      cost_best = cost;
      best = s;
    }
  }
  return best;
}

// Splits for linear_wgrad_wide_kernel, 0 where linear_wgrad_kernel is the better one: below 8 G multiply-adds (profiles/linear_train_products.txt, with column
// sums, there against here: 768 x 768 M 12288 31.4 against 29.9 us, M 16384 36.7 -> 34.7; 1152 x 1152 M 6144 35.1 -> 32.9; 2304 x 768 M 5120 33.3 -> 34.8, M 6144 36.5 ->
// 37.0, M 8192 44.3 -> 43.9; the kernel taken is 0.5 % slower than the faster in the mean).  Estimates fitted to 160 such products, in 10 ns; all work-groups at
// once; chains of sums no longer than that kernel's.
static int wgrad_wide_splits(int64_t M, int64_t N, int64_t K) {
  if (M * N < 8000000000 / K) return 0;
  const int64_t cus = compute_units(), tiles = ((N + WgradWide::BM - 1) / WgradWide::BM) * ((K + WgradWide::BN - 1) / WgradWide::BN), total = (M + 63) / 64;
  int best = 0;
  int64_t cost_best = INT64_MAX;
  for (int64_t s = wgrad_splits(M, N, K); s <= 64 && s <= total && tiles * s <= cus; ++s) {
    const int64_t per = (total + s - 1) / s;
    if ((s - 1) * per >= total) continue;   // (a split would be empty)
    int64_t cost = per * (77 * cus + 46 * tiles * s) / cus + 173 * tiles * s / cus;
    if (s > 1) cost += N * K * 4 * (2 * s + 1) / 152000 + 396;
    if (cost < cost_best) {
      cost_best = cost;
      best = (int)s;
    }
  }
  return best;
}

static bool wgrad_shape_ok(int64_t M, int64_t N, int64_t K) {
  if (M < 1 || N < 8 || N % 8 || K < 8 || K % 8 || M * K >= (int64_t)1 << 30 || N * K >= (int64_t)1 << 30 || M * N >= (int64_t)1 << 30) return false;
  // rows up to the end of the last step are addressed too, in 32 bits: wrapped around, one past the last would be read, not be zero
  return (M + 63) / 64 * 64 * std::max(N, K) < (int64_t)1 << 31;
}

}  // namespace dmf

extern "C" int64_t dmf_linear_wgrad_workspace_floats(int64_t M, int N, int K) {
  if (M > INT32_MAX || !dmf::wgrad_shape_ok(M, N, K)) return -1;
  const int wide = dmf::wgrad_wide_splits(M, N, K), s = wide ? wide : dmf::wgrad_splits(M, N, K);
  return s > 1 ? (int64_t)s * N * (K + 1) : 0;
}

// Which weight gradients without column sums these kernels are the faster ones for (us, library -> here, of profiles/linear_train_products.txt; the library's
// launch alone takes 20 us of host time): those of layers without a bias, which the models do not have.
//   up to M 1472 on every result of the models with a column sum beside the library's (next rule); without one the GPU alone takes 5 to 30 % more here
//   for 768 x 768 and smaller (M 512 8.7 against 10.6, M 1000 13.8 against 14.7), which the host's share outweighs, and less for large results
//   (4608 x 1152 M 512 17.1 -> 13.3, M 1000 28.4 -> 19.6);
//   M 2048: 1152 x 1152 21 against 23, 2304 x 768 20.5 against 22.9, 3456 x 1152 28 against 34;
//   M 4096: 3072 x 768 43 -> 34, 1152 x 1152 34 -> 25, 3072 x 1024 43 -> 42, 4608 x 1152 60 -> 53, but 3456 x 1152 45 against 46, 4096 x 1024 45 against 47;
//   M 6144: 3456 x 1152 63 -> 57, 4608 x 1152 86 -> 69, 4096 x 1024 64 -> 62, 1024 x 4096 64 -> 60;
//   M 8192: 3456 x 1152 83 -> 69, 4608 x 1152 112 -> 85, 4096 x 1024 84 -> 76, 1152 x 1152 61 -> 36, 768 x 768 49 -> 23;  M 16384: 3072 x 768 147 ->
//   82, 4608 x 1152 320 -> 158 (1100 TFLOP/s).  The largest result measured is 6912 x 1152 (8 M elements); beyond it the library's products are kept.
extern "C" int dmf_linear_wgrad_plan(int64_t M, int N, int K) {
  if (M > INT32_MAX || !dmf::wgrad_shape_ok(M, N, K)) return 0;
  const int64_t result = (int64_t)N * K;
  if (result > 8000000) return 0;
  if (M < 1536) return 1;
  if (M < 4096) return result <= 600000;
  return M >= 6144 || result <= 3200000 || (result >= 5000000 && K % dmf::kWgK == 0);
}

// ... and with the column sums, where the library's product has a column sum beside it (two launches, 8 to 11 us): on every result of the models, 0.62 of the
// library's time in the mean of 320 (us, library and column sum -> here): M 1: 768 x 768 9.3 -> 5.7;  M 256: 4608 x 768 19.8 -> 10.3, 6912 x 1152 24.1 -> 13.4;  M 512:
// 768 x 768 15.6 -> 12.3;  M 1536: 2304 x 768 27.2 -> 23.3, 3072 x 1024 31.5 -> 29.0;  M 2048: 3072 x 768 36.0 -> 28.4, 3072 x 1024 36.4 -> 36.3, 1152 x 1152 31.3 ->
// 23.4, 4608 x 1152 45.3 -> 38.4;  M 4096: 3456 x 1152 54.8 -> 47.6, 4096 x 1024 56.3 -> 51.6;  M 5120: 3456 x 1152 64.5 -> 53.7, 1024 x 4096 63.7 -> 57.8.
extern "C" int dmf_linear_wgrad_sums_plan(int64_t M, int N, int K) { return M <= INT32_MAX && dmf::wgrad_shape_ok(M, N, K) && (int64_t)N * K <= 8000000; }

extern "C" int dmf_linear_train_plan(int which, int64_t M, int N, int K, char* buf, int buflen) {
  const bool ok = which == 0 ? M <= INT32_MAX && dmf_linear_gelu_plan(M, N, K) : which == 1 ? dgrad_shape_ok(M, N, K) : which == 2 && M <= INT32_MAX && dmf::wgrad_shape_ok(M, N, K);
  if (!ok) return DMF_ATTN_ESHAPE;
  if (buf == nullptr || buflen < 1) return DMF_ATTN_ENULL;
  if (which == 2) {
    const int wide = dmf::wgrad_wide_splits(M, N, K);
    snprintf(buf, (size_t)buflen, "dmf::linear_wgrad_%skernel, %d splits", wide ? "wide_" : "", wide ? wide : dmf::wgrad_splits(M, N, K));
    return DMF_ATTN_OK;
  }
  const char* tile[7] = {"", "", "", "4, 3, 2, 3, 2", "4, 2, 2, 3, 3", "", "4, 4, 2, 3, 2"};
  snprintf(buf, (size_t)buflen, "dmf::linear_%s_kernel<dmf::WalkTile<%s> >", which ? "dgrad" : "walk_pre", tile[which ? dgrad_tile(M, N, K) : dmf::linear_tile(M, N, K, true, true)]);
  return DMF_ATTN_OK;
}

extern "C" int dmf_linear_wgrad(const void* g, const void* x, float* gw, float* gbias, float* workspace, int M, int N, int K, void* stream) {
  if (g == nullptr || x == nullptr || gw == nullptr) return DMF_ATTN_ENULL;
  if (!dmf::wgrad_shape_ok(M, N, K)) return DMF_ATTN_ESHAPE;
  const int wide = dmf::wgrad_wide_splits(M, N, K), splits = wide ? wide : dmf::wgrad_splits(M, N, K);
  if (splits > 1 && workspace == nullptr) return DMF_ATTN_ENULL;
  for (const void* q : {g, x, (const void*)gw, (const void*)gbias, (const void*)workspace})
    if (reinterpret_cast<uintptr_t>(q) % 16) return DMF_ATTN_EALIGN;
  dmf::WgradParams p{};
  p.g = static_cast<const __bf16*>(g);
  p.x = static_cast<const __bf16*>(x);
  p.out = splits > 1 ? workspace : gw;
  p.bias = gbias == nullptr ? nullptr : splits > 1 ? workspace + (int64_t)splits * N * K : gbias;
  p.M = M; p.N = N; p.K = K;
  const int columns = wide ? dmf::WgradWide::BM : dmf::kWgN;
  p.ntiles = (N + columns - 1) / columns;
  p.ktiles = (K + dmf::kWgK - 1) / dmf::kWgK;
  p.splits = splits;
  p.per = ((M + 63) / 64 + splits - 1) / splits;
  static bool lds_ok[64] = {}, lds_ok_wide[64] = {};
  if (!(wide ? dmf::ensure_dynamic_lds(dmf::linear_wgrad_wide_kernel, dmf::WgradWide::STAGES, lds_ok_wide)
             : dmf::ensure_dynamic_lds(dmf::linear_wgrad_kernel, 2 * dmf::kWgStage, lds_ok)))
    return -7;
  auto stm = static_cast<hipStream_t>(stream);
  const dim3 grid((uint32_t)p.ntiles * p.ktiles * splits);
  const int rc = wide ? dmf::launch_kernel(dmf::linear_wgrad_wide_kernel, grid, dim3(256), dmf::WgradWide::STAGES, stm, p)
                      : dmf::launch_kernel(dmf::linear_wgrad_kernel, grid, dim3(256), 2 * dmf::kWgStage, stm, p);
  if (rc != 0 || splits == 1) return rc;
  const int64_t n4 = (int64_t)N * K / 4, b4 = gbias == nullptr ? 0 : N / 4;
  const dmf::SumSplitsParams q{reinterpret_cast<const f32x4*>(workspace), reinterpret_cast<f32x4*>(gw), reinterpret_cast<f32x4*>(gbias), n4, b4, splits};
  return dmf::launch_kernel(dmf::sum_splits_kernel, dim3((uint32_t)((n4 + b4 + 255) / 256)), dim3(256), 0, stm, q);
}
