// y = x W^T + b and, with tangents, ty = tx W^T: the linear layers' forward, bf16 with fp32 accumulation.  With GELU (tanh form) the
// activation is applied in the epilogue, to the primal and, through its derivative, to the tangent, so that neither pre-activation
// travels to HBM and back.
//
// The library ran the two products of a layer one after the other (two partly empty last rounds), in tiles that fit these widths
// badly, and spent 18 us of host time on each.  Here both are one grid; 192 columns divide every layer width of the models, so the
// 128 x 192 tile fills whole rounds.
#include <type_traits>
#include "attn_common.h"
#include "attn_kernels.h"
#include "../../include/dmf_fused.h"

namespace dmf {

struct LinearParams {
  const __bf16 *x[2], *w, *bias;   // x[1]: the tangent's rows (second half of the grid), no bias
  __bf16* y[2];
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
enum LinMode { kLinPlain, kLinGelu, kLinGeluJvp };

// sigma = 1 / (1 + exp(-2 u)), u = sqrt(2 / pi) (v + 0.044715 v^3): gelu(v) = 0.5 v (1 + tanh u) = v sigma
__device__ __forceinline__ float gelu_sigma(float v) {
  const float u2 = 1.5957691216057308f * v * fmaf(0.044715f, v * v, 1.f);
  return __builtin_amdgcn_rcpf(1.f + fast_exp2(-kLog2e * u2));
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
            else v[e] *= sg * fmaf(x * (1.f - sg), 1.5957691216057308f * fmaf(3.f * 0.044715f, x * x, 1.f), 1.f);
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

// Tile policy: the shortest of four estimates, a K step (64) and a work-group's start and end taking `a` and `b` (in 10 ns) with one, two,
// three work-groups on a CU -- fitted to K = 384 .. 4608 on MI355X (us: 128 x 192, 768 columns, 48 steps: 43.6 for 128 work-groups, 47 for 256,
// 68.4 for 512; 12 steps, 1536 work-groups: 63.9):
struct LinTile { int bm, bn, per_cu, a[3], b[3]; };
constexpr LinTile kLinTiles[4] = {
    {128, 192, 2, {90, 140, 0}, {350, 450, 0}}, {128, 128, 2, {77, 95, 0}, {120, 400, 0}},
    {128, 64, 3, {61, 63, 93}, {60, 200, 250}}, {64, 64, 2, {20, 36, 0}, {320, 320, 0}}};

static int linear_tile(int64_t M, int N, int K, bool jvp) {
  const int64_t cus = compute_units(), steps = K / kLinK;
  int best = 0;
  int64_t cost_best = INT64_MAX;
  for (int t = 0; t < 4; ++t) {
    const LinTile& c = kLinTiles[t];
    const int64_t wgs = ((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn) * (jvp ? 2 : 1), slots = cus * c.per_cu, rest = wgs % slots;
    auto full = [&](int64_t occ) { return c.a[occ] * steps + c.b[occ]; };
    auto round = [&](int64_t n) {   // some CUs with one work-group more than the others: the step up, and the rest by their share
      const int64_t o = (n + cus - 1) / cus - 1, over = n - o * cus;
      return o == 0 || over == cus ? full(o) : full(o - 1) + (full(o) - full(o - 1)) * (35 * cus + 65 * over) / (100 * cus);
    };
    const int64_t cost = wgs / slots * round(slots) + (rest ? round(rest) : 0);
    if (cost < cost_best) {
      cost_best = cost;
      best = t;
    }
  }
  return best;
}

template <int MODE>
static int launch_linear_tile(int tile, LinearParams& p, bool jvp, hipStream_t stream) {
  switch (tile) {
    case 0: return launch_linear<128, 192, 2, MODE>(p, jvp, stream);
    case 1: return launch_linear<128, 128, 2, MODE>(p, jvp, stream);
    case 2: return launch_linear<128, 64, 2, MODE>(p, jvp, stream);
    default: return launch_linear<64, 64, 4, MODE>(p, jvp, stream);
  }
}

}  // namespace dmf

// Which calls this kernel is the faster one for (us, library -> here; C: model width, M rows):
//   pairs: C768 M16384 N 3C 133 -> 120, N C 48 -> 43, K 4C 130 -> 130; C1152 M8192 158 -> 124, 64 -> 47, N 4C 171 -> 161, K 4C 166 -> 160;
//     M4096 82 -> 69, 40 -> 26, 114 -> 82, 94 -> 80;
//   single: C768 M2048 N 3C 16.4 -> 13.1, M4096 N 3C 19.9 -> 20.5, N C 12.0 -> 9.4, gelu N 4C 29.5 -> 26.0; C1152 M8192 N 3C 79 -> 70;
//   the library keeps single products with few columns for their depth (K 4C: M4096 C768 26.9 against 31.3, C1152 48 against 56), pairs
//   that spread a short K over a large result (N 4C M16384: C768 141 against 155, C1152 296 against 317; C768 with gelu 86 against 90)
//   and outputs narrower than a tile.
extern "C" int dmf_linear_plan(int64_t M, int N, int K, int jvp, int gelu) {
  if (M < 1 || N < 64 || N % 8 || K < 64 || K % 64 || M * K > (int64_t)1 << 30 || (int64_t)N * K > (int64_t)1 << 30 || M * N > (int64_t)1 << 30) return 0;
  if (jvp && gelu) return 1;
  if (!jvp && K >= 2 * N) return 0;
  if (M * N > 40000000 && N > 3 * K && (jvp || K < 1024)) return 0;
  return 1;
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
  if (jvp && gelu) return dmf::launch_linear<128, 192, 2, dmf::kLinGeluJvp>(p, true, stm);
  const int tile = dmf::linear_tile(M, N, K, jvp);
  return gelu ? dmf::launch_linear_tile<dmf::kLinGelu>(tile, p, false, stm) : dmf::launch_linear_tile<dmf::kLinPlain>(tile, p, jvp, stm);
}
