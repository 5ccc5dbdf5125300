// Projections of few tokens (decode steps) on gfx950 matrix cores: y = x . w^T and the gated
// gate/up form of gemm.hip, for at most kSkinnyTokens rows of x; and f32 projections of any
// number of tokens, with true f32 products (v_mfma_f32_16x16x4).
//
// Bound by reading the weight once.  gemm.hip's 256 x 256 tiles leave most of the device idle
// here (4096 x 14336: 16 workgroups, each walking all of K: 293 us at 32 tokens); this kernel
// gives every 16 to 64 weight rows a workgroup whose 8 waves split K:
//   * wave w takes the 64-wide slices w, w + 8, ...: together the waves read 1 KB runs of each
//     weight row, and no wave waits for another before the end;
//   * a slice goes global -> LDS in loads of 8 rows x 128 bytes and from there into fragments.
//     Loading fragments straight from memory (16 rows at a 16-byte column per quarter wave)
//     was 1.3 to 1.9 times slower: 64 line lookups for a load's 1 KB instead of 8;
//   * each wave refills its own ring and waits on its own loads, so the loop has no barrier;
//     two workgroups share a compute unit where the ring allows it;
//   * the waves' f32 sums are added in LDS, wave 0 first: the order of a sum depends on K alone.
// Measured (MI355X, us a call, distinct weights each call; before: the tile kernel): gated
// 2 x 14336 x 4096 at 32 tokens 98 -> 48 (4.9 TB/s), 4096 x 14336 293 -> 29; at 1 token 44 and
// 23 (5.3 TB/s); 2048 x 2048 at 1 token 37 -> 5.
#include <algorithm>

#include "cea_lds_dma.hpp"
#include "gemm_common.hpp"

namespace cea {
namespace {

constexpr int S_WAVES = 8;
constexpr int S_THREADS = S_WAVES * 64;
constexpr int S_ROW = 128;   // bytes of a slice row: a cache line (64 of K in 16 bits, 32 in f32)

// RB: 16-row weight blocks of a workgroup (gated: RB / 2 of the gate and the matching RB / 2 of
// the up rows), TB: 16-token blocks of x.
template <int RB, int TB> struct SkinnyLds {
  static constexpr int SLICE = (RB + TB) * 16 * S_ROW;   // bytes of one wave's slice
  static constexpr int PD = 2 * S_WAVES * SLICE <= 80 * 1024 ? 2 : 1;   // ring stages
  static constexpr int RING = S_WAVES * PD * SLICE;
  static constexpr int RED = S_WAVES * RB * TB * 1024;
  static constexpr int BYTES = RING > RED ? RING : RED;
};

template <typename T, int MODE, int ACT, int RB, int TB>
__global__ __launch_bounds__(S_THREADS, 2) void gemm_skinny_kernel(const GemmParams p) {
  typedef typename GMfma<T>::frag frag;
  typedef SkinnyLds<RB, TB> L;
  constexpr int ESZ = sizeof(T);
  constexpr int BK = S_ROW / ESZ;   // K per slice
  constexpr int NB = MODE == kGated ? RB / 2 : RB;   // output column blocks
  constexpr int PD = L::PD;
  extern __shared__ __attribute__((aligned(16))) char smem[];

  const int wave = uniform(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int n0 = blockIdx.x * NB * 16;
  const int K = p.K;
  const int KT = (K + BK - 1) / BK;
  const int rows = min(NB * 16, p.N - n0);
  const int m0 = blockIdx.y * TB * 16;
  const int toks = min(TB * 16, p.M - m0);

  const i32x4 rx = make_rsrc((const char*)p.x + (int64_t)m0 * p.ldx * ESZ,
                             (uint32_t)((int64_t)(toks - 1) * p.ldx * ESZ + (int64_t)K * ESZ));
  const uint32_t wbytes = (uint32_t)((int64_t)(rows - 1) * p.ldw * ESZ + (int64_t)K * ESZ);
  const i32x4 rg = make_rsrc((const char*)p.wg + (int64_t)n0 * p.ldw * ESZ, wbytes);
  const i32x4 ru = MODE == kGated ? make_rsrc((const char*)p.wu + (int64_t)n0 * p.ldw * ESZ, wbytes) : rg;

  // one load: 8 rows x 128 bytes, lane l the 16-byte group (l & 7) ^ swizzle of row l >> 3
  int kcol[2];
  uint32_t off_w[2], off_x[2];   // rows 0-7 and 8-15 of a block
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = 8 * i + (lane >> 3);
    const int grp = (lane & 7) ^ g_swz(row);
    kcol[i] = grp * (16 / ESZ);
    off_w[i] = (uint32_t)((int64_t)row * p.ldw * ESZ) + grp * 16;
    off_x[i] = (uint32_t)((int64_t)row * p.ldx * ESZ) + grp * 16;
  }
  const uint32_t blk_w = (uint32_t)(16 * p.ldw * ESZ), blk_x = (uint32_t)(16 * p.ldx * ESZ);
  char* ring = smem + wave * (PD * L::SLICE);
  const uint32_t ring_lds = lds_addr(ring);
  auto load = [&](int d, int s) {   // slice s into ring stage d
    const uint32_t kb = (uint32_t)s * S_ROW;
    const uint32_t base = ring_lds + (uint32_t)d * L::SLICE;
    const bool kin[2] = {s * BK + kcol[0] < K, s * BK + kcol[1] < K};
#pragma unroll
    for (int f = 0; f < RB; ++f)
#pragma unroll
      for (int i = 0; i < 2; ++i)
        buffer_load_lds16_m0_so(f < NB ? rg : ru, base + (2 * f + i) * 1024,
                                kin[i] ? off_w[i] + (f % NB) * blk_w : kOutOfRange, kb);
#pragma unroll
    for (int t = 0; t < TB; ++t)
#pragma unroll
      for (int i = 0; i < 2; ++i)
        buffer_load_lds16_m0_so(rx, base + (2 * (RB + t) + i) * 1024,
                                kin[i] ? off_x[i] + t * blk_x : kOutOfRange, kb);
  };

  f32x4 acc[RB][TB];
#pragma unroll
  for (int f = 0; f < RB; ++f)
#pragma unroll
    for (int t = 0; t < TB; ++t) acc[f][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  uint32_t rd[2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
    rd[h] = (lane & 15) * S_ROW + (((4 * h + (lane >> 4)) ^ g_swz(lane & 15)) << 4);

#pragma unroll
  for (int d = 0; d < PD; ++d) load(d, wave + d * S_WAVES);
  for (int s0 = wave; s0 < KT; s0 += PD * S_WAVES) {
#pragma unroll
    for (int d = 0; d < PD; ++d) {
      wait_vmcnt<(PD - 1) * 2 * (RB + TB)>();
      frag a[2][RB], b[2][TB];
      const char* st = ring + d * L::SLICE;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int f = 0; f < RB; ++f) a[h][f] = *(const frag*)(st + f * 16 * S_ROW + rd[h]);
#pragma unroll
        for (int t = 0; t < TB; ++t) b[h][t] = *(const frag*)(st + (RB + t) * 16 * S_ROW + rd[h]);
      }
      wait_lgkmcnt0();   // the stage is read: refill it
      __builtin_amdgcn_sched_barrier(0);
      load(d, s0 + (d + PD) * S_WAVES);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int f = 0; f < RB; ++f)
#pragma unroll
          for (int t = 0; t < TB; ++t) acc[f][t] = GMfma<T>::run(a[h][f], b[h][t], acc[f][t]);
    }
  }
  wait_vmcnt<0>();   // no load into the ring is left when the sums take its place
  __syncthreads();
  f32x4 (*red)[RB * TB][64] = (f32x4 (*)[RB * TB][64])smem;

  // the waves' sums, wave 0 first, then the epilogue of 4 consecutive features of one token
#pragma unroll
  for (int f = 0; f < RB; ++f)
#pragma unroll
    for (int t = 0; t < TB; ++t) red[wave][f * TB + t][lane] = acc[f][t];
  __syncthreads();
  const bool vec = p.vec_out != 0;
  for (int i = wave; i < NB * TB; i += S_WAVES) {
    const int f = i / TB, t = i % TB;
    f32x4 g = red[0][i][lane], u = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 1; w < S_WAVES; ++w) g += red[w][i][lane];
    if constexpr (MODE == kGated) {
      u = red[0][NB * TB + i][lane];
#pragma unroll
      for (int w = 1; w < S_WAVES; ++w) u += red[w][NB * TB + i][lane];
    }
    const int tok = m0 + t * 16 + (lane & 15);
    const int col = n0 + f * 16 + 4 * (lane >> 4);
    if (tok >= p.M || col >= p.N) continue;
    float gv[4], uv[4], bgv[4], buv[4] = {0.0f, 0.0f, 0.0f, 0.0f}, v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) gv[j] = g[j], uv[j] = u[j];
    bias4<T, float>(p.bg, col, p.N, vec, bgv);
    if constexpr (MODE == kGated) bias4<T, float>(p.bu, col, p.N, vec, buv);
    finish4<T, MODE, ACT, true, float>(gv, uv, bgv, buv, v);
    store4<T, float>((T*)p.y + (int64_t)tok * p.ldy, col, p.N, vec, v);
  }
}

template <typename T, int MODE, int ACT, int RB, int TB>
int launch_shape(const GemmParams& p, hipStream_t st) {
  constexpr int NB = MODE == kGated ? RB / 2 : RB;
  constexpr int lds = SkinnyLds<RB, TB>::BYTES;
  const hipError_t e = reserve_lds<gemm_skinny_kernel<T, MODE, ACT, RB, TB>>(lds);
  CEA_REQUIRE(e == hipSuccess, CEA_ELAUNCH, "linear: cannot reserve %d bytes of LDS: %s", lds,
              hipGetErrorString(e));
  hipLaunchKernelGGL((gemm_skinny_kernel<T, MODE, ACT, RB, TB>), dim3(ceil_div(p.N, NB * 16), ceil_div(p.M, TB * 16)),
                     dim3(S_THREADS), lds, st, p);
  CEA_CHECK_LAUNCH(MODE == kGated ? "linear_gated" : "linear");
  return CEA_OK;
}

// Weight blocks per workgroup: the count with the least bytes through the busiest compute unit,
// rounds of workgroups times (RB weight blocks + M / 16 token blocks), since every workgroup
// reads all of x and a unit takes in at most about 57 B/ns however the loads are arranged (over
// whole launches at 32 tokens, by the L2's read requests, 43 for 4096 x 14336, of which two thirds
// are x, and 29 for gated 2 x 14336 x 4096, whose 448 workgroups run in 1.75 rounds).  Measured
// (us, RB 1 / 2 / 4): 4096 x 14336, 32 tokens 28.7 / 35.7 / 50.6; 6144 x 4096, 16 tokens 15.6 /
// 13.1 / 16.0; gated 2 x 4864 x 896, 20 tokens - / 10.3 / 7.3.
template <int MODE> int weight_blocks(const GemmParams& p) {
  const int cus = std::max(device_cus(), 1);
  int best = 1;
  double least = 0;
  for (int rb = MODE == kGated ? 2 : 1; rb <= 4; rb *= 2) {
    const int wgs = ceil_div(p.N, (MODE == kGated ? rb / 2 : rb) * 16);
    const double cost = (double)ceil_div(wgs, cus) * (rb + p.M / 16.0);
    if (least == 0 || cost < least) best = rb, least = cost;
  }
  return best;
}

template <typename T, int MODE, int ACT, int RB>
int launch_tokens(const GemmParams& p, int tb, hipStream_t st) {
  switch (tb) {
    case 1: return launch_shape<T, MODE, ACT, RB, 1>(p, st);
    case 2: return launch_shape<T, MODE, ACT, RB, 2>(p, st);
    case 3: return launch_shape<T, MODE, ACT, RB, 3>(p, st);
    default: return launch_shape<T, MODE, ACT, RB, 4>(p, st);
  }
}

// f32: weight and token blocks per workgroup.  A compute unit needs about 36 ns per block pair
// and slice for the matrix instructions and 36 ns per block for its 2 KB; a round of workgroups
// costs about 2 us more for its first loads and its sums.  Measured (us, generic kernel before ->
// this rule; RB x TB 2 x 2 / 2 x 3 / 4 x 4): 512 tokens 1536 x 512 73 -> 14.8 (13.5 / 17.6 /
// 14.8), 512 x 512 71 -> 6.0 (6.0 / 7.2 / 13.2), 2400 tokens 6144 x 2048 1293 -> 519 (521 / 497 /
// 519; 116 of 157 TFLOP/s).
template <int MODE> void blocks_f32(const GemmParams& p, int& rb, int& tb) {
  const int cus = std::max(device_cus(), 1);
  const double slices = ceil_div(p.K, S_ROW / 4);
  double least = 0;
  for (int r = MODE == kGated ? 2 : 1; r <= 4; r *= 2)
    for (int t = 1; t <= 4; ++t) {
      const int64_t wgs = (int64_t)ceil_div(p.N, (MODE == kGated ? r / 2 : r) * 16) * ceil_div(p.M, t * 16);
      const double us = (double)((wgs + cus - 1) / cus) *
                        (2.0 + slices * 0.036 * std::max(r * t, r + t));
      if (least == 0 || us < least) rb = r, tb = t, least = us;
    }
}

template <int MODE, int ACT>
int launch_f32(const GemmParams& p, hipStream_t st) {
  int rb = 4, tb = 4;
  blocks_f32<MODE>(p, rb, tb);
  if (ceil_div(p.M, tb * 16) > 65535) tb = 4;   // the second grid dimension
  CEA_REQUIRE(ceil_div(p.M, tb * 16) <= 65535, CEA_EUNSUPPORTED, "linear: %d rows exceed the f32 kernel's grid",
              p.M);
  if constexpr (MODE == kPlain)
    if (rb == 1) return launch_tokens<float, MODE, ACT, 1>(p, tb, st);
  if (rb == 2) return launch_tokens<float, MODE, ACT, 2>(p, tb, st);
  return launch_tokens<float, MODE, ACT, 4>(p, tb, st);
}

template <typename T, int MODE, int ACT>
int launch_act(const GemmParams& p, hipStream_t st) {
  if constexpr (sizeof(T) == 4) return launch_f32<MODE, ACT>(p, st);
  const int rb = weight_blocks<MODE>(p), tb = ceil_div(p.M, 16);
  if constexpr (MODE == kPlain)
    if (rb == 1) return launch_tokens<T, MODE, ACT, 1>(p, tb, st);
  if (rb == 2) return launch_tokens<T, MODE, ACT, 2>(p, tb, st);
  return launch_tokens<T, MODE, ACT, 4>(p, tb, st);
}

template <typename T>
int launch_typed(const GemmParams& p, int mode, int act, hipStream_t st) {
  if (mode == kPlain) return launch_act<T, kPlain, 0>(p, st);
  switch (act) {
    case CEA_ACT_SILU: return launch_act<T, kGated, CEA_ACT_SILU>(p, st);
    case CEA_ACT_GELU: return launch_act<T, kGated, CEA_ACT_GELU>(p, st);
    case CEA_ACT_GELU_TANH: return launch_act<T, kGated, CEA_ACT_GELU_TANH>(p, st);
    case CEA_ACT_RELU: return launch_act<T, kGated, CEA_ACT_RELU>(p, st);
  }
  set_error("linear_gated: unknown activation %d", act);
  return CEA_EUNSUPPORTED;
}

}  // namespace

int launch_linear_skinny(const GemmParams& p, int dtype, int mode, int act, hipStream_t st) {
  switch (dtype) {
    case CEA_BF16: return launch_typed<bf16>(p, mode, act, st);
    case CEA_F16: return launch_typed<f16>(p, mode, act, st);
    default: return launch_typed<float>(p, mode, act, st);
  }
}

}  // namespace cea
