// Column-parallel projection GEMMs on gfx950 matrix cores.
//
//   plain  y[M, N] = x[M, K] . w[N, K]^T (+ bias[N]), f32 accumulation rounded once to the
//          input dtype: F.linear(x, self.weight, self.bias) of FusedColumnParallelLinear
//          (collab_infer/parallel/tensor_parallel.py:294-295); the per-projection outputs of
//          .split(local_sizes, dim=-1) are column views of y.
//   gated  the gated MLP's gate/up projection and activation in one pass
//          (collab_infer/models/llama.py:298-305, and its replicated-token branch :309-316):
//          gate = T(x . w_g^T + b_g), up = T(x . w_u^T + b_u), y = T(T(act(gate)) * up), with
//          w_g / w_u any two row ranges of one weight (the fused [gate; up] parameter); the
//          [M, 2I] gate/up intermediate never reaches memory.
//
// Matrix-core kernel (bf16 / f16, 16-byte aligned rows, K a multiple of 8):
//   * one workgroup = 8 waves, two per SIMD (256 registers each), computes 256 tokens (160 or
//     128 where those pad or quantise less: plan_tiles) x 256 weight rows; each wave owns 128
//     tokens x 64 weight rows, 32 accumulators of v_mfma_f32_16x16x32 (128 registers); with
//     two waves per SIMD one wave's stalls (load issue, barrier, the activation epilogue's
//     transcendental latencies) leave the matrix core to the other;
//   * the MFMA's A operand is the weight (16 rows) and B the tokens (16 columns), so the 4
//     accumulator values of a lane are 4 consecutive output features of one token;
//   * 64-wide K slices of both operands go global -> LDS directly (buffer_load ... lds) into
//     two stages (three for the lower tiles); a slice row is one 128-byte cache line, so each
//     load instruction touches 8 lines (the address unit's cost is per line touched); rows are
//     XOR-swizzled in 16-byte groups so that the fragment reads (ds_read_b128) hit distinct
//     banks;
//   * one barrier per slice, between its two 32-wide steps; a step's 32 matrix instructions
//     run token-block major and each carries a share of the rest: every token fragment is
//     reloaded for the next step right after its last use (so only one token set is held),
//     the next weight fragments go into a second set, and in the second step the 8 loads
//     refilling the buffer just freed go out one per 4 instructions, so neither the LDS nor
//     the address unit sees a burst;
//   * rows past M / N and columns past K read as zero through the buffer resources' range
//     check, so ragged tiles take no branches in the loop; slices past K load as zeros, so the
//     loop runs uniformly;
//   * the output block goes through LDS and leaves as whole 16-byte row chunks, so each
//     cache line of y is written by one store instruction;
//   * tiles too few to fill the device split K: each workgroup writes its f32 sums in lane order
//     and gemm_reduce_kernel adds them, split 0 first, and runs the epilogue;
//   * at most kSkinnyTokens tokens, and f32 operands, go to gemm_skinny.hip;
//   * workgroups are dealt to the 8 XCDs round robin; tiles are renumbered so that each XCD
//     works through a compact group of tiles that share operand rows in its L2.
// Generic kernel (any dtype, stride or alignment): LDS-tiled FMA loop with f32 accumulation
// (f64 for f64 tensors).
#include <algorithm>
#include <type_traits>

#include "cea_lds_dma.hpp"
#include "gemm_common.hpp"

namespace cea {
namespace {

constexpr int G_THREADS = 512;                       // 8 waves, two per SIMD
constexpr int G_BW = 256;                            // weight rows per tile
constexpr int G_BK = 64;                             // K per LDS slice
constexpr int G_ROW = G_BK * 2;                      // bytes of one row of a slice: a cache line
constexpr int G_WBYTES = G_BW * G_ROW;               // weight part of a stage
constexpr int G_WLOADS = G_WBYTES / (G_THREADS * 16);  // weight loads per wave and slice
constexpr int kLgkm0 = 0xC07F;   // s_waitcnt lgkmcnt(0), vmcnt / expcnt left at their maximum

// TB: 16-token blocks per wave; a tile holds 2 waves of them.
template <int TB> struct Tile {
  static constexpr int BM = 32 * TB;                         // tokens per tile
  static constexpr int STAGE = G_WBYTES + BM * G_ROW;        // weight slice, then token slice
  static constexpr int NST = 160 * 1024 / STAGE >= 3 ? 3 : 2;  // LDS stages
  static constexpr int LDS = NST * STAGE;
  static constexpr int XLOADS = (TB + 1) / 2;   // token loads per wave (odd TB: the last by waves 0-3)
  static constexpr int LOADS = G_WLOADS + XLOADS;
};

// Tile (token block, weight block) and K split of this workgroup.
__device__ __forceinline__ void tile_of(const GemmParams& p, int& tm, int& tn, int& split) {
  const int nwg = gridDim.x;
  int b = blockIdx.x;
  // one contiguous run per XCD, the first nwg % 8 runs one longer.  (Without it for counts that
  // are not multiples of 8, the workgroups that share weight rows sat on different XCDs and read
  // them several times: 700 tokens x 32000 x 2048 in 750 tiles 122.6 -> 90.1 us, 129 tokens in 250
  // 43.8 -> 29.0; 4096 tokens of gated 2 x 4864 x 896 in 988 93.2 -> 81.4.)
  b = (b & 7) * (nwg >> 3) + min(b & 7, nwg & 7) + (b >> 3);
  const int tiles = p.tiles_m * p.tiles_n;
  split = b / tiles;
  b -= split * tiles;
  const int per_group = p.group_m * p.tiles_n;                // group_m token blocks wide
  const int grp = b / per_group;
  const int first = grp * p.group_m;
  const int gm = min(p.tiles_m - first, p.group_m);
  const int r = b - grp * per_group;
  tm = first + r % gm;
  tn = r / gm;
}

template <typename T, int MODE, int ACT, int TB>
__global__ __launch_bounds__(G_THREADS, 1) void gemm_mfma_kernel(const GemmParams p) {
  typedef typename GMfma<T>::frag frag;
  typedef Tile<TB> L;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int ESZ = sizeof(T);
  constexpr int OUT_N = MODE == kGated ? G_BW / 2 : G_BW;   // output columns per tile
  constexpr int NST = L::NST;

  const int tid = threadIdx.x;
  const int wave = uniform(tid >> 6);
  const int lane = tid & 63;
  const int wm = wave & 1;    // token half of the tile
  const int wn = wave >> 1;   // weight quarter (gated: output-column quarter)
  int tm, tn, split;
  tile_of(p, tm, tn, split);
  const int m0 = tm * L::BM;
  const int n0 = tn * OUT_N;
  const int K = p.K;
  const int s_begin = split * p.split_slices;
  const int s_end = min((K + G_BK - 1) / G_BK, s_begin + p.split_slices);
  const int kend = min(K, s_end * G_BK);

  const int rows_x = min(L::BM, p.M - m0);
  const i32x4 rx = make_rsrc((const char*)p.x + (int64_t)m0 * p.ldx * ESZ,
                             (uint32_t)((int64_t)(rows_x - 1) * p.ldx * ESZ + (int64_t)K * ESZ));
  const int rows_w = min(OUT_N, p.N - n0);
  const uint32_t wbytes = (uint32_t)((int64_t)(rows_w - 1) * p.ldw * ESZ + (int64_t)K * ESZ);
  const i32x4 rg = make_rsrc((const char*)p.wg + (int64_t)n0 * p.ldw * ESZ, wbytes);
  const i32x4 ru = MODE == kGated ? make_rsrc((const char*)p.wu + (int64_t)n0 * p.ldw * ESZ, wbytes) : rg;

  // slice loads: load i of wave w fills rows [64 i + 8 w, 64 i + 8 w + 8) of an operand, 8 rows x
  // 128 bytes; the swizzle depends on the row modulo 16, so on the wave alone
  const int lrow = 8 * wave + (lane >> 3);
  const int grp = (lane & 7) ^ g_swz(lrow);
  const int kcol = grp * 8;
  uint32_t off_w[G_WLOADS], off_x[L::XLOADS];
#pragma unroll
  for (int i = 0; i < G_WLOADS; ++i) {   // gated: loads 0, 1 the 128 gate rows, 2, 3 the up rows
    const int row = lrow + 64 * (MODE == kGated ? i & 1 : i);
    off_w[i] = (uint32_t)((int64_t)row * p.ldw * ESZ) + grp * 16;
  }
#pragma unroll
  for (int i = 0; i < L::XLOADS; ++i)
    off_x[i] = (uint32_t)((int64_t)(lrow + 64 * i) * p.ldx * ESZ) + grp * 16;
  const uint32_t lds_wave = lds_addr(smem) + wave * 1024;
  auto issue_one = [&](int s, int stage, int i) {   // i < G_WLOADS: weight rows, else token rows
    const uint32_t sb = lds_wave + (uint32_t)stage * L::STAGE;
    const uint32_t kb = (uint32_t)s * G_ROW;
    const bool kin = s * G_BK + kcol < kend;
    if (i < G_WLOADS) {
      buffer_load_lds16_m0_so(MODE == kGated && i >= 2 ? ru : rg, sb + i * 8192,
                              kin ? off_w[i] : kOutOfRange, kb);
    } else {
      const int li = i - G_WLOADS;
      if ((TB & 1) && li == L::XLOADS - 1 && wave >= 4) return;
      buffer_load_lds16_m0_so(rx, sb + G_WBYTES + li * 8192, kin ? off_x[li] : kOutOfRange, kb);
    }
  };
  // this wave's loads of all but the newest slice have landed
  auto wait_slice = [&] {
    if constexpr (NST == 2) wait_vmcnt<0>();
    else if (!(TB & 1) || wave < 4) wait_vmcnt<(NST - 2) * L::LOADS>();
    else wait_vmcnt<(NST - 2) * (L::LOADS - 1)>();
  };

  // fragments: 4 weight blocks and TB token blocks of 16 rows per 32-wide step
  uint32_t rd[2];
#pragma unroll
  for (int q = 0; q < 2; ++q)
    rd[q] = (lane & 15) * G_ROW + (((4 * q + (lane >> 4)) ^ g_swz(lane & 15)) << 4);
  auto read_a = [&](int stage, int q, int j, frag (&fa)[4]) {
    const int row = MODE == kGated ? (j >> 1) * 128 + wn * 32 + (j & 1) * 16 : wn * 64 + j * 16;
    fa[j] = *(const frag*)(smem + stage * L::STAGE + rd[q] + row * G_ROW);
  };
  auto read_b = [&](int stage, int q, int t, frag (&fb)[TB]) {
    fb[t] = *(const frag*)(smem + stage * L::STAGE + G_WBYTES + rd[q] + (wm * (16 * TB) + t * 16) * G_ROW);
  };

  f32x4 acc[4][TB];
#pragma unroll
  for (int f = 0; f < 4; ++f)
#pragma unroll
    for (int t = 0; t < TB; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[f][t][e] = 0.0f;

  // One 32-wide step: 4 TB matrix instructions token-block major; each token fragment is
  // reloaded for the next step (stage rs, step rq) right after its last use, the next
  // weight fragments go into the other set early, and with DMA the loads of slice ls (into
  // stage lst) are spread evenly.
  frag fa0[4], fa1[4], fb[TB];
  auto step = [&](const frag (&fa)[4], int rs, int rq, frag (&na)[4], auto dma, int ls, int lst) {
#pragma unroll
    for (int t = 0; t < TB; ++t)
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        const int i = t * 4 + f;
        acc[f][t] = GMfma<T>::run(fa[f], fb[t], acc[f][t]);
        if (f == 3) read_b(rs, rq, t, fb);
        if ((i & 3) == 1 && i < 16) read_a(rs, rq, i >> 2, na);
        if constexpr (decltype(dma)::value) {
#pragma unroll
          for (int l = 0; l < L::LOADS; ++l)
            if (i == l * 4 * TB / L::LOADS + 2) issue_one(ls, lst, l);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
  };

#pragma unroll
  for (int s = 0; s < NST; ++s)
#pragma unroll
    for (int i = 0; i < L::LOADS; ++i) issue_one(s_begin + s, s, i);
  if (!(TB & 1) || wave < 4) wait_vmcnt<(NST - 1) * L::LOADS>();
  else wait_vmcnt<(NST - 1) * (L::LOADS - 1)>();
  barrier_no_fence();
#pragma unroll
  for (int j = 0; j < 4; ++j) read_a(0, 0, j, fa0);
#pragma unroll
  for (int t = 0; t < TB; ++t) read_b(0, 0, t, fb);
  __builtin_amdgcn_sched_barrier(0);
  int st = 0;   // stage of slice s
  for (int s = s_begin; s < s_end; ++s) {
    step(fa0, st, 1, fa1, std::integral_constant<bool, false>(), 0, 0);
    wait_slice();
    __builtin_amdgcn_s_waitcnt(kLgkm0);
    barrier_no_fence();
    __builtin_amdgcn_sched_barrier(0);
    const int nx = NST == 2 ? st ^ 1 : (st == NST - 1 ? 0 : st + 1);
    step(fa1, nx, 0, fa0, std::integral_constant<bool, true>(), s + NST, st);
    st = nx;
  }
  wait_vmcnt<0>();

  if (p.partial != nullptr) {
    // one of several K splits: the raw sums, 1 KB per 16 x 16 block in lane order, for
    // gemm_reduce_kernel
    f32x4* dst = (f32x4*)p.partial +
                 ((((int64_t)split * p.tiles_n + tn) * p.tiles_m + tm) * 8 + wave) * (4 * TB * 64) + lane;
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
      for (int t = 0; t < TB; ++t) dst[(f * TB + t) * 64] = acc[f][t];
    return;
  }

  // epilogue: block (f, t) holds token t * 16 + (l & 15) and weight rows f * 16 + 4 (l >> 4) ..
  const int q4 = lane >> 4;
  const bool vec = p.vec_out != 0;
  T* y = (T*)p.y;
  constexpr int NF = MODE == kGated ? 2 : 4;   // output column blocks of 16 per wave
  constexpr int NCOL = NF * 16;
  const int col0 = n0 + wn * NCOL;
  auto values = [&](int f, int t, const float (&bgv)[4], const float (&buv)[4], float (&v)[4],
                    auto bias) {
    float gv[4], uv[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      gv[j] = acc[f][t][j];
      uv[j] = MODE == kGated ? acc[f + 2][t][j] : 0.0f;
    }
    finish4<T, MODE, ACT, decltype(bias)::value, float>(gv, uv, bgv, buv, v);
  };
  if (p.vec_out == 2) {
    constexpr int RB = NCOL * 2;
    constexpr int CPR = RB / 16;
    constexpr int RPI = 64 / CPR;
    auto row_swz = [](int r) { return CPR == 8 ? ((r >> 1) & 7) : ((r >> 2) & 3); };
    __builtin_amdgcn_s_waitcnt(kLgkm0);
    barrier_no_fence();
    char* stage = smem + wave * (16 * TB * RB);
    auto to_lds = [&](auto bias) {
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        const int c4 = f * 16 + 4 * q4;
        float bgv[4] = {0.0f, 0.0f, 0.0f, 0.0f}, buv[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if constexpr (decltype(bias)::value) {
          bias4<T, float>(p.bg, col0 + c4, p.N, true, bgv);
          if constexpr (MODE == kGated) bias4<T, float>(p.bu, col0 + c4, p.N, true, buv);
        }
#pragma unroll
        for (int t = 0; t < TB; ++t) {
          float v[4];
          values(f, t, bgv, buv, v, bias);
          T o[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) o[j] = store_cast<T, float>(v[j]);
          uint2 raw;
          __builtin_memcpy(&raw, o, 8);
          const int row = t * 16 + (lane & 15);
          const int chunk = (c4 >> 3) ^ row_swz(row);
          *(uint2*)(stage + row * RB + chunk * 16 + (q4 & 1) * 8) = raw;
        }
      }
    };
    if (p.bg != nullptr) to_lds(std::integral_constant<bool, true>());
    else to_lds(std::integral_constant<bool, false>());
#pragma unroll
    for (int k = 0; k < 16 * TB / RPI; ++k) {
      const int row = k * RPI + lane / CPR;
      const int c = lane % CPR;
      const uint4 raw = *(const uint4*)(stage + row * RB + ((c ^ row_swz(row)) * 16));
      const int tok = m0 + wm * (16 * TB) + row;
      const int col = col0 + c * 8;
      if (tok < p.M && col < p.N) *(uint4*)(y + (int64_t)tok * p.ldy + col) = raw;
    }
    return;
  }
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const int col = col0 + f * 16 + 4 * q4;
    if (col >= p.N) continue;
    float bgv[4], buv[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    bias4<T, float>(p.bg, col, p.N, vec, bgv);
    if constexpr (MODE == kGated) bias4<T, float>(p.bu, col, p.N, vec, buv);
#pragma unroll
    for (int t = 0; t < TB; ++t) {
      const int tok = m0 + wm * (16 * TB) + t * 16 + (lane & 15);
      if (tok >= p.M) continue;
      float v[4];
      values(f, t, bgv, buv, v, std::integral_constant<bool, true>());
      store4<T, float>(y + (int64_t)tok * p.ldy, col, p.N, vec, v);
    }
  }
}

// The sum of a split launch's partials (split 0 first) and the epilogue: one wave per 16 x 16
// block, in the layout the tiles wrote, so the reads (all but a few percent of the bytes) are
// whole kilobytes.  Bound by those reads, which mostly still sit in the Infinity Cache: 42 MB of
// partials (300 tokens x 4096 x 14336, 8 splits) add about 10 us to a call of 50 us that took
// 285 us unsplit.
template <typename T, int MODE, int ACT>
__global__ __launch_bounds__(256) void gemm_reduce_kernel(const GemmParams p, int tb, int splits) {
  const int lane = threadIdx.x & 63;
  const int nf = MODE == kGated ? 2 : 4;   // output column blocks of a tile's wave
  const int per_wave = nf * tb;
  const int64_t blk = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int64_t tw = blk / per_wave;       // (weight block, token block, wave) of the tile grid
  const int r = (int)(blk - tw * per_wave);
  const int f = r / tb, t = r - f * tb;
  const int64_t tiles = (int64_t)p.tiles_m * p.tiles_n;
  if (tw >= tiles * 8) return;
  const int wave = (int)(tw & 7);
  const int tm = (int)((tw >> 3) % p.tiles_m), tn = (int)((tw >> 3) / p.tiles_m);
  const int tok = tm * 32 * tb + (wave & 1) * 16 * tb + t * 16 + (lane & 15);
  const int col = tn * (nf * 64) + (wave >> 1) * (nf * 16) + f * 16 + 4 * (lane >> 4);
  if (tok >= p.M || col >= p.N) return;
  const int64_t per_split = tiles * 8 * (4 * tb * 64);
  const f32x4* src = (const f32x4*)p.partial + tw * (4 * tb * 64) + (f * tb + t) * 64 + lane;
  f32x4 g = src[0], u = {0.0f, 0.0f, 0.0f, 0.0f};
  if constexpr (MODE == kGated) u = src[2 * tb * 64];
  for (int i = 1; i < splits; ++i) {
    g += src[i * per_split];
    if constexpr (MODE == kGated) u += src[i * per_split + 2 * tb * 64];
  }
  const bool vec = p.vec_out != 0;
  float gv[4], uv[4], bgv[4], buv[4] = {0.0f, 0.0f, 0.0f, 0.0f}, v[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) gv[j] = g[j], uv[j] = u[j];
  bias4<T, float>(p.bg, col, p.N, vec, bgv);
  if constexpr (MODE == kGated) bias4<T, float>(p.bu, col, p.N, vec, buv);
  finish4<T, MODE, ACT, true, float>(gv, uv, bgv, buv, v);
  store4<T, float>((T*)p.y + (int64_t)tok * p.ldy, col, p.N, vec, v);
}

// ---------------------------------------------------------------------------------------
// generic kernel: 64 tokens x 64 output columns per 256-thread block, 4 x 4 per thread
// ---------------------------------------------------------------------------------------
constexpr int GG_T = 64;
constexpr int GG_N = 64;
constexpr int GG_K = 16;

template <typename A> __device__ __forceinline__ A fma_acc(A a, A b, A c);
template <> __device__ __forceinline__ float fma_acc<float>(float a, float b, float c) {
  return __builtin_fmaf(a, b, c);
}
template <> __device__ __forceinline__ double fma_acc<double>(double a, double b, double c) {
  return __builtin_fma(a, b, c);
}

template <typename T, int MODE, int ACT>
__global__ __launch_bounds__(256) void gemm_generic_kernel(const GemmParams p) {
  typedef typename acc_of<T>::type A;
  constexpr int NW = MODE == kGated ? 2 : 1;   // weight operands
  __shared__ A xs[GG_K][GG_T + 1];
  __shared__ A ws[NW][GG_K][GG_N + 1];
  const int tid = threadIdx.x;
  const int tx = tid & 15, ty = tid >> 4;
  const int n0 = blockIdx.x * GG_N;
  const int m0 = blockIdx.y * GG_T;
  const T* x = (const T*)p.x;
  A acc[NW][4][4];
#pragma unroll
  for (int w = 0; w < NW; ++w)
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[w][i][j] = A(0);

  for (int k0 = 0; k0 < p.K; k0 += GG_K) {
    for (int e = tid; e < GG_T * GG_K; e += 256) {
      const int r = e / GG_K, c = e % GG_K;
      const int k = k0 + c;
      const int tok = m0 + r, col = n0 + r;
      xs[c][r] = (tok < p.M && k < p.K) ? load_acc<T, A>(x + (int64_t)tok * p.ldx + k) : A(0);
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const T* wp = (const T*)(w == 0 ? p.wg : p.wu);
        ws[w][c][r] = (col < p.N && k < p.K) ? load_acc<T, A>(wp + (int64_t)col * p.ldw + k) : A(0);
      }
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < GG_K; ++c) {
      A xv[4], wv[NW][4];
#pragma unroll
      for (int i = 0; i < 4; ++i) xv[i] = xs[c][ty * 4 + i];
#pragma unroll
      for (int w = 0; w < NW; ++w)
#pragma unroll
        for (int j = 0; j < 4; ++j) wv[w][j] = ws[w][c][tx * 4 + j];
#pragma unroll
      for (int w = 0; w < NW; ++w)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[w][i][j] = fma_acc<A>(xv[i], wv[w][j], acc[w][i][j]);
    }
    __syncthreads();
  }

  const int col = n0 + tx * 4;
  if (col >= p.N) return;
  A bgv[4], buv[4] = {A(0), A(0), A(0), A(0)};
  bias4<T, A>(p.bg, col, p.N, false, bgv);
  if constexpr (MODE == kGated) bias4<T, A>(p.bu, col, p.N, false, buv);
  T* y = (T*)p.y;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int tok = m0 + ty * 4 + i;
    if (tok >= p.M) continue;
    A gv[4], uv[4], v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      gv[j] = acc[0][i][j];
      uv[j] = MODE == kGated ? acc[NW - 1][i][j] : A(0);
    }
    finish4<T, MODE, ACT, true, A>(gv, uv, bgv, buv, v);
    store4<T, A>(y + (int64_t)tok * p.ldy, col, p.N, false, v);
  }
}

// ---------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------
constexpr int kGroupM = 8;   // token blocks per tile group

// Tile height and K splits of a launch.
struct TilePlan {
  int tb, splits, split_slices;
  size_t ws;   // bytes of partial sums
};
constexpr size_t kMaxPartials = (size_t)128 << 20;

// The launch of least modelled time: rounds of workgroups over the compute units, times the
// slices each walks at its tile height's pace, plus the partial sums' way out and back.  Measured
// pace (us per 64-wide slice with every unit busy): 0.94 / 1.11 / 1.69 at 128 / 160 / 256 tokens;
// 192 (1.41) and 224 (1.50) are slower per token than 256 and are not built.  A small tile wins
// where 256 tokens leave a last round nearly empty or pad much (3001 x 6144 x 4096: 288 tiles in
// two rounds 172 us, 456 of 160 tokens 136 us; 300 tokens x 2 x 14336: 105 -> 81 us), splits
// where the tiles are fewer than the units (4096 x 14336, 300 tokens: 32 tiles unsplit 163 us
// and up, 8 splits 51 us).  A split keeps at least 512 of K.
TilePlan plan_tiles(int64_t M, int64_t rows, int64_t K, size_t ws_bytes) {
  static constexpr struct { int tb; double pace; } kHeights[] = {{8, 1.69}, {5, 1.11}, {4, 0.94}};
  constexpr double kEnds = 5.0;      // prologue and epilogue of a workgroup, us
  constexpr double kLaunch = 3.0;    // the reduction's launch, us
  constexpr double kBytesUs = 6e6;   // partial sums written or read, bytes per us
  const int cus = device_cus() > 0 ? device_cus() : 256;
  const int kt = (int)((K + G_BK - 1) / G_BK);
  TilePlan best{8, 1, kt, 0};
  double least = 0;
  for (const auto& h : kHeights) {
    const int64_t tiles = ((M + 32 * h.tb - 1) / (32 * h.tb)) * ((rows + G_BW - 1) / G_BW);
    for (int want = 1; want <= 16; ++want) {
      const int slices = (kt + want - 1) / want;
      if (want > 1 && (slices < 8 || tiles * want > 2 * cus)) break;
      const int splits = want == 1 ? 1 : (kt + slices - 1) / slices;
      const size_t ws = splits == 1 ? 0 : (size_t)(tiles * splits) * (size_t)(32 * h.tb * G_BW * 4);
      if (ws > std::min(ws_bytes, kMaxPartials)) break;
      const double rounds = (double)((tiles * splits + cus - 1) / cus);
      const double us = rounds * (slices * h.pace + kEnds) + (splits > 1 ? kLaunch + 2.0 * ws / kBytesUs : 0);
      if (least == 0 || us < least) least = us, best = {h.tb, splits, slices, ws};
    }
  }
  return best;
}

bool mfma_path(const GemmParams& p, int dtype, int mode) {
  if (dtype != CEA_BF16 && dtype != CEA_F16 && dtype != CEA_F32) return false;
  const int64_t esz = dtype_size(dtype), per16 = 16 / esz;
  if (p.K % per16 || p.ldx % per16 || p.ldw % per16) return false;
  auto al16 = [](const void* q) { return ((uintptr_t)q & 15) == 0; };
  if (!al16(p.x) || !al16(p.wg) || (mode == kGated && !al16(p.wu))) return false;
  // every byte offset of a tile's rows must stay below the out-of-range marker
  const int64_t lim = (int64_t)kOutOfRange;
  const int wrows = mode == kGated ? G_BW / 2 : G_BW;
  if ((int64_t)(Tile<8>::BM - 1) * p.ldx * esz + (int64_t)p.K * esz >= lim) return false;
  if ((int64_t)(wrows - 1) * p.ldw * esz + (int64_t)p.K * esz >= lim) return false;
  return true;
}

// f32 products of few terms each, bound by writing them: the matrix-core kernel, whose waves split
// K, has waves without work there and adds their sums through LDS all the same.  Measured (us,
// generic / matrix cores): 2048 x 2048 products of 16 11.7 / 25.1, of 64 19.2 / 25.4, of 96 25.8 /
// 25.6; 512 x 2048 of 16 6.0 / 7.4, of 32 8.0 / 7.4; 8192 x 8192 of 64 203 / 356, of 128 356 / 367,
// of 192 513 / 490.
bool f32_output_bound(int64_t M, int64_t rows, int64_t K) {
  return K <= 128 && M * rows >= (K <= 96 ? K << 16 : (int64_t)1 << 25);
}

template <typename T, int MODE, int ACT, int TB>
int launch_tiles(GemmParams p, const TilePlan& pl, hipStream_t st) {
  typedef Tile<TB> L;
  const int out_n = MODE == kGated ? G_BW / 2 : G_BW;
  p.tiles_m = (p.M + L::BM - 1) / L::BM;
  p.tiles_n = (p.N + out_n - 1) / out_n;
  p.group_m = kGroupM;
  p.split_slices = pl.split_slices;
  const int64_t tiles = (int64_t)p.tiles_m * p.tiles_n;
  CEA_REQUIRE(tiles * pl.splits <= INT32_MAX, CEA_EUNSUPPORTED, "linear: problem too large");
  if (pl.splits == 1) p.partial = nullptr;
  const hipError_t e = reserve_lds<gemm_mfma_kernel<T, MODE, ACT, TB>>(L::LDS);
  CEA_REQUIRE(e == hipSuccess, CEA_ELAUNCH, "linear: cannot reserve %d bytes of LDS: %s", L::LDS,
              hipGetErrorString(e));
  hipLaunchKernelGGL((gemm_mfma_kernel<T, MODE, ACT, TB>), dim3((unsigned)(tiles * pl.splits)),
                     dim3(G_THREADS), L::LDS, st, p);
  CEA_CHECK_LAUNCH(MODE == kGated ? "linear_gated" : "linear");
  if (pl.splits > 1) {
    const int64_t blocks = tiles * 8 * (MODE == kGated ? 2 : 4) * TB;
    hipLaunchKernelGGL((gemm_reduce_kernel<T, MODE, ACT>), dim3((unsigned)((blocks + 3) / 4)),
                       dim3(256), 0, st, p, TB, pl.splits);
    CEA_CHECK_LAUNCH(MODE == kGated ? "linear_gated" : "linear");
  }
  return CEA_OK;
}

template <typename T, int MODE, int ACT>
int launch_one(GemmParams p, bool mfma, hipStream_t st) {
  if constexpr (sizeof(T) == 2) {
    if (mfma) {
      const int64_t rows = (int64_t)p.N * (MODE == kGated ? 2 : 1);
      const bool ws16 = ((uintptr_t)p.partial & 15) == 0;
      const TilePlan pl = plan_tiles(p.M, rows, p.K, p.partial && ws16 ? p.ws_bytes : 0);
      switch (pl.tb) {
        case 4: return launch_tiles<T, MODE, ACT, 4>(p, pl, st);
        case 5: return launch_tiles<T, MODE, ACT, 5>(p, pl, st);
        default: return launch_tiles<T, MODE, ACT, 8>(p, pl, st);
      }
    }
  }
  const int64_t gy = (p.M + GG_T - 1) / GG_T;
  CEA_REQUIRE(gy <= 65535, CEA_EUNSUPPORTED, "linear: %d rows exceed the generic kernel's grid",
              p.M);
  hipLaunchKernelGGL((gemm_generic_kernel<T, MODE, ACT>),
                     dim3((unsigned)((p.N + GG_N - 1) / GG_N), (unsigned)gy), dim3(256), 0, st, p);
  CEA_CHECK_LAUNCH(MODE == kGated ? "linear_gated" : "linear");
  return CEA_OK;
}

template <typename T>
int launch_typed(const GemmParams& p, int mode, int act, bool mfma, hipStream_t st) {
  if (mode == kPlain) return launch_one<T, kPlain, 0>(p, mfma, st);
  switch (act) {
    case CEA_ACT_SILU: return launch_one<T, kGated, CEA_ACT_SILU>(p, mfma, st);
    case CEA_ACT_GELU: return launch_one<T, kGated, CEA_ACT_GELU>(p, mfma, st);
    case CEA_ACT_GELU_TANH: return launch_one<T, kGated, CEA_ACT_GELU_TANH>(p, mfma, st);
    case CEA_ACT_RELU: return launch_one<T, kGated, CEA_ACT_RELU>(p, mfma, st);
  }
  set_error("linear_gated: unknown activation %d", act);
  return CEA_EUNSUPPORTED;
}

}  // namespace

// x [M, K], w_gate / w_up [N, K] (one row stride), biases [N] or null, y [M, N]; shapes and
// dtypes validated by the caller.  mode: 0 plain (w_up / b_up unused), 1 gated.
int launch_linear(const cea_tensor* x, const cea_tensor* wg, const cea_tensor* wu,
                  const cea_tensor* bg, const cea_tensor* bu, cea_tensor* y, int mode, int act,
                  void* ws, size_t ws_bytes, hipStream_t st) {
  GemmParams p{};
  p.partial = (float*)ws;
  p.ws_bytes = ws ? ws_bytes : 0;
  p.x = x->data;
  p.wg = wg->data;
  p.wu = wu ? wu->data : nullptr;
  p.bg = bg ? bg->data : nullptr;
  p.bu = bu ? bu->data : nullptr;
  p.y = y->data;
  p.M = (int32_t)x->size[0];
  p.K = (int32_t)x->size[1];
  p.N = (int32_t)wg->size[0];
  p.ldx = x->size[0] > 1 ? x->stride[0] : p.K;
  p.ldw = wg->size[0] > 1 ? wg->stride[0] : p.K;
  p.ldy = y->size[0] > 1 ? y->stride[0] : p.N;
  // output stores: 2 = whole 16-byte chunks staged through LDS, 1 = 8-byte stores,
  // 0 = element stores
  const bool v8 = p.N % 4 == 0 && p.ldy % 4 == 0 && ((uintptr_t)p.y & 7) == 0 &&
                  (p.bg == nullptr || ((uintptr_t)p.bg & 7) == 0) &&
                  (p.bu == nullptr || ((uintptr_t)p.bu & 7) == 0);
  const bool v16 = v8 && p.N % 8 == 0 && p.ldy % 8 == 0 && ((uintptr_t)p.y & 15) == 0;
  p.vec_out = v16 ? 2 : v8 ? 1 : 0;
  if (p.M == 0 || p.N == 0) return CEA_OK;
  bool mfma = mfma_path(p, x->dtype, mode);
  if (x->dtype == CEA_F32 && f32_output_bound(p.M, (int64_t)p.N * (mode == kGated ? 2 : 1), p.K))
    mfma = false;
  if (mfma && (p.M <= kSkinnyTokens || x->dtype == CEA_F32))
    return launch_linear_skinny(p, x->dtype, mode, act, st);
  switch (x->dtype) {
    case CEA_BF16: return launch_typed<bf16>(p, mode, act, mfma, st);
    case CEA_F16: return launch_typed<f16>(p, mode, act, mfma, st);
    case CEA_F32: return launch_typed<float>(p, mode, act, false, st);
    case CEA_F64: return launch_typed<double>(p, mode, act, false, st);
  }
  set_error("linear: unsupported dtype %s", dtype_name(x->dtype));
  return CEA_EUNSUPPORTED;
}

size_t linear_workspace_bytes(int64_t M, int64_t N, int64_t K, int dtype, int mode) {
  if ((dtype != CEA_BF16 && dtype != CEA_F16) || M <= kSkinnyTokens || K % 8) return 0;
  return plan_tiles(M, N * (mode == kGated ? 2 : 1), K, SIZE_MAX).ws;
}

}  // namespace cea
