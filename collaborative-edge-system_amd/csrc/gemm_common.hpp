// Shared by the projection GEMM kernels (gemm.hip, gemm_skinny.hip): operand block, matrix-core
// wrappers and the epilogue of four consecutive output columns.
#pragma once

#include "cea_kernels.hpp"

namespace cea {

struct GemmParams {
  const void* x;    // [M, K], row stride ldx
  const void* wg;   // [N, K], row stride ldw (gated: the gate rows)
  const void* wu;   // gated: the up rows, same row stride
  const void* bg;   // [N] or null (gated: gate bias)
  const void* bu;   // gated: up bias or null
  void* y;          // [M, N], row stride ldy
  int64_t ldx, ldw, ldy;
  int32_t M, N, K;  // N = output columns
  int32_t tiles_m, tiles_n, group_m;
  int32_t vec_out;  // 2: 16-byte row chunks, 1: 4-element stores, 0: element stores
  // K splits of the tile kernel: 64-wide slices per split, f32 sums (null: one split) and the
  // caller's scratch size
  int32_t split_slices;
  float* partial;
  size_t ws_bytes;
};

// Rows of x the skinny kernel takes (4 blocks of 16).
constexpr int kSkinnyTokens = 64;
// Operands as gemm.hip's matrix-core path; bf16 / f16 with M <= kSkinnyTokens, or f32.
int launch_linear_skinny(const GemmParams& p, int dtype, int mode, int act, hipStream_t st);

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <typename T> struct GMfma;
template <> struct GMfma<bf16> {
  typedef bf16x8 frag;
  static __device__ __forceinline__ f32x4 run(frag a, frag b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct GMfma<f16> {
  typedef f16x8 frag;
  static __device__ __forceinline__ f32x4 run(frag a, frag b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

enum { kPlain = 0, kGated = 1 };
// f32: a fragment holds 4 consecutive K per lane, multiplied in 4 steps of v_mfma_f32_16x16x4.
template <> struct GMfma<float> {
  typedef f32x4 frag;
  static __device__ __forceinline__ f32x4 run(frag a, frag b, f32x4 c) {
#pragma unroll
    for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], c, 0, 0, 0);
    return c;
  }
};

constexpr uint32_t kOutOfRange = 0x80000000u;        // above every resource's range

// 16-byte group swizzle of a slice row (8 groups of 16 bytes): group c of row r sits at group
// c ^ g_swz(r).  A fragment read has 16 rows per 16-lane quarter and the quarters read groups
// c, c+1, c+2, c+3.  Measured on gfx950 (LDS bank-conflict counter), the reads behave as if 32
// lanes share a 512-byte bank window; this swizzle gives distinct 16-byte slots for any 32
// lanes (rows of equal r & 3 in one window), for any 16 lanes within 256 bytes and for any 8
// within 128 bytes.  Depends on r & 15 only.
__device__ __forceinline__ int g_swz(int r) { return ((r >> 1) & 7) ^ ((r & 1) << 2); }

template <typename T, typename A> __device__ __forceinline__ A rnd_acc(A v) {
  if constexpr (sizeof(T) >= sizeof(A)) return v;
  else return (A)round_to<T>((float)v);
}

// Bias of 4 consecutive columns (zero without a bias, or past n).
template <typename T, typename A>
__device__ __forceinline__ void bias4(const void* b, int col, int n, bool vec, A (&v)[4]) {
  const T* bp = (const T*)b;
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = A(0);
  if (bp == nullptr) return;
  if (vec && col + 3 < n) {
    T t[4];
    __builtin_memcpy(t, bp + col, sizeof(t));
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = (A)to_f32<T>(t[j]);
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (col + j < n) v[j] = load_acc<T, A>(bp + col + j);
  }
}

// Stores 4 consecutive columns of one output row.
template <typename T, typename A>
__device__ __forceinline__ void store4(T* row, int col, int n, bool vec, const A (&v)[4]) {
  T t[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) t[j] = store_cast<T, A>(v[j]);
  if (vec && col + 3 < n) {
    if constexpr (sizeof(T) == 2) {
      uint2 raw;
      __builtin_memcpy(&raw, t, 8);
      *(uint2*)(row + col) = raw;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) row[col + j] = t[j];
    }
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (col + j < n) row[col + j] = t[j];
  }
}

// The epilogue of 4 consecutive columns: plain y = acc + bias; gated
// y = T(act(T(gate + b_g))) * T(up + b_u).
template <typename T, int MODE, int ACT, bool BIAS, typename A>
__device__ __forceinline__ void finish4(const A (&g)[4], const A (&u)[4], const A (&bg)[4],
                                        const A (&bu)[4], A (&v)[4]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if constexpr (MODE == kPlain) {
      v[j] = BIAS ? add_rn(g[j], bg[j]) : g[j];
    } else {
      const A gate = rnd_acc<T, A>(BIAS ? add_rn(g[j], bg[j]) : g[j]);
      const A up = rnd_acc<T, A>(BIAS ? add_rn(u[j], bu[j]) : u[j]);
      v[j] = mul_rn(rnd_acc<T, A>(gate_act<ACT, A>(gate)), up);
    }
  }
}

}  // namespace

// ceil(a / b) for positive b
__host__ __device__ constexpr int ceil_div(int a, int b) { return (a + b - 1) / b; }

}  // namespace cea
