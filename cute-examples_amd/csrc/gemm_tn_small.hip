// Small products on fp32 sums whose operands have rows of any alignment: one wave per block of 4 x 4 outputs, K spread over its lanes.
// For e4m3, whose sums on the matrix cores are coarser (16-bit products run on gemm_tn_slices, where their rows are in its reach).
//
// What the streaming and tile kernels cannot address (K*elem_bytes or a row stride not a multiple of 16, A or B misaligned)
// and is too small to be worth repacking used to run one serial chain of K additions per thread, bound by the latency of
// two element loads per step.  Here lane l takes the 16-byte pieces l, l + 64, ... of the rows (global loads need no
// alignment on this target), 4 + 4 of them per step, multiplies in fp32 (products of 16- and 8-bit values are exact) and the
// 64 partial sums are added in a fixed tree at the end: the error grows with K / 64 where the serial chain's grows with K.
// What bounds it is the latency of K * elem_bytes / 1024 dependent rounds of loads, two in flight.  Counterpart in the
// reference: none (its only kernel rejects such shapes, kernels/gemm_kernels/sm90a/gemm_test.cu:33-41).
#include "cdna4_primitives.h"
#include "gemm_launch.h"

namespace mi355 {
namespace {

// 16 bytes -> kPer floats.
template <class T> struct Piece;
template <> struct Piece<BF16> {
  static constexpr int kPer = 8;
  typedef uint16_t Element;
  static __device__ __forceinline__ void decode(u32x4 a, float* v) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[2 * k] = __builtin_bit_cast(float, a[k] << 16);
      v[2 * k + 1] = __builtin_bit_cast(float, a[k] & 0xffff0000u);
    }
  }
};
template <> struct Piece<F16> {
  static constexpr int kPer = 8;
  typedef uint16_t Element;
  static __device__ __forceinline__ void decode(u32x4 a, float* v) {
    const f16x8 h = __builtin_bit_cast(f16x8, a);
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = (float)h[k];
  }
};
template <> struct Piece<E4M3> {
  static constexpr int kPer = 16;
  typedef uint8_t Element;
  static __device__ __forceinline__ void decode(u32x4 a, float* v) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      typedef __attribute__((ext_vector_type(2))) float f2;
      const f2 lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)a[k], false), hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)a[k], true);
      v[4 * k] = lo[0]; v[4 * k + 1] = lo[1]; v[4 * k + 2] = hi[0]; v[4 * k + 3] = hi[1];
    }
  }
};

// Elements [k, k + kPer) of a row of K, zeros from K on; no byte outside the row is read.
template <class T>
__device__ __forceinline__ u32x4 row_piece(const void* row, int64_t k, int64_t K) {
  typedef typename Piece<T>::Element E;
  constexpr int kPer = Piece<T>::kPer;
  u32x4 out = {0u, 0u, 0u, 0u};
  const E* p = (const E*)row + k;
  if (k + kPer <= K) {
    __builtin_memcpy(&out, p, 16);
  } else {
#pragma unroll
    for (int e = 0; e < kPer; ++e)
      if (k + e < K) out[e * (int)sizeof(E) / 4] |= (uint32_t)p[e] << (8 * (e * (int)sizeof(E) % 4));
  }
  return out;
}

constexpr int kSide = 4;   // outputs per wave: kSide x kSide

template <class T, class OutT>
__global__ __launch_bounds__(256) void gemm_tn_small(GemmArgs g) {
  constexpr int kPer = Piece<T>::kPer;
  const uint32_t lane = threadIdx.x & 63u;
  const int64_t blocks_n = (g.N + kSide - 1) / kSide, blocks = blocks_n * ((g.M + kSide - 1) / kSide);
  const int64_t block = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (block >= blocks) return;
  const int64_t m0 = block / blocks_n * kSide, n0 = block % blocks_n * kSide;
  const uint8_t *rows_a[kSide], *rows_b[kSide];
#pragma unroll
  for (int i = 0; i < kSide; ++i) {   // rows past the edge repeat the last one; their outputs are not stored
    rows_a[i] = (const uint8_t*)g.A + (m0 + i < g.M ? m0 + i : g.M - 1) * g.lda * T::kBytes;
    rows_b[i] = (const uint8_t*)g.B + (n0 + i < g.N ? n0 + i : g.N - 1) * g.ldb * T::kBytes;
  }
  const float scale = output_scale(g);
  float acc[kSide][kSide] = {};
  u32x4 a[2][kSide], b[2][kSide];
  auto load = [&](int s, int64_t k) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kSide; ++i) {
      a[s][i] = row_piece<T>(rows_a[i], k, g.K);
      b[s][i] = row_piece<T>(rows_b[i], k, g.K);
    }
  };
  auto multiply = [&](int s) __attribute__((always_inline)) {
    float va[kSide][kPer], vb[kPer];
#pragma unroll
    for (int i = 0; i < kSide; ++i) Piece<T>::decode(a[s][i], va[i]);
#pragma unroll
    for (int j = 0; j < kSide; ++j) {
      Piece<T>::decode(b[s][j], vb);
#pragma unroll
      for (int i = 0; i < kSide; ++i)
#pragma unroll
        for (int k = 0; k < kPer; ++k) acc[i][j] = __builtin_fmaf(va[i][k], vb[k], acc[i][j]);
    }
  };
  constexpr int64_t kStep = 64 * kPer;
  int64_t k = lane * kPer;
  for (; k + kStep < g.K; k += 2 * kStep) {
    load(0, k);
    load(1, k + kStep);
    multiply(0);
    multiply(1);
  }
  if (k < g.K) {
    load(0, k);
    multiply(0);
  }
  // Sum over the lanes; afterwards lane 4 * i + j keeps output (i, j).
  float mine = 0.f;
#pragma unroll
  for (int i = 0; i < kSide; ++i)
#pragma unroll
    for (int j = 0; j < kSide; ++j) {
      float s = acc[i][j];
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
      mine = lane == (uint32_t)(kSide * i + j) ? s : mine;
    }
  const int64_t m = m0 + lane / kSide, n = n0 + lane % kSide;
  if (lane < kSide * kSide && m < g.M && n < g.N) ((uint16_t*)g.C)[m * g.ldc + n] = Pack4<OutT>::one(mine * scale);
}

template <class T, class OutT>
int launch(const GemmArgs& g, hipStream_t stream) {
  const int64_t blocks = ((g.N + kSide - 1) / kSide) * ((g.M + kSide - 1) / kSide), grid = (blocks + 3) / 4;
  if (grid >= ((int64_t)1 << 31)) return -1;
  hipLaunchKernelGGL((gemm_tn_small<T, OutT>), dim3((unsigned)grid), dim3(256), 0, stream, g);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace

int launch_small(const GemmArgs& g, int in_dtype, int out_dtype, hipStream_t stream) {
  const bool out_bf16 = out_dtype == 0;
  switch (in_dtype) {
    case 0: return out_bf16 ? launch<BF16, BF16>(g, stream) : launch<BF16, F16>(g, stream);
    case 1: return out_bf16 ? launch<F16, BF16>(g, stream) : launch<F16, F16>(g, stream);
    case 2: return out_bf16 ? launch<E4M3, BF16>(g, stream) : launch<E4M3, F16>(g, stream);
  }
  return -1;
}

}  // namespace mi355
