// One thread per output element: C[m][n] = rne(scale * sum_k A[m][k] * B[n][k]) with a serial
// fp32 fused-multiply-add chain over k.  Handles every shape, stride and dtype the ABI accepts;
// it is the library's on-device cross-check for the MFMA kernels and the path for shapes they
// reject.  Also here: the copy kernels with which the library repacks the operands of such a problem
// into aligned ones, and its output out of an aligned one, when the caller lends it the memory (gemm_api.hip).  Counterpart in the reference:
// none (its only kernel rejects such shapes, kernels/gemm_kernels/sm90a/gemm_test.cu:33-41).
#include "cdna4_primitives.h"
#include "gemm_launch.h"

namespace mi355 {
namespace {

template <class T, class OutT>
__global__ __launch_bounds__(256) void gemm_tn_simple(GemmArgs g) {
  // 16 x 16 outputs per workgroup; the workgroups walk the blocks of C in one dimension (the y and z
  // dimensions of a grid hold 65535 entries only), striding when there are more than 2^31 - 1.
  const int64_t blocks_n = (g.N + 15) / 16, blocks = blocks_n * ((g.M + 15) / 16);
  for (int64_t b = blockIdx.x; b < blocks; b += gridDim.x) {
    const int64_t n = (b % blocks_n) * 16 + (threadIdx.x & 15);
    const int64_t m = (b / blocks_n) * 16 + (threadIdx.x >> 4);
    if (m >= g.M || n >= g.N) continue;
    const int64_t a0 = m * g.lda, b0 = n * g.ldb;
    float acc = 0.f;
    for (int64_t k = 0; k < g.K; ++k)
      acc = __builtin_fmaf(Decode<T>::run(g.A, a0 + k), Decode<T>::run(g.B, b0 + k), acc);
    ((uint16_t*)g.C)[m * g.ldc + n] = Pack4<OutT>::one(acc * output_scale(g));
  }
}

// Sixteen source bytes of a row from byte `at` on, zeros from row_bytes on.  The source has only element alignment: the
// compiler may use one wide load (global accesses need no alignment on this target).
template <class E>
__device__ __forceinline__ u32x4 row_chunk(const uint8_t* row, uint32_t at, uint32_t row_bytes) {
  u32x4 out = {0u, 0u, 0u, 0u};
  if (at + 16 <= row_bytes) {
    __builtin_memcpy(&out, row + at, 16);
  } else if (at < row_bytes) {
    E v[16 / sizeof(E)];
#pragma unroll
    for (uint32_t i = 0; i < 16 / sizeof(E); ++i) {
      const uint32_t byte = at + i * (uint32_t)sizeof(E);
      v[i] = byte < row_bytes ? *(const E*)(row + byte) : (E)0;
    }
    __builtin_memcpy(&out, v, 16);
  }
  return out;
}

// Bound by its read and its write: kChunks 16-byte chunks of the destination per thread, all loads out before the first
// store; one or two operands per launch.
constexpr int kChunks = 4;
template <class E>
__global__ __launch_bounds__(256) void repack_rows(RepackOperand first, RepackOperand second, uint32_t row_bytes,
                                                   uint32_t first_blocks) {
  const bool is_second = blockIdx.x >= first_blocks;
  const RepackOperand& op = is_second ? second : first;
  const uint32_t per_row = (uint32_t)(op.dst_ld / 16);
  const uint32_t begin = (is_second ? blockIdx.x - first_blocks : blockIdx.x) * (256 * kChunks) + threadIdx.x;
  const uint32_t total = (uint32_t)op.rows * per_row;      // below 2^31 (launch_repack_rows)
  u32x4 v[kChunks];
  int64_t to[kChunks];
#pragma unroll
  for (int i = 0; i < kChunks; ++i) {
    const uint32_t id = begin + i * 256;
    const uint32_t row = id / per_row, at = (id % per_row) * 16;
    to[i] = id < total ? (int64_t)row * op.dst_ld + at : -1;
    if (id < total) v[i] = row_chunk<E>(op.src + (int64_t)row * op.src_ld, at, row_bytes);
  }
#pragma unroll
  for (int i = 0; i < kChunks; ++i)
    if (to[i] >= 0) *(u32x4*)(op.dst + to[i]) = v[i];
}

// Bound by its read and its write: one wave per run of kRunColumns columns of a row, cut where the destination is 16-byte
// aligned, so that it writes whole lines (a load needs no alignment on this target, and a misaligned one costs less than a
// misaligned store); four loads in flight per lane.  4096 x 14337 bf16 8 us less than with 8-byte pieces cut at the source's
// alignment.
constexpr uint32_t kRunChunks = 4 * 64, kRunColumns = 8 * kRunChunks;
__global__ __launch_bounds__(256) void copy_out(const uint16_t* __restrict__ src, int64_t waves, int64_t runs_per_row, int64_t cols,
                                                int64_t src_ld, uint16_t* __restrict__ dst, int64_t dst_ld) {
  const int64_t wave = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (wave >= waves) return;
  const int64_t row = wave / runs_per_row, run = wave % runs_per_row;
  const uint16_t* from = src + row * src_ld;
  uint16_t* to = dst + row * dst_ld;
  const int64_t first = run * kRunColumns - (int64_t)((uintptr_t)to % 16 / 2);   // the first chunk of a row may begin before it
  u32x4 v[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t col = first + (int64_t)(i * 64 + (threadIdx.x & 63)) * 8;
    if (col >= 0 && col + 8 <= cols) __builtin_memcpy(&v[i], from + col, 16);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t col = first + (int64_t)(i * 64 + (threadIdx.x & 63)) * 8;
    if (col >= 0 && col + 8 <= cols) {
      *(u32x4*)(to + col) = v[i];
    } else if (col + 8 > 0 && col < cols) {
      for (int64_t c = col < 0 ? 0 : col; c < col + 8 && c < cols; ++c) to[c] = from[c];
    }
  }
}

template <class T, class OutT>
int launch(const GemmArgs& g, hipStream_t stream) {
  const int64_t blocks = ((g.N + 15) / 16) * ((g.M + 15) / 16);
  const int64_t grid = blocks < 0x7fffffff ? blocks : 0x7fffffff;
  hipLaunchKernelGGL((gemm_tn_simple<T, OutT>), dim3((unsigned)grid), dim3(256), 0, stream, g);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace

int launch_repack_rows(const RepackOperand& first, const RepackOperand& second, int64_t row_bytes, int elem_bytes, hipStream_t stream) {
  const auto kernel = elem_bytes == 2 ? repack_rows<uint16_t> : repack_rows<uint8_t>;
  constexpr int64_t kMaxChunks = ((int64_t)1 << 31) - 1;   // of a launch and operand; a larger copy goes in runs of rows
  RepackOperand rest[2] = {first, second};
  while (rest[0].rows > 0 || rest[1].rows > 0) {
    RepackOperand part[2];
    uint32_t blocks[2];
    for (int i = 0; i < 2; ++i) {
      part[i] = rest[i];
      blocks[i] = 0;
      if (rest[i].rows == 0) continue;
      const int64_t per_row = rest[i].dst_ld / 16;
      if (rest[i].dst_ld % 16 != 0 || per_row > kMaxChunks) return -1;
      if (part[i].rows > kMaxChunks / per_row) part[i].rows = kMaxChunks / per_row;
      blocks[i] = (uint32_t)((part[i].rows * per_row + 256 * kChunks - 1) / (256 * kChunks));
      rest[i].rows -= part[i].rows;
      rest[i].src += part[i].rows * rest[i].src_ld;
      rest[i].dst += part[i].rows * rest[i].dst_ld;
    }
    hipLaunchKernelGGL(kernel, dim3(blocks[0] + blocks[1]), dim3(256), 0, stream, part[0], part[1], (uint32_t)row_bytes, blocks[0]);
    if (hipGetLastError() != hipSuccess) return -1;
  }
  return 0;
}

int launch_copy_out(const void* src, int64_t rows, int64_t cols, int64_t src_ld, void* dst, int64_t dst_ld, hipStream_t stream) {
  if (rows == 0 || cols == 0) return 0;
  const int64_t runs = (cols + 7 + kRunColumns - 1) / kRunColumns, waves = rows * runs, blocks = (waves + 3) / 4;
  if (blocks >= ((int64_t)1 << 31)) return -1;
  hipLaunchKernelGGL(copy_out, dim3((unsigned)blocks), dim3(256), 0, stream, (const uint16_t*)src, waves, runs, cols, src_ld,
                     (uint16_t*)dst, dst_ld);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_simple(const GemmArgs& g, int in_dtype, int out_dtype, hipStream_t stream) {
  const bool out_bf16 = out_dtype == 0;
  switch (in_dtype) {
    case 0: return out_bf16 ? launch<BF16, BF16>(g, stream) : launch<BF16, F16>(g, stream);
    case 1: return out_bf16 ? launch<F16, BF16>(g, stream) : launch<F16, F16>(g, stream);
    case 2: return out_bf16 ? launch<E4M3, BF16>(g, stream) : launch<E4M3, F16>(g, stream);
  }
  return -1;
}

}  // namespace mi355
