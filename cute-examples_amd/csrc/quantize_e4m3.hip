// Per-tensor fp8 quantisation on the device: the step in front of the fp8 GEMM.
//
//   amax  = max |x|
//   scale = amax / 448  (1 if amax == 0)  (OCP e4m3 has no infinities; 448 is its largest value)
//   x_q   = e4m3_rne(clamp(x / scale, -448, 448))
//
// so that x ~= scale * x_q.  Launches on the caller's stream, no host synchronisation: the scale stays in device memory
// and the GEMM reads it from there.  One launch for small tensors (bound by its latency: bf16 16 x 4096 9.1 -> 3.8 us), two
// for larger ones, or three where the caller has no scratch memory for the maxima of the workgroups.  Large tensors are
// bound by their two reads and one write: bf16 8192 x 8192 65.6 -> 53.6 us, 6.3 TB/s (the maximum 22.7 us; the rest was
// 47.7 us long on its divisions, see codes_of).  The reference has no fp8 path;
// the contract is the benchmark configuration's (operands quantised with per-tensor fp32 scales
// amax/448) and is checked against torch's float8_e4m3fn cast and the C restatement in the tests.
#include "cdna4_primitives.h"
#include "gemm_launch.h"
#include "quantize_convert.h"

namespace mi355 {
namespace {

constexpr float kE4m3Max = 448.0f;
// Up to here one launch does it all, every workgroup reading the whole tensor (bf16, per call back to back: 65536 elements
// 3.8 us against 6.6 in two launches and 9.1 in the three with an atomic maximum; 131072 4.8 against 6.9; with 524288 bytes
// read by every workgroup the two launches are ahead, fp32 131072 6.0 against 6.9).
constexpr int64_t kSmallBytes = 262144;
// Workgroups of the maximum, and floats of scratch memory: 512 read at full rate (bf16 8192 x 8192 22.7 us; 256, 1024 and
// 2048 workgroups 24.8...25.3).
constexpr int64_t kAmaxBlocks = 512;
// Codes of larger tensors are stored non-temporally, which leaves the Infinity Cache to the second read of x: bf16
// 8192 x 8192 53.6 us against 60.0, 48 Mi elements 41.4 against 46.5; at 32 Mi elements and below the two are within 1 %,
// and the GEMM that reads the codes next would rather find them there: fp8 8192^3 behind its quantiser takes 383 us when they
// are, 394 when not (traced), which leaves 8 us of the quantiser's gain to the two together (422 -> 415 us back to back).
constexpr int64_t kStreamElements = 32 << 20;
// 1024...8192 workgroups are within 2 % of each other on large tensors.  What the L2s hold together is better read by fewer with
// more in flight (4096 against 1024, with scratch memory: bf16 8 and 12 Mi elements 9.8 / 8.3 and 11.3 / 10.6 us, fp32 6 Mi 8.6 / 7.7).
constexpr int64_t kQuantizeBlocks = 4096, kQuantizeBlocksInL2 = 1024, kL2Bytes = 32 << 20;

__global__ void amax_init(float* out) { out[0] = 1.0f; out[1] = 0.0f; }

__device__ __forceinline__ float scale_of(float amax) { return amax > 0.f ? amax / kE4m3Max : 1.0f; }

// max |x[i]| over the groups of eight elements first, first + stride, ... below n / 8; kFlight loads in flight.
template <class In, int kFlight>
__device__ __forceinline__ float groups_amax(const void* x, int64_t n, int64_t first, int64_t stride) {
  float m = 0.f;
  const int64_t groups = n / 8;
  int64_t g = first;
  for (; g + (kFlight - 1) * stride < groups; g += kFlight * stride) {
    float v[kFlight][8];
#pragma unroll
    for (int u = 0; u < kFlight; ++u) Load8<In>::run(x, (g + u * stride) * 8, v[u]);
#pragma unroll
    for (int u = 0; u < kFlight; ++u)
#pragma unroll
      for (int k = 0; k < 8; ++k) m = __builtin_fmaxf(m, __builtin_fabsf(v[u][k]));
  }
  for (; g < groups; g += stride) {
    float v[8];
    Load8<In>::run(x, g * 8, v);
#pragma unroll
    for (int k = 0; k < 8; ++k) m = __builtin_fmaxf(m, __builtin_fabsf(v[k]));
  }
  if (first < n % 8) m = __builtin_fmaxf(m, __builtin_fabsf(Load8<In>::one(x, groups * 8 + first)));   // the last, partial group
  return m;
}

// The maximum over a workgroup of kWaves waves, in every thread.
template <int kWaves>
__device__ __forceinline__ float workgroup_max(float m) {
  __shared__ float wave_max[kWaves];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = __builtin_fmaxf(m, __shfl_xor(m, off));
  if ((threadIdx.x & 63) == 0) wave_max[threadIdx.x >> 6] = m;
  __syncthreads();
  m = wave_max[0];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) m = __builtin_fmaxf(m, wave_max[w]);
  return m;
}

// x / scale for eight elements -> eight codes, the same bits whichever way is taken.
//   kDivide   the IEEE division: about a dozen instructions, one of them quarter rate, per element; alone it takes longer
//             than the memory traffic of the pass (bf16 8192 x 8192: 47.7 us of vector instructions)
//   else      Markstein's correction (IBM J. Res. Dev. 34, 1990) of x * y, y = 1 / scale correctly rounded: with
//             r = x - (x*y) * scale, which one fused multiply-add gives exactly, x*y + r*y is the correctly rounded quotient:
//             three instructions.  It needs r free of underflow for every quotient that does not round to code 0 (from 2^-11 on
//             r is a multiple of 2^-57 times scale), hence the range of `scale` in markstein_ok.  The sign is taken from x (a
//             negative zero would lose it).  amax is finite here, so no quotient exceeds 448 * (1 + 2^-23), which the
//             conversion rounds to 448: no clamp.  NaN stays NaN through all of it.
__device__ __forceinline__ bool markstein_ok(float scale) { return scale >= 0x1p-60f && scale <= 0x1p100f; }

template <bool kDivide>
__device__ __forceinline__ u32x2 codes_of(const float (&v)[8], float scale, float inv) {
  if constexpr (kDivide) {
    return (u32x2){to_e4m3x4(v[0] / scale, v[1] / scale, v[2] / scale, v[3] / scale),
                   to_e4m3x4(v[4] / scale, v[5] / scale, v[6] / scale, v[7] / scale)};
  } else {
    float q[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float q0 = v[k] * inv;
      const float r = __builtin_fmaf(-q0, scale, v[k]);
      q[k] = __builtin_copysignf(__builtin_fmaf(r, inv, q0), v[k]);
    }
    return (u32x2){to_e4m3x4_bounded(q[0], q[1], q[2], q[3]), to_e4m3x4_bounded(q[4], q[5], q[6], q[7])};
  }
}

template <bool kStream>
__device__ __forceinline__ void store_codes(uint8_t* q, int64_t group, u32x2 codes) {
  if constexpr (kStream) __builtin_nontemporal_store(codes, (u32x2*)q + group);
  else ((u32x2*)q)[group] = codes;
}

// Groups of eight elements first, first + stride, ... and, thread by thread, the partial group behind the last one.
template <class In, bool kDivide>
__device__ __forceinline__ void quantize_groups(const void* x, int64_t n, uint8_t* q, float scale, float inv, int64_t first,
                                                int64_t stride, int64_t thread) {
  const int64_t groups = n / 8;
  for (int64_t g = first; g < groups; g += stride) {
    float v[8];
    Load8<In>::run(x, g * 8, v);
    ((u32x2*)q)[g] = codes_of<kDivide>(v, scale, inv);
  }
  if (thread < n % 8) {
    const int64_t i = groups * 8 + thread;
    q[i] = (uint8_t)to_e4m3(Load8<In>::one(x, i) / scale);
  }
}

// Pieces of 256 groups, four loads in flight per thread.  Streamed tensors go in runs of four pieces: a workgroup reads and writes
// one stretch of memory at a time.  In smaller ones a workgroup's pieces are as far apart as the maximum's were, which finds again
// what that left in the XCD's L2, and there are enough workgroups to fill the chip (us, runs against this, with scratch memory:
// bf16 8, 12 and 16 Mi elements 10.3 / 8.3, 13.8 / 10.6, 16.9 / 14.3, fp32 6, 8 and 12 Mi 12.3 / 7.7, 16.1 / 9.4, 21.9 / 17.9;
// without: bf16 1 Mi 12.0 / 11.4, fp32 8 Mi 17.0 / 14.5, but bf16 8 Mi 10.8 / 13.9).
template <class In, bool kDivide, bool kStream>
__device__ __forceinline__ void quantize_all(const void* x, int64_t n, uint8_t* q, float scale) {
  constexpr int kRun = kDivide ? 1 : 4;
  const float inv = 1.0f / scale;
  const int64_t pieces = n / (8 * 256), block = blockIdx.x, blocks = gridDim.x, step = kStream ? 1 : blocks;
  int64_t p = kStream ? block * kRun : block;
  for (; p + (kRun - 1) * step < pieces; p += kRun * blocks) {
    float v[kRun][8];
#pragma unroll
    for (int u = 0; u < kRun; ++u) Load8<In>::run(x, ((p + u * step) * 256 + threadIdx.x) * 8, v[u]);
#pragma unroll
    for (int u = 0; u < kRun; ++u)
      store_codes<kStream>(q, (p + u * step) * 256 + threadIdx.x, codes_of<kDivide>(v[u], scale, inv));
  }
  // what is left: in runs the pieces behind the last whole one, otherwise this workgroup's own and the groups behind the last piece
  const int64_t thread = block * 256 + threadIdx.x;
  const int64_t first = kStream ? pieces / kRun * kRun * 256 + thread : p * 256 + threadIdx.x;
  quantize_groups<In, kDivide>(x, n, q, scale, inv, first, blocks * 256, thread);
}

// The maximum of each workgroup to partial[blockIdx.x]; without that scratch memory, to the atomic maximum out[1]: for
// non-negative floats the unsigned order of the bit patterns is the numeric order.
template <class In>
__global__ __launch_bounds__(256) void amax_kernel(const void* x, int64_t n, float* out, float* partial) {
  const float m = workgroup_max<4>(
      groups_amax<In, 4>(x, n, (int64_t)blockIdx.x * 256 + threadIdx.x, (int64_t)gridDim.x * 256));
  if (threadIdx.x != 0) return;
  if (partial) {
    partial[blockIdx.x] = m;
    return;
  }
  // Thousands of atomics on one address take tens of microseconds, one after the other.  The maximum only grows, so a
  // workgroup whose own maximum is not above what it reads there has nothing to add; on ordinary data a handful are.
  const unsigned mine = __builtin_bit_cast(unsigned, m);
  if (mine > __hip_atomic_load((unsigned*)(out + 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
    atomicMax((unsigned*)(out + 1), mine);
}

// partials > 0: out[1] is not set yet, every workgroup takes the maximum of partial[0 .. partials) first.
template <class In, bool kStream>
__global__ __launch_bounds__(256) void quantize_kernel(const void* x, int64_t n, uint8_t* q, float* out, const float* partial,
                                                       int partials) {
  float amax;
  if (partials > 0) {
    float m = 0.f;
    for (int i = threadIdx.x; i < partials; i += 256) m = __builtin_fmaxf(m, partial[i]);
    amax = workgroup_max<4>(m);
  } else {
    amax = out[1];
  }
  const float scale = scale_of(amax);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    out[0] = scale;
    if (partials > 0) out[1] = amax;
  }
  if (markstein_ok(scale)) quantize_all<In, false, kStream>(x, n, q, scale);
  else quantize_all<In, true, kStream>(x, n, q, scale);   // tiny or infinite scales
}

// Small tensors in one launch: every workgroup takes the maximum of the whole tensor, out of its XCD's L2, and then
// quantises its own share.
template <class In>
__global__ __launch_bounds__(1024) void quantize_small_kernel(const void* x, int64_t n, uint8_t* q, float* out) {
  const float amax = workgroup_max<16>(groups_amax<In, 4>(x, n, threadIdx.x, 1024));
  const float scale = scale_of(amax);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    out[0] = scale;
    out[1] = amax;
  }
  const float inv = 1.0f / scale;
  const int64_t thread = (int64_t)blockIdx.x * 1024 + threadIdx.x, stride = (int64_t)gridDim.x * 1024;
  if (markstein_ok(scale)) quantize_groups<In, false>(x, n, q, scale, inv, thread, stride, thread);
  else quantize_groups<In, true>(x, n, q, scale, inv, thread, stride, thread);
}

template <class In>
int run(const void* x, int64_t n, void* q, float* out, float* partial, int64_t partials, hipStream_t stream) {
  if (n * (int64_t)sizeof(typename Load8<In>::Element) <= kSmallBytes) {
    const int64_t want = (n / 8 + 1023) / 1024;
    hipLaunchKernelGGL((quantize_small_kernel<In>), dim3((unsigned)(want < 1 ? 1 : want)), dim3(1024), 0, stream, x, n, (uint8_t*)q, out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
  }
  const int64_t want = (n / 8 + 255) / 256;
  const int64_t most = n * (int64_t)sizeof(typename Load8<In>::Element) <= kL2Bytes ? kQuantizeBlocksInL2 : kQuantizeBlocks;
  const unsigned blocks = (unsigned)(want > most ? most : want);
  if (!partial || partials < 1) {
    hipLaunchKernelGGL(amax_init, dim3(1), dim3(1), 0, stream, out);
    partial = nullptr;
    partials = kAmaxBlocks;
  }
  const unsigned amax_blocks = (unsigned)(blocks < partials ? blocks : partials);
  hipLaunchKernelGGL((amax_kernel<In>), dim3(amax_blocks), dim3(256), 0, stream, x, n, out, partial);
  const auto kernel = n > kStreamElements ? quantize_kernel<In, true> : quantize_kernel<In, false>;
  hipLaunchKernelGGL(kernel, dim3(blocks), dim3(256), 0, stream, x, n, (uint8_t*)q, out, (const float*)partial,
                     partial ? (int)amax_blocks : 0);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace

int64_t quantize_e4m3_partials(int64_t n) { return n <= kSmallBytes / 4 ? 0 : kAmaxBlocks; }

// in_dtype: 0 bf16, 1 fp16, 3 fp32.
int launch_quantize_e4m3(const void* x, int in_dtype, int64_t n, void* q, float* scale_amax, float* partial, int64_t partials,
                         hipStream_t stream) {
  if (partials > kAmaxBlocks) partials = kAmaxBlocks;
  switch (in_dtype) {
    case 0: return run<BF16>(x, n, q, scale_amax, partial, partials, stream);
    case 1: return run<F16>(x, n, q, scale_amax, partial, partials, stream);
    case 3: return run<float>(x, n, q, scale_amax, partial, partials, stream);
  }
  return -1;
}

}  // namespace mi355
