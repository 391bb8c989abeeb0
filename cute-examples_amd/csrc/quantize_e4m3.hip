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
// 47.7 us long on its divisions, see codes4), but for those that the chip holds: 41.8 us (quantize_resident_kernel).  The reference
// has no fp8 path;
// the contract is the benchmark configuration's (operands quantised with per-tensor fp32 scales
// amax/448) and is checked against torch's float8_e4m3fn cast and the C restatement in the tests.
#include "cdna4_primitives.h"
#include "gemm_launch.h"
#include "quantize_convert.h"
#include "ring_common.h"

#include <cstdlib>

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

// x / scale for four elements -> four codes, the same bits whichever way is taken.
//   kDivide     the IEEE division: about a dozen instructions, one of them quarter rate, per element; alone it takes longer
//             than the memory traffic of the pass (bf16 8192 x 8192: 47.7 us of vector instructions)
//   kCorrected  Markstein's correction (IBM J. Res. Dev. 34, 1990) of x * y, y = 1 / scale correctly rounded: with
//             r = x - (x*y) * scale, which one fused multiply-add gives exactly, x*y + r*y is the correctly rounded quotient:
//             three instructions.  It needs r free of underflow for every quotient that does not round to code 0 (from 2^-11 on
//             r is a multiple of 2^-57 times scale), hence the range of `scale` in markstein_ok.  The sign is taken from x (a
//             negative zero would lose it).  amax is finite here, so no quotient exceeds 448 * (1 + 2^-23), which the
//             conversion rounds to 448: no clamp.  NaN stays NaN through all of it.
__device__ __forceinline__ bool markstein_ok(float scale) { return scale >= 0x1p-60f && scale <= 0x1p100f; }

//   kProduct, kTwoProducts  for 16-bit x without NaN, see factors_for
enum Quotient { kDivide, kCorrected, kProduct, kTwoProducts };
// inv: 1 / scale, or factors_for's first factor; `more` its second.
template <Quotient kQuotient>
__device__ __forceinline__ uint32_t codes4(const float* v, float scale, float inv, float more = 0.f) {
  if constexpr (kQuotient == kProduct) {
    return to_e4m3x4_numbers(v[0] * inv, v[1] * inv, v[2] * inv, v[3] * inv);
  } else if constexpr (kQuotient == kTwoProducts) {
    return to_e4m3x4_numbers(__builtin_fmaf(v[0], inv, v[0] * more), __builtin_fmaf(v[1], inv, v[1] * more),
                             __builtin_fmaf(v[2], inv, v[2] * more), __builtin_fmaf(v[3], inv, v[3] * more));
  } else if constexpr (kQuotient == kDivide) {
    return to_e4m3x4(v[0] / scale, v[1] / scale, v[2] / scale, v[3] / scale);
  } else {
    float q[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float q0 = v[k] * inv;
      const float r = __builtin_fmaf(-q0, scale, v[k]);
      q[k] = __builtin_copysignf(__builtin_fmaf(r, inv, q0), v[k]);
    }
    return to_e4m3x4_bounded(q[0], q[1], q[2], q[3]);
  }
}
template <bool kDivides>
__device__ __forceinline__ u32x2 codes_of(const float (&v)[8], float scale, float inv) {
  constexpr Quotient kQuotient = kDivides ? kDivide : kCorrected;
  return (u32x2){codes4<kQuotient>(v, scale, inv), codes4<kQuotient>(v + 4, scale, inv)};
}

// The codes of 16-bit x without NaN from one or two products per element (x * first, or x * first + x * more, rounded once, where
// first + more is 1 / scale to 48 bits) instead of the corrected quotient.  They are off the quotient by less than 2^-21.9 of it, which
// changes a code only if one of the codes' midpoints (odd m up to 31 times a power of two) lies that close to x / scale, that is, m *
// scale that close to a value of so few bits as x has: at most one value per m (they are 2^-11 apart), and which side of the midpoint
// it falls on does not depend on its power of two.  So those sixteen values are tried against the corrected quotient, with four first
// factors within two units of the last place of 1 / scale and with the two products; what agrees on all sixteen will do for every x.
// (m = 7 always is such a case, amax / 448 being amax / 7 but for a power of two.  One of the four factors does for 94 % of all amax.)
// markstein_ok keeps the factors normal; a quotient below that rounds to a zero of x's sign either way, since more is not negative.
struct Factors {
  float first, more;   // first == 0: none
};
template <class In>
__device__ __forceinline__ Factors factors_for(float scale, float inv) {
  constexpr uint32_t kDropped = 24 - (std::is_same<In, BF16>::value ? 8 : 11);   // bits of a significand that x does not have
  const uint32_t lane = threadIdx.x & 63u, pick = lane >> 4;
  const float p = (float)(int)(2 * (lane & 15u) + 1) * scale * 0x1p-10f;
  const uint32_t near = (__builtin_bit_cast(uint32_t, p) + (1u << (kDropped - 1))) & ~((1u << kDropped) - 1);
  const float x = __builtin_bit_cast(float, near);
  const auto ulps = [&](int n) { return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, inv) + (uint32_t)n); };
  const auto candidate = [&](uint32_t c) { return ulps(c == 3 ? 2 : c == 2 ? -1 : (int)c); };
  const float v[4] = {x, x, x, x};
  const uint32_t want = codes4<kCorrected>(v, scale, inv);
  const uint64_t agree = __ballot(codes4<kProduct>(v, scale, candidate(pick)) == want);
  for (uint32_t c = 0; c < 4; ++c)
    if ((agree >> (16 * c) & 0xffffu) == 0xffffu) return {candidate(c), 0.f};
  const float below = __builtin_fmaf(-inv, scale, 1.0f) < 0.f ? ulps(-1) : inv;   // the largest number not above 1 / scale
  const float more = __builtin_fmaf(-below, scale, 1.0f) * inv;
  return {__all(codes4<kTwoProducts>(v, scale, below, more) == want) ? below : 0.f, more};
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

// Tensors of kResidentFrom bytes to what the chip holds, read once.  One workgroup per CU keeps its pieces of 8 KiB on the chip
// between the maximum and the codes, 48 in registers (192 of a lane's 256) and 16 in LDS: 512 KiB per CU, 128 MiB in all.  Between the
// two halves every workgroup waits for the maxima of all others, one word each in `slots`.  That they all run at the same time is how
// the chip fills when nothing else does; it is not relied on: the wait is bounded by about what the second read costs (40 us, ten
// times the usual wait), and a workgroup that gives up leaves its pieces to quantize_left_kernel behind it, which finds nothing to do
// otherwise.  A stream with a CU mask, where workgroups would always be waiting for others that cannot start, reads twice (has_all_cus;
// bf16 8192 x 8192 on 255, 224 or 128 CUs 53 us, 115...119 this way, 275 with a bound of 200 us).  Beside other work, this against two
// reads (us): two such quantisers on two streams 74 / 99 the pair, two beside a bf16 4096^3 product 170 / 190 in all, six beside products
// of several rounds (8192^3, 8192^2 x 1024, 4352^2 x 4096, 8192 x 16384 x 256) 0.90...1.02 of the time in all, 2048 x 14336 x 4096 1.06...1.12.
// bf16 8192 x 8192 (128 MiB) 53.4 -> 41.8 us, of which reading 20, waiting 4, codes 11 (19 with the corrected quotient, see factors_for),
// the two small launches around it 5; 96 MiB 41.2 -> 34.6, 80 MiB 35.7 -> 31.1, 64 MiB 30.8 / 30.1, 32 MiB 16.6 / 23.8; fp32 128 MiB 52.7 ->
// 40.3, 80 MiB 33.2 -> 30.2, 64 MiB 28.2 / 29.3; with a part of 224 MiB read twice 89.5 / 104.  fp8 layer 8192^3 421 -> 406 us.
constexpr int kHeld = 48, kHeldInLds = 16, kResident = kHeld + kHeldInLds, kResidentThreads = 512, kResidentBlocks = 256;
constexpr int64_t kResidentFrom = (int64_t)80 << 20;
constexpr int64_t kWaitTicks = 4000;       // of the 100 MHz clock: 40 us
constexpr uint32_t kUnset = 0xffffffffu;   // no maximum: those are numbers, this is the pattern of a NaN
typedef __attribute__((ext_vector_type(32))) uint32_t u32x32;

template <class In> struct Chunk {   // 16 bytes of x
  static constexpr int kPer = 16 / sizeof(typename Load8<In>::Element);
  static __device__ __forceinline__ void decode(u32x4 a, float* v) {
    if constexpr (std::is_same<In, float>::value) {
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = __builtin_bit_cast(float, (uint32_t)a[k] + 0u);   // (of an element itself, the first one's bits)
    } else if constexpr (std::is_same<In, BF16>::value) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        v[2 * k] = __builtin_bit_cast(float, a[k] << 16);
        v[2 * k + 1] = __builtin_bit_cast(float, a[k] & 0xffff0000u);
      }
    } else {
      const f16x8 h = __builtin_bit_cast(f16x8, a);
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = (float)h[k];
    }
  }
  static __device__ __forceinline__ float amax(u32x4 a, float m) {
    float v[kPer];
    decode(a, v);
#pragma unroll
    for (int k = 0; k < kPer; ++k) m = __builtin_fmaxf(m, __builtin_fabsf(v[k]));
    return m;
  }
  // Chunk `tid` of piece `piece`: the piece's address is the workgroup's, the chunk's a lane's 32-bit offset.
  static __device__ __forceinline__ u32x4 load(const void* x, int64_t piece, uint32_t tid) {
    return ((const u32x4*)x + piece * kResidentThreads)[tid];
  }
  template <Quotient kQuotient>
  static __device__ __forceinline__ void store(uint8_t* q, int64_t piece, uint32_t tid, u32x4 a, float scale, float inv, float more = 0.f) {
    float v[kPer];
    decode(a, v);
    // Written through the L2s and past the Infinity Cache (nt sc1), at once: what the L2s still hold when the kernel ends, the next one
    // waits for, and lines left in the Infinity Cache cost other passes 8 us (bf16 8192 x 8192 43.7 or 51.5 us, by what came before;
    // written through 41.3).
    const __amdgpu_buffer_rsrc_t to = make_raw_buffer(q + piece * (kResidentThreads * kPer), kResidentThreads * kPer);
    const uint32_t low = codes4<kQuotient>(v, scale, inv, more);
    if constexpr (kPer == 8) __builtin_amdgcn_raw_buffer_store_b64((u32x2){low, codes4<kQuotient>(v + 4, scale, inv, more)}, to, tid * 8, 0, 18);
    else __builtin_amdgcn_raw_buffer_store_b32(low, to, tid * 4, 0, 18);
  }
};

// The largest magnitude of chunks.  16-bit values by their bits, two at a time (for magnitudes the order of the bits is that of the
// numbers, with NaN above infinity): half the instructions of the decoded ones.
template <class In> struct Largest {
  typedef __attribute__((ext_vector_type(2))) uint16_t u16x2;
  u16x2 most = {0, 0};
  __device__ __forceinline__ void add(u32x4 a) {
#pragma unroll
    for (int k = 0; k < 4; ++k) most = __builtin_elementwise_max(most, __builtin_bit_cast(u16x2, (uint32_t)(a[k] & 0x7fff7fffu)));
  }
  __device__ __forceinline__ uint16_t bits() const { return most[0] > most[1] ? most[0] : most[1]; }
  __device__ __forceinline__ bool has_nan() const { return bits() > (std::is_same<In, BF16>::value ? 0x7f80 : 0x7c00); }
  __device__ __forceinline__ float value() const {
    const uint16_t b = bits();
    return Decode<In>::run(&b, 0);
  }
};
template <> struct Largest<float> {
  float most = 0.f;
  __device__ __forceinline__ void add(u32x4 a) { most = Chunk<float>::amax(a, most); }
  __device__ __forceinline__ bool has_nan() const { return false; }   // ignored by add, put right by the conversion
  __device__ __forceinline__ float value() const { return most; }
};

// Pieces of workgroup b of `blocks`: b, b + blocks, ...  Whole pieces only; the elements behind the last one are workgroup 0's.
template <class In>
__device__ __forceinline__ int64_t pieces_of(int64_t n, int64_t b, int64_t blocks) {
  const int64_t pieces = n / (Chunk<In>::kPer * kResidentThreads);
  return (pieces - b + blocks - 1) / blocks;
}

template <class In, Quotient kQuotient>
__device__ __forceinline__ void quantize_pieces(const void* x, int64_t n, uint8_t* q, float scale, float inv, int64_t mine) {
#pragma unroll 4
  for (int64_t i = 0; i < mine; ++i) {
    const int64_t piece = i * gridDim.x + blockIdx.x;
    Chunk<In>::template store<kQuotient>(q, piece, threadIdx.x, Chunk<In>::load(x, piece, threadIdx.x), scale, inv);
  }
}
template <class In>
__device__ __forceinline__ void quantize_rest(const void* x, int64_t n, uint8_t* q, float scale) {
  if (blockIdx.x != 0) return;
  constexpr int64_t kPiece = Chunk<In>::kPer * kResidentThreads;
  for (int64_t i = n / kPiece * kPiece + threadIdx.x; i < n; i += kResidentThreads) q[i] = (uint8_t)to_e4m3(Load8<In>::one(x, i) / scale);
}

__global__ __launch_bounds__(2 * kResidentBlocks) void resident_init(uint32_t* slots) { slots[threadIdx.x] = threadIdx.x < kResidentBlocks ? kUnset : 0u; }

// slots: kResidentBlocks maxima, then as many words that say whose pieces are done.
template <class In>
__global__ __launch_bounds__(kResidentThreads, 2) void quantize_resident_kernel(const void* x, int64_t n, uint8_t* q, float* out,
                                                                                uint32_t* slots, int64_t wait_ticks) {
  __shared__ __attribute__((aligned(1024))) uint8_t kept[kHeldInLds * kResidentThreads * 16];
  const int64_t b = blockIdx.x, blocks = gridDim.x, mine = pieces_of<In>(n, b, blocks);
  const uint32_t tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const auto piece = [&](int64_t i) __attribute__((always_inline)) { return i * blocks + b; };

  Largest<In> most;
  // kResident pieces; past the workgroup's last one, that one again.
  const int64_t step = blocks * (kResidentThreads * 16);   // bytes from one of the workgroup's pieces to its next
  const uint8_t* from = (const uint8_t*)x + b * (kResidentThreads * 16);
  int left = (int)mine - 1;
  const auto next = [&]() __attribute__((always_inline)) {
    const uint8_t* p = from;
    from += left > 0 ? step : 0;
    --left;
    return p;
  };
  u32x32 held[kHeld / 8];
#pragma unroll
  for (int j = 0; j < kHeld; ++j) {
    const u32x4 a = ((const u32x4*)next())[tid];
#pragma unroll
    for (int k = 0; k < 4; ++k) held[j / 8][j % 8 * 4 + k] = a[k];
  }
#pragma unroll
  for (int j = 0; j < kHeldInLds; ++j)
    dma_16B_to_lds(__builtin_amdgcn_readfirstlane(lds_address(kept) + j * (kResidentThreads * 16) + wave * 1024), tid * 16,
                   make_raw_buffer(next(), kResidentThreads * 16), 0);
#pragma unroll
  for (int g = 0; g < kHeld / 8; ++g) {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      most.add((u32x4){held[g][4 * j], held[g][4 * j + 1], held[g][4 * j + 2], held[g][4 * j + 3]});
    asm volatile("" : "+v"(held[g]));   // what is kept are the chunks, not their elements
  }
  wait_vmcnt<0>();
  const u32x4* const in_lds = (const u32x4*)kept + tid;   // a lane reads what its own copies brought
#pragma unroll 4
  for (int j = 0; j < kHeldInLds; ++j) most.add(in_lds[j * kResidentThreads]);
  const bool numbers = !__syncthreads_or(most.has_nan());
  float m = most.value();
  if (!numbers) {   // the maximum of the numbers among them
    m = 0.f;
    for (int64_t i = 0; i < mine; ++i) m = Chunk<In>::amax(Chunk<In>::load(x, piece(i), tid), m);
  }
  if (b == 0) {
    constexpr int64_t kPiece = Chunk<In>::kPer * kResidentThreads;
    for (int64_t i = n / kPiece * kPiece + tid; i < n; i += kResidentThreads) m = __builtin_fmaxf(m, __builtin_fabsf(Load8<In>::one(x, i)));
  }
  m = workgroup_max<8>(m);
  if (tid == 0) __hip_atomic_store(slots + b, __builtin_bit_cast(uint32_t, m), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

  // The values travel in the words themselves, so no order with other memory is needed.
  uint32_t theirs = 0;
  if (tid < blocks) {
    const int64_t until = (int64_t)__builtin_amdgcn_s_memrealtime() + wait_ticks;
    for (;;) {
      theirs = __hip_atomic_load(slots + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (theirs != kUnset || (int64_t)__builtin_amdgcn_s_memrealtime() >= until) break;
      __builtin_amdgcn_s_sleep(1);
    }
  }
  if (!__syncthreads_and(theirs != kUnset)) return;
  const float amax = workgroup_max<8>(__builtin_bit_cast(float, theirs)), scale = scale_of(amax), inv = 1.0f / scale;
  if (tid == 0) {
    slots[kResidentBlocks + b] = 1u;
    if (b == 0) {
      out[0] = scale;
      out[1] = amax;
    }
  }
  const auto store_all = [&](auto quotient, float inv, float more) __attribute__((always_inline)) {
    constexpr Quotient kQuotient = decltype(quotient)::value;
    // loops over registers by a scalar index: unrolled, these are tens of KB of code that run once
#pragma unroll
    for (int g = 0; g < kHeld / 8; ++g) {
#pragma unroll 2
      for (int j = 0; j < 8; ++j) {
        const u32x4 a = {held[g][4 * j], held[g][4 * j + 1], held[g][4 * j + 2], held[g][4 * j + 3]};
        if (8 * g + j < mine) Chunk<In>::template store<kQuotient>(q, piece(8 * g + j), tid, a, scale, inv, more);
      }
    }
#pragma unroll 2
    for (int j = 0; j < kHeldInLds; ++j)
      if (kHeld + j < mine) Chunk<In>::template store<kQuotient>(q, piece(kHeld + j), tid, in_lds[j * kResidentThreads], scale, inv, more);
  };
  Factors f = {0.f, 0.f};
  if constexpr (!std::is_same<In, float>::value)
    if (numbers && markstein_ok(scale)) f = factors_for<In>(scale, inv);
  if (!markstein_ok(scale)) {   // tiny or infinite scales
    quantize_pieces<In, kDivide>(x, n, q, scale, inv, mine);
  } else if constexpr (std::is_same<In, float>::value) {
    store_all(std::integral_constant<Quotient, kCorrected>{}, inv, 0.f);
  } else if (f.first != 0.f && f.more == 0.f) {
    store_all(std::integral_constant<Quotient, kProduct>{}, f.first, 0.f);
  } else if (f.first != 0.f) {
    store_all(std::integral_constant<Quotient, kTwoProducts>{}, f.first, f.more);
  } else {
    quantize_pieces<In, kCorrected>(x, n, q, scale, inv, mine);
  }
  quantize_rest<In>(x, n, q, scale);
}

template <class In>
__global__ __launch_bounds__(kResidentThreads) void quantize_left_kernel(const void* x, int64_t n, uint8_t* q, float* out, const uint32_t* slots) {
  if (slots[kResidentBlocks + blockIdx.x]) return;
  const float amax = workgroup_max<8>(threadIdx.x < gridDim.x ? __builtin_bit_cast(float, slots[threadIdx.x]) : 0.f);
  const float scale = scale_of(amax), inv = 1.0f / scale;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    out[0] = scale;
    out[1] = amax;
  }
  const int64_t mine = pieces_of<In>(n, blockIdx.x, gridDim.x);
  if (markstein_ok(scale)) quantize_pieces<In, kCorrected>(x, n, q, scale, inv, mine);
  else quantize_pieces<In, kDivide>(x, n, q, scale, inv, mine);
  quantize_rest<In>(x, n, q, scale);
}

// Whether the stream's kernels may run on all `cus` compute units; false where that cannot be told.
bool has_all_cus(hipStream_t stream, int64_t cus) {
  uint32_t mask[32] = {};
  if (hipExtStreamGetCUMask(stream, 32, mask) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  int64_t on = 0;
  for (const uint32_t word : mask) on += __builtin_popcount(word);
  return on >= cus;
}

template <class In>
int run_resident(const void* x, int64_t n, void* q, float* out, uint32_t* slots, hipStream_t stream) {
  const char* wait = std::getenv("MI355_QUANTIZE_WAIT_US");   // for tests, up to the bound: 0 has the second kernel do what is left
  const int64_t asked = wait ? std::atoll(wait) : kWaitTicks / 100, ticks = asked < kWaitTicks / 100 ? asked * 100 : kWaitTicks;
  const dim3 grid((unsigned)compute_units());   // at most kResidentBlocks (run)
  hipLaunchKernelGGL(resident_init, dim3(1), dim3(2 * kResidentBlocks), 0, stream, slots);
  hipLaunchKernelGGL((quantize_resident_kernel<In>), grid, dim3(kResidentThreads), 0, stream, x, n, (uint8_t*)q, out, slots, ticks);
  hipLaunchKernelGGL((quantize_left_kernel<In>), grid, dim3(kResidentThreads), 0, stream, x, n, (uint8_t*)q, out, (const uint32_t*)slots);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <class In>
int run(const void* x, int64_t n, void* q, float* out, float* partial, int64_t partials, hipStream_t stream) {
  if (n * (int64_t)sizeof(typename Load8<In>::Element) <= kSmallBytes) {
    const int64_t want = (n / 8 + 1023) / 1024;
    hipLaunchKernelGGL((quantize_small_kernel<In>), dim3((unsigned)(want < 1 ? 1 : want)), dim3(1024), 0, stream, x, n, (uint8_t*)q, out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
  }
  const int64_t bytes = n * (int64_t)sizeof(typename Load8<In>::Element);
  if (bytes >= kResidentFrom && partial && partials >= 2 * kResidentBlocks) {
    const int64_t cus = compute_units();
    if (cus <= kResidentBlocks && bytes < cus * kResident * kResidentThreads * 16 + kResidentThreads * 16 &&   // whole pieces fit
        has_all_cus(stream, cus))
      return run_resident<In>(x, n, q, out, (uint32_t*)partial, stream);
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
