// Products of few outputs under MI355_VARIANT_AUTO: one workgroup per tile of 16...64 rows and columns, whose waves share out K.
//
// The tile and streaming kernels occupy the CUs with such a product only by cutting K over workgroups, and then a second launch
// adds the partial sums: half of the time of a product that takes 7 us.  Tiles this small are enough of
// them to go round without that, and K is cut inside the workgroup instead: wave w takes the k-steps w, w + waves, ... of all
// rows and columns of the tile, copies them straight into a ring of two stages in LDS that is its own (8 rows of 128 bytes per
// copy, the swizzle of the other kernels), and needs no barrier until the waves' accumulators are added, in the order of the
// waves, at the end.  What bounds it is a CU's intake: (rows + columns) x K bytes per tile at up to 140 KB per us, half of that
// where they come from HBM, and about 2.5 us of launch, first load and reduction; matrix cores are idle most of the time.
// Two stages are as good as three or four, since eight waves keep more lines requested than the L1 has room for
// (105 to 123 lines of 128 bytes per CU), and the LDS they leave holds a second workgroup.
//
// In a replayed graph, operands rotated, before (a K split and its reduction, or 128 x 128 tiles on few CUs) and now: bf16 3 x 1952 x
// 2048 7.0 -> 4.3 us, 66 x 2064 x 768 9.8 -> 4.2, 579 x 208 x 2304 14.4 -> 6.2, e4m3 55 x 2144 x 6144 10.3 -> 7.2, MXFP8 368 x 224 x 2816
// 13.8 -> 5.1, bf16 53 x 1120 x 8448 11.6 -> 13.4 (not taken); calls back to back, fp16 512^3 6.1 -> 4.3, an fp8 layer of 16 x 6144 x
// 4096 with its quantiser 13.6 -> 11.0.  Over 800 problems of M = 1...5800, N = 128...46000, K = 128...14000 the rule of slices_config leaves
// 0.71 of the time before on average, the better choice on each of them 0.70.  Rows of any alignment (kAnyRows) spare such products
// the repacking, or the kernel that computes 4 x 4 outputs per wave: bf16 10 x 10028 x 12846 146 -> 70 us, 112 x 154 x 3092 13.5 -> 5.9,
// fp16 515 x 2050 x 4100 30 -> 26; what bounds them is the same intake, at 50-80 KB per us since most pieces of rows straddle lines.
//
// Counterpart in the reference: none (its launcher rejects shapes that are not multiples of its tile,
// kernels/gemm_kernels/sm90a/gemm_test.cu:33-41); the arithmetic is gemm.cuh:352-377: fp32 accumulation, one rounding.
#include "gemm_launch.h"
#include "ring_common.h"
#include "tile_map.h"

#include <cstdlib>
#include <type_traits>

namespace mi355 {
namespace {

template <class T> struct SliceGeo { typedef Geo<T> type; };
template <> struct SliceGeo<E4M3> { typedef GeoE4M3Rows type; };
template <> struct SliceGeo<MxE4M3> { typedef GeoMxE4M3Rows type; };

constexpr int kDepth = 2;           // stages of a wave's ring
constexpr uint32_t kMxUnit = 512;   // block scales: bytes of one (128 rows, k-step) unit, see gemm_tn_stream.hip

// kMB x kNB blocks of 16 x 16 outputs per workgroup.  kRaggedC: rows of C at any 2-byte alignment (g.c_ragged).
// kAnyRows: rows of A and B at any alignment of their elements.  They cannot be copied straight into LDS then, and go through
// registers instead: global loads of 16 bytes need no alignment on this target, and a wave's accesses to LDS keep their order, so
// that one stage does.  A row has at least 16 bytes (host check).
template <class T, class OutT, int kMB, int kNB, int kWaves, bool kRaggedC, bool kAnyRows>
__global__ __launch_bounds__(64 * kWaves) void gemm_tn_slices(GemmArgs g) {
  typedef typename SliceGeo<T>::type G;
  typedef typename G::Frag Frag;
  static_assert(G::kBlk == 16, "16x16 MFMA blocks");
  constexpr int kSliceChunks = G::kGroups * G::kCpl;
  constexpr int kSlices = 8 / kSliceChunks;
  constexpr bool kMx = G::kMx;
  constexpr int kTm = 16 * kMB, kTn = 16 * kNB;
  constexpr int kDataBytes = (kTm + kTn) * kRowBytes;
  constexpr int kStageBytes = kDataBytes + (kMx ? 512 : 0);
  constexpr int kCopies = (kTm + kTn) / 8;
  constexpr int kVm = kCopies + (kMx ? 2 : 0);
  constexpr int kStages = kAnyRows ? 1 : kDepth;
  constexpr int kRingBytes = kWaves * kStages * kStageBytes, kSumBytes = kWaves * kMB * kNB * 1024;
  static_assert(kVm * (kDepth - 1) < 64, "vmcnt is a 6-bit counter");
  static_assert(kRingBytes <= 160 * 1024 && kSumBytes <= 160 * 1024, "LDS of a CU");
  __shared__ __attribute__((aligned(1024))) uint8_t ring[kRingBytes > kSumBytes ? kRingBytes : kSumBytes];

  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t tiles_m = (uint32_t)g.tiles_m, tiles_n = (uint32_t)g.tiles_n;
  uint32_t tile_m, tile_n;
  tile_coord_t<uint32_t>(blockIdx.x, tiles_m, tiles_n, &tile_m, &tile_n);
  const int64_t m0 = (int64_t)tile_m * kTm, n0 = (int64_t)tile_n * kTn;

  const uint32_t lda_b = (uint32_t)(g.lda * T::kBytes), ldb_b = (uint32_t)(g.ldb * T::kBytes);
  const uint32_t k_bytes = (uint32_t)(g.K * T::kBytes);
  const uint32_t steps = __builtin_amdgcn_readfirstlane((k_bytes + kRowBytes - 1) / kRowBytes);
  const uint32_t tail_bytes = __builtin_amdgcn_readfirstlane(k_bytes % kRowBytes);
  const int64_t rows_x = g.M - m0 < kTm ? g.M - m0 : kTm;
  const int64_t left_n = g.N - n0;
  const int64_t rows_w = left_n < kTn ? left_n : kTn;
  const __amdgpu_buffer_rsrc_t rsrc_x = make_raw_buffer((const uint8_t*)g.A + m0 * (int64_t)lda_b, (uint32_t)((rows_x - 1) * lda_b + k_bytes));
  const __amdgpu_buffer_rsrc_t rsrc_w = make_raw_buffer((const uint8_t*)g.B + n0 * (int64_t)ldb_b, (uint32_t)((rows_w - 1) * ldb_b + k_bytes));
  const uint32_t scale_units_x = kMx ? (uint32_t)((g.M + 255) / 256) * 2u * steps * kMxUnit : 0u;
  const uint32_t scale_units_w = kMx ? (uint32_t)((g.N + 255) / 256) * 2u * steps * kMxUnit : 0u;
  const __amdgpu_buffer_rsrc_t rsrc_sx = make_raw_buffer(g.mx_a, scale_units_x);
  const __amdgpu_buffer_rsrc_t rsrc_sw = make_raw_buffer(g.mx_b, scale_units_w);
  const uint32_t voff_sx = (uint32_t)(m0 / 128) * steps * kMxUnit + lane * 8 + (uint32_t)(m0 % 128) / 64 * 4;
  const uint32_t voff_sw = (uint32_t)(n0 / 128) * steps * kMxUnit + lane * 8 + (uint32_t)(n0 % 128) / 64 * 4;

  const uint32_t r8 = lane >> 3, c8 = lane & 7u;
  const uint32_t ring0 = __builtin_amdgcn_readfirstlane(lds_address(ring) + wave * (kStages * kStageBytes));
  uint32_t voff_x[2], voff_w[2], chunk16[2];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    chunk16[p] = (c8 ^ swizzle(p * 8 + r8)) * 16;
    voff_x[p] = (p * 8 + r8) * lda_b + chunk16[p];
    voff_w[p] = (p * 8 + r8) * ldb_b + chunk16[p];
  }
  // Tiles start their k-steps evenly spread and wrap around, as in the streaming kernel: rows a power of two apart would otherwise
  // be read from the same few memory channels by everybody at once.
  const uint32_t rot = __builtin_amdgcn_readfirstlane(tile_n * steps / tiles_n);
  // The wave's copies of k-step `at`; past the end, as many that fetch nothing (out-of-range offsets), so that one count fits all.
  auto issue_step = [&](uint32_t stage, uint32_t at) __attribute__((always_inline)) {
    uint32_t kk = at + rot;
    kk = kk >= steps ? kk - steps : kk;
    const bool past = at >= steps;
    kk = past ? 0u : kk;
    const uint32_t soff = __builtin_amdgcn_readfirstlane(kk * kRowBytes);
    const bool ragged = tail_bytes != 0 && kk == steps - 1;
    const uint32_t dst = ring0 + stage * kStageBytes;
    uint32_t drop[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) drop[p] = past || (ragged && chunk16[p] >= tail_bytes) ? 0x80000000u : 0u;
#pragma unroll
    for (int c = 0; c < kCopies; ++c) {
      if (c < kTm / 8) dma_16B_to_lds(dst + c * 1024, (voff_x[c & 1] + (uint32_t)(c / 2) * 16u * lda_b) | drop[c & 1], rsrc_x, soff);
      else dma_16B_to_lds(dst + c * 1024, (voff_w[c & 1] + (uint32_t)((c - kTm / 8) / 2) * 16u * ldb_b) | drop[c & 1], rsrc_w, soff);
    }
    if constexpr (kMx) {
      dma_4B_to_lds(dst + kDataBytes, voff_sw, rsrc_sw, kk * kMxUnit);
      dma_4B_to_lds(dst + kDataBytes + 256, voff_sx, rsrc_sx, kk * kMxUnit);
    }
  };

  // Fragments as in gemm_tn_stream.hip.
  const uint32_t rblk = lane & 15u, grp = lane >> 4;
  const uint32_t swz = swizzle(rblk);
  auto frag = [&](const uint8_t* rows, int blk, int s) __attribute__((always_inline)) -> Frag {
    const uint8_t* p = rows + (blk * 16 + rblk) * kRowBytes;
    if constexpr (G::kCpl == 1) {
      return *(const i32x4*)(p + (((uint32_t)(s * kSliceChunks) + grp) ^ swz) * 16);
    } else {
      const i32x4 lo = *(const i32x4*)(p + ((grp ^ swz) * 16));
      const i32x4 hi = *(const i32x4*)(p + (((grp + 4) ^ swz) * 16));
      return (i32x8){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    }
  };

  f32x4 acc[kMB][kNB];
#pragma unroll
  for (int i = 0; i < kMB; ++i)
#pragma unroll
    for (int j = 0; j < kNB; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

  uint8_t* const mine = ring + wave * (kStages * kStageBytes);
  const auto multiply = [&](const uint8_t* base) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < kSlices; ++s) {
      Frag fx[kMB], fw[kNB];
#pragma unroll
      for (int i = 0; i < kMB; ++i) fx[i] = frag(base, i, s);
#pragma unroll
      for (int j = 0; j < kNB; ++j) fw[j] = frag(base + kTm * kRowBytes, j, s);
      if constexpr (kMx) {
        const uint32_t sw = *(const uint32_t*)(base + kDataBytes + lane * 4) >> ((uint32_t)(n0 / 16) % 4u * 8u);
        const uint32_t sx = *(const uint32_t*)(base + kDataBytes + 256 + lane * 4) >> ((uint32_t)(m0 / 16) % 4u * 8u);
        static_for<kMB>([&](auto ic) __attribute__((always_inline)) {
          static_for<kNB>([&](auto jc) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value, j = decltype(jc)::value;
            G::template mfma_scaled_inplace<j, i>(fw[j], fx[i], acc[i][j], sw, sx);
          });
        });
      } else {
#pragma unroll
        for (int i = 0; i < kMB; ++i)
#pragma unroll
          for (int j = 0; j < kNB; ++j) acc[i][j] = G::mfma(fw[j], fx[i], acc[i][j]);
      }
    }
  };
  if constexpr (kAnyRows) {
    typedef typename std::conditional<T::kBytes == 2, uint16_t, uint8_t>::type E;
    const uint8_t* const base_x = (const uint8_t*)g.A + m0 * (int64_t)lda_b;
    const uint8_t* const base_w = (const uint8_t*)g.B + n0 * (int64_t)ldb_b;
    uint32_t off[kCopies];   // rows past the end repeat the last one: nothing of them is stored
#pragma unroll
    for (int c = 0; c < kCopies; ++c) {
      const uint32_t row = c * 8 + r8, last_x = (uint32_t)rows_x - 1, last_w = (uint32_t)rows_w - 1;
      off[c] = (c < kTm / 8 ? (row < last_x ? row : last_x) * lda_b : (row - kTm < last_w ? row - kTm : last_w) * ldb_b) + chunk16[c & 1];
    }
    u32x4 next[kCopies];
    const auto load = [&](uint32_t at) __attribute__((always_inline)) {
      uint32_t kk = at + rot;
      kk = kk >= steps ? kk - steps : kk;
      const uint32_t soff = __builtin_amdgcn_readfirstlane(kk * kRowBytes);
      if (tail_bytes == 0 || kk != steps - 1) {
#pragma unroll
        for (int c = 0; c < kCopies; ++c)
          __builtin_memcpy(&next[c], (const E*)((c < kTm / 8 ? base_x : base_w) + soff + (uint64_t)off[c]), 16);
      } else {
        // Chunks up to the row's end as they are; the one that straddles it from the row's last 16 bytes, moved down; zeros behind.
        const uint32_t drop = 16u - tail_bytes % 16u;   // bytes of a chunk past the row's end; 16: none straddles it
#pragma unroll
        for (int c = 0; c < kCopies; ++c) {
          const uint32_t chunk = chunk16[c & 1];
          const bool whole = chunk + 16 <= tail_bytes, straddles = !whole && chunk < tail_bytes;
          const int64_t to_end = whole ? 0 : (int64_t)tail_bytes - 16 - (int64_t)chunk;
          u32x4 v;
          __builtin_memcpy(&v, (const E*)((c < kTm / 8 ? base_x : base_w) + soff + (uint64_t)off[c] + to_end), 16);
          u32x4 d = v;
          if (drop & 8u) d = (u32x4){d[2], d[3], 0u, 0u};
          if (drop & 4u) d = (u32x4){d[1], d[2], d[3], 0u};
          d = (u32x4){__builtin_amdgcn_alignbyte(d[1], d[0], drop), __builtin_amdgcn_alignbyte(d[2], d[1], drop),
                      __builtin_amdgcn_alignbyte(d[3], d[2], drop), __builtin_amdgcn_alignbyte(0u, d[3], drop)};
#pragma unroll
          for (int i = 0; i < 4; ++i) next[c][i] = whole ? v[i] : straddles ? d[i] : 0u;
        }
      }
    };
    if (wave < steps) load(wave);
    for (uint32_t at = wave; at < steps; at += kWaves) {
#pragma unroll
      for (int c = 0; c < kCopies; ++c) *(u32x4*)(mine + c * 1024 + lane * 16) = next[c];
      if (at + kWaves < steps) load(at + kWaves);
      multiply(mine);
    }
  } else {
    issue_step(0, wave);
    uint32_t stage = 0;
    for (uint32_t at = wave; at < steps; at += kWaves) {
      issue_step(stage ^ 1u, at + kWaves);
      wait_vmcnt<kVm>();
      multiply(mine + stage * kStageBytes);
      wait_lgkmcnt0();   // the reads are back before the next turn refills a stage
      stage ^= 1u;
    }
    wait_vmcnt<0>();
  }
  // the scaled MFMAs are inline assembly: the compiler does not know how long their results take
  if constexpr (kMx) asm volatile("s_nop 15\n\ts_nop 15\n\ts_nop 15" ::: "memory");
  __syncthreads();
  f32x4* const sums = (f32x4*)ring;
#pragma unroll
  for (int i = 0; i < kMB; ++i)
#pragma unroll
    for (int j = 0; j < kNB; ++j) sums[(wave * (kMB * kNB) + i * kNB + j) * 64 + lane] = acc[i][j];
  __syncthreads();
  const float scale = output_scale(g);
#pragma unroll
  for (uint32_t q0 = 0; q0 < kMB * kNB * 64; q0 += 64 * kWaves) {
    const uint32_t q = q0 + tid;
    if (kMB * kNB * 64 % (64 * kWaves) != 0 && q >= kMB * kNB * 64) break;
    f32x4 sum = sums[q];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) sum += sums[w * (kMB * kNB * 64) + q];
    const uint32_t blk = q >> 6, ln = q & 63u;
    const uint32_t m = (blk / kNB) * 16 + (ln & 15u), n = (blk % kNB) * 16 + (ln >> 4) * 4;
    if (m < rows_x && n < rows_w) {
      u32x2 out = Pack4<OutT>::run(sum[0] * scale, sum[1] * scale, sum[2] * scale, sum[3] * scale);
      asm volatile("" : "+v"(out));
      uint16_t* c = (uint16_t*)g.C + (m0 + m) * g.ldc + n0 + n;
      if constexpr (kRaggedC) store_ragged_quad(c, out, left_n - n);
      else *(u32x2*)c = out;
      hold_last(out);
    }
  }
}

// Forms of the kernel: blocks of rows and columns, waves, and what a launch takes (slices_config).
//   us = launch + per_step x k-steps of a wave + round_mb x MB taken in by the busiest CU were the tiles of one round spread evenly
//        + mean_mb x MB taken in by the mean CU + unique_mb x MB of operands + round x further rounds of resident workgroups
// Least squares (relative error) over 740-800 problems each, 60 % of them fitted and the rest predicted equally well (7-10 % rms).
struct Form {
  int mb, nb, waves;
  double launch, per_step, round_mb, mean_mb, unique_mb, round;
};
constexpr Form kForms[] = {
    {1, 1, 4, 2.54, 0.081, 5.70, 4.26, 0.090, 1.54}, {1, 1, 8, 2.77, 0.082, 4.35, 5.15, 0.083, 1.47},
    {1, 2, 4, 2.63, 0.051, 6.83, 2.93, 0.107, 1.49}, {2, 2, 2, 2.56, 0.160, 6.01, 3.92, 0.078, 2.49},
    {2, 2, 4, 2.79, 0.085, 5.76, 4.26, 0.087, 1.63}, {2, 4, 4, 3.08, 0.178, 4.55, 5.30, 0.088, 2.00},
    {4, 4, 4, 3.74, 0.281, 5.08, 6.84, 0.036, 2.68}};

// With rows of any alignment (420 problems, 9-12 % rms): a CU takes in less, as most pieces of rows straddle cache lines (rows at
// multiples of 4 bytes and more as below, of 2 bytes 1.25 times the MB, of 1 byte 1.6 times).
constexpr Form kAnyRowsForms[] = {
    {1, 1, 4, 2.41, 0.158, 10.1, 3.56, 0.080, 0.65}, {1, 1, 8, 2.74, 0.010, 11.7, 1.83, 0.089, 0.88},
    {1, 2, 4, 2.61, 0.089, 11.4, 3.21, 0.105, 0.56}, {2, 2, 2, 2.65, 0.239, 9.87, 4.95, 0.068, 1.50},
    {2, 2, 4, 2.97, 0.069, 11.1, 3.70, 0.087, 1.09}, {4, 4, 4, 4.32, 0.158, 10.8, 5.78, 0.071, 2.95},
    {5, 4, 4, 4.67, 0.224, 10.5, 7.01, 0.043, 3.19}};

constexpr int64_t kCuSlots = 256;
int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

double form_us(const Form& f, int stages, int64_t M, int64_t N, int64_t steps, bool mx, double intake = 1.0) {
  const int64_t tiles = ceil_div(M, 16 * f.mb) * ceil_div(N, 16 * f.nb);
  const int64_t lds = (int64_t)f.waves * stages * (16 * (f.mb + f.nb) * kRowBytes + (mx ? 512 : 0));
  const int64_t by_lds = 163840 / lds, by_waves = 32 / f.waves, resident = by_lds < by_waves ? by_lds : by_waves;
  const double tile_mb = intake * 16e-6 * (f.mb + f.nb) * kRowBytes * (double)steps;
  return f.launch + f.per_step * (double)ceil_div(steps, f.waves) + f.round_mb * (double)ceil_div(tiles, kCuSlots) * tile_mb +
         f.mean_mb * (double)tiles / kCuSlots * tile_mb + f.unique_mb * 1e-6 * kRowBytes * (double)((M + N) * steps) +
         f.round * (double)(ceil_div(tiles, kCuSlots * resident) - 1);
}

// The shortest of `n` forms and its estimate.
int shortest_form(const Form* forms, int n, int stages, int64_t M, int64_t N, int64_t steps, bool mx, double intake, double* us) {
  int best = 0;
  for (int f = 0; f < n; ++f) {
    const double e = form_us(forms[f], stages, M, N, steps, mx, intake);
    if (f == 0 || e < *us) {
      *us = e;
      best = f;
    }
  }
  return best;
}
constexpr int kFormCount = sizeof(kForms) / sizeof(kForms[0]), kAnyRowsFormCount = sizeof(kAnyRowsForms) / sizeof(kAnyRowsForms[0]);

// The same for the route the problem takes otherwise, fitted on the same problems (5-9 % rms): the streaming kernel or 128 x 128
// tiles, with or without a K split.
double other_us(const SlicesAlternative& o, int64_t M, int64_t N, int64_t steps) {
  const int64_t tiles = ceil_div(M, o.tile_rows) * ceil_div(N, o.tile_cols), items = tiles * o.splits, item_steps = ceil_div(steps, o.splits);
  const double unique_mb = 1e-6 * kRowBytes * (double)((M + N) * steps), planes_mb = 4e-6 * (double)(o.splits * M * N);
  const double rounds = (double)ceil_div(items, kCuSlots), round_steps = rounds * (double)item_steps, mean_steps = (double)items / kCuSlots * (double)item_steps;
  if (o.streams) {
    const double step_mb = 1e-6 * kRowBytes * (double)(o.tile_rows + o.tile_cols);
    if (o.splits == 1) return 3.01 + (20.5 * round_steps + 12.5 * mean_steps) * step_mb;
    return 4.79 + 22.6 * round_steps * step_mb + 0.051 * unique_mb + 0.507 * planes_mb + 0.021 * (double)item_steps;
  }
  if (o.splits == 1) return 0.379 * round_steps + 0.009 * mean_steps + 0.0645 * unique_mb + 3.90 * rounds + 0.265e-6 * 2.0 * (double)(M * N);
  return 4.98 + 0.479 * round_steps + 0.108 * unique_mb + 0.323 * planes_mb;
}

template <class T, class OutT, bool kAnyRows, int kForm>
int launch_form(GemmArgs g, hipStream_t stream) {
  constexpr Form f = kAnyRows ? kAnyRowsForms[kForm] : kForms[kForm];
  g.tiles_m = (g.M + 16 * f.mb - 1) / (16 * f.mb);
  g.tiles_n = (g.N + 16 * f.nb - 1) / (16 * f.nb);
  const dim3 grid((unsigned)(g.tiles_m * g.tiles_n)), threads(64 * f.waves);
  if constexpr (!std::is_same<T, MxE4M3>::value) {
    if (kAnyRows || g.c_ragged) {   // one form for every C beside rows of A and B of any alignment
      hipLaunchKernelGGL((gemm_tn_slices<T, OutT, f.mb, f.nb, f.waves, true, kAnyRows>), grid, threads, 0, stream, g);
      return hipGetLastError() == hipSuccess ? 0 : -1;
    }
  }
  if constexpr (!kAnyRows) hipLaunchKernelGGL((gemm_tn_slices<T, OutT, f.mb, f.nb, f.waves, false, false>), grid, threads, 0, stream, g);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <class T, class OutT, bool kAnyRows>
int launch_any(const GemmArgs& g, int form, hipStream_t s) {
  static_assert(kFormCount == 7 && kAnyRowsFormCount == 7, "one case per form");
  switch (form) {
    case 0: return launch_form<T, OutT, kAnyRows, 0>(g, s);
    case 1: return launch_form<T, OutT, kAnyRows, 1>(g, s);
    case 2: return launch_form<T, OutT, kAnyRows, 2>(g, s);
    case 3: return launch_form<T, OutT, kAnyRows, 3>(g, s);
    case 4: return launch_form<T, OutT, kAnyRows, 4>(g, s);
    case 5: return launch_form<T, OutT, kAnyRows, 5>(g, s);
    case 6: return launch_form<T, OutT, kAnyRows, 6>(g, s);
  }
  return -1;
}

template <class T, bool kAnyRows>
int launch_out(const GemmArgs& g, int out_dtype, int form, hipStream_t s) {
  return out_dtype == 0 ? launch_any<T, BF16, kAnyRows>(g, form, s) : launch_any<T, F16, kAnyRows>(g, form, s);
}

bool on_this_route(const SlicesAlternative& other) { return other.streams || other.tile_rows <= 128; }

}  // namespace

// Rows of B of more than 32 MiB (48 MiB up to 16 rows of A) are left to the streaming kernel, which HBM bounds there as it would this
// one (M <= 16: 10-20 % faster here between 24 and 48 MiB, 4 % from there to 90).  MI355_RING_TILE, which forces a tile for
// measurements, keeps problems off this kernel as well.
double slices_us(int64_t M, int64_t N, int64_t K, int elem_bytes, bool mx, int* form) {
  *form = -1;
  if (M <= 0 || N <= 0 || K <= 0 || (double)M * (double)N * (double)K > kSlicesMaxProducts || (double)M * (double)N > kSlicesMaxOutputs) return 1e30;
  if ((double)N * (double)K * elem_bytes > (M <= 16 ? 48.0 : 32.0) * 1048576.0 || std::getenv("MI355_RING_TILE")) return 1e30;
  double us = 0;
  *form = shortest_form(kForms, kFormCount, kDepth, M, N, ceil_div(K * elem_bytes, kRowBytes), mx, 1.0, &us);
  return us;
}

// Taken where the estimate is 15 % below the other route's, and not where the plan has tiles of 256 rows.  Of the 800 problems, 8 are
// more than 2 % slower than on the other route (10 % at most; with a tenth below, 17 and 33 %, and 0.704 for 0.707 of the time).
int slices_config(int64_t M, int64_t N, int64_t K, int elem_bytes, bool mx, const SlicesAlternative& other, double* route_us) {
  const int64_t steps = ceil_div(K * elem_bytes, kRowBytes);
  const double limit = on_this_route(other) ? other_us(other, M, N, steps) : ring_shortest_us(M, N, K, elem_bytes);
  if (route_us) *route_us = limit;
  if (!on_this_route(other)) return -1;
  int form;
  const double us = slices_us(M, N, K, elem_bytes, mx, &form);
  if (us >= 0.85 * limit) return -1;
  if (route_us) *route_us = us;
  return form;
}

// The other route of a product with rows of any alignment is `other` (or this kernel, whichever is shorter) behind a repacking of
// `copied` bytes: us = 6.4 + 0.36 x MB + 0.75 x product + 0.25 x million outputs (296 problems, 11 % rms).  Taken from 0.97 of it:
// 0.66 of the time before on average over those, as the better choice on each would leave, 4 of them 4-24 % slower; with more than four
// million outputs, whose stores the estimate does not know, not at all (e4m3 4150 x 4115 x 174 32.5 us repacked, 40.9 as it is).  Small 16-bit
// products (copied == 0) have none but one thread or a sixteenth of a wave per output, which was slower on all of 124 problems.
int slices_any_rows_config(int64_t M, int64_t N, int64_t K, int elem_bytes, int alignment, int64_t copied, const SlicesAlternative& other) {
  if (M <= 0 || N <= 0 || K * elem_bytes < 16 || (double)M * (double)N * (double)K > kSlicesMaxProductsAnyRows) return -1;
  if (std::getenv("MI355_RING_TILE")) return -1;
  double us = 0, product = 0;
  const int form = shortest_form(kAnyRowsForms, kAnyRowsFormCount, 1, M, N, ceil_div(K * elem_bytes, kRowBytes), false,
                                 alignment % 4 == 0 ? 1.0 : alignment % 2 == 0 ? 1.25 : 1.6, &us);
  if (copied == 0) return form;
  if ((double)M * (double)N > kSlicesMaxOutputsAnyRows) return -1;
  slices_config(M, N, K, elem_bytes, false, other, &product);
  return us < 0.97 * (6.44 + 0.357e-6 * (double)copied + 0.751 * product + 0.25e-6 * (double)M * (double)N) ? form : -1;
}

int launch_slices(const GemmArgs& g, int in_dtype, int out_dtype, int config, hipStream_t stream) {
  switch (in_dtype) {
    case 0: return launch_out<BF16, false>(g, out_dtype, config, stream);
    case 1: return launch_out<F16, false>(g, out_dtype, config, stream);
    case 2: return g.mx_a ? launch_out<MxE4M3, false>(g, out_dtype, config, stream) : launch_out<E4M3, false>(g, out_dtype, config, stream);
  }
  return -1;
}

int launch_slices_any_rows(const GemmArgs& g, int in_dtype, int out_dtype, int config, hipStream_t stream) {
  switch (in_dtype) {
    case 0: return launch_out<BF16, true>(g, out_dtype, config, stream);
    case 1: return launch_out<F16, true>(g, out_dtype, config, stream);
    case 2: return launch_out<E4M3, true>(g, out_dtype, config, stream);
  }
  return -1;
}

}  // namespace mi355
