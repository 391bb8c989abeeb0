// Single-group tile kernel (gemm_tn_ring.h), fp16 operands, storing rows of C at any 2-byte alignment.
#include "gemm_tn_ring.h"

namespace mi355 {

int launch_tile_ring_f16_ragged(const GemmArgs& g, int out_dtype, int tile, hipStream_t stream) {
  return out_dtype == 0 ? launch<F16, BF16, true>(g, tile, stream) : launch<F16, F16, true>(g, tile, stream);
}

}  // namespace mi355
