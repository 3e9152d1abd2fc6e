// Quantised products of 2 to 32 rows whose slice of the contraction fits the registers (kernel: mfma_slab_impl.h, one unit per width).
#pragma once
#include "mfma_common.h"

namespace gbx {

// hipErrorInvalidValue: not a shape of this kernel.  With a.ws a slice of a.ksplit leaves its fp32 sums in ws[slice][M][N].
hipError_t launch_qgemm_slab(const MfmaArgs& a, int bits, bool bf16, hipStream_t s);
template <int BITS> hipError_t launch_slab_bits(const MfmaArgs& a, bool bf16, hipStream_t s);

}  // namespace gbx
