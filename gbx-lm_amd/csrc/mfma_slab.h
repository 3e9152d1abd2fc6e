// Quantised products of up to 32 rows (one matrix: 1023, in groups) that fit the registers, contractions of 1024 to 4096 (kernel: mfma_slab_impl.h, one unit per width; launch: mfma_rows.hip).
#pragma once
#include "mfma_common.h"

namespace gbx {

// hipErrorInvalidValue: not a shape of this kernel
hipError_t launch_qgemm_slab(const MfmaArgs& a, int bits, bool bf16, hipStream_t s);
template <int BITS> hipError_t launch_slab_bits(const MfmaArgs& a, bool bf16, hipStream_t s);

}  // namespace gbx
