// Quantised products whose rows fit the registers (kernel: mfma_slab_impl.h, one unit per width; launch: mfma_rows.hip): up to 32 rows with contractions of 1024 to 4096, more in groups of
// up to 32 with contractions of 128 to 4096 -- 4096 rows of one matrix, 64 of two or three.
#pragma once
#include "mfma_common.h"

namespace gbx {

// hipErrorInvalidValue: not a shape of this kernel
hipError_t launch_qgemm_slab(const MfmaArgs& a, int bits, bool bf16, hipStream_t s);
template <int BITS> hipError_t launch_slab_bits(const MfmaArgs& a, bool bf16, hipStream_t s);

}  // namespace gbx
