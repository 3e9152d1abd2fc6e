// 2-bit instantiations of the register-resident rows kernel.
#include "mfma_slab_impl.h"
namespace gbx {
template hipError_t launch_slab_bits<2>(const MfmaArgs& a, bool bf16, hipStream_t s);
}  // namespace gbx
