// Head dim 128, fp16: see fa2_d128_kernel.h.

#include "fa2_d128_kernel.h"

namespace fl {

hipError_t launch_d128_f16(const FwdArgs& a, int cfg, hipStream_t stream) {
  return launch_d128_t<_Float16>(a, cfg, stream);
}

}  // namespace fl
