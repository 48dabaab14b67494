// Residual-stack kernels, bf16 weights.
#include "residual_stack.h"

namespace omni_stack {

template int launch_stack96<false>(const StackParams&, int, int, hipStream_t);

}  // namespace omni_stack
