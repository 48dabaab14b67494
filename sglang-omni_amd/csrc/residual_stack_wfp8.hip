// Residual-stack kernels, E4M3 weights.
#include "residual_stack.h"

namespace omni_stack {

template int launch_stack96<true>(const StackParams&, int, int, hipStream_t);

}  // namespace omni_stack
