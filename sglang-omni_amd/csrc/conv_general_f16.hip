// The matrix-core general conv for _Float16 activations.
#include "conv_general_mfma.h"

namespace omni_general {

int launch_mfma_f16(const GeneralParams& p, bool transposed, hipStream_t stream) {
  return launch_mfma<_Float16>(p, transposed, stream);
}

}  // namespace omni_general
