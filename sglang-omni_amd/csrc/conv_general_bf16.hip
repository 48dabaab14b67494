// The matrix-core general conv for __bf16 activations.
#include "conv_general_mfma.h"

namespace omni_general {

int launch_mfma_bf16(const GeneralParams& p, bool transposed, hipStream_t stream) {
  return launch_mfma<__bf16>(p, transposed, stream);
}

}  // namespace omni_general
