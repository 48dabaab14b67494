// The matrix-core general conv for float activations.
#include "conv_general_mfma.h"

namespace omni_general {

int launch_mfma_f32(const GeneralParams& p, bool transposed, hipStream_t stream) {
  return launch_mfma<float>(p, transposed, stream);
}

}  // namespace omni_general
