// The small-call residual unit (conv_small.h), 192 channels.
#include "conv_small.h"

namespace omni_conv {

int launch_small_unit(const ConvParams& p, double than, Choice& ch, hipStream_t stream) {
  // 32 positions, weights one group ahead: three groups ahead, or 64 positions, spill
  return launch_small_list<SmallUnitConfig<2, 12, 2>>(p, than, ch, stream);
}

}  // namespace omni_conv
