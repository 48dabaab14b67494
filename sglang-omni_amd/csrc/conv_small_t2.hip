// The small-call convolution kernels (conv_small.h) of 2 taps.
#include "conv_small.h"

namespace omni_conv {

int launch_small_taps2(const ConvParams& p, double than, Choice& ch, hipStream_t stream) {
  return launch_small_list<SmallConfig<2, 1, 1, 3, 7>, SmallConfig<2, 1, 2, 3, 7>,
                           SmallConfig<2, 1, 4, 3, 7>, SmallConfig<2, 2, 1, 3, 7>,
                           SmallConfig<2, 2, 2, 3, 7>, SmallConfig<2, 2, 4, 3, 7>,
                           SmallConfig<2, 4, 1, 3, 7>, SmallConfig<2, 4, 2, 3, 7>,
                           SmallConfig<2, 4, 4, 3, 7>>(p, than, ch, stream);
}

}  // namespace omni_conv
