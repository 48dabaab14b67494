// The small-call convolution kernels (conv_small.h) of 7 taps.
#include "conv_small.h"

namespace omni_conv {

int launch_small_taps7(const ConvParams& p, double than, Choice& ch, hipStream_t stream) {
  return launch_small_list<SmallConfig<7, 1, 1, 1, 6>, SmallConfig<7, 1, 2, 1, 6>,
                           SmallConfig<7, 1, 4, 1, 6>, SmallConfig<7, 2, 1, 1, 6>,
                           SmallConfig<7, 2, 2, 1, 6>, SmallConfig<7, 2, 4, 1, 6>,
                           SmallConfig<7, 4, 1, 1, 6>, SmallConfig<7, 4, 2, 1, 6>,
                           SmallConfig<7, 4, 4, 1, 6>>(p, than, ch, stream);
}

}  // namespace omni_conv
