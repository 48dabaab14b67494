// The small-call convolution kernels (conv_small.h) of 1 tap.
#include "conv_small.h"

namespace omni_conv {

int launch_small_taps1(const ConvParams& p, double than, Choice& ch, hipStream_t stream) {
  return launch_small_list<SmallConfig<1, 1, 1, 3, 8>, SmallConfig<1, 1, 2, 3, 8>,
                           SmallConfig<1, 1, 4, 3, 8>, SmallConfig<1, 2, 1, 3, 8>,
                           SmallConfig<1, 2, 2, 3, 8>, SmallConfig<1, 2, 4, 3, 8>,
                           SmallConfig<1, 4, 1, 3, 8>, SmallConfig<1, 4, 2, 3, 8>,
                           SmallConfig<1, 4, 4, 3, 8>>(p, than, ch, stream);
}

}  // namespace omni_conv
