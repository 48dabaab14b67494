// LDS-DMA convolution kernels for k = 1 convs: the tiles between the loaded step's and the
// small-call kernel (bf16 operand and weights).
#include "conv_dma.h"

namespace omni_conv {

int launch_mid_taps1(const ConvParams& p, Choice& ch, hipStream_t stream) {
  // 96 columns x 64, 128 or 256 positions: 8, 8 and 16 waves
  // (measured in one round, us at 24 / 12 chunks: 12 / 8.5, 15.5 / 12, 20 / 15.5). 768 -> 768
  // columns at 2 000 positions 19 -> 12.4 us, at 8 000 34.6 -> 22.3; 384 -> 384 at 16 000
  // positions 25.6 -> 17.2.
  return launch_least<DmaConfig<2, 4, 3, 1, 64, 1, 4>, DmaConfig<2, 4, 3, 2, 128, 1, 3>,
                      DmaConfig<2, 8, 3, 2, 256, 1, 3>>(p, {{5.5, 0.26}, {7.5, 0.33}, {11, 0.4}}, ch, stream);
}

}  // namespace omni_conv
