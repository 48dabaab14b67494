// LDS-DMA convolution kernels for k = 7 convs: the tiles between the loaded step's and the
// small-call kernel (bf16 operand and weights).
#include "conv_dma.h"

namespace omni_conv {

int launch_mid_taps7(const ConvParams& p, Choice& ch, hipStream_t stream) {
  // 96 columns x 64, 128 or 256 positions: 8, 8 and 16 waves
  // (measured in one round, us at 24 / 12 chunks: 30 / 17, 36 / 22, 49 / 30; 16 waves of 48 x 32
  // in the last, which 8 waves of 48 x 64 take 53 / 32 for). 768 -> 768 columns at 2 000 positions
  // 45 -> 30.5 us (88 workgroups of 96 x 192, 256 of 96 x 64), 384 -> 384 at 16 000 positions
  // 52 -> 35 (336 of 96 x 192 in two rounds, 252 of 96 x 256 in one). 96 x 96, 48 x 192, 48 x 256
  // and 64 x 192 tiles are no faster than these three anywhere by more than 5 %.
  return launch_least<DmaConfig<2, 4, 3, 1, 176, 7, 1>, DmaConfig<2, 4, 3, 2, 240, 7, 1>,
                      DmaConfig<2, 8, 3, 2, 368, 7, 1>>(p, {{4, 1.1}, {7.5, 1.25}, {11.5, 1.6}}, ch, stream);
}

}  // namespace omni_conv
