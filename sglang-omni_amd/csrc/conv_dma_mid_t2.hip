// LDS-DMA convolution kernels for two-tap convs (transposed convs of kernel 2 * stride): the tiles between the loaded step's and the
// small-call kernel (bf16 operand and weights).
#include "conv_dma.h"

namespace omni_conv {

int launch_mid_taps2(const ConvParams& p, Choice& ch, hipStream_t stream) {
  // 96 columns x 64, 128 or 256 positions: 8, 8 and 16 waves
  // (measured in one round, us at 48 / 24 / 12 chunks: 26 - 28 / 15 / 8.5, 33 / 20 / 12, 45 / 28 /
  // 19). 1536 -> 6144 columns at 250 positions 39.7 -> 27.9 us, at 1 000 75 -> 48; 768 -> 3072 at
  // 2 000 positions 45 -> 30.
  return launch_least<DmaConfig<2, 4, 3, 1, 96, 2, 2>, DmaConfig<2, 4, 3, 2, 160, 2, 2>,
                      DmaConfig<2, 8, 3, 2, 288, 2, 1>>(p, {{3, 0.52}, {4.5, 0.62}, {9, 0.75}}, ch, stream);
}

}  // namespace omni_conv
