// General Conv1d / ConvTranspose1d of channels-last activations: what omni_conv1d_general launches.
#pragma once

#include <type_traits>

#include "common.h"

namespace omni_general {

struct GeneralParams {
  const void* x;
  int64_t x_sb, x_st, x_sc;
  int64_t batch, length_in, c_in;
  const void* w;
  int64_t w_s0, w_s1, w_s2, taps;
  const void* bias;
  int64_t c_out, groups, stride, dilation, pad_left;
  void* y;
  int64_t y_sb, y_st, y_sc, length_out;
};

template <typename T>
__device__ __forceinline__ float load_as_float(const void* base, int64_t i) {
  if constexpr (std::is_same<T, float>::value) {
    return reinterpret_cast<const float*>(base)[i];
  } else if constexpr (std::is_same<T, __bf16>::value) {
    return bits_to_float_bf16(reinterpret_cast<const u16*>(base)[i]);
  } else {
    return bits_to_float_f16(reinterpret_cast<const u16*>(base)[i]);
  }
}

template <typename T>
__device__ __forceinline__ void store_from_float(void* base, int64_t i, float v) {
  if constexpr (std::is_same<T, float>::value) {
    reinterpret_cast<float*>(base)[i] = v;
  } else if constexpr (std::is_same<T, __bf16>::value) {
    reinterpret_cast<u16*>(base)[i] = float_to_bits_bf16(v);
  } else {
    reinterpret_cast<u16*>(base)[i] = float_to_bits_f16(v);
  }
}

// The matrix-core kernel (conv_general_mfma.h) of each dtype, one translation unit each;
// OMNI_ERR_UNSUPPORTED, before any launch, for what it does not take.
int launch_mfma_f32(const GeneralParams& p, bool transposed, hipStream_t stream);
int launch_mfma_bf16(const GeneralParams& p, bool transposed, hipStream_t stream);
int launch_mfma_f16(const GeneralParams& p, bool transposed, hipStream_t stream);

}  // namespace omni_general
