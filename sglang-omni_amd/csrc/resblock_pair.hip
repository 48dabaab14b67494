// A HiFiGAN ResBlock pair of the 32-channel stage in one launch (gfx950 bf16 MFMA):
//
//   h = act1(c1(x))                    c1: k taps, dilation d, "same" zero padding
//   y = c2(h) (+ residual, mix, ...)   c2: k taps, dilation 1; the conv epilogue of omni_conv1d
//
// (ResBlock of sglang_omni/models/minicpm_o/components/token2wav/hift_layers.py:95-110, as
// hift.py:255-281 runs it: xt = act(x); xt = c1(xt); xt = act(xt); xt = c2(xt); x = xt + x.)
// Run as two launches, h goes to HBM as bf16 and comes back (4 bytes per element); here h stays in
// LDS. A pair then moves 256 bytes a position (x, the float16 stream in and out, the next
// operand), and what bounds it is that stream: 3.84 M positions, 983 MB, 187 us at k = 3.
//
// Workgroup: 8 waves by roles, so that the matrix work, the LDS exchange and the HBM traffic of
// different tiles overlap: waves 0 - 3 compute h of one tile while waves 4 - 7 run c2 and its
// epilogue on the tile before, one barrier per tile, the tiles one after another (a grid of one
// workgroup per resident slot). Each SIMD holds one wave of either role. A wave keeps its conv's
// whole weights in registers (K x 2 column tiles), so the only LDS reads are the operand rows, one
// per two MFMAs; with the weights in LDS too, three reads per two MFMAs kept the matrix cores
// waiting. The x rows reach LDS by DMA, one tile ahead, and the residual rows are loaded under the
// convs. k = 3 leaves room for two workgroups per CU; k = 7 and 11 take one (at two, their weights
// spill: k = 7 250 us, k = 11 460).
//
// us per pair at 16 x 240 000 positions, weights in LDS -> by roles (k = 11: two launches -> by
// roles; its weights-in-LDS pair took 456): k = 3 200 -> 187, k = 7 314 -> 198, k = 11 400 - 440
// -> 235; with the mix 334 -> 235, 507 -> 275, 436 -> 275; one row of 24 000 positions 10.4 ->
// 8.3, 13.2 -> 10.0, 18 -> 11.5.
//
// A tile is 256 h rows (16 groups of 16, 4 per wave) and so BP = 256 - (k - 1) output positions.
// LDS rows are 64 bytes, 16-byte slot s of row r at s ^ ((r / 2) % 4), at which the MFMA operand
// reads meet no bank conflict. h rows outside [0, length) are zeros (c2's padding). Each
// accumulator takes its MFMAs in the order of the LDS-DMA conv kernel's (taps ascending), h rounds
// the way that kernel's epilogue rounds its bf16 output, and c2's accumulators go through
// conv_epilogue's arithmetic: the pair gives the bits of the two launches.
#include "conv_kernel.h"
#include "omni_codec.h"

namespace omni_conv {
int make_conv_params(const omni_conv_args* a, ConvParams& p, bool& x_f32, bool& fp8, bool& fuse2);
}

namespace {

using namespace omni_conv;

constexpr int kC = 32;      // channels: one 32-channel chunk
constexpr int kMaxDil = 5;  // the largest c1 dilation the LDS is sized for

// element offset of 16-byte slot `slot` of 64-byte row `row`
__device__ __forceinline__ int row_slot(int row, int slot) {
  return row * kC + ((slot ^ ((row >> 1) & 3)) << 3);
}

template <int K>
struct PairTile {
  static constexpr int R2 = (K - 1) / 2;
  static constexpr int HR = 256;            // h rows of a tile: 4 waves x 4 groups of 16
  static constexpr int BP = HR - 2 * R2;    // output positions of a tile
  static constexpr int XROWS = (HR + (K - 1) * kMaxDil + 15) / 16 * 16;  // staged x rows
  static constexpr int XP = (XROWS / 16 + 3) / 4;  // DMA instructions per wave (16 rows each)
  static constexpr int HROWS = HR + 16;  // + the rows c2 reads for its positions past BP (unused)
  static constexpr size_t x_bytes = (size_t)XROWS * kC * 2;
  static constexpr size_t h_bytes = (size_t)HROWS * kC * 2;
  static constexpr size_t coef_offset = 2 * (x_bytes + h_bytes);
  static constexpr size_t lds_bytes = coef_offset + (size_t)(kNumCoefRows + 1) * kC * 4;
};

template <int K, int OCC, int GP, bool F16, bool MIX>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2 * OCC, 2 * OCC)))
    resblock_pair_kernel(const ConvParams c1, const ConvParams c2, int tiles_per_row) {
  using T = PairTile<K>;
  extern __shared__ __attribute__((aligned(16))) u16 lds[];
  float* coef = reinterpret_cast<float*>(reinterpret_cast<uint8_t*>(lds) + T::coef_offset);
  float* bias1 = coef + kNumCoefRows * kC;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int pw = wave & 3;
  const bool first = wave < 4;  // the c1 waves
  const int lrow = lane & 15;
  const int q = lane >> 4;
  const int L = c2.length;

  // the wave's conv: all K taps x 32 columns in registers. Row i of column tile c is column
  // 8 (i / 4) + 4 c + i % 4, so a lane's accumulators of the two tiles are 8 consecutive columns
  // of its position: one 16-byte slot of an h row, 16 bytes of an output row
  bf16x8 w[K][2];
  {
    const auto wr = buffer_rsrc(first ? c1.weight : c2.weight, (uint32_t)(kC * K * kC * 2));
#pragma unroll
    for (int j = 0; j < K; ++j)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int n = 8 * (lrow >> 2) + 4 * c + (lrow & 3);
        w[j][c] = __builtin_bit_cast(
            bf16x8, __builtin_amdgcn_raw_buffer_load_b128(wr, (uint32_t)((n * K + j) * kC + q * 8) * 2u, 0, 0));
      }
  }
  stage_coefficients<kC, 512, false>(c2, coef, 0);
  for (int n = tid; n < kC; n += 512) bias1[n] = c1.bias ? c1.bias[n] : 0.f;
  __syncthreads();

  const int tiles = tiles_per_row * c2.batch;
  const int tile0 = xcd_tile(blockIdx.x, gridDim.x);
  const int count = tile0 < tiles ? (tiles - tile0 + (int)gridDim.x - 1) / (int)gridDim.x : 0;
  auto xs_of = [&](int b) __attribute__((always_inline)) { return lds + (b & 1) * (T::x_bytes / 2); };
  auto hs_of = [&](int b) __attribute__((always_inline)) {
    return lds + T::x_bytes + (b & 1) * (T::h_bytes / 2);
  };
  // step it: the c1 waves' tile it, the c2 waves' tile it - 1. The barrier before it: the c1
  // waves' DMA of tile it has landed, h of tile it - 1 is whole, and both buffers about to be
  // refilled (x of tile it - 1, h of tile it - 2) have been read.
  if (first) {
    const int d = c1.dil;
    const int R = c1.lpad + T::R2;
    const auto xr = buffer_rsrc(c1.x, c1.x_bytes);
    const int rel0 = (lane >> 2) * (int)c1.x_st + (((lane & 3) ^ ((lane >> 3) & 3)) << 3);
    const int span = T::HR + (K - 1) * d;  // rows the tile reads
    auto send_x = [&](int it) __attribute__((always_inline)) {
      const int tile = tile0 + it * (int)gridDim.x;
      const int b = tile / tiles_per_row;
      const int p0 = (tile - b * tiles_per_row) * T::BP - R;
      const int base = (int)((int64_t)b * c1.x_sb + (int64_t)p0 * c1.x_st) + rel0;
      u16* xs = xs_of(it);
#pragma unroll
      for (int u = 0; u < T::XP; ++u) {
        const int ii = pw + 4 * u;
        if (ii * 16 < span) {
          const int row = ii * 16 + (lane >> 2);
          const bool ok = (unsigned)(p0 + row) < (unsigned)c1.x_length;
          const uint32_t off = ok ? (uint32_t)(base + ii * 16 * (int)c1.x_st) * 2u : kOutOfRange;
          __builtin_amdgcn_raw_ptr_buffer_load_lds(
              xr, (__attribute__((address_space(3))) void*)(xs + ii * 512), 16, (int)off, 0, 0, 0);
        }
      }
    };
    f32x4 b1[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) b1[c] = *reinterpret_cast<const f32x4*>(bias1 + 8 * q + 4 * c);
    if (count > 0) send_x(0);
    for (int it = 0; it <= count; ++it) {
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      asm volatile("s_barrier" ::: "memory");
      if (it == count) break;
      if (it + 1 < count) send_x(it + 1);
      const int tile = tile0 + it * (int)gridDim.x;
      const int b = tile / tiles_per_row;
      const int h0 = (tile - b * tiles_per_row) * T::BP - T::R2;  // position of h row 0
      const u16* xs = xs_of(it);
      u16* hs = hs_of(it);
#pragma unroll
      for (int gp = 0; gp < 4 / GP; ++gp) {
        f32x4 acc[GP][2];
#pragma unroll
        for (int t = 0; t < GP; ++t)
#pragma unroll
          for (int c = 0; c < 2; ++c) acc[t][c] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int hr0 = (pw * 4 + gp * GP) * 16 + lrow;
#pragma unroll
        for (int j = 0; j < K; ++j)
#pragma unroll
          for (int t = 0; t < GP; ++t) {
            const bf16x8 xv = *reinterpret_cast<const bf16x8*>(xs + row_slot(hr0 + t * 16 + j * d, q));
#pragma unroll
            for (int c = 0; c < 2; ++c)
              acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j][c], xv, acc[t][c], 0, 0, 0);
          }
        // acc + bias, then the activation, rounded to bf16; zeros outside [0, length)
#pragma unroll
        for (int t = 0; t < GP; ++t) {
          const int hr = hr0 + t * 16;
          const bool inside = (unsigned)(h0 + hr) < (unsigned)L;
          u32x4 o;
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            f32x4 v = acc[t][c] + b1[c];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              if (c1.act == OMNI_ACT_LEAKY_RELU) v[e] = v[e] >= 0.f ? v[e] : v[e] * c1.slope;
              if (!inside) v[e] = 0.f;
            }
            o[2 * c] = pack_bf16x2(v[0], v[1]);
            o[2 * c + 1] = pack_bf16x2(v[2], v[3]);
          }
          *reinterpret_cast<u32x4*>(hs + row_slot(hr, q)) = o;
        }
      }
    }
    return;
  }

  f32x4 b2[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) b2[c] = *reinterpret_cast<const f32x4*>(coef + kBias * kC + 8 * q + 4 * c);
  const auto rr = buffer_rsrc(c2.residual, c2.residual ? c2.r_bytes : 0);
  const auto ra = buffer_rsrc(c2.mix_a, c2.mix_a ? c2.r_bytes : 0);
  const auto rb = buffer_rsrc(c2.mix_b, c2.mix_a ? c2.r_bytes : 0);
  const auto rs = buffer_rsrc(c2.sum_out, c2.sum_out ? c2.r_bytes : 0);
  const auto ro = buffer_rsrc(c2.out, c2.out ? c2.o_bytes : 0);
  constexpr int RW = F16 ? 1 : 2;  // 16-byte pieces of 8 residual-stream elements
  auto widen = [&](const u32x4 (&raw)[RW], f32x4 (&v)[2]) __attribute__((always_inline)) {
    if constexpr (F16) {
      v[0] = widen_residual4(u32x4{raw[0][0], raw[0][1], 0u, 0u}, 1);
      v[1] = widen_residual4(u32x4{raw[0][2], raw[0][3], 0u, 0u}, 1);
    } else {
      v[0] = widen_residual4(raw[0], 0);
      v[1] = widen_residual4(raw[RW - 1], 0);
    }
  };
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  asm volatile("s_barrier" ::: "memory");
  for (int it = 0; it < count; ++it) {
    const int tile = tile0 + it * (int)gridDim.x;
    const int b = tile / tiles_per_row;
    const int i0 = (tile - b * tiles_per_row) * T::BP;
    // the tile's residual rows, in flight under the barrier and the convs
    uint32_t roff[4], ooff[4];
    u32x4 res[4][RW];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int o = (pw * 4 + t) * 16 + lrow;
      const int i = i0 + o;
      const bool ok = o < T::BP && i < L;
      roff[t] = ok ? (uint32_t)((int64_t)b * c2.r_sb + (int64_t)i * c2.r_st + 8 * q) * (F16 ? 2u : 4u)
                   : kOutOfRange;
      ooff[t] = ok ? (uint32_t)((int64_t)b * c2.o_sb + (int64_t)i * c2.o_st + 8 * q) *
                         (c2.out_bf16 ? 2u : 4u)
                   : kOutOfRange;
#pragma unroll
      for (int k = 0; k < RW; ++k)
        res[t][k] = __builtin_amdgcn_raw_buffer_load_b128(rr, ok ? roff[t] + 16u * k : kOutOfRange, 0, 0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    asm volatile("s_barrier" ::: "memory");
    const u16* hs = hs_of(it);
#pragma unroll
    for (int gp = 0; gp < 4 / GP; ++gp) {
      u32x4 wa[GP][RW], wb[GP][RW];
      if constexpr (MIX) {
#pragma unroll
        for (int t = 0; t < GP; ++t)
#pragma unroll
          for (int k = 0; k < RW; ++k) {
            const uint32_t r0 = roff[gp * GP + t];
            const uint32_t off = r0 == kOutOfRange ? kOutOfRange : r0 + 16u * k;
            wa[t][k] = __builtin_amdgcn_raw_buffer_load_b128(ra, off, 0, 0);
            wb[t][k] = __builtin_amdgcn_raw_buffer_load_b128(rb, off, 0, 0);
          }
      }
      f32x4 acc[GP][2];
#pragma unroll
      for (int t = 0; t < GP; ++t)
#pragma unroll
        for (int c = 0; c < 2; ++c) acc[t][c] = f32x4{0.f, 0.f, 0.f, 0.f};
      const int o0 = (pw * 4 + gp * GP) * 16 + lrow;
#pragma unroll
      for (int j = 0; j < K; ++j)
#pragma unroll
        for (int t = 0; t < GP; ++t) {
          const bf16x8 hv = *reinterpret_cast<const bf16x8*>(hs + row_slot(o0 + t * 16 + j, q));
#pragma unroll
          for (int c = 0; c < 2; ++c)
            acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j][c], hv, acc[t][c], 0, 0, 0);
        }
      // conv_epilogue's arithmetic, 8 columns of a position per lane
#pragma unroll
      for (int t = 0; t < GP; ++t) {
        const int g = gp * GP + t;
        f32x4 v[2] = {acc[t][0] + b2[0], acc[t][1] + b2[1]};
        if (c2.residual) {
          f32x4 r[2];
          widen(res[g], r);
          v[0] += r[0];
          v[1] += r[1];
        }
        if constexpr (MIX) {
          f32x4 ma[2], mb[2];
          widen(wa[t], ma);
          widen(wb[t], mb);
#pragma unroll
          for (int c = 0; c < 2; ++c) v[c] = ((ma[c] + mb[c]) + v[c]) * c2.mix_scale;
        }
        if (c2.sum_out) {
          if constexpr (F16) {
            const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_convertvector(v[0], f16x4));
            const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_convertvector(v[1], f16x4));
            __builtin_amdgcn_raw_buffer_store_b128(u32x4{lo[0], lo[1], hi[0], hi[1]}, rs, roff[g], 0, 0);
          } else {
#pragma unroll
            for (int c = 0; c < 2; ++c)
              __builtin_amdgcn_raw_buffer_store_b128(
                  __builtin_bit_cast(u32x4, v[c]), rs,
                  roff[g] == kOutOfRange ? kOutOfRange : roff[g] + 16u * c, 0, 0);
          }
        }
        if (c2.out != nullptr) {
          const int act = c2.act;
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            if (act == OMNI_ACT_SNAKE) {
              const f32x4 aa = *reinterpret_cast<const f32x4*>(coef + kActA * kC + 8 * q + 4 * c);
              const f32x4 ab = *reinterpret_cast<const f32x4*>(coef + kActB * kC + 8 * q + 4 * c);
#pragma unroll
              for (int e = 0; e < 4; ++e) v[c][e] = snake_rev(v[c][e], aa[e], ab[e]);
            } else if (act == OMNI_ACT_LEAKY_RELU) {
#pragma unroll
              for (int e = 0; e < 4; ++e) v[c][e] = v[c][e] >= 0.f ? v[c][e] : v[c][e] * c2.slope;
            } else if (act != OMNI_ACT_NONE) {
#pragma unroll
              for (int e = 0; e < 4; ++e) v[c][e] = apply_act(act, v[c][e], 0.f, 0.f, c2.slope);
            }
          }
          if (c2.out_bf16) {
            __builtin_amdgcn_raw_buffer_store_b128(
                u32x4{pack_bf16x2(v[0][0], v[0][1]), pack_bf16x2(v[0][2], v[0][3]),
                      pack_bf16x2(v[1][0], v[1][1]), pack_bf16x2(v[1][2], v[1][3])},
                ro, ooff[g], 0, 0);
          } else {
#pragma unroll
            for (int c = 0; c < 2; ++c)
              __builtin_amdgcn_raw_buffer_store_b128(
                  __builtin_bit_cast(u32x4, v[c]), ro,
                  ooff[g] == kOutOfRange ? kOutOfRange : ooff[g] + 16u * c, 0, 0);
          }
        }
      }
    }
  }
}

template <int K, int OCC, int GP, bool F16, bool MIX>
int launch_as(const ConvParams& p1, const ConvParams& p2, hipStream_t stream) {
  using T = PairTile<K>;
  const int64_t tiles_per_row = (p2.length + T::BP - 1) / T::BP;
  const int64_t tiles = tiles_per_row * p2.batch;
  if (tiles > 0x7fffffffLL) return OMNI_ERR_UNSUPPORTED;
  auto k = resblock_pair_kernel<K, OCC, GP, F16, MIX>;
  static const bool raised = hipFuncSetAttribute((const void*)k,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 (int)T::lds_bytes) == hipSuccess;
  if (!raised) return OMNI_ERR_LAUNCH;
  static const int64_t slots = [] {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        cus <= 0)
      cus = 256;
    return (int64_t)cus * OCC;
  }();
  hipLaunchKernelGGL(k, dim3((unsigned)(tiles < slots ? tiles : slots)), dim3(512), T::lds_bytes,
                     stream, p1, p2, (int)tiles_per_row);
  OMNI_LAUNCH_CHECK();
  return OMNI_OK;
}

// GP: the 16-row groups a wave takes through a conv at once (as many as the registers hold: with
// the float16 stream four at k = 11, two otherwise, but one at k = 3 with the float32 mix, where two
// spill 20 registers at two workgroups a CU: 4 x 325 366 positions 167 us, with one 130).
template <int K, int OCC, int GP16>
int launch(const ConvParams& p1, const ConvParams& p2, hipStream_t s) {
  if (p2.r_f16)
    return p2.mix_a ? launch_as<K, OCC, GP16, true, true>(p1, p2, s)
                    : launch_as<K, OCC, GP16, true, false>(p1, p2, s);
  return p2.mix_a ? launch_as<K, OCC, K == 3 ? 1 : 2, false, true>(p1, p2, s)
                  : launch_as<K, OCC, 2, false, false>(p1, p2, s);
}

}  // namespace

extern "C" int omni_resblock_pair(const omni_conv_args* c1, const omni_conv_args* c2,
                                  omni_stream_t stream) {
  if (!c1 || !c2) return OMNI_ERR_INVALID_ARG;
  // c1 writes no tensor (h stays on chip) and c2 reads none (its operand is h): validate each as
  // a conv with c1's operand standing in
  if (c1->out || c1->sum_out || c1->residual || c1->mix_a || c2->x) return OMNI_ERR_INVALID_ARG;
  omni_conv_args a1 = *c1, a2 = *c2;
  a1.out = const_cast<void*>(c1->x);
  a1.out_dtype = OMNI_DTYPE_BF16;
  a1.out_stride_b = c1->x_stride_b;
  a1.out_stride_t = c1->x_stride_t;
  a2.x = c1->x;
  a2.x_dtype = c1->x_dtype;
  a2.x_stride_b = c1->x_stride_b;
  a2.x_stride_t = c1->x_stride_t;
  a2.x_length = 0;
  ConvParams p1, p2;
  bool f32a, fp8a, fuse2a, f32b, fp8b, fuse2b;
  int st = make_conv_params(&a1, p1, f32a, fp8a, fuse2a);
  if (st > 0) return st;
  const int st2 = make_conv_params(&a2, p2, f32b, fp8b, fuse2b);
  if (st2 > 0) return st2;
  // the shapes the kernel takes: 32 channels, bf16 operand and weights, k = 3 / 7 / 11 with
  // "same" padding, c1 dilation <= 5, c2 dilation 1, no input activation, history or fused conv
  const int64_t k = c1->taps;
  if (c1->c_in != kC || c1->n_cols != kC || c1->c_out != kC || c2->c_in != kC ||
      c2->n_cols != kC || c2->c_out != kC || c2->taps != k || c2->dilation != 1 ||
      (k != 3 && k != 7 && k != 11) || c1->dilation > kMaxDil ||
      c1->left_pad != (k - 1) * c1->dilation / 2 || c2->left_pad != (k - 1) / 2 ||
      f32a || fp8a || fp8b || fuse2a || fuse2b || c1->in_activation != OMNI_ACTIVATION_NONE ||
      c2->in_activation != OMNI_ACTIVATION_NONE || c1->hist_pool || c2->hist_pool ||
      (c1->activation != OMNI_ACTIVATION_NONE && c1->activation != OMNI_ACTIVATION_LEAKY_RELU) ||
      c1->batch != c2->batch || c1->length != c2->length ||
      (c1->x_length != 0 && c1->x_length != c1->length))
    return OMNI_ERR_UNSUPPORTED;
  if (st < 0 || st2 < 0) return OMNI_OK;  // nothing to do
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  switch (k) {
    case 3: return launch<3, 2, 2>(p1, p2, s);
    case 7: return launch<7, 1, 2>(p1, p2, s);
    default: return launch<11, 1, 4>(p1, p2, s);
  }
}
