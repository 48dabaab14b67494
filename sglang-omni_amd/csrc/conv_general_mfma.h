// Conv1d / ConvTranspose1d of channels-last activations on the matrix cores, for what the packed
// bf16 kernels (conv_dma.h, conv_kernel.h) do not take: float16 and float32 activations, grouped
// convs of wide groups, strides, channel counts off their grid, weights in the module's layout.
//
// An implicit GEMM per (batch row, group, output phase): output channels are the MFMA M dimension,
// positions N, (chunk of input channels, tap) K. A transposed conv runs one phase of its stride
// per workgroup, with the phase's own taps only (outputs s u + r - pad take the taps j with
// (r - j dil) % s == 0, input u + (r - j dil) / s), so no product with a structural zero exists.
//
// A stage is a chunk of 64 bytes of channels (32 of 2-byte types, 16 float32) and up to G taps:
// the input rows every tap reads (shifted) and the taps' weights go through registers into LDS as
// 64-byte rows, 16-byte quarters rotated by (row / 2) % 4 so that the 16-row operand reads meet no
// bank conflict; the next stage's global loads are in flight during this stage's MFMAs. float32
// runs on v_mfma_f32_16x16x4_f32 (full float32 products and sums): a lane's 16-byte read feeds
// four MFMAs, element e of both operands in the e-th. Every output sums its products in the order
// (chunk, tap), whatever the tile and the taps per stage, starting from the bias, in float32, rounded once.
//
// Bound by: float16, the LDS operand reads (6 of 1 KiB per 8 MFMAs of a wave) and the stage
// barriers; float32, the matrix cores and, with two or three taps a stage, the latency of the next
// stage's loads. Measured against one thread per output (conv_general.hip), 4 x 4801 positions of
// 192 channels: float16 k = 7, d = 3 16 015 -> 22.2 us (445 TFLOP/s), k = 1 1 769 -> 11.6 us;
// float32 16 863 -> 110 us (90 TFLOP/s), 2 360 -> 28 us; transposed 256 -> 128, k = 11, s = 5, 2 x
// 2003 positions: float16 390 -> 19.4 us, float32 465 -> 50.7 us. The VALU work of addressing was
// half of the time until each piece's offset was computed once and a stage added a uniform base.
#pragma once

#include <cmath>

#include "conv_general.h"

namespace omni_general {

constexpr int kRowBytes = 64;   // an LDS row: one chunk of one position's or column's channels
constexpr int kMaxRows = 208;   // staged input rows: a tile's positions and the taps' reach
constexpr int kThreads = 256;

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

template <typename T>
__device__ __forceinline__ f32x4 mfma64(u32x4 a, u32x4 b, f32x4 acc) {
  if constexpr (std::is_same<T, float>::value) {
    const f32x4 fa = __builtin_bit_cast(f32x4, a), fb = __builtin_bit_cast(f32x4, b);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[e], fb[e], acc, 0, 0, 0);
    return acc;
  } else if constexpr (std::is_same<T, __bf16>::value) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), acc, 0, 0, 0);
  }
}

struct MfmaParams {
  GeneralParams g;
  int transposed;
  int cin_g, cout_g;
  int phases;                // output phases: the stride of a transposed conv, 1 of a conv
  int u_count;               // positions per phase (a conv's outputs)
  int u_tiles, n_tiles;
  int u_step;                // input rows between positions: a conv's stride, 1 transposed
  int group_taps;            // taps per stage
  int s_dil_gcd, dil_inv;    // transposed: gcd(stride, dilation), 1 / (dilation / gcd) mod stride / gcd
  uint32_t x_bytes, w_bytes; // extents of one batch row of x and of the weight
};

// A 16-byte piece on its way from global memory to LDS: loaded whole (VEC), or element by element
// (any stride), the elements of a 2-byte type kept apart until they are stored.
template <typename T, bool VEC>
struct Piece {
  static constexpr int E = 16 / sizeof(T);
  static constexpr int NR = VEC ? 4 : E;
  uint32_t r[NR];

  // the E channels from byte offset off + base on (base uniform), `step` bytes apart; off =
  // kOutOfRange reads zeros, as do channels from `have` on
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rsrc, uint32_t off, uint32_t base,
                                       uint32_t step, int have) {
    if constexpr (VEC) {
      const u32x4 v =
          __builtin_amdgcn_raw_buffer_load_b128(rsrc, have > 0 ? off : kOutOfRange, base, 0);
#pragma unroll
      for (int e = 0; e < 4; ++e) r[e] = v[e];
    } else {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const uint32_t o = off != kOutOfRange && e < have ? off + e * step : kOutOfRange;
        if constexpr (sizeof(T) == 4)
          r[e] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, o, base, 0);
        else
          r[e] = __builtin_amdgcn_raw_buffer_load_b16(rsrc, o, base, 0);
      }
    }
  }
  __device__ __forceinline__ u32x4 packed() const {
    if constexpr (VEC || sizeof(T) == 4)
      return u32x4{r[0], r[1], r[2], r[3]};
    else
      return u32x4{(r[0] & 0xffffu) | (r[1] << 16), (r[2] & 0xffffu) | (r[3] << 16),
                   (r[4] & 0xffffu) | (r[5] << 16), (r[6] & 0xffffu) | (r[7] << 16)};
  }
};

template <typename T, int WCO, int WP, int TCO, int TP, bool VX, bool VW>
struct GeneralTile {
  static constexpr int BCO = WCO * TCO * 16;
  static constexpr int BP = WP * TP * 16;
  static constexpr int KC = kRowBytes / sizeof(T);
  static constexpr int E = 16 / sizeof(T);
  // taps per stage: a thread holds G * BCO / 64 weight pieces while they are on their way (8
  // registers each where 2-byte elements travel one by one)
  static constexpr int G = VW || sizeof(T) == 4 ? 8 : 4;
  static constexpr int X_PIECES = (kMaxRows * 4 + kThreads - 1) / kThreads;
  static constexpr int W_PIECES = (G * BCO * 4 + kThreads - 1) / kThreads;
  static constexpr int lds_bytes(int taps) { return (kMaxRows + taps * BCO) * kRowBytes; }
  static_assert(WCO * WP * 64 == kThreads, "four waves");
};

template <typename T, int WCO, int WP, int TCO, int TP, bool VX, bool VW>
__global__ void __launch_bounds__(kThreads) conv_general_mfma_kernel(const MfmaParams p) {
  using Tile = GeneralTile<T, WCO, WP, TCO, TP, VX, VW>;
  constexpr int BCO = Tile::BCO, BP = Tile::BP, KC = Tile::KC, E = Tile::E;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds_general[];
  uint8_t* xs = lds_general;
  uint8_t* ws = lds_general + kMaxRows * kRowBytes;
  const GeneralParams& g = p.g;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wave_co = wave % WCO, wave_p = wave / WCO;

  // column tile fastest: the workgroups that share input rows run together on one XCD
  int t = xcd_tile(blockIdx.x, gridDim.x);
  const int n_tile = t % p.n_tiles;
  t /= p.n_tiles;
  const int u_tile = t % p.u_tiles;
  t /= p.u_tiles;
  const int phase = t % p.phases;
  t /= p.phases;
  const int group = t % (int)g.groups;
  const int b = t / (int)g.groups;
  const int n0 = n_tile * BCO, u0 = u_tile * BP;
  const int cin_g = p.cin_g, cout_g = p.cout_g;

  // the phase's taps j0 + n * j_step, reading input rows u * u_step + d0 + n * d_step
  const int s = (int)g.stride, dil = (int)g.dilation, taps = (int)g.taps;
  int j0 = 0, j_step = 1, d0 = -(int)g.pad_left, d_step = dil, nt = taps;
  if (p.transposed) {
    // tap j reaches phase r when j * dil = r (mod s): every j_step-th tap from j0 on
    const int a = p.s_dil_gcd;
    j_step = s / a;
    d_step = -(dil / a);
    j0 = phase / a * p.dil_inv % j_step;
    if (phase % a != 0 || j0 >= taps) nt = 0, j0 = 0;
    else nt = (taps - 1 - j0) / j_step + 1;
    d0 = nt ? (phase - j0 * dil) / s : 0;
  }

  const int ci0 = group * cin_g;
  const auto x_rsrc = buffer_rsrc(reinterpret_cast<const T*>(g.x) + (int64_t)b * g.x_sb, p.x_bytes);
  const auto w_rsrc = buffer_rsrc(g.w, p.w_bytes);
  // weight element (column n, channel c, tap j): n * w_n + c * w_c + j * w_j bytes past w_base
  const uint32_t w_c = (uint32_t)((p.transposed ? g.w_s0 : g.w_s1) * sizeof(T));
  const uint32_t w_n = (uint32_t)((p.transposed ? g.w_s1 : g.w_s0) * sizeof(T));
  const uint32_t w_j = (uint32_t)(g.w_s2 * sizeof(T));
  const uint32_t w_base = p.transposed ? ci0 * w_c : (uint32_t)(group * cout_g) * w_n;
  const uint32_t x_t = (uint32_t)(g.x_st * sizeof(T)), x_c = (uint32_t)(g.x_sc * sizeof(T));

  const int chunks = (cin_g + KC - 1) / KC;
  const int gt = p.group_taps;
  const int tap_groups = nt > 0 ? (nt + gt - 1) / gt : 0;

  Piece<T, VX> xr[Tile::X_PIECES];
  Piece<T, VW> wr[Tile::W_PIECES];
  // rows a stage of `count` taps reads, from the input row of the lowest tap on
  auto stage_rows = [&](int count) __attribute__((always_inline)) {
    return (BP - 1) * p.u_step + (count - 1) * (d_step < 0 ? -d_step : d_step) + 1;
  };
  // A piece's byte offset at chunk 0 of the first tap group; a stage adds its uniform base (range
  // checks look at the offset alone: an offset is kOutOfRange, or in bounds with every base used)
  uint32_t xoff[Tile::X_PIECES], woff[Tile::W_PIECES];
  const int xq = (tid & 3) * E;  // the piece's channel within a chunk
  auto place_rows = [&](int tap0, int count) __attribute__((always_inline)) {
    const int low = d0 + (d_step < 0 ? tap0 + count - 1 : tap0) * d_step;
    const int first = u0 * p.u_step + low, rows = stage_rows(count);
#pragma unroll
    for (int i = 0; i < Tile::X_PIECES; ++i) {
      const int row = (tid + i * kThreads) >> 2, pos = first + row;
      xoff[i] = row < rows && pos >= 0 && pos < (int)g.length_in
                    ? (uint32_t)pos * x_t + (uint32_t)(ci0 + xq) * x_c : kOutOfRange;
    }
  };
  place_rows(0, min(gt, nt));
#pragma unroll
  for (int i = 0; i < Tile::W_PIECES; ++i) {
    const int piece = tid + i * kThreads;
    const int quarter = VW ? piece & 3 : piece / BCO & 3;
    const int n = VW ? (piece >> 2) % BCO : piece % BCO;
    const int k = piece / (BCO * 4);
    woff[i] = n0 + n < cout_g ? w_base + (uint32_t)(n0 + n) * w_n + (uint32_t)(quarter * E) * w_c +
                                    (uint32_t)((j0 + k * j_step) * (int64_t)w_j)
                              : kOutOfRange;
  }
  // stage (chunk c, tap group tg)
  auto load_stage = [&](int c, int tg) __attribute__((always_inline)) {
    const int c0 = c * KC, tap0 = tg * gt, count = min(gt, nt - tap0);
    if (tap_groups > 1) place_rows(tap0, count);
    const uint32_t xbase = (uint32_t)c0 * x_c;
#pragma unroll
    for (int i = 0; i < Tile::X_PIECES; ++i)
      xr[i].load(x_rsrc, xoff[i], xbase, x_c, cin_g - c0 - xq);
    const int pieces = count * BCO * 4;
    const uint32_t wbase = (uint32_t)c0 * w_c + (uint32_t)(tap0 * j_step) * w_j;
#pragma unroll
    for (int i = 0; i < Tile::W_PIECES; ++i) {
      if (i * kThreads < pieces) {
        const int piece = tid + i * kThreads;
        const int quarter = VW ? piece & 3 : piece / BCO & 3;
        wr[i].load(w_rsrc, piece < pieces ? woff[i] : kOutOfRange, wbase, w_c,
                   cin_g - c0 - quarter * E);
      }
    }
  };
  auto store_stage = [&](int tg) __attribute__((always_inline)) {
    const int count = min(gt, nt - tg * gt), pieces = count * BCO * 4;
    const int x_pieces = stage_rows(count) * 4;
#pragma unroll
    for (int i = 0; i < Tile::X_PIECES; ++i) {
      const int piece = tid + i * kThreads, row = piece >> 2;
      if (piece < x_pieces)
        *reinterpret_cast<u32x4*>(xs + row * kRowBytes + (((piece ^ (row >> 1)) & 3) << 4)) =
            xr[i].packed();
    }
#pragma unroll
    for (int i = 0; i < Tile::W_PIECES; ++i) {
      const int piece = tid + i * kThreads;
      if (piece < pieces) {
        const int quarter = VW ? piece & 3 : piece / BCO & 3;
        const int n = VW ? (piece >> 2) % BCO : piece % BCO;
        const int k = piece / (BCO * 4);
        *reinterpret_cast<u32x4*>(ws + (k * BCO + n) * kRowBytes + (((quarter ^ (n >> 1)) & 3) << 4)) =
            wr[i].packed();
      }
    }
  };

  const int lrow = lane & 15, lq = lane >> 4;
  const int co_wave = wave_co * TCO * 16, u_wave = wave_p * TP * 16;
  f32x4 acc[TCO][TP];
#pragma unroll
  for (int c = 0; c < TCO; ++c) {
    f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
    if (g.bias) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int n = n0 + co_wave + c * 16 + lq * 4 + e;
        if (n < cout_g) v[e] = load_as_float<T>(g.bias, group * cout_g + n);
      }
    }
#pragma unroll
    for (int u = 0; u < TP; ++u) acc[c][u] = v;
  }

  const int last_chunk = tap_groups ? chunks : 0;  // (a phase without taps has no stages)
  if (last_chunk) load_stage(0, 0);
  for (int c = 0, tg = 0; c < last_chunk;) {
    __syncthreads();  // the previous stage's operand reads are done
    store_stage(tg);
    __syncthreads();
    const int count = min(gt, nt - tg * gt);
    if (++tg == tap_groups) tg = 0, ++c;
    if (c < last_chunk) load_stage(c, tg);
    for (int k = 0; k < count; ++k) {
      // tap k's input row for position u: d_step < 0 stages the last tap's rows first
      const int shift = d_step < 0 ? (count - 1 - k) * -d_step : k * d_step;
      u32x4 a[TCO], bv[TP];
#pragma unroll
      for (int c = 0; c < TCO; ++c) {
        const int n = co_wave + c * 16 + lrow;
        a[c] = *reinterpret_cast<const u32x4*>(ws + (k * BCO + n) * kRowBytes +
                                               (((lq ^ (n >> 1)) & 3) << 4));
      }
#pragma unroll
      for (int u = 0; u < TP; ++u) {
        const int row = (u_wave + u * 16 + lrow) * p.u_step + shift;
        bv[u] = *reinterpret_cast<const u32x4*>(xs + row * kRowBytes + (((lq ^ (row >> 1)) & 3) << 4));
      }
#pragma unroll
      for (int c = 0; c < TCO; ++c)
#pragma unroll
        for (int u = 0; u < TP; ++u) acc[c][u] = mfma64<T>(a[c], bv[u], acc[c][u]);
    }
  }

  // A tap outside the row adds nothing, but the matrix cores multiply its staged zeros all the same,
  // which an infinite or NaN weight turns into NaN: at a row's ends an output with a tap outside that
  // is not finite is summed again, without the taps outside (`again`: bit 4 TCO u + 4 c + e).
  const int d_last = d0 + (nt - 1) * d_step;
  const bool edge = u0 * p.u_step + min(d0, d_last) < 0 ||
                    (min(u0 + BP, p.u_count) - 1) * p.u_step + max(d0, d_last) >= (int)g.length_in;
  uint64_t again = 0;
  static_assert(4 * TCO * TP <= 64, "a bit for each of a lane's outputs");
  if (edge) {
#pragma unroll
    for (int u = 0; u < TP; ++u) {
      const int pos = (u0 + u_wave + u * 16 + lrow) * p.u_step;
      const bool outside = pos + min(d0, d_last) < 0 || pos + max(d0, d_last) >= (int)g.length_in;
#pragma unroll
      for (int c = 0; c < TCO; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (outside && !__builtin_isfinite(acc[c][u][e])) again |= 1ull << (4 * (TCO * u + c) + e);
    }
  }

  // lane: position lrow of a group of 16, output channels 4 lq .. 4 lq + 3 of 16
  T* y = reinterpret_cast<T*>(g.y) + (int64_t)b * g.y_sb;
  const bool vec = g.y_sc == 1 && g.y_st % 4 == 0 && g.y_sb % 4 == 0 && (group * cout_g) % 4 == 0 &&
                   (reinterpret_cast<uintptr_t>(g.y) & (4 * sizeof(T) - 1)) == 0;
#pragma unroll
  for (int u = 0; u < TP; ++u) {
    const int uu = u0 + u_wave + u * 16 + lrow;
    const int64_t i = p.transposed ? (int64_t)uu * s + phase - g.pad_left : uu;
    if (uu >= p.u_count || i < 0 || i >= g.length_out) continue;
#pragma unroll
    for (int c = 0; c < TCO; ++c) {
      const int n = n0 + co_wave + c * 16 + lq * 4;
      const int64_t o = i * g.y_st + (int64_t)(group * cout_g + n) * g.y_sc;
      if (vec && n + 3 < cout_g) {
        if constexpr (sizeof(T) == 4) {
          *reinterpret_cast<f32x4*>(y + o) = acc[c][u];
        } else {
          u16 h[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) store_from_float<T>(h, e, acc[c][u][e]);
          *reinterpret_cast<u32x2*>(y + o) = u32x2{h[0] | (uint32_t)h[1] << 16, h[2] | (uint32_t)h[3] << 16};
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < cout_g) store_from_float<T>(y, o + e * g.y_sc, acc[c][u][e]);
      }
    }
  }
  while (again) {
    const int bit = __builtin_ctzll(again);
    again &= again - 1;
    const int uu = u0 + u_wave + bit / (4 * TCO) * 16 + lrow;
    const int n = n0 + co_wave + bit / 4 % TCO * 16 + lq * 4 + bit % 4;
    const int64_t i = p.transposed ? (int64_t)uu * s + phase - g.pad_left : uu;
    if (uu >= p.u_count || i < 0 || i >= g.length_out || n >= cout_g) continue;
    float sum = g.bias ? load_as_float<T>(g.bias, group * cout_g + n) : 0.f;
    for (int k = 0; k < nt; ++k) {
      const int64_t pos = (int64_t)uu * p.u_step + d0 + (int64_t)k * d_step;
      if (pos < 0 || pos >= g.length_in) continue;
      const int64_t xo = (int64_t)b * g.x_sb + pos * g.x_st + ci0 * g.x_sc;
      const int64_t wo = (int64_t)(p.transposed ? ci0 : group * cout_g + n) * g.w_s0 +
                         (p.transposed ? n * g.w_s1 : 0) + (int64_t)(j0 + k * j_step) * g.w_s2;
      const int64_t wc = p.transposed ? g.w_s0 : g.w_s1;
      for (int c = 0; c < cin_g; ++c)
        sum = fmaf(load_as_float<T>(g.w, wo + c * wc), load_as_float<T>(g.x, xo + c * g.x_sc), sum);
    }
    store_from_float<T>(y, i * g.y_st + (int64_t)(group * cout_g + n) * g.y_sc, sum);
  }
}

template <typename T, int WCO, int WP, int TCO, int TP, bool VX, bool VW>
int launch_tile(MfmaParams p, int max_taps, int reach_step, hipStream_t stream) {
  using Tile = GeneralTile<T, WCO, WP, TCO, TP, VX, VW>;
  // as many taps per stage as the staged rows hold
  const int64_t base = (int64_t)(Tile::BP - 1) * p.u_step + 1;
  if (base > kMaxRows) return OMNI_ERR_UNSUPPORTED;
  const int64_t fit = reach_step ? (kMaxRows - base) / reach_step + 1 : Tile::G;
  int taps = max_taps < Tile::G ? max_taps : Tile::G;
  if (fit < taps) taps = (int)fit;
  p.group_taps = taps < 1 ? 1 : taps;
  p.u_tiles = (p.u_count + Tile::BP - 1) / Tile::BP;
  p.n_tiles = (p.cout_g + Tile::BCO - 1) / Tile::BCO;
  const int64_t wgs = (int64_t)p.u_tiles * p.n_tiles * p.phases * p.g.groups * p.g.batch;
  if (wgs > 0x7fffffffLL) return OMNI_ERR_UNSUPPORTED;
  hipLaunchKernelGGL((conv_general_mfma_kernel<T, WCO, WP, TCO, TP, VX, VW>), dim3((unsigned)wgs),
                     dim3(kThreads), Tile::lds_bytes(p.group_taps), stream, p);
  OMNI_LAUNCH_CHECK();
  return OMNI_OK;
}

// The choice between this kernel and one thread per output (conv_general.hip) compares estimates of
// both at this many rows, whatever the call's own number: the two sum in different orders, and a
// row's result must not depend on the rows beside it.
constexpr int kEstimateRows = 16;

// One thread per output, us: its chain of dependent loads, and the loads' traffic at the 64-byte
// lines that a wave's 64 weights and inputs spread over.
inline double estimate_scalar(const MfmaParams& p, int max_taps, int size) {
  const GeneralParams& g = p.g;
  const double outputs = 1e-6 * kEstimateRows * g.length_out * g.c_out;
  const double macs = (double)g.taps / p.phases * p.cin_g;  // of an output
  const double wave_groups = fmin((double)g.groups, fmax(1, 64.0 / p.cout_g));
  const double wave_pos = fmax(1, 64.0 / g.c_out);
  const double weights = p.transposed
      ? wave_groups * fmax(1, (double)p.cout_g * g.taps * size / 64)
      : 64 / wave_pos * fmin(1, (double)p.cin_g * g.taps * size / 64);
  const double lines = fmin(64, weights + wave_groups * wave_pos * fmin(1, p.cin_g * size / 64.0));
  const double chain = 0.1 * max_taps * p.cin_g + (p.transposed ? 0.29 * g.taps : 0);
  return 2.1 + chain + outputs * (2.9 + 0.68 * g.taps + macs * (0.33 + 1.45 * lines / 64) *
                                                            (size == 4 ? 1.16 : 1));
}

constexpr int kTiles[6][2] = {{96, 128}, {64, 128}, {32, 128}, {96, 64}, {64, 64}, {32, 32}};

// Workgroups of tile k at `rows` rows.
inline int64_t tile_workgroups(const MfmaParams& p, int k, int64_t rows) {
  return (int64_t)((p.u_count + kTiles[k][1] - 1) / kTiles[k][1]) *
         ((p.cout_g + kTiles[k][0] - 1) / kTiles[k][0]) * p.phases * p.g.groups * rows;
}

// The tile of the least time: rounds of 256 workgroups times a stage's cost, its padded columns
// and positions included, in units of 16 x 16 accumulators plus the staging a tile of any size
// pays (fitted to the measurements above: float32's MFMAs take 8 times as long). -1: none fits.
inline int pick_tile(const MfmaParams& p, int64_t rows, int size) {
  int best = -1;
  int64_t least = 0;
  for (int k = 0; k < 6; ++k) {
    if ((int64_t)(kTiles[k][1] - 1) * p.u_step + 1 > kMaxRows) continue;
    const int64_t cost = ((tile_workgroups(p, k, rows) + 255) / 256) *
                         (kTiles[k][0] * kTiles[k][1] / 256 + (size == 4 ? 4 : 16));
    if (best < 0 || cost < least) best = k, least = cost;
  }
  return best;
}

// This kernel on the tile k, us: a workgroup's setup, its stages and their MFMAs, one workgroup after
// another on each CU.
inline double estimate_tile(const MfmaParams& p, int k, int max_taps, int reach_step,
                            int stage_taps, int size) {
  const int base = (kTiles[k][1] - 1) * p.u_step + 1;
  int taps = max_taps < stage_taps ? max_taps : stage_taps;
  if (reach_step && (kMaxRows - base) / reach_step + 1 < taps) taps = (kMaxRows - base) / reach_step + 1;
  const double chunks = (p.cin_g * size + kRowBytes - 1) / kRowBytes;
  const double stages = chunks * ((max_taps + taps - 1) / taps);
  const double workgroup = 0.45 + stages * (size == 4 ? 0.39 : 0.61) +
                           chunks * max_taps * (kTiles[k][0] * kTiles[k][1] / 256) *
                               (size == 4 ? 0.039 : 0.025);
  return 3.1 + workgroup * fmax(1, tile_workgroups(p, k, kEstimateRows) / (256 * 1.3));
}

template <typename T, bool VX, bool VW>
int launch_tiles(const MfmaParams& p, int max_taps, int reach_step, hipStream_t stream) {
  constexpr int size = sizeof(T);
  const int fit = pick_tile(p, kEstimateRows, size);
  if (fit < 0) return OMNI_ERR_UNSUPPORTED;
  // Many small workgroups of little work each (grouped convs of a few positions, transposed convs
  // with fewer taps than phases) take longer than one thread per output: 58 rows of 2 positions,
  // 64 groups of 24 -> 5 channels, 2 taps at stride 8 are 29 696 workgroups, 88 us against 6.9.
  // Over 1 636 drawn forms at a few hundred products and fewer an output the choice lies within
  // 1.6 % of the better kernel in the mean (this kernel always: 4.4 %).
  constexpr int stage_taps = GeneralTile<T, 2, 2, 1, 1, VX, VW>::G;
  if (estimate_scalar(p, max_taps, size) < estimate_tile(p, fit, max_taps, reach_step, stage_taps, size))
    return OMNI_ERR_UNSUPPORTED;
  switch (pick_tile(p, p.g.batch, size)) {
    case 0: return launch_tile<T, 2, 2, 3, 4, VX, VW>(p, max_taps, reach_step, stream);
    case 1: return launch_tile<T, 2, 2, 2, 4, VX, VW>(p, max_taps, reach_step, stream);
    case 2: return launch_tile<T, 1, 4, 2, 2, VX, VW>(p, max_taps, reach_step, stream);
    case 3: return launch_tile<T, 2, 2, 3, 2, VX, VW>(p, max_taps, reach_step, stream);
    case 4: return launch_tile<T, 2, 2, 2, 2, VX, VW>(p, max_taps, reach_step, stream);
    default: return launch_tile<T, 2, 2, 1, 1, VX, VW>(p, max_taps, reach_step, stream);
  }
}

template <typename T>
int launch_mfma(const GeneralParams& g, bool transposed, hipStream_t stream) {
  constexpr int64_t kBig = 0x3fffffffLL;  // indices inside the kernel are 32-bit
  const int64_t cin_g = g.c_in / g.groups, cout_g = g.c_out / g.groups;
  // Groups of fewer channels leave the 16 x 16 x 64-byte steps mostly empty, and one thread per
  // output is as fast or faster (2 x 4000 or 40000 positions, this kernel against that one, us:
  // float16 8 -> 4 channels 4.3 / 6.6, 4 -> 8 6.7 / 4.8, 2 -> 16 6.6 / 4.8; float32 4 -> 6 4.6 /
  // 5.2, 4 -> 4 8.0 / 5.7; 16 groups of 4 -> 4 float16 12.4 / 16.9, 8 of 8 -> 8 6.1 / 32.1)
  if (cout_g < 4 || cin_g * (int64_t)sizeof(T) < 16 || cin_g * cout_g < 24)
    return OMNI_ERR_UNSUPPORTED;
  if (g.length_in < 1 || g.length_in > kBig || g.length_out > kBig || g.c_in > kBig || g.c_out > kBig ||
      g.taps > kBig || g.stride > kBig || g.dilation > kBig || g.pad_left > kBig ||
      g.taps * g.dilation > kBig || (g.length_out + g.pad_left) > kBig ||
      (g.length_out + 128) * g.stride > kBig || (transposed && g.stride > 32768))
    return OMNI_ERR_UNSUPPORTED;
  constexpr int64_t kLimit = 0x7fffffffLL;  // byte offsets are 32-bit
  if (g.x_st > kLimit || g.x_sc > kLimit || g.w_s0 > kLimit || g.w_s1 > kLimit || g.w_s2 > kLimit)
    return OMNI_ERR_UNSUPPORTED;
  const int64_t w_rows = transposed ? g.c_in : g.c_out, w_cols = transposed ? cout_g : cin_g;
  const int64_t size = sizeof(T);
  const int64_t x_bytes = ((g.length_in - 1) * g.x_st + (g.c_in - 1) * g.x_sc + 1) * size;
  const int64_t w_bytes =
      ((w_rows - 1) * g.w_s0 + (w_cols - 1) * g.w_s1 + (g.taps - 1) * g.w_s2 + 1) * size;
  if (x_bytes > kLimit || w_bytes > kLimit) return OMNI_ERR_UNSUPPORTED;
  MfmaParams p{};
  p.g = g;
  p.transposed = transposed;
  p.cin_g = (int)cin_g;
  p.cout_g = (int)cout_g;
  p.x_bytes = (uint32_t)x_bytes;
  p.w_bytes = (uint32_t)w_bytes;
  int max_taps = (int)g.taps, reach_step = (int)g.dilation;
  if (transposed) {
    int a = (int)g.stride, c = (int)(g.dilation % g.stride);
    while (c) { const int m = a % c; a = c; c = m; }
    const int j_step = (int)g.stride / a;
    p.s_dil_gcd = a;
    // 1 / (dilation / a) mod j_step (Euclid)
    int64_t r0 = j_step, r1 = g.dilation / a % j_step, t0 = 0, t1 = 1;
    while (r1) {
      const int64_t q = r0 / r1, r = r0 - q * r1, t = t0 - q * t1;
      r0 = r1, r1 = r, t0 = t1, t1 = t;
    }
    p.dil_inv = (int)(t0 < 0 ? t0 + j_step : t0);
    max_taps = ((int)g.taps + j_step - 1) / j_step;
    reach_step = (int)g.dilation / a;
    p.phases = (int)g.stride;
    // the last output length_out - 1 = s u + r - pad
    p.u_count = (int)((g.length_out - 1 + g.pad_left) / g.stride) + 1;
    p.u_step = 1;
  } else {
    p.phases = 1;
    p.u_count = (int)g.length_out;
    p.u_step = (int)g.stride;
  }
  // whole 16-byte pieces of a chunk's channels: unit stride, aligned, whole pieces per group
  constexpr int64_t E = 16 / sizeof(T);
  auto aligned = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  const bool vx = g.x_sc == 1 && g.x_st % E == 0 && g.x_sb % E == 0 && cin_g % E == 0 && aligned(g.x);
  const int64_t wc = transposed ? g.w_s0 : g.w_s1, wn = transposed ? g.w_s1 : g.w_s0;
  const bool vw = wc == 1 && wn % E == 0 && (g.taps == 1 || g.w_s2 % E == 0) && cin_g % E == 0 && aligned(g.w);
  if (vx && vw) return launch_tiles<T, true, true>(p, max_taps, reach_step, stream);
  if (vx) return launch_tiles<T, true, false>(p, max_taps, reach_step, stream);
  return launch_tiles<T, false, false>(p, max_taps, reach_step, stream);
}

}  // namespace omni_general
