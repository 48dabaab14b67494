// Polyphase convolution for few positions (a streaming step of a few streams, a short utterance),
// where the LDS-DMA tiles of conv_dma.h leave most of the GPU idle and a workgroup's chain of
// staged weights is waited on stage by stage.
//
// The arithmetic is conv_dma_kernel's, in its order (chunks of 32 input channels ascending, taps
// ascending, one 16x16x32 bf16 MFMA a step, then scale, bias, residual, mix, activation), so an
// output has the same bits whichever kernel computes it: a stream decoded a few frames at a time
// equals its whole decode. What differs is how the operands arrive:
//
//   * a wave owns 16 output columns and 16 TP positions, and reads its columns' weights straight
//     from memory into the MFMA's operand registers, D - 1 groups of GC chunks ahead (GC x taps
//     loads of 1 KiB a group: 21 in flight a wave at one tap, 36 at two, 35 at seven, 7 in the
//     residual unit, whose twelve waves share a workgroup), with no barrier and no LDS on the way:
//     the weights, which nobody else in the workgroup needs, are what such a call is bound by;
//   * the tile's input rows (positions plus halos) of every channel that fits the LDS are staged
//     once, by LDS DMA, before the first MFMA (one slab for the decoders' layers at one to a few
//     row segments; more slabs, each behind a barrier, otherwise).
//
// A layer that runs in K slices (omni_conv1d_splitk) adds its slices up in registers, in slice
// order, as the reduction launch does: no partials and no second launch.
//
// Bound by: the 30 B per clock a CU reads through its L1 in the MFMA operand layout (64-byte
// pieces of 16 columns; one-wave workgroups spread a layer over more CUs), the latency of the first
// loads (about 1 us, then the slab's), and for one wave a SIMD by instructions at four cycles each.
// Measured, us per launch with weights from the Infinity Cache, LDS-DMA tile -> this kernel: at 32
// positions (4 frames of one stream in block 0) 768 channels k = 7 d = 9 59.7 -> 11.3, k = 1 12.6 ->
// 5.1; up conv 1536 -> 6144 columns at 4 positions 29.4 -> 11.2; 384 channels at 256 positions k =
// 7 24.6 -> 8.8, k = 1 10.9 -> 4.6; the 192-channel unit at 1 280 positions 35.7 -> 16.6 (the
// LDS-DMA unit's tiles of 64 positions: 19.1). The
// crossing lies near 1 000 to 2 000 positions at 768 channels and 4 000 to 8 000 at 192.
#pragma once

#include "conv_kernel.h"

namespace omni_conv {

constexpr int kSmallLdsBytes = 152 * 1024;

template <int TAPS, int TP, int NW, int GC, int D>
struct SmallTile {
  static constexpr int NT = 64 * NW;
  static constexpr int BCO = 16 * NW;
  static constexpr int BP = 16 * TP;
  static constexpr int kMaxRows = 16 * 4 * NW < 128 ? 128 : 16 * 4 * NW;  // staged rows (16 per DMA instruction)
  static constexpr int X_PIECES = (kMaxRows / 16 + NW - 1) / NW;
  static constexpr int STEPS = GC * TAPS;                    // MFMA steps of a group
  static constexpr int ES = 64;                              // weight bytes of a step and column
};

template <int TAPS, int TP, int NW, int GC, int D, bool SPLIT, bool UNIT>
__global__ void __launch_bounds__(64 * NW, 1)
    conv_small_kernel(const ConvParams p, int rows16, int slab_chunks) {
  using Tile = SmallTile<TAPS, TP, NW, GC, D>;
  extern __shared__ __attribute__((aligned(16))) u16 lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // position tile fastest: the workgroups that read the same weights run on one XCD, back to back
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int p_tile = tile % p.p_tiles, n_tile = tile / p.p_tiles;
  const int dil = p.dil, lpad = p.lpad, halo = p.halo, L = p.length, XL = p.x_length, H = lpad;
  const int c_in = p.c_in, n_cols = p.n_cols;
  const int n_wave = n_tile * Tile::BCO + wave * 16;  // the wave's first column
  const int chunks = c_in / kChunk;
  const int groups = chunks / GC;  // the launcher requires whole groups

  const auto w_rsrc = buffer_rsrc(p.weight, p.w_bytes);
  // The wave's weights: column n_wave + lane % 16, channels 8 (lane / 16) .. + 7 of each step. Their
  // first loads go out before anything else.
  const int lrow = lane & 15, lq = lane >> 4;
  const int n_w = n_wave + lrow;
  const uint32_t w_off = n_w < n_cols ? (uint32_t)(n_w * TAPS * Tile::ES + lq * (Tile::ES / 4))
                                      : kOutOfRange;
  typedef u32x4 wreg_t;
  wreg_t w[D][Tile::STEPS];
  // group g's weights; past the last group nothing is read, but the loads are issued all the same:
  // a load under a branch would have every wait count the fewest that may be in flight
  auto load_group = [&](int g, wreg_t (&dst)[Tile::STEPS]) __attribute__((always_inline)) {
    const uint32_t row = (uint32_t)n_cols * TAPS * Tile::ES;  // a chunk of the packed weights
    const uint32_t off = g < groups ? w_off : kOutOfRange;
#pragma unroll
    for (int k = 0; k < Tile::STEPS; ++k) {
      // (the tap's offset is an immediate of the load)
      const uint32_t base = (uint32_t)(g * GC + k / TAPS) * row;
      dst[k] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, off + k % TAPS * Tile::ES, base, 0);
    }
  };
#pragma unroll
  for (int i = 0; i < D - 1; ++i)
    load_group(i, w[i]);

  const int M = p.batch * L;
  const int m0 = p_tile * Tile::BP;
  const int m_end = min(m0 + Tile::BP, M);
  const int b0 = m0 / L;
  const int lo0 = m0 - b0 * L;
  const int first = min(L - lo0, m_end - m0);
  const int nseg = (m_end - 1) / L - b0 + 1;
  const int rows = (m_end - m0) + nseg * halo;
  const int seg_rows = L + halo;

  // The staged rows, as conv_dma_kernel describes them: piece u of a thread is LDS slot tid % 4 of
  // row r = tid / 4 + 16 NW u, which holds the quarter (tid % 4) ^ ((r / 2) % 4) of the row.
  const int q8 = (tid & 3) * 8;
  const int pieces = (rows16 / 16 + NW - 1) / NW;  // uniform: the pieces any thread has
  int xoff[Tile::X_PIECES], hwoff[Tile::X_PIECES];
  unsigned xmode = 0;  // 2 bits a piece: 0 zeros, 1 x, 2 history, 3 not staged
  const bool hist_rows = p.hist != nullptr && !p.hist_cold;
  const bool may_write_history = p.hist != nullptr && n_tile == 0 && H > 0;
#pragma unroll
  for (int u = 0; u < Tile::X_PIECES; ++u) {
    const int r = (tid >> 2) + u * 16 * NW;
    const int lq8 = ((tid & 3) ^ ((r >> 1) & 3)) * 8;
    int off = 0, hw = -1;
    unsigned mode = 3;
    if (u < pieces && r < rows) {
      mode = 0;
      int b, pos;
      bool row_start;  // the tile holds position 0 of row b
      if (r < first + halo) {
        b = b0;
        pos = lo0 - lpad + r;
        row_start = lo0 == 0;
      } else {
        const int rr = r - (first + halo);
        const int s = rr / seg_rows;
        b = b0 + 1 + s;
        pos = rr - s * seg_rows - lpad;
        row_start = true;
      }
      int64_t slot = -1, parity = 0;
      if (p.hist != nullptr) {
        slot = p.slot_index[b];
        if (slot >= p.hist_slots) slot = -1;
        if (slot >= 0) parity = p.slot_parity[slot] & 1;
      }
      if (pos >= 0 && pos < XL) {
        off = (int)(b * p.x_sb + (int64_t)pos * p.x_st) + lq8;
        mode = 1;
      } else if (pos < 0 && slot >= 0 && !p.hist_cold) {
        off = (int)(slot * p.hist_slot_stride + (parity * H + (H + pos)) * (int64_t)c_in) + lq8;
        mode = 2;
      }
      if (may_write_history && slot >= 0 && pos >= XL - H && pos < XL) {
        const int64_t m = (int64_t)b * L + pos;
        const bool owned = pos >= 0 ? (m >= m0 && m < m_end) : row_start;
        if (owned)
          hw = (int)(slot * p.hist_slot_stride +
                     ((1 - parity) * H + (pos - (XL - H))) * (int64_t)c_in) + lq8;
      }
    }
    xoff[u] = off;
    hwoff[u] = hw;
    xmode |= mode << (2 * u);
  }

  const auto x_rsrc = buffer_rsrc(p.x, p.x_bytes);
  const auto h_rsrc = buffer_rsrc(p.hist, p.hist_bytes);
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  auto xs_of = [&](int c) __attribute__((always_inline)) -> u16* { return lds + c * rows16 * kChunk; };

  // chunks c0 .. of the input rows into the LDS: the rows from x, those of the history (their DMA
  // with the non-temporal hint: see conv_dma_kernel), and zeros for the rows left of the stream
  // (and past x). Piece by piece, each lane's choice made once for all chunks: made per chunk, its
  // branches took 350 cycles a chunk.
  auto stage_slab = [&](int c0) __attribute__((always_inline)) {
    const int count = min(slab_chunks, chunks - c0);
    const int step = rows16 * kChunk;  // LDS elements of a chunk
#pragma unroll
    for (int u = 0; u < Tile::X_PIECES; ++u) {
      if (u >= pieces) break;
      u16* dst = lds + (wave + u * NW) * 64 * 8;
      const unsigned mode = (xmode >> (2 * u)) & 3u;
      if (mode == 1u) {
#pragma unroll 4
        for (int c = 0; c < count; ++c)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(x_rsrc, (lds_ptr_t)(dst + c * step), 16,
                                                   (int)((uint32_t)xoff[u] * 2u),
                                                   (int)((uint32_t)(c0 + c) * (kChunk * 2)), 0, 0);
      } else if (mode == 2u) {
#pragma unroll 4
        for (int c = 0; c < count; ++c)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(h_rsrc, (lds_ptr_t)(dst + c * step), 16,
                                                   (int)((uint32_t)xoff[u] * 2u),
                                                   (int)((uint32_t)(c0 + c) * (kChunk * 2)), 0, 2);
      } else if (mode == 0u && c0 == 0) {
        u16* zero = lds + ((tid >> 2) + u * 16 * NW) * kChunk + q8;
#pragma unroll 4
        for (int c = 0; c < slab_chunks; ++c)
          *reinterpret_cast<u32x4*>(zero + c * step) = u32x4{0u, 0u, 0u, 0u};
      }
    }
  };
  // the slab's new history samples, from LDS to the slot's other copy
  auto write_history = [&](int c0) __attribute__((always_inline)) {
    const int count = min(slab_chunks, chunks - c0);
#pragma unroll
    for (int u = 0; u < Tile::X_PIECES; ++u)
      if (u < pieces && may_write_history && hwoff[u] >= 0)
        for (int c = 0; c < count; ++c)
          __builtin_amdgcn_raw_buffer_store_b128(
              *reinterpret_cast<const u32x4*>(xs_of(c) + ((tid >> 2) + u * 16 * NW) * kChunk + q8),
              h_rsrc, (uint32_t)(hwoff[u] + (c0 + c) * kChunk) * 2, 0, 0);
  };
  stage_slab(0);

  // This lane's epilogue coefficients (columns n .. n + 3) and its positions
  const int n = n_wave + lq * 4;
  const bool live = n < n_cols;  // n_cols is a multiple of 16
  const int co = live ? n % p.c_out : 0;
  f32x4 sc = f32x4{1.f, 1.f, 1.f, 1.f}, bi = f32x4{0.f, 0.f, 0.f, 0.f}, aa = bi, ab = bi;
  if (live) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (p.wscale) sc[e] = p.wscale[n + e];
      if (p.bias) bi[e] = p.bias[co + e];
      if (p.act_a) aa[e] = p.act_a[co + e] * kInvTwoPi;
      if (p.act_b) ab[e] = p.act_b[co + e];
    }
  }
  // byte offset in a chunk's rows of what the lane reads for each tap and position (computed once:
  // a wave alone on its SIMD issues an instruction every four cycles at best, so the steps are
  // bound by their instructions)
  uint32_t xread[TAPS][TP];
  uint32_t roff[TP], ooff[TP];
  const uint32_t rsize = p.r_f16 ? 2u : 4u, osize = p.out_bf16 ? 2u : 4u;
#pragma unroll
  for (int t = 0; t < TP; ++t) {
    const int m = m0 + t * 16 + lrow;
    const bool ok = m < m_end;
    const int b = ok ? m / L : b0, i = ok ? m - b * L : lo0;
#pragma unroll
    for (int j = 0; j < TAPS; ++j) {
      const int row = (ok ? (m - m0) + (b - b0) * halo : 0) + j * dil;
      xread[j][t] = (uint32_t)(row * kChunk * 2 + (((lq ^ (row >> 1)) & 3) << 4));
    }
    const bool st = ok && live;
    roff[t] = st ? (uint32_t)(b * p.r_sb + (int64_t)i * p.r_st + n) * rsize : kOutOfRange;
    ooff[t] = st ? (uint32_t)(b * p.o_sb + (int64_t)i * p.o_st + n) * osize : kOutOfRange;
  }
  u32x4 res[TP];
  if (p.residual) {
    const auto rr = buffer_rsrc(p.residual, p.r_bytes);
#pragma unroll
    for (int t = 0; t < TP; ++t) res[t] = load_residual4_raw(rr, roff[t], p.r_f16);
  }

  f32x4 acc[TP], total[TP];
#pragma unroll
  for (int t = 0; t < TP; ++t) acc[t] = total[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int split_groups = SPLIT ? groups / p.k_splits : 0;
  int slab0 = 0, split_end = split_groups;

  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the slab (and the first weights) are in
  __syncthreads();
  // UNIT: the k = 1 conv's weights for the wave's columns, all on their way under the k = 7 conv
  constexpr int kUnitChunks = UNIT ? 16 * NW / kChunk : 1;
  u32x4 w2[kUnitChunks];
  if constexpr (UNIT) {
    const auto w2_rsrc = buffer_rsrc(p.weight2, p.w2_bytes);
#pragma unroll
    for (int c = 0; c < kUnitChunks; ++c)
      w2[c] = __builtin_amdgcn_raw_buffer_load_b128(w2_rsrc, (uint32_t)(n_w * 64 + lq * 16),
                                                    (uint32_t)(c * 16 * NW * 64), 0);
  }
  typedef bf16x8 xreg_t[Tile::STEPS][TP];
  auto read_rows = [&](int g, xreg_t& bv) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < Tile::STEPS; ++k) {
      const uint8_t* xs = reinterpret_cast<const uint8_t*>(xs_of(g * GC - slab0 + k / TAPS));
#pragma unroll
      for (int t = 0; t < TP; ++t)
        bv[k][t] = *reinterpret_cast<const bf16x8*>(xs + xread[k % TAPS][t]);
    }
  };
  auto multiply = [&](int g, const wreg_t (&wg)[Tile::STEPS], const xreg_t& bv)
      __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < Tile::STEPS; ++k) {
      const bf16x8 a = __builtin_bit_cast(bf16x8, wg[k]);
#pragma unroll
      for (int t = 0; t < TP; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bv[k][t], acc[t], 0, 0, 0);
    }
    if (SPLIT && g + 1 == split_end) {
      // a K slice is done: slices add up in order, each summed from zero
#pragma unroll
      for (int t = 0; t < TP; ++t) {
        total[t] = split_end == split_groups ? acc[t] : total[t] + acc[t];
        acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
      split_end += split_groups;
    }
  };
  // (three waves a SIMD hide each other's LDS reads, and have no registers to read ahead)
  constexpr bool AHEAD = !UNIT;
  xreg_t bv[AHEAD ? 2 : 1];
  // whole blocks of D groups: the weights D - 1 groups ahead, the rows one group ahead
  const int blocks = groups / D;
  for (int blk = 0; blk < blocks; ++blk) {
    if (blk * D * GC == slab0 + slab_chunks) {
      // the next slab (of whole blocks): every wave has read this one, its history rows are out
      write_history(slab0);
      __syncthreads();
      slab0 += slab_chunks;
      stage_slab(slab0);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
    }
    if (AHEAD) read_rows(blk * D, bv[0]);
#pragma unroll
    for (int i = 0; i < D; ++i) {
      const int g = blk * D + i;
      load_group(g + D - 1, w[(i + D - 1) % D]);
      if constexpr (AHEAD) {
        if (i + 1 < D) read_rows(g + 1, bv[(i + 1) & 1]);
        multiply(g, w[i], bv[i & 1]);
      } else {
        read_rows(g, bv[0]);
        multiply(g, w[i], bv[0]);
      }
    }
  }
  // the last groups, their weights on the way already
  if (blocks * D < groups && blocks * D * GC == slab0 + slab_chunks) {
    write_history(slab0);
    __syncthreads();
    slab0 += slab_chunks;
    stage_slab(slab0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < D - 1; ++i)
    if (blocks * D + i < groups) {
      read_rows(blocks * D + i, bv[0]);
      multiply(blocks * D + i, w[i], bv[0]);
    }
  write_history(slab0);

  if constexpr (UNIT) {
    // h = mid_act(acc * scale + bias) as bf16 rows beside the slab, then the k = 1 conv over it
    u16* hs = lds + slab_chunks * rows16 * kChunk;
    f32x4 ma = f32x4{0.f, 0.f, 0.f, 0.f}, mb = ma;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (p.mid_a) ma[e] = p.mid_a[co + e] * kInvTwoPi;
      if (p.mid_b) mb[e] = p.mid_b[co + e];
    }
#pragma unroll
    for (int t = 0; t < TP; ++t) {
      float y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        y[e] = operand_act(p.mid_act, acc[t][e] * sc[e] + bi[e], ma[e], mb[e], p.mid_slope);
      const int pos = t * 16 + lrow;
      const int slot = ((n & 31) >> 3) ^ ((pos >> 1) & 3);
      *reinterpret_cast<u32x2*>(hs + ((n >> 5) * Tile::BP + pos) * kChunk + slot * 8 + (n & 7)) =
          u32x2{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
      acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      sc[e] = p.wscale2 ? p.wscale2[n + e] : 1.f;
      bi[e] = p.bias2 ? p.bias2[co + e] : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < kUnitChunks; ++c)
#pragma unroll
      for (int t = 0; t < TP; ++t) {
        const int pos = t * 16 + lrow;
        const bf16x8 hv = *reinterpret_cast<const bf16x8*>(
            hs + (c * Tile::BP + pos) * kChunk + ((lq ^ ((pos >> 1) & 3)) << 3));
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w2[c]), hv,
                                                         acc[t], 0, 0, 0);
      }
  }

  // conv_epilogue's arithmetic on the accumulator layout: lane = position, 4 columns
  const auto ra = buffer_rsrc(p.mix_a, p.mix_a ? p.r_bytes : 0);
  const auto rb = buffer_rsrc(p.mix_b, p.mix_a ? p.r_bytes : 0);
  const auto rs = buffer_rsrc(p.sum_out, p.sum_out ? p.r_bytes : 0);
  const auto ro = buffer_rsrc(p.out, p.o_bytes);
#pragma unroll
  for (int t = 0; t < TP; ++t) {
    f32x4 v = SPLIT ? total[t] : acc[t];
    v = v * sc + bi;
    if (p.residual) v += widen_residual4(res[t], p.r_f16);
    if (p.mix_a) {
      const f32x4 ma = load_residual4(ra, roff[t], p.r_f16);
      const f32x4 mb = load_residual4(rb, roff[t], p.r_f16);
      v = ((ma + mb) + v) * p.mix_scale;
    }
    if (p.sum_out) store_residual4(v, rs, roff[t], p.r_f16);
    if (p.out != nullptr) {
      const int act = p.act;
      if (act == OMNI_ACT_SNAKE) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = snake_rev(v[e], aa[e], ab[e]);
      } else if (act == OMNI_ACT_LEAKY_RELU) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = v[e] >= 0.f ? v[e] : v[e] * p.slope;
      } else if (act != OMNI_ACT_NONE) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = apply_act(act, v[e], 0.f, 0.f, p.slope);
      }
      if (p.out_bf16)
        __builtin_amdgcn_raw_buffer_store_b64(
            u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])}, ro, ooff[t], 0, 0);
      else
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), ro, ooff[t], 0, 0);
    }
  }
}

template <int TAPS, int TP, int NW, int GC, int D>
struct SmallConfig {
  using Tile = SmallTile<TAPS, TP, NW, GC, D>;

  static int64_t rows_needed(const ConvParams& p) {
    int64_t nseg = (Tile::BP + p.length - 2) / p.length + 1;
    if (nseg > p.batch) nseg = p.batch;
    return Tile::BP + nseg * p.halo;
  }
  // chunks staged at once: all of them, or as many whole blocks of D groups as the LDS holds
  static int slab_chunks(const ConvParams& p) {
    const int64_t rows16 = (rows_needed(p) + 15) / 16 * 16;
    const int64_t most = kSmallLdsBytes / (rows16 * kChunk * 2);
    const int64_t chunks = p.c_in / kChunk;
    return (int)(most >= chunks ? chunks : most / (GC * D) * (GC * D));
  }
  static bool fits(const ConvParams& p) {
    return p.taps == TAPS && p.c_in % (kChunk * GC) == 0 &&
           p.c_in / (kChunk * GC) % p.k_splits == 0 && rows_needed(p) <= Tile::kMaxRows &&
           slab_chunks(p) > 0 && (p.k_splits == 1 || TAPS == 7);
  }
  static int64_t workgroups(const ConvParams& p) {
    const int64_t positions = (int64_t)p.batch * p.length;
    return ((positions + Tile::BP - 1) / Tile::BP) * ((p.n_cols + Tile::BCO - 1) / Tile::BCO);
  }
  // The launch's time in us, fitted to measurements over the decoder's layers (1 x 4 to 32 x 12
  // frames; within 25 %): what a workgroup reads at 80 KB per us, its steps' instructions, its
  // epilogue, times the workgroups of the fullest CU (also where its LDS holds several at once: 288
  // of 4 waves at 768 -> 3072 columns, two taps, 96 positions take 19.6 us, 192 of 2 waves 12.1).
  // A CU holds eight waves of one tap (two a SIMD): further workgroups start, and wait for their
  // first loads, when those are done (192 -> 192 columns, 4 waves of 32 positions: 237 workgroups
  // 6.1 us, 471 7.1, 564 10.2; the LDS-DMA tile of 96 x 192 9.5).
  static double microseconds(const ConvParams& p) {
    const double rows = (double)rows_needed(p), steps = (double)(p.c_in / kChunk) * TAPS;
    const double us = (steps * Tile::BCO * Tile::ES + rows * p.c_in * 2) / 80e3 +
                      TP * (0.018 * steps + 0.4);
    const int64_t per_cu = (workgroups(p) + 255) / 256;
    const int64_t starts = TAPS == 1 ? (per_cu * NW + 7) / 8 : 1;
    return 3.0 * starts + us * per_cu;
  }
  static int launch(ConvParams p, hipStream_t stream) {
    const int64_t positions = (int64_t)p.batch * p.length;
    p.p_tiles = (int)((positions + Tile::BP - 1) / Tile::BP);
    p.n_tiles = (int)((p.n_cols + Tile::BCO - 1) / Tile::BCO);
    const int rows16 = (int)((rows_needed(p) + 15) / 16 * 16), slab = slab_chunks(p);
    constexpr bool kSplits = TAPS == 7;  // the layers that run in K slices
    auto k = kSplits && p.k_splits > 1 ? conv_small_kernel<TAPS, TP, NW, GC, D, kSplits, false>
                                       : conv_small_kernel<TAPS, TP, NW, GC, D, false, false>;
    static const bool raised =
        raise_lds_limit((const void*)conv_small_kernel<TAPS, TP, NW, GC, D, kSplits, false>) &&
        raise_lds_limit((const void*)conv_small_kernel<TAPS, TP, NW, GC, D, false, false>);
    (void)raised;
    hipLaunchKernelGGL(k, dim3((unsigned)(p.p_tiles * p.n_tiles)), dim3(Tile::NT),
                       (size_t)rows16 * slab * kChunk * 2, stream, p, rows16, slab);
    OMNI_LAUNCH_CHECK();
    return OMNI_OK;
  }
};

// A residual unit (k = 7 conv, activation, k = 1 conv) of 16 NW channels in one workgroup per tile
// of positions: every column's wave keeps its part of h in LDS for the others.
template <int TP, int NW, int D>
struct SmallUnitConfig {
  using Tile = SmallTile<7, TP, NW, 1, D>;
  using Conv = SmallConfig<7, TP, NW, 1, D>;

  static size_t lds_bytes(const ConvParams& p) {
    const size_t rows16 = (Conv::rows_needed(p) + 15) / 16 * 16;
    return (rows16 + Tile::BP) * p.c_in * 2;  // every channel's rows, then h
  }
  static bool fits(const ConvParams& p) {
    return p.taps == 7 && p.k_splits == 1 && p.c_in == Tile::BCO && p.n_cols == Tile::BCO &&
           p.c_out == Tile::BCO && p.weight2 != nullptr &&
           Conv::rows_needed(p) <= Tile::kMaxRows && lds_bytes(p) <= 160 * 1024;
  }
  static int64_t workgroups(const ConvParams& p) {
    return ((int64_t)p.batch * p.length + Tile::BP - 1) / Tile::BP;
  }
  // 16.4 to 18.9 us a round as it fills (18.6 to 22 in the LDS-DMA form's tiles of 64 positions)
  static double microseconds(const ConvParams& p) { return 17.0 * ((workgroups(p) + 255) / 256); }
  static int launch(ConvParams p, hipStream_t stream) {
    p.p_tiles = (int)workgroups(p);
    p.n_tiles = 1;
    const int rows16 = (int)((Conv::rows_needed(p) + 15) / 16 * 16);
    auto k = conv_small_kernel<7, TP, NW, 1, D, false, true>;
    static const bool raised = raise_lds_limit((const void*)k);
    (void)raised;
    hipLaunchKernelGGL(k, dim3((unsigned)p.p_tiles), dim3(Tile::NT), lds_bytes(p), stream, p, rows16,
                       p.c_in / kChunk);
    OMNI_LAUNCH_CHECK();
    return OMNI_OK;
  }
};

// Launch the entry of the least time if that is well below `than` us (the estimates are good to 15 %
// near the crossing; a forced entry runs whatever it takes); OMNI_ERR_UNSUPPORTED otherwise.
template <typename... Cfgs>
int launch_small_list(const ConvParams& p, double than, Choice& ch, hipStream_t stream) {
  constexpr int n = sizeof...(Cfgs);
  const bool fits[n] = {Cfgs::fits(p)...};
  const int64_t wgs[n] = {Cfgs::workgroups(p)...};
  int (*const launch[n])(ConvParams, hipStream_t) = {&Cfgs::launch...};
  int pick = -1;
  if (ch.force == 0) {
    than /= 1.15;
    double (*const microseconds[n])(const ConvParams&) = {&Cfgs::microseconds...};
    for (int i = 0; i < n; ++i) {
      if (!fits[i]) continue;
      const double us = microseconds[i](p);
      if (us < than) pick = i, than = us;
    }
    if (pick < 0) return OMNI_ERR_UNSUPPORTED;
  }
  return choose_and_launch(ch, n, fits, wgs, launch, pick, p, stream);
}

// 16, 32 or 64 positions by one, two or four waves of 16 columns, one translation unit per tap
// count, and the residual unit.
int launch_small_taps1(const ConvParams& p, double than, Choice& ch, hipStream_t stream);
int launch_small_taps2(const ConvParams& p, double than, Choice& ch, hipStream_t stream);
int launch_small_taps7(const ConvParams& p, double than, Choice& ch, hipStream_t stream);
int launch_small_unit(const ConvParams& p, double than, Choice& ch, hipStream_t stream);

}  // namespace omni_conv
