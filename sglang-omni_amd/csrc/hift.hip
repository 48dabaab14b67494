// HiFT's short-time Fourier transform and its inverse (the iSTFT tail of the CosyVoice3 /
// MiniCPM-o vocoders), on gfx950. Both are near HBM-bound: a 16-point transform does 16 MACs per
// output component, so the kernels read their input once, keep the workgroup's window of frames
// in LDS, and give every output one fixed summation order (so a row's result does not depend on
// the batch or the tiling). HiFT's geometry (n_fft 16, hop 4) has its
// own instantiation with the loops unrolled; other sizes take the runtime-sized kernels.
//
//   short_time_spectrum: spectrum[r, c, f] = sum_{k < n_fft} x[r, f * hop + k - pad] * basis[c, k]
//     (c < bins the windowed cosines, c >= bins the windowed negative sines; pad = n_fft / 2 with
//     reflection when centring, else the caller's signal is already padded)
//   overlap_add_inverse: y[r, i] = (sum_{frames f over i} sum_{b < bins} re[r, b, f] *
//     ibasis[b, t] + im[r, b, f] * ibasis[bins + b, t]) / (sum_f window[t]^2), t = i + n_fft / 2 -
//     f * hop (torch.istft with center = True)
//   istft_tail: the same inverse fed straight from the vocoder's last conv, channels-last
//     h[r, f, 2 * bins]: magnitude = min(exp(h[.., b]), mag_clip), phase = sin(h[.., bins + b]),
//     re = magnitude * cos(phase), im = magnitude * sin(phase), and the output clamped to
//     +-audio_limit (hift_channels_last.py:269-276 with hift_channels_last.py:117-125).
#include "common.h"

namespace {

constexpr int kMaxFft = 64;
constexpr int kThreads = 256;
constexpr int kFramesPerBlock = 256;   // spectrum: frames per workgroup (one per thread)
constexpr int kSamplesPerBlock = 256;  // inverse: output samples per workgroup (one per thread)

// Reflection of index i into [0, n) (torch's "reflect" padding: the edge sample is not repeated).
__device__ __forceinline__ int64_t reflect(int64_t i, int64_t n) {
  if (n == 1) return 0;
  const int64_t period = 2 * (n - 1);
  i = i % period;
  if (i < 0) i += period;
  return i < n ? i : period - i;
}

struct StftParams {
  const float* x;
  int64_t x_stride;  // elements between rows
  int64_t samples;   // samples per row of x
  int center;        // 1: reflect-pad by n_fft / 2 here; 0: x is already padded
  const float* basis;  // [2 * bins][n_fft]
  int n_fft, hop, bins;
  int64_t frames;
  float* out;  // [rows][2 * bins][frames]
};

// Dynamic LDS: the basis [2 * bins][n_fft], then the block's signal span.
size_t stft_lds_bytes(int n_fft, int hop, int bins) {
  return (size_t)(2 * bins * n_fft + (kFramesPerBlock - 1) * hop + n_fft) * sizeof(float);
}

// NF, HP: the transform's n_fft and hop when known at compile time (the loops unroll and the
// frame's samples stay in registers), 0 for the runtime values of the parameters.
template <int NF, int HP>
__global__ void __launch_bounds__(kThreads) short_time_spectrum_kernel(const StftParams p) {
  extern __shared__ float smem[];
  const int n_fft = NF ? NF : p.n_fft;
  const int hop = HP ? HP : p.hop;
  const int bins = n_fft / 2 + 1;
  const int comps = 2 * bins;
  float* basis = smem;
  float* seg = smem + comps * n_fft;
  const int tid = threadIdx.x;
  const int64_t row = blockIdx.y;
  const int64_t f0 = (int64_t)blockIdx.x * kFramesPerBlock;
  if constexpr (NF == 0)
    for (int e = tid; e < comps * n_fft; e += kThreads) basis[e] = p.basis[e];
  // the block's signal span: frames f0 .. f0 + kFramesPerBlock - 1 read padded samples
  // f0 * hop .. (f0 + kFramesPerBlock - 1) * hop + n_fft - 1
  const int64_t nframes = min((int64_t)kFramesPerBlock, p.frames - f0);
  const int span = (int)((nframes - 1) * hop + n_fft);
  const int pad = p.center ? n_fft / 2 : 0;
  const float* xr = p.x + row * p.x_stride;
  for (int e = tid; e < span; e += kThreads) {
    int64_t i = f0 * hop + e - pad;
    if (p.center) i = reflect(i, p.samples);
    seg[e] = xr[i];
  }
  __syncthreads();
  if (tid >= nframes) return;
  float* o = p.out + (row * comps) * p.frames + f0 + tid;
  if constexpr (NF != 0) {
    // the bases are the same for every thread: read through the constant address space, they
    // arrive by scalar loads and feed the FMAs as scalar operands (no LDS traffic)
    typedef __attribute__((address_space(4))) const float cfloat;
    cfloat* gbasis = (cfloat*)(p.basis);
    float s[NF];
#pragma unroll
    for (int k = 0; k < NF; ++k) s[k] = seg[tid * hop + k];
#pragma unroll 2
    for (int c = 0; c < comps; ++c) {
      cfloat* b = gbasis + c * NF;
      float acc = 0.f;
#pragma unroll
      for (int k = 0; k < NF; ++k) acc = __builtin_fmaf(s[k], b[k], acc);
      o[(int64_t)c * p.frames] = acc;
    }
  } else {
    const float* s = seg + tid * hop;
    for (int c = 0; c < comps; ++c) {
      const float* b = basis + c * n_fft;
      float acc = 0.f;
      for (int k = 0; k < n_fft; ++k) acc = __builtin_fmaf(s[k], b[k], acc);
      o[(int64_t)c * p.frames] = acc;
    }
  }
}

struct IstftParams {
  // spectrum source: either separate real / imaginary [rows][bins][frames] (tail = 0), or the
  // vocoder's channels-last conv output h [rows][frames][h_stride] (tail = 1)
  const float* re;
  const float* im;
  const float* h;
  int64_t h_row_stride, h_frame_stride;
  int tail;
  float mag_clip, audio_limit;
  const float* basis;     // [2 * bins][n_fft], the one-sided inverse's windowed bases / n_fft
  const float* win2;      // [n_fft] squared window
  int n_fft, hop, bins;
  int64_t frames, samples;
  float* out;  // [rows][out_stride]
  int64_t out_stride;
};

// The frames one inverse workgroup reads: its samples' padded positions span
// (kSamplesPerBlock - 1) / hop + 1 frame starts, plus n_fft / hop - 1 earlier overlapping frames.
int inverse_frames_per_block(int n_fft, int hop) {
  return (kSamplesPerBlock - 1) / hop + n_fft / hop + 1;
}

// Dynamic LDS: the basis [2 * bins][n_fft], the squared window [n_fft], then the workgroup's
// frames [nf][2 * bins].
size_t inverse_lds_bytes(int n_fft, int hop, int bins) {
  return (size_t)(2 * bins * n_fft + n_fft + inverse_frames_per_block(n_fft, hop) * 2 * bins) *
         sizeof(float);
}

template <int NF, int HP>
__global__ void __launch_bounds__(kThreads) overlap_add_inverse_kernel(const IstftParams p) {
  extern __shared__ float smem[];
  const int n_fft = NF ? NF : p.n_fft;
  const int hop = HP ? HP : p.hop;
  const int bins = n_fft / 2 + 1;
  const int comps = 2 * bins;
  const int half = n_fft / 2;
  const int overlaps = n_fft / hop;
  float* basis = smem;
  float* win2 = basis + comps * n_fft;
  float* spec = win2 + n_fft;
  const int tid = threadIdx.x;
  const int64_t row = blockIdx.y;
  const int64_t i0 = (int64_t)blockIdx.x * kSamplesPerBlock;
  for (int e = tid; e < comps * n_fft; e += kThreads) basis[e] = p.basis[e];
  for (int e = tid; e < n_fft; e += kThreads) win2[e] = p.win2[e];
  // frames whose window covers samples i0 .. i0 + kSamplesPerBlock - 1 (padded positions
  // i + half): from (i0 + half) / hop - (overlaps - 1) to (i0 + kSamplesPerBlock - 1 + half) / hop
  const int64_t fa = (i0 + half) / hop - (overlaps - 1);
  const int64_t fb = (i0 + kSamplesPerBlock - 1 + half) / hop;
  const int nf = (int)(fb - fa + 1);
  if (p.tail) {
    // one thread per (frame, bin): magnitude and phase once, both parts out
    for (int e = tid; e < nf * bins; e += kThreads) {
      const int j = e / bins;  // frame within the window
      const int b = e - j * bins;
      const int64_t f = fa + j;
      float re = 0.f, im = 0.f;
      if (f >= 0 && f < p.frames) {
        const float* hf = p.h + row * p.h_row_stride + f * p.h_frame_stride;
        const float mag = fminf(expf(hf[b]), p.mag_clip);
        const float phase = sinf(hf[bins + b]);
        re = mag * cosf(phase);
        im = mag * sinf(phase);
      }
      spec[j * comps + b] = re;
      spec[j * comps + bins + b] = im;
    }
  } else {
    for (int e = tid; e < nf * comps; e += kThreads) {
      const int j = e / comps;  // frame within the window
      const int c = e - j * comps;
      const int64_t f = fa + j;
      float v = 0.f;
      if (f >= 0 && f < p.frames) {
        const float* src = c < bins ? p.re : p.im;
        const int b = c < bins ? c : c - bins;
        v = src[(row * bins + b) * p.frames + f];
      }
      spec[j * comps + c] = v;
    }
  }
  __syncthreads();
  const int64_t i = i0 + tid;
  if (i >= p.samples) return;
  const int64_t pos = i + half;
  float signal = 0.f, envelope = 0.f;
#pragma unroll
  for (int o = 0; o < (NF ? NF / HP : kMaxFft); ++o) {
    if (!NF && o >= overlaps) break;
    const int64_t f = pos / hop - o;
    if (f < 0 || f >= p.frames) continue;
    const int t = (int)(pos - f * hop);
    const float* s = spec + (int)(f - fa) * comps;
#pragma unroll
    for (int b = 0; b < (NF ? NF / 2 + 1 : kMaxFft / 2 + 1); ++b) {
      if (!NF && b >= bins) break;
      signal += __builtin_fmaf(s[b], basis[b * n_fft + t],
                               s[bins + b] * basis[(bins + b) * n_fft + t]);
    }
    envelope += win2[t];
  }
  float y = signal / envelope;
  if (p.tail) y = fminf(fmaxf(y, -p.audio_limit), p.audio_limit);
  p.out[row * p.out_stride + i] = y;
}

// The tail's exp, sin and cos. The general library functions took 27 of the tail's 44 us (every
// call carries its argument's whole range reduction and, for sine and cosine, both polynomials).
// These take fewer instructions and are no further from the true value: in units of the last place,
// largest and root mean square error over 2^24 arguments, library and here: exp on [-103, 88] 0.89,
// 0.300 and 0.89, 0.300; sin to 2^15 1.58, 0.375 and 1.52, 0.360; of [-1, 1] the sine 1.05, 0.307
// and 0.76, 0.292, the cosine 0.87, 0.340 and 0.78, 0.299.

// exp(x) = 2^k 2^f: x log2 e as a rounded product and what it lost (log2 e in two floats), k the
// integer next to it, f the rest, rounded once. x is clamped to where exp is 0 or infinite beyond;
// NaN gives what the caller's clip makes of infinity.
__device__ __forceinline__ float tail_exp(float x) {
#pragma clang fp contract(off)
  x = fmaxf(fminf(x, 150.f), -150.f);
  const float hi = x * 1.4426950216293335f;
  const float lo = __builtin_fmaf(x, 1.925963033500011e-08f,
                                  __builtin_fmaf(x, 1.4426950216293335f, -hi));
  const float k = rintf(hi);
  return __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f((hi - k) + lo), (int)k);
}

// sin(x): r = x - k pi / 2 in three fused steps (pi / 2 as three floats), then on [-pi/4, pi/4] an
// odd polynomial of r where k is even and an even one where it is odd (least maximum relative errors,
// 4e-9 and 1e-10, fitted with the leading coefficients fixed), the sign of k / 2's parity. (One
// polynomial on [-pi/2, pi/2] is off by 2.1 units near pi/2 however well it is fitted: its terms
// cancel there.) Beyond 2^15, and for infinities and NaN, the library's.
__device__ __forceinline__ float tail_sin(float x) {
  if (!(fabsf(x) < 32768.f)) return sinf(x);
  const float k = rintf(x * 0.6366197466850281f);
  float r = __builtin_fmaf(-k, 1.5707963705062866f, x);
  r = __builtin_fmaf(-k, -4.371138828673793e-08f, r);
  r = __builtin_fmaf(-k, -1.7151245100058819e-15f, r);
  const uint32_t n = (uint32_t)(int)k;
  const bool odd = n & 1u;
  const float z = r * r;
  float q = __builtin_fmaf(z, odd ? 2.4432327336398885e-05f : 0.f,
                           odd ? -0.0013887309469282627f : -0.00019518287444952875f);
  q = __builtin_fmaf(z, q, odd ? 0.04166664555668831f : 0.008332189172506332f);
  q = __builtin_fmaf(z, q, odd ? -0.5f : -0.16666655242443085f);
  r = __builtin_fmaf(odd ? z : r * z, q, odd ? 1.f : r);
  return __uint_as_float(__float_as_uint(r) ^ (n >> 1 << 31));
}

// sin and cos of p in [-1, 1] (a sine's value): polynomials fitted there (3e-10 and 1.5e-9). The cosine
// adds 1 - p^2 / 2 and what its rounding lost apart from the rest.
__device__ __forceinline__ void tail_sincos(float p, float& sn, float& cs) {
  const float z = p * p;
  float q = __builtin_fmaf(z, 2.7262710773356957e-06f, -0.00019842384790536016f);
  q = __builtin_fmaf(z, q, 0.008333354257047176f);
  q = __builtin_fmaf(z, q, -0.1666666716337204f);
  sn = __builtin_fmaf(p * z, q, p);
  float c = __builtin_fmaf(z, 2.4201613996410742e-05f, -0.001388469710946083f);
  c = __builtin_fmaf(z, c, 0.04166657477617264f);
  const float h = __builtin_fmaf(z, -0.5f, 1.f);
  const float lost = __builtin_fmaf(z, -0.5f, 1.f - h);
  cs = h + __builtin_fmaf(z * z, c, lost);
}

// HiFT's geometry (n_fft 16, hop 4, 9 bins), 1 024 samples a workgroup. The window's frames go to
// LDS as rows of 18 components (the tail's input first as it lies in memory, coalesced, then each
// (frame, bin) pair replaced by its real and imaginary part); each 16 frames are transformed on the
// matrix cores (v_mfma_f32_16x16x4_f32, float32 products and sums: D[t][frame] over 20 components,
// two of them zero), which leaves a lane the four consecutive values 4 o .. 4 o + 3 of one frame:
// what that frame adds to the four samples of the quad o hops later. The quads' four parts meet
// through LDS, overlaps ascending, and leave as 16-byte stores. Before, every sample read its four
// frames' 72 components from LDS (16 us of LDS traffic at the size below) and multiplied them on
// the VALU. An output's sum order is fixed: components in the MFMA's order within a frame, then
// overlaps. Bound by: the tail's VALU work per (frame, bin); the inverse, HBM.
// Measured, 16 x 240 000 samples: tail 43.8 -> 28.7 us (84 MB: 2.9 TB/s), inverse 47 -> 23.4
// us; 3 x 5 frames 3.5 and 4.0 -> 3.8 (5.6 and 4.4 with the tail's functions over the whole window).
constexpr int kInv16Quads = kThreads;                  // quads of samples per workgroup
constexpr int kInv16Samples = 4 * kInv16Quads;
constexpr int kInv16Frames = kInv16Quads + 3;          // frames that reach them
constexpr int kInv16Groups = (kInv16Frames + 15) / 16;  // MFMA groups of 16 frames

template <bool TAIL>
__global__ void __launch_bounds__(kThreads) overlap_add_inverse16_kernel(const IstftParams p) {
  constexpr int NF = 16, BINS = 9, COMPS = 18, OV = 4, ROWS = kInv16Groups * 16;
  // the spectra, then (once every wave holds its groups' results) the quads' parts [OV][ROWS]: one
  // buffer, so eight workgroups share a CU
  __shared__ __attribute__((aligned(16))) float spec[ROWS * COMPS];
  static_assert(OV * ROWS * 4 <= ROWS * COMPS, "the parts fit the spectra's buffer");
  f32x4* parts = reinterpret_cast<f32x4*>(spec);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t row = blockIdx.y;
  const int64_t i0 = (int64_t)blockIdx.x * kInv16Samples;
  const int64_t q0 = i0 / 4 + 2;  // the first quad: padded position / 4
  const int64_t fa = q0 - (OV - 1);
  // the window's frames inside the row: lo .. hi - 1 of its kInv16Frames
  const int lo = fa < 0 ? (int)-fa : 0;
  const int hi = (int)min((int64_t)kInv16Frames, p.frames - fa);
  if constexpr (TAIL) {
    const float* hr = p.h + row * p.h_row_stride + fa * p.h_frame_stride;
    if (p.h_frame_stride == COMPS && (reinterpret_cast<uintptr_t>(hr) & 7) == 0) {
      // packed frames: one run of memory, 8 bytes a load, all in flight together
      constexpr int N = kInv16Frames * COMPS / 2, U = (N + kThreads - 1) / kThreads;
      const uint2* src = reinterpret_cast<const uint2*>(hr);
      uint2 v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = tid + u * kThreads;
        v[u] = e >= lo * (COMPS / 2) && e < hi * (COMPS / 2) ? src[e] : uint2{0u, 0u};
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (tid + u * kThreads < N) reinterpret_cast<uint2*>(spec)[tid + u * kThreads] = v[u];
    } else {
      for (int e = lo * COMPS + tid; e < hi * COMPS; e += kThreads) {
        const int j = e / COMPS;
        spec[e] = hr[j * p.h_frame_stride + (e - j * COMPS)];
      }
    }
    __syncthreads();
    // (the row's own frames only: what lies in LDS for the others meets its own column of the
    // product, which nothing reads)
    int j = lo + tid / BINS, b = tid % BINS;
#pragma unroll 3
    for (int e = lo * BINS + tid; e < hi * BINS; e += kThreads) {
      float* s = spec + j * COMPS + b;
      const float mag = fminf(tail_exp(s[0]), p.mag_clip);
      float sn, cs;
      tail_sincos(tail_sin(s[BINS]), sn, cs);
      s[0] = mag * cs;
      s[BINS] = mag * sn;
      j += kThreads / BINS;
      b += kThreads % BINS;
      if (b >= BINS) b -= BINS, ++j;
    }
  } else {
    // component c's run of frames, a thread's frames of every component in flight together
    const int64_t first = row * BINS * p.frames + fa;
    for (int j = tid; j < kInv16Frames; j += kThreads) {
      float v[COMPS];
      const bool real = j >= lo && j < hi;
#pragma unroll
      for (int c = 0; c < COMPS; ++c) {
        const float* src = c < BINS ? p.re : p.im;
        v[c] = real ? src[first + (c % BINS) * p.frames + j] : 0.f;
      }
#pragma unroll
      for (int c = 0; c < COMPS; ++c) spec[j * COMPS + c] = v[c];
    }
  }
  // operand lanes: output t (or frame) lane % 16, component 4 s + lane / 16 of step s
  const int ln = lane & 15, lq = lane >> 4;
  float basis[5];
#pragma unroll
  for (int s = 0; s < 5; ++s) basis[s] = 4 * s + lq < COMPS ? p.basis[(4 * s + lq) * NF + ln] : 0.f;
  __syncthreads();
  constexpr int GROUPS = (kInv16Groups + kThreads / 64 - 1) / (kThreads / 64);  // of a wave
  f32x4 acc[GROUPS];
#pragma unroll
  for (int k = 0; k < GROUPS; ++k) {
    acc[k] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int g = wave + k * (kThreads / 64);
    if (g * 16 >= hi) break;
    const float* sp = spec + (g * 16 + ln) * COMPS + lq;
#pragma unroll
    for (int s = 0; s < 5; ++s) {
      const float v = s < 4 || lq < 2 ? sp[4 * s] : 0.f;  // components 18 and 19 do not exist
      acc[k] = __builtin_amdgcn_mfma_f32_16x16x4f32(basis[s], v, acc[k], 0, 0, 0);
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < GROUPS; ++k) {
    const int g = wave + k * (kThreads / 64);
    if (g * 16 < hi) parts[lq * ROWS + g * 16 + ln] = acc[k];
  }
  __syncthreads();
  const int64_t i = i0 + 4 * tid;
  if (i >= p.samples) return;  // samples come in whole quads: hop * (frames - 1)
  f32x4 signal = f32x4{0.f, 0.f, 0.f, 0.f}, envelope = signal;
#pragma unroll
  for (int o = 0; o < OV; ++o) {
    const int64_t f = q0 + tid - o;
    if (f < 0 || f >= p.frames) continue;
    signal += parts[o * ROWS + tid + OV - 1 - o];
#pragma unroll
    for (int r = 0; r < 4; ++r) envelope[r] += p.win2[4 * o + r];
  }
  float* out = p.out + row * p.out_stride + i;
  f32x4 y;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    y[r] = signal[r] / envelope[r];
    if (TAIL) y[r] = fminf(fmaxf(y[r], -p.audio_limit), p.audio_limit);
  }
  if ((reinterpret_cast<uintptr_t>(out) & 15) == 0) {
    *reinterpret_cast<f32x4*>(out) = y;
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r) out[r] = y[r];
  }
}

bool valid_fft(int64_t n_fft, int64_t hop, int64_t bins) {
  return n_fft >= 2 && n_fft <= kMaxFft && hop >= 1 && hop <= n_fft && n_fft % hop == 0 &&
         bins == n_fft / 2 + 1;
}

}  // namespace

extern "C" int omni_short_time_spectrum(const float* signal, int64_t rows, int64_t samples,
                                        int64_t signal_stride_row, int center,
                                        const float* basis, int64_t bins, int64_t n_fft,
                                        int64_t hop, float* spectrum, int64_t frames,
                                        omni_stream_t stream) {
  if (!signal || !basis || !spectrum) return OMNI_ERR_INVALID_ARG;
  if (rows < 0 || samples < 1 || signal_stride_row < samples || !valid_fft(n_fft, hop, bins))
    return OMNI_ERR_INVALID_ARG;
  const int64_t padded = center ? samples + n_fft : samples;  // 2 * (n_fft / 2) padding
  if (padded < n_fft || frames != (padded - n_fft) / hop + 1) return OMNI_ERR_INVALID_ARG;
  if (center && samples <= n_fft / 2) return OMNI_ERR_INVALID_ARG;  // reflect needs pad < samples
  if (rows == 0) return OMNI_OK;
  if (rows > 65535 || frames > 0x7fffffffLL / kFramesPerBlock) return OMNI_ERR_UNSUPPORTED;
  StftParams p{};
  p.x = signal;
  p.x_stride = signal_stride_row;
  p.samples = samples;
  p.center = center;
  p.basis = basis;
  p.n_fft = (int)n_fft;
  p.hop = (int)hop;
  p.bins = (int)bins;
  p.frames = frames;
  p.out = spectrum;
  dim3 grid((unsigned)((frames + kFramesPerBlock - 1) / kFramesPerBlock), (unsigned)rows);
  const size_t lds = stft_lds_bytes(p.n_fft, p.hop, p.bins);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (p.n_fft == 16 && p.hop == 4)
    hipLaunchKernelGGL((short_time_spectrum_kernel<16, 4>), grid, dim3(kThreads), lds, s, p);
  else
    hipLaunchKernelGGL((short_time_spectrum_kernel<0, 0>), grid, dim3(kThreads), lds, s, p);
  OMNI_LAUNCH_CHECK();
  return OMNI_OK;
}

namespace {

int launch_inverse(IstftParams& p, int64_t rows, omni_stream_t stream) {
  // a workgroup's frame window in LDS stays within the default 64 KiB (HiFT: n_fft 16, hop 4
  // takes 6 KiB)
  if (inverse_lds_bytes(p.n_fft, p.hop, p.bins) > 64 * 1024) return OMNI_ERR_UNSUPPORTED;
  if (rows == 0 || p.samples == 0) return OMNI_OK;
  if (rows > 65535 || p.samples > 0x7fffffffLL - kSamplesPerBlock) return OMNI_ERR_UNSUPPORTED;
  dim3 grid((unsigned)((p.samples + kSamplesPerBlock - 1) / kSamplesPerBlock), (unsigned)rows);
  const size_t lds = inverse_lds_bytes(p.n_fft, p.hop, p.bins);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (p.n_fft == 16 && p.hop == 4) {
    dim3 grid16((unsigned)((p.samples + kInv16Samples - 1) / kInv16Samples), (unsigned)rows);
    hipLaunchKernelGGL(p.tail ? overlap_add_inverse16_kernel<true> : overlap_add_inverse16_kernel<false>,
                       grid16, dim3(kThreads), 0, s, p);
  } else {
    hipLaunchKernelGGL((overlap_add_inverse_kernel<0, 0>), grid, dim3(kThreads), lds, s, p);
  }
  OMNI_LAUNCH_CHECK();
  return OMNI_OK;
}

}  // namespace

extern "C" int omni_overlap_add_inverse(const float* real, const float* imag, int64_t rows,
                                        int64_t bins, int64_t frames, const float* basis,
                                        const float* squared_window, int64_t n_fft, int64_t hop,
                                        float* out, int64_t out_stride_row,
                                        omni_stream_t stream) {
  if (!real || !imag || !basis || !squared_window || !out) return OMNI_ERR_INVALID_ARG;
  if (rows < 0 || frames < 1 || !valid_fft(n_fft, hop, bins)) return OMNI_ERR_INVALID_ARG;
  const int64_t samples = hop * (frames - 1);
  if (out_stride_row < samples) return OMNI_ERR_INVALID_ARG;
  IstftParams p{};
  p.re = real;
  p.im = imag;
  p.basis = basis;
  p.win2 = squared_window;
  p.n_fft = (int)n_fft;
  p.hop = (int)hop;
  p.bins = (int)bins;
  p.frames = frames;
  p.samples = samples;
  p.out = out;
  p.out_stride = out_stride_row;
  return launch_inverse(p, rows, stream);
}

extern "C" int omni_istft_tail(const float* h, int64_t rows, int64_t frames, int64_t h_stride_row,
                               int64_t h_stride_frame, const float* basis,
                               const float* squared_window, int64_t bins, int64_t n_fft,
                               int64_t hop, float magnitude_clip, float audio_limit, float* out,
                               int64_t out_stride_row, omni_stream_t stream) {
  if (!h || !basis || !squared_window || !out) return OMNI_ERR_INVALID_ARG;
  if (rows < 0 || frames < 1 || !valid_fft(n_fft, hop, bins)) return OMNI_ERR_INVALID_ARG;
  if (h_stride_frame < 2 * bins || h_stride_row < frames * h_stride_frame)
    return OMNI_ERR_INVALID_ARG;
  if (!(magnitude_clip > 0.f) || !(audio_limit > 0.f)) return OMNI_ERR_INVALID_ARG;
  const int64_t samples = hop * (frames - 1);
  if (out_stride_row < samples) return OMNI_ERR_INVALID_ARG;
  IstftParams p{};
  p.h = h;
  p.h_row_stride = h_stride_row;
  p.h_frame_stride = h_stride_frame;
  p.tail = 1;
  p.mag_clip = magnitude_clip;
  p.audio_limit = audio_limit;
  p.basis = basis;
  p.win2 = squared_window;
  p.n_fft = (int)n_fft;
  p.hop = (int)hop;
  p.bins = (int)bins;
  p.frames = frames;
  p.samples = samples;
  p.out = out;
  p.out_stride = out_stride_row;
  return launch_inverse(p, rows, stream);
}
