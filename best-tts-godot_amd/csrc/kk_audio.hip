// The waveform's output stage, as runtime/audio.gd:59-106 drives it: the
// notch FIR (kernels/fir.glsl:35-47) and the float -> 16-bit PCM conversion
// (kernels/pcm16.glsl:28-46), separately or fused into one pass.
//
// FIR: y[i] = sum_k h[k] x[clamp(i - center + k, 0, n - 1)], each output's
// taps accumulated in order (k = 0, 1, ...) in fp32 with one fused
// multiply-add per tap: on the fp32 matrix cores (fir_mfma_kernel), and with
// fewer than 32 taps, where that product would be half padding, on the VALU
// (fir_kernel: a block of 256 threads computes 2048 consecutive outputs from
// a window staged in LDS; each thread keeps a 16-sample register window over
// its 8 outputs and slides it 8 taps at a time, the taps coming from the
// scalar cache).
//
// PCM16: round(clamp(x * gain, -1, 1) * 32767) as int16, written as the
// little-endian byte stream the reference reads back (two bytes per
// sample).  GLSL's round() leaves a .5 tie to the implementation; roundf
// rounds it away from zero.
#include <algorithm>
#include <type_traits>

#include "kk_internal.h"

namespace kk {
namespace audio {  // named: the kernels keep readable names in profiles

constexpr int kThreads = 256;
constexpr int kPerThread = 8;                        // consecutive outputs per thread
constexpr int kTile = kThreads * kPerThread;         // outputs per block
constexpr int kMaxTaps = 4096;
constexpr int kMfmaMinTaps = 32;                     // from here on the matrix cores
constexpr int kWindow = kTile + kMfmaMinTaps + 16;   // fir_kernel's: outputs, taps rounded up, slack

__device__ __forceinline__ int16_t to_pcm16(float v, float gain) {
  const float c = fminf(fmaxf(v * gain, -1.0f), 1.0f);
  return static_cast<int16_t>(roundf(c * 32767.0f));
}

// PCM: pcm16 bytes out instead of fp32 (the fused form).
template <bool PCM>
__global__ void __launch_bounds__(kThreads) fir_kernel(const float* __restrict__ x, int64_t n,
                                                       const float* __restrict__ h, int taps,
                                                       int center, float* __restrict__ y,
                                                       int16_t* __restrict__ pcm, float gain) {
  __shared__ __align__(16) float xs[kWindow];
  const int64_t i0 = static_cast<int64_t>(blockIdx.x) * kTile;
  const int taps8 = (taps + 7) & ~7;
  const int span = kTile + taps8 + 8;  // the window the threads read
  for (int j = threadIdx.x; j < span; j += kThreads) {
    int64_t s = i0 - center + j;
    s = s < 0 ? 0 : (s >= n ? n - 1 : s);
    xs[j] = x[s];
  }
  __syncthreads();
  const int j0 = threadIdx.x * kPerThread;
  float acc[kPerThread];
#pragma unroll
  for (int r = 0; r < kPerThread; ++r) acc[r] = 0.0f;
  float win[16];
  {
    const float4 a = *reinterpret_cast<const float4*>(&xs[j0]);
    const float4 b = *reinterpret_cast<const float4*>(&xs[j0 + 4]);
    win[0] = a.x; win[1] = a.y; win[2] = a.z; win[3] = a.w;
    win[4] = b.x; win[5] = b.y; win[6] = b.z; win[7] = b.w;
  }
  // eight taps: slide the window by 8 and accumulate (the taps are the same
  // address in every lane: scalar loads); `tail` guards a partial last chunk
  auto chunk = [&](int k0, auto tail) {
    const float4 a = *reinterpret_cast<const float4*>(&xs[j0 + k0 + 8]);
    const float4 b = *reinterpret_cast<const float4*>(&xs[j0 + k0 + 12]);
    win[8] = a.x; win[9] = a.y; win[10] = a.z; win[11] = a.w;
    win[12] = b.x; win[13] = b.y; win[14] = b.z; win[15] = b.w;
    float hk[8];
#pragma unroll
    for (int kk = 0; kk < 8; ++kk)
      hk[kk] = (!decltype(tail)::value || k0 + kk < taps) ? h[k0 + kk] : 0.0f;
#pragma unroll
    for (int kk = 0; kk < 8; ++kk)
#pragma unroll
      for (int r = 0; r < kPerThread; ++r) acc[r] = __builtin_fmaf(hk[kk], win[r + kk], acc[r]);
#pragma unroll
    for (int q = 0; q < 8; ++q) win[q] = win[q + 8];
  };
  const int full = taps & ~7;
  for (int k0 = 0; k0 < full; k0 += 8) chunk(k0, std::false_type{});
  if (full < taps) chunk(full, std::true_type{});
  const int64_t o = i0 + j0;
  if (o + kPerThread <= n) {
    if (PCM) {
      uint32_t w[4];
#pragma unroll
      for (int q = 0; q < 4; ++q)
        w[q] = static_cast<uint16_t>(to_pcm16(acc[2 * q], gain)) |
               (static_cast<uint32_t>(static_cast<uint16_t>(to_pcm16(acc[2 * q + 1], gain))) << 16);
      *reinterpret_cast<uint4*>(pcm + o) = make_uint4(w[0], w[1], w[2], w[3]);
    } else {
      st_stream4(y + o, make_float4(acc[0], acc[1], acc[2], acc[3]));
      st_stream4(y + o + 4, make_float4(acc[4], acc[5], acc[6], acc[7]));
    }
  } else {
#pragma unroll
    for (int r = 0; r < kPerThread; ++r) {
      if (o + r >= n) break;
      if (PCM) pcm[o + r] = to_pcm16(acc[r], gain);
      else y[o + r] = acc[r];
    }
  }
}

// The FIR on the fp32 matrix cores, for kMfmaMinTaps taps and more.  Outputs in
// tiles of 16 x 16, y[o + 16 i + r] = sum_s T[r][s] x[o + 16 i + s] with the
// Toeplitz matrix T[r][s] = h[s - r] (0 outside the filter): taps + 15 terms
// of which taps count, 1.5% more at 1023 taps.  v_mfma_f32_16x16x4_f32 adds
// its four terms one after another, each a fused multiply-add, so an output
// is the chain of the kernel above, bit for bit (the zeros before and after
// its taps leave it as it is), at twice the VALU's fp32 rate.  (On the bf16
// matrix cores, samples and taps split in three, it took 31 us; its sums are
// closer to 64 bits, but another rounding than the chain's puts 0.23% of the
// PCM16 samples on another step.)
//
// Lane (n, g) = (lane % 16, lane / 16) holds row / column n of k = g, i.e.
// the terms s = 4 j + g of steps j, so the window is kept as four sequences of
// every fourth sample and a lane reads four steps at once; column n's unit of
// four is n after column 0's.  The taps likewise, in four copies shifted by 0
// .. 3 units' quarters, so that row r's reads are aligned too; the sixteen
// sequences start on different banks.
//
// Bound by the matrix cores (2,029,200 samples x 1023 taps: 27.7 us at their
// rate).  A wave takes NC tiles, which share the taps' reads.  Measured, 1023
// taps: 2,029,200 samples 67.4 -> 40.0 us (PCM16 65.1 -> 38.8), 1,060,000
// 52.7 -> 29.5, 400,000 36.0 -> 16.4, 2400 32.1 -> 10.3; 64 taps over
// 1,060,000 7.1 either way, over 24,000 5.2 -> 3.8.
typedef float fir_f4 __attribute__((ext_vector_type(4)));

__host__ __device__ constexpr int fir_units(int taps) { return (taps + 15 + 15) / 16; }  // of four steps
// 16-byte units of a sequence of taps (= 1 mod 16) and of samples (= 4 mod 16:
// the window's writes fall on all banks)
__host__ __device__ constexpr int fir_tap_pitch(int units) { return (units + 15) / 16 * 16 + 1; }
__host__ __device__ constexpr int fir_win_pitch(int tile, int units) {
  return (tile / 16 + units - 4 + 15) / 16 * 16 + 4;
}
__host__ __device__ constexpr int fir_lds(int tile, int units) {
  return 16 * (16 * fir_tap_pitch(units) + 4 * fir_win_pitch(tile, units));
}

// one output from its own samples, taps in order
__device__ __attribute__((noinline)) float fir_direct(const float* x, int64_t n, const float* h, int taps,
                                                      int64_t first) {
  float acc = 0.0f;
  for (int k = 0; k < taps; ++k) {
    int64_t s = first + k;
    s = s < 0 ? 0 : (s >= n ? n - 1 : s);
    acc = __builtin_fmaf(h[k], x[s], acc);
  }
  return acc;
}

template <int NC, bool PCM>
__global__ void __launch_bounds__(kThreads) fir_mfma_kernel(const float* __restrict__ x, int64_t n,
                                                            const float* __restrict__ h, int taps,
                                                            int center, float* __restrict__ y,
                                                            int16_t* __restrict__ pcm, float gain) {
  constexpr int kOut = 256 * NC * 4;  // outputs per block
  extern __shared__ __align__(16) unsigned char fir_mem[];
  const int units = fir_units(taps), VP = fir_tap_pitch(units), XP = fir_win_pitch(kOut, units);
  float* ht = reinterpret_cast<float*>(fir_mem);  // [s % 4][copy][4 VP]
  float* xt = ht + 16 * 4 * VP;                   // [s % 4][4 XP]
  const int64_t i0 = static_cast<int64_t>(blockIdx.x) * kOut;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  // the window: samples i0 - center + t
  const int span = kOut + 16 * units;
#pragma unroll 4
  for (int t = tid; t < span; t += kThreads) {
    int64_t s = i0 - center + t;
    s = s < 0 ? 0 : (s >= n ? n - 1 : s);
    xt[(t & 3) * 4 * XP + (t >> 2)] = x[s];
  }
  // copy c of residue q: place m holds h[4 (m - 4 - c) + q]
#pragma unroll 4
  for (int it = tid; it < 16 * 4 * (units + 1); it += kThreads) {
    const int a = it & 15, m = it >> 4, q = a >> 2, c = a & 3;
    const int k = 4 * (m - 4 - c) + q;
    ht[a * 4 * VP + m] = k >= 0 && k < taps ? h[k] : 0.0f;
  }
  __syncthreads();
  const int r = lane & 15, g = lane >> 4;
  const int o_w = wv * 256 * NC;
  // row r's term s = 4 j + g is h[4 (j - c) + q], q = (g - r) mod 4
  const int q = (g - r) & 3, c = (r - g + q) >> 2;  // c = 0 .. 4
  const fir_f4* ha = reinterpret_cast<const fir_f4*>(ht + (q * 4 + (c & 3)) * 4 * VP) + 1 - (c >> 2);
  const fir_f4* xa = reinterpret_cast<const fir_f4*>(xt + g * 4 * XP) + o_w / 16 + r;
  fir_f4 acc[NC] = {};
  fir_f4 a[2], b[2][NC];
  auto fetch = [&](int u, int slot) {
    a[slot] = ha[u];
#pragma unroll
    for (int t = 0; t < NC; ++t) b[slot][t] = xa[16 * t + u];
  };
  auto mma = [&](int slot) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int t = 0; t < NC; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[slot][e], b[slot][t][e], acc[t], 0, 0, 0);
  };
  fetch(0, 0);
  for (int u = 0; u < units; u += 2) {  // (fetches past the last unit read it again)
    fetch(min(u + 1, units - 1), 1);
    mma(0);
    if (u + 1 < units) {
      fetch(min(u + 2, units - 1), 0);
      mma(1);
    }
  }
  // D: column lane % 16, rows 4 (lane / 16) + 0 .. 3: four consecutive outputs a lane
#pragma unroll
  for (int t = 0; t < NC; ++t) {
    const int64_t o = i0 + o_w + 256 * t + 16 * r + 4 * g;
    if (o >= n) continue;
    float v[4] = {acc[t][0], acc[t][1], acc[t][2], acc[t][3]};
    // not finite: an infinity or NaN beside the output's own samples may have
    // met a zero of T
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (!(fabsf(v[e]) < INFINITY) && o + e < n) v[e] = fir_direct(x, n, h, taps, o + e - center);
    if (o + 4 <= n) {
      if (PCM) {
        uint32_t w[2];
#pragma unroll
        for (int e = 0; e < 2; ++e)
          w[e] = static_cast<uint16_t>(to_pcm16(v[2 * e], gain)) |
                 (static_cast<uint32_t>(static_cast<uint16_t>(to_pcm16(v[2 * e + 1], gain))) << 16);
        *reinterpret_cast<uint2*>(pcm + o) = make_uint2(w[0], w[1]);
      } else {
        st_stream4(y + o, make_float4(v[0], v[1], v[2], v[3]));
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (o + e < n) {
          if (PCM) pcm[o + e] = to_pcm16(v[e], gain);
          else y[o + e] = v[e];
        }
    }
  }
}

// Eight samples per thread: two 16-byte loads, one 16-byte store.
__global__ void __launch_bounds__(256) pcm16_kernel(const float* __restrict__ x, int64_t n,
                                                    float gain, int16_t* __restrict__ pcm) {
  const int64_t n8 = n / 8;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < n8; i += stride) {
    const float4 a = ld_stream4(x + 8 * i);
    const float4 b = ld_stream4(x + 8 * i + 4);
    const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    uint32_t w[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
      w[q] = static_cast<uint16_t>(to_pcm16(v[2 * q], gain)) |
             (static_cast<uint32_t>(static_cast<uint16_t>(to_pcm16(v[2 * q + 1], gain))) << 16);
    *reinterpret_cast<uint4*>(pcm + 8 * i) = make_uint4(w[0], w[1], w[2], w[3]);
  }
  // the last n % 8 samples, one per thread of the grid's first threads
  const int64_t t = 8 * n8 + blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  if (t < n) pcm[t] = to_pcm16(x[t], gain);
}

}  // namespace audio
using namespace audio;

// x: contiguous fp32 waveform (any shape); out_bytes: contiguous uint8 with
// 2 * numel(x) elements.
static int check_wave(const kk_tensor* x, const char* who) {
  KK_TRY(require_ready());
  KK_TRY(check_tensor(x, "x"));
  if (x->dtype != KK_F32 || !is_contiguous(x))
    return set_error(KK_E_ARG, "%s: x must be a contiguous fp32 waveform", who);
  if (reinterpret_cast<uintptr_t>(x->data) % 16)
    return set_error(KK_E_ARG, "%s: x must be 16-byte aligned", who);
  return KK_OK;
}

static int check_pcm_out(const kk_tensor* out, int64_t n, const char* who) {
  KK_TRY(check_tensor(out, "out"));
  if (out->dtype != KK_U8 || !is_contiguous(out) || numel(out) != 2 * n)
    return set_error(KK_E_ARG, "%s: out must be contiguous uint8 with 2 * %lld bytes", who,
                     (long long)n);
  if (reinterpret_cast<uintptr_t>(out->data) % 16)
    return set_error(KK_E_ARG, "%s: out must be 16-byte aligned", who);
  return KK_OK;
}

static int check_taps(const kk_tensor* taps, int* center, const char* who) {
  KK_TRY(check_tensor(taps, "taps"));
  const int64_t t = numel(taps);
  if (taps->dtype != KK_F32 || !is_contiguous(taps) || t < 1 || t > kMaxTaps)
    return set_error(KK_E_ARG, "%s: taps must be contiguous fp32 with 1..%d values", who, kMaxTaps);
  if (*center < 0) *center = static_cast<int>((t - 1) / 2);
  if (*center >= t) return set_error(KK_E_ARG, "%s: center %d outside the %lld taps", who, *center,
                                     (long long)t);
  return KK_OK;
}

template <int NC, bool PCM>
static int launch_mfma(const float* x, int64_t n, const float* h, int taps, int center, float* y,
                       int16_t* pcm, float gain) {
  constexpr int kOut = 256 * NC * 4;
  const int64_t blocks = ceil_div(n, kOut);
  if (blocks > 0x7fffffff) return set_error(KK_E_UNSUPPORTED, "FIR: waveform too long");
  const size_t lds = static_cast<size_t>(fir_lds(kOut, fir_units(taps)));
  if (lds > 65536) KK_TRY(allow_large_lds(reinterpret_cast<const void*>(fir_mfma_kernel<NC, PCM>)));
  KK_LAUNCH((fir_mfma_kernel<NC, PCM>), dim3(static_cast<unsigned>(blocks)), dim3(kThreads), lds,
            ctx().stream, x, n, h, taps, center, y, pcm, gain);
  return check_launch("fir_mfma_kernel");
}

static int launch_fir(const kk_tensor* x, const kk_tensor* taps, int center, float* y, int16_t* pcm,
                      float gain) {
  const int64_t n = numel(x);
  const float* xp = static_cast<const float*>(x->data);
  const float* hp = static_cast<const float*>(taps->data);
  const int t = static_cast<int>(numel(taps));
  if (t >= kMfmaMinTaps) {
    // Tiles a wave: blocks of one, two or four go round the CUs whole.  Costs
    // of a round (0.1 us at 1023 taps), measured from 32 to 4096 taps and 20,000
    // to 8,000,000 samples:
    //  - three blocks and more a CU by their LDS: 47, 87 and 167 (51, 98, 183 for
    //    the first block of a CU, alone there; 80 for two below 64 taps).  Four
    //    are not worth their registers below 192 taps (800,000 samples x 128:
    //    8.5, 8.6 and 9.3 us; 8,000,000: 34.6, 32.8, 34.7).
    //  - from about 2,700 taps two blocks, from 3,800 one, whose window and
    //    taps are staged with less or nothing in their shadow: half or all of a
    //    tile's time more (4096 taps x 600,000: 99, 98 and 78 us; 1,060,000:
    //    159, 142, 152; 3000 taps x 2,154,000: 161, 148, 153).
    // 1023 taps: 400,000 samples 16.4, 18.0 and 25.4 us, 800,000 25.8, 25.9, 26.6,
    // 1,060,000 32.1, 33.7, 40.8, 1,500,000 37.8, 34.7, 41.4, 2,029,200 48.4, 43.1,
    // 42.7.  (32 to 47 taps over 2,000,000 to 2,600,000 samples take up to 1.06
    // times the VALU kernel's time, below and above that less.)
    const int64_t cus = ctx().num_cus > 0 ? ctx().num_cus : 256;
    const int resident = 163840 / fir_lds(1024, fir_units(t));
    auto cost = [&](int64_t nc) {
      const int64_t rounds = ceil_div(ceil_div(n, 1024 * nc), cus);
      if (resident < 3) return rounds * (nc * 50 + (resident < 2 ? 50 : 25));
      if (rounds <= 1) return nc == 1 ? int64_t{51} : nc == 2 ? int64_t{98} : int64_t{183};
      return rounds * (nc == 1 ? 47 : nc == 2 ? (t < 64 ? 80 : 87) : 167);
    };
    const int64_t c1 = cost(1), c2 = cost(2), c4 = t < 192 ? INT64_MAX : cost(4);
    auto run = [&](auto nc) {
      constexpr int kNc = decltype(nc)::value;
      return pcm ? launch_mfma<kNc, true>(xp, n, hp, t, center, y, pcm, gain)
                 : launch_mfma<kNc, false>(xp, n, hp, t, center, y, pcm, gain);
    };
    if (c4 <= c2 && c4 <= c1) return run(std::integral_constant<int, 4>{});
    if (c2 <= c1) return run(std::integral_constant<int, 2>{});
    return run(std::integral_constant<int, 1>{});
  }
  const int64_t blocks = ceil_div(n, kTile);
  if (blocks > 0x7fffffff) return set_error(KK_E_UNSUPPORTED, "FIR: waveform too long");
  if (pcm)
    KK_LAUNCH(fir_kernel<true>, dim3(static_cast<unsigned>(blocks)), dim3(kThreads), 0,
                       ctx().stream, xp, n, hp, t, center, nullptr, pcm, gain);
  else
    KK_LAUNCH(fir_kernel<false>, dim3(static_cast<unsigned>(blocks)), dim3(kThreads), 0,
                       ctx().stream, xp, n, hp, t, center, y, nullptr, 0.0f);
  return check_launch("fir_kernel");
}

}  // namespace kk

using namespace kk;

extern "C" {

int kk_fir(const kk_tensor* out, const kk_tensor* x, const kk_tensor* taps, int center) {
  KK_TRY(check_wave(x, "kk_fir"));
  KK_TRY(check_taps(taps, &center, "kk_fir"));
  KK_TRY(check_tensor(out, "out"));
  if (out->dtype != KK_F32 || !is_contiguous(out) || numel(out) != numel(x) ||
      reinterpret_cast<uintptr_t>(out->data) % 16)
    return set_error(KK_E_ARG, "kk_fir: out must be a 16-byte-aligned contiguous fp32 tensor of x's size");
  if (numel(x) == 0) return KK_OK;
  return launch_fir(x, taps, center, static_cast<float*>(out->data), nullptr, 0.0f);
}

int kk_pcm16(const kk_tensor* out_bytes, const kk_tensor* x, float gain) {
  KK_TRY(check_wave(x, "kk_pcm16"));
  const int64_t n = numel(x);
  KK_TRY(check_pcm_out(out_bytes, n, "kk_pcm16"));
  if (n == 0) return KK_OK;
  const unsigned g = static_cast<unsigned>(std::max<int64_t>(1, std::min<int64_t>(ceil_div(n, 8 * 256), 4096)));
  KK_LAUNCH(pcm16_kernel, dim3(g), dim3(256), 0, ctx().stream,
                     static_cast<const float*>(x->data), n, gain, static_cast<int16_t*>(out_bytes->data));
  return check_launch("pcm16_kernel");
}

int kk_fir_pcm16(const kk_tensor* out_bytes, const kk_tensor* x, const kk_tensor* taps, int center,
                 float gain) {
  KK_TRY(check_wave(x, "kk_fir_pcm16"));
  KK_TRY(check_taps(taps, &center, "kk_fir_pcm16"));
  const int64_t n = numel(x);
  KK_TRY(check_pcm_out(out_bytes, n, "kk_fir_pcm16"));
  if (n == 0) return KK_OK;
  return launch_fir(x, taps, center, nullptr, static_cast<int16_t*>(out_bytes->data), gain);
}

}  // extern "C"
