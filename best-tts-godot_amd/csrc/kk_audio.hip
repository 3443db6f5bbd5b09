// The waveform's output stage, as runtime/audio.gd:59-106 drives it: the
// notch FIR (kernels/fir.glsl:35-47) and the float -> 16-bit PCM conversion
// (kernels/pcm16.glsl:28-46), separately or fused into one pass.
//
// FIR: y[i] = sum_k h[k] x[clamp(i - center + k, 0, n - 1)], each output's
// taps accumulated in order (k = 0, 1, ...) in fp32 with one fused
// multiply-add per tap.  A block of 256 threads computes 2048 consecutive
// outputs: it stages the input window they read (2048 + taps - 1 samples,
// edges clamped) in LDS once; each thread keeps a 16-sample register window
// over its 8 consecutive outputs and slides it 8 taps at a time (two 16-byte
// LDS reads per 64 FMAs), the taps coming from the scalar cache (the same
// address in every lane).  1023 taps over 2.15M samples are 2.2 G FMAs:
// bound by the VALU's fp32 FMA rate, not by HBM (17 MB in and out).
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
constexpr int kMaxTaps = 4096;                       // window: kTile + taps rounded up + slack
constexpr int kWindow = kTile + kMaxTaps + 16;

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

// The FIR on the matrix cores, for kMfmaMinTaps .. kMfmaTaps taps (the split
// copies of the taps take 54 KB of LDS at 1023; below 256 taps forming them
// costs more than the sum: 128 taps over 1,060,000 samples 12.2 us, 10.4 on
// the VALU, 513 taps 19.1 and 29.4).  Outputs in tiles of
// 32 x 32, y[o + 32 i + r] = sum_s T[r][s] x[o + 32 i + s] with the Toeplitz
// matrix T[r][s] = h[s - r] (0 outside the filter): taps + 31 terms of which
// taps count, 3% more at 1023 taps.  Samples and taps are split into three
// bf16 parts (round to nearest, exact: 3 x 8 significant bits) and the six
// products of parts above 2^-26 of the whole run on
// v_mfma_f32_32x32x16_bf16 (2.5 PF/s dense, so 417 TF/s of fp32-accurate work
// against 79 on the VALU); the sum of the leading products and that of the
// other five are kept apart until the end.  Its 66 steps round less than the
// chain of 1023 fused multiply-adds: the notch filter's relative error
// against 64 bits is 2.1e-7 (6.8e-8 with the sum shared by four waves)
// where that chain's is 5.7e-7, 1.2e-7 against 4.0e-7 at 513 taps and 2.3e-7
// against 7.0e-7 at 1536.  Measured, 1023 taps: 2,029,200 samples 67.4 ->
// 31.5 us (PCM16 65 -> 30), 400,000 33.8 -> 12.9, 2400 32.1 -> 8.3; bound by
// LDS reads and their latency (nine fragments for twelve matrix
// instructions, one wave a SIMD), the products alone taking 10.5 us.
//
// LDS: the taps in eight copies shifted by 0 .. 7 (row r of T reads copy
// r % 8, so every operand fragment is one aligned 16-byte read), and the
// block's window of x, in units of eight bf16 dealt round over four regions,
// so the 32 columns of a fragment -- four units apart in time -- read
// consecutive units.
//
// A wave takes NC tiles and one of WK shares of the sum; with WK = 4 the four
// waves' partial tiles are added through LDS in wave order.  Where an output
// is not finite (an infinity or NaN in its tile's window, or a sample above
// bf16's range), it is formed again as the kernel above does.
constexpr int kMfmaMinTaps = 256, kMfmaTaps = 1536;
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef float f16v __attribute__((ext_vector_type(16)));

__host__ __device__ constexpr int fir_steps(int taps, int wk) {  // of 16 terms, a multiple of wk
  return ((taps + 31 + 15) / 16 + wk - 1) / wk * wk;
}
// units a copy of the taps takes: -3 .. 2 steps - 1; = 4 mod 16 (the copies
// of a row octet fall on different banks)
__host__ __device__ constexpr int fir_tap_pitch(int steps) { return (2 * steps + 3 - 4 + 15) / 16 * 16 + 4; }
// units of a region of the window (a quarter of the window's)
__host__ __device__ constexpr int fir_win_pitch(int tile, int steps) { return (tile / 8 + 2 * steps + 3) / 4; }
__host__ __device__ constexpr int fir_lds(int tile, int steps, int wk) {
  const int w = 3 * 4 * fir_win_pitch(tile, steps) * 16, red = wk > 1 ? wk * tile * 4 : 0;
  return 3 * 8 * fir_tap_pitch(steps) * 16 + (w > red ? w : red);
}

// v = p[0] + p[1] + p[2] (up to 2^-26 of v), each a bf16
__device__ __forceinline__ void split3(float v, __bf16 (&p)[3]) {
  p[0] = static_cast<__bf16>(v);
  const float r1 = v - static_cast<float>(p[0]);
  p[1] = static_cast<__bf16>(r1);
  p[2] = static_cast<__bf16>(r1 - static_cast<float>(p[1]));
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

template <int NC, int WK, bool PCM>
__global__ void __launch_bounds__(kThreads) fir_mfma_kernel(const float* __restrict__ x, int64_t n,
                                                            const float* __restrict__ h, int taps,
                                                            int center, float* __restrict__ y,
                                                            int16_t* __restrict__ pcm, float gain) {
  constexpr int kOut = 1024 * NC * (4 / WK);  // outputs per block
  extern __shared__ __align__(16) unsigned char fir_mem[];
  const int steps = fir_steps(taps, WK), VP = fir_tap_pitch(steps), XP = fir_win_pitch(kOut, steps);
  bf8* ht = reinterpret_cast<bf8*>(fir_mem);  // [part][copy][VP]
  bf8* xt = ht + 3 * 8 * VP;                  // [part][unit % 4][XP]
  const int64_t i0 = static_cast<int64_t>(blockIdx.x) * kOut;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  // the window: unit u holds samples i0 - center + 8 u ..
  for (int u = tid; u < 4 * XP; u += kThreads) {
    bf8 q[3];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      int64_t s = i0 - center + 8 * u + e;
      s = s < 0 ? 0 : (s >= n ? n - 1 : s);
      __bf16 p[3];
      split3(x[s], p);
#pragma unroll
      for (int k = 0; k < 3; ++k) q[k][e] = p[k];
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) xt[(k * 4 + (u & 3)) * XP + (u >> 2)] = q[k];
  }
  // the taps: copy c, unit v holds h[8 (v - 3) - c + 0 .. 7]
  for (int it = tid; it < 8 * VP; it += kThreads) {
    const int c = it & 7, v = it >> 3, k0 = 8 * (v - 3) - c;
    bf8 q[3];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int k = k0 + e;
      __bf16 p[3];
      split3(k >= 0 && k < taps ? h[k] : 0.0f, p);
#pragma unroll
      for (int t = 0; t < 3; ++t) q[t][e] = p[t];
    }
#pragma unroll
    for (int t = 0; t < 3; ++t) ht[(t * 8 + c) * VP + v] = q[t];
  }
  __syncthreads();
  const int r = lane & 31, g = lane >> 5;
  const int kp = wv % WK, o_w = (wv / WK) * 1024 * NC;  // this wave's share of the sum, its outputs
  const int per = steps / WK, st0 = kp * per;
  // lane (r, g) of step st: taps unit 2 st + g - r / 8 (+ 3) of copy r % 8;
  // window unit o_w / 8 + 128 c + 2 st + g + 4 r of tile c
  const bf8* ha = ht + (r & 7) * VP + g - (r >> 3) + 3;
  auto xaddr = [&](int st, int c) {
    const int u0 = 2 * st + g;
    return xt + (u0 & 3) * XP + (u0 >> 2) + o_w / 32 + 32 * c + r;
  };
  f16v big[NC] = {}, small[NC] = {};
  bf8 a[2][3], b[2][NC][3];
  auto fetch = [&](int st, bf8 (&fa)[3], bf8 (&fb)[NC][3]) {
#pragma unroll
    for (int k = 0; k < 3; ++k) fa[k] = ha[k * 8 * VP + 2 * st];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const bf8* p = xaddr(st, c);
#pragma unroll
      for (int k = 0; k < 3; ++k) fb[c][k] = p[k * 4 * XP];
    }
  };
  auto mma = [&](const bf8 (&fa)[3], const bf8 (&fb)[NC][3]) {
#define KK_FIR_MMA(D, P, Q) \
  _Pragma("unroll") for (int c = 0; c < NC; ++c) D[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[P], fb[c][Q], D[c], 0, 0, 0)
    KK_FIR_MMA(small, 2, 0);
    KK_FIR_MMA(big, 0, 0);
    KK_FIR_MMA(small, 0, 2);
    KK_FIR_MMA(small, 1, 1);
    KK_FIR_MMA(small, 1, 0);
    KK_FIR_MMA(small, 0, 1);
#undef KK_FIR_MMA
  };
  fetch(st0, a[0], b[0]);
  for (int st = 0; st < per; st += 2) {  // (fetches past the share read its last step again)
    fetch(st0 + min(st + 1, per - 1), a[1], b[1]);
    mma(a[0], b[0]);
    if (st + 1 < per) {
      fetch(st0 + min(st + 2, per - 1), a[0], b[0]);
      mma(a[1], b[1]);
    }
  }
  // D(i, j): lane j + 32 ((i / 4) % 2), register (i / 8) 4 + i % 4: four
  // consecutive outputs a register quad
  auto put4 = [&](int64_t o, float4 v4) {
    if (o >= n) return;
    float v[4] = {v4.x, v4.y, v4.z, v4.w};
#pragma unroll
    for (int t = 0; t < 4; ++t)
      if (!(fabsf(v[t]) < INFINITY) && o + t < n) v[t] = fir_direct(x, n, h, taps, o + t - center);
    if (o + 4 <= n) {
      if (PCM) {
        uint32_t w[2];
#pragma unroll
        for (int t = 0; t < 2; ++t)
          w[t] = static_cast<uint16_t>(to_pcm16(v[2 * t], gain)) |
                 (static_cast<uint32_t>(static_cast<uint16_t>(to_pcm16(v[2 * t + 1], gain))) << 16);
        *reinterpret_cast<uint2*>(pcm + o) = make_uint2(w[0], w[1]);
      } else {
        *reinterpret_cast<float4*>(y + o) = make_float4(v[0], v[1], v[2], v[3]);
      }
    } else {
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if (o + t < n) {
          if (PCM) pcm[o + t] = to_pcm16(v[t], gain);
          else y[o + t] = v[t];
        }
    }
  };
  if constexpr (WK == 1) {
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        put4(i0 + o_w + 1024 * c + 32 * r + 8 * q + 4 * g,
             make_float4(big[c][4 * q] + small[c][4 * q], big[c][4 * q + 1] + small[c][4 * q + 1],
                         big[c][4 * q + 2] + small[c][4 * q + 2], big[c][4 * q + 3] + small[c][4 * q + 3]));
  } else {
    __syncthreads();  // every wave is done with the window
    float4* red = reinterpret_cast<float4*>(xt);  // [wave][outputs / 4]
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        red[kp * (kOut / 4) + o_w / 4 + 256 * c + 8 * r + 2 * q + g] =
            make_float4(big[c][4 * q] + small[c][4 * q], big[c][4 * q + 1] + small[c][4 * q + 1],
                        big[c][4 * q + 2] + small[c][4 * q + 2], big[c][4 * q + 3] + small[c][4 * q + 3]);
    __syncthreads();
    for (int t = tid; t < kOut / 4; t += kThreads) {
      float4 v = red[t];
#pragma unroll
      for (int w = 1; w < WK; ++w) {
        const float4 p = red[w * (kOut / 4) + t];
        v = make_float4(v.x + p.x, v.y + p.y, v.z + p.z, v.w + p.w);
      }
      put4(i0 + 4 * t, v);
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

template <int NC, int WK, bool PCM>
static int launch_mfma(const float* x, int64_t n, const float* h, int taps, int center, float* y,
                       int16_t* pcm, float gain) {
  constexpr int kOut = 1024 * NC * (4 / WK);
  const int64_t blocks = ceil_div(n, kOut);
  if (blocks > 0x7fffffff) return set_error(KK_E_UNSUPPORTED, "FIR: waveform too long");
  const size_t lds = static_cast<size_t>(fir_lds(kOut, fir_steps(taps, WK), WK));
  // above 64 KB of dynamic LDS a kernel needs the attribute (per device: set
  // on each call, a host-side store)
  KK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(fir_mfma_kernel<NC, WK, PCM>),
                             hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
  KK_LAUNCH((fir_mfma_kernel<NC, WK, PCM>), dim3(static_cast<unsigned>(blocks)), dim3(kThreads), lds,
            ctx().stream, x, n, h, taps, center, y, pcm, gain);
  return check_launch("fir_mfma_kernel");
}

static int launch_fir(const kk_tensor* x, const kk_tensor* taps, int center, float* y, int16_t* pcm,
                      float gain) {
  const int64_t n = numel(x);
  const float* xp = static_cast<const float*>(x->data);
  const float* hp = static_cast<const float*>(taps->data);
  const int t = static_cast<int>(numel(taps));
  if (t >= kMfmaMinTaps && t <= kMfmaTaps) {
    // 8192 outputs a block, one block a CU (1,500,000 samples 28.9 us) where
    // its rounds over the CUs are at least two thirds full: it takes as long
    // at 1,060,000 (27.7 us) and twice as long at 2,154,000 (52 us).  Else
    // 1024 outputs a block, the waves sharing the sum (1,040,000 samples 23.6
    // us, 2400 8.3 us).
    const int64_t cus = ctx().num_cus > 0 ? ctx().num_cus : 256;
    const int64_t b8 = ceil_div(n, 8192), rounds = ceil_div(b8, cus);
    if (3 * b8 >= 2 * rounds * cus)
      return pcm ? launch_mfma<2, 1, true>(xp, n, hp, t, center, y, pcm, gain)
                 : launch_mfma<2, 1, false>(xp, n, hp, t, center, y, pcm, gain);
    return pcm ? launch_mfma<1, 4, true>(xp, n, hp, t, center, y, pcm, gain)
               : launch_mfma<1, 4, false>(xp, n, hp, t, center, y, pcm, gain);
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
