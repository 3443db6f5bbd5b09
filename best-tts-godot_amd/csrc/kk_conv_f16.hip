// Conv1d and ConvTranspose1d with fp16 or 8-bit weights on the fp16 matrix
// cores (v_mfma_f32_32x32x16_f16), fp32 results, in one launch (8-bit weights
// over multiples of 128 channels: convq_kernel below, on the bf16 ones).
//
// Exact operands.  An fp16 weight is exact in fp16, and so is an 8-bit
// weight less its zero point (|q - zp| <= 255); the 8-bit weights' scale,
// per tensor or per output channel, multiplies the fp32 sum
// (sum (q - zp) s x = s sum (q - zp) x up to fp32 rounding).  Every output
// column (time step) scales its activations by its own power of two, 2^k,
// chosen from the largest |x| its receptive field has shown so far: with m
// that maximum, m 2^k first lies in [2^10, 2^11) (exact in fp32), and a
// scaled y = x 2^k is split into hi = fp16(y) and lo = fp16(y - hi) (y - hi
// is exact in fp32).  For |y| >= 2^-3 lo is a normal fp16 number and hi + lo
// equals y to within 2^-22 |y|; below that the error is at most 2^-25 in
// scaled units, m 2^-35 or less.  Every product w hi and w lo is exact in
// fp32 (11 + 11 significant bits) and the matrix cores accumulate them in
// fp32.  Only when a column's maximum grows past 2^15 in scaled units (a
// value 16 to 32 times the first maximum) does its k fall afresh; its
// accumulators (all in the lanes that hold that column) are then multiplied
// by 2^(k_new - k_old), exact for a power of two.  The sums are scaled back
// by 2^-k at the end.  A column whose receptive field holds an infinity or
// a NaN is recomputed with scalar fp32 products and sums, which give numpy's
// inf / NaN pattern.
//
// Both operations are one implicit GEMM with rows m = co P + r (output
// channel co, phase r < P) and columns q, the reduction index k running over
// (input channel ci, tap t') with TP in {2, 4, 8} taps a channel (T taps
// used, the rest weigh 0):
//   out[co, q os + r + oph] = sum_ci sum_t' Wv[m][ci][t'] x[ci, q qs + ta + t' tm]
//   Conv1d (P = 1): t' = the tap, qs = stride, ta = -pad0, tm = dilation,
//     os = 1, oph = 0, Wv[co][ci][t'] = W[co][ci][t'].
//   ConvTranspose1d (dilation 1), P = stride phases, T = ceil(K / P) taps a
//     phase, read in increasing position: x[ci, q - (T - 1) + t'] (qs = 1,
//     ta = 1 - T, tm = 1), os = stride, oph = -pad0,
//     Wv[co P + r][ci][t'] = W[ci][co][r + P (T - 1 - t')] (0 past K).
// A 16-deep reduction slice s holds channels 16 s / TP .. + 16 / TP - 1, each
// with its TP taps, so a lane's eight operand values of a slice are TP
// consecutive taps of 8 / TP channels: for Conv1d with dilation 1 and for
// ConvTranspose1d, consecutive x positions of each channel.
//
// Packed weights (kk_conv_pack, or per call into the context scratch): fp16
// values (W less its zero point) in the matrix cores' operand order: the
// 16-byte unit (mt KS + s) 64 + l holds lane l's operand of slice s for rows
// 32 mt .. 32 mt + 31: row 32 mt + l % 32, k = 8 (l / 32) + 0..7 (KS slices;
// zeros past M, past Cin and past T).
//
// A block owns 32 MI rows x 32 WN columns; its 4 waves are WN (columns) x
// WK (reduction ranges).  A wave holds MI 32 x 32 accumulator tiles of its
// 32 columns: lane (n, g) = (lane % 32, lane / 32) loads its column's eight
// x values of a slice straight from memory (bounds-checked buffer loads: 0
// outside the signal, past Cin and past T), the two lanes of a column agree
// on its scale (one lane swap), and split, and the weights' operands come
// as 1 KB fragments; both run three slices ahead in a register ring, with
// no LDS and no barrier in the reduction loop.  The WK waves of a column
// range add their unscaled partial tiles through LDS in wave order.
#include <algorithm>
#include <climits>
#include <mutex>
#include <unordered_map>
#include <utility>

#include "kk_internal.h"

namespace kk {
namespace convh {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f16v __attribute__((ext_vector_type(16)));

constexpr int kThreads = 256;

// Taps a channel spans in the reduction order: T rounded up to 2, 4 or 8 (0:
// more than 8 taps, which this path does not take).
static int taps_padded(int64_t T) { return T <= 2 ? 2 : T <= 4 ? 4 : T <= 8 ? 8 : 0; }

// The packed geometry: what a pack and a convolution must agree on.
struct Geo {
  int transposed;
  int64_t Cin, Cout, Kw, P;  // P: phases (the stride) of a transposed conv, else 1
  int64_t T, TP;             // taps a row reads; taps a channel spans (0: unsupported)
  int64_t M, MT, KS;         // rows, 32-row tiles, 16-deep slices
  int64_t bytes;             // packed size
};

static Geo geometry(bool transposed, int64_t Cin, int64_t Cout, int64_t Kw, int64_t stride) {
  Geo g{};
  g.transposed = transposed ? 1 : 0;
  g.Cin = Cin; g.Cout = Cout; g.Kw = Kw;
  g.P = transposed ? stride : 1;
  g.T = transposed ? ceil_div(Kw, stride) : Kw;
  g.TP = taps_padded(g.T);
  g.M = g.P * Cout;
  g.MT = ceil_div(g.M, 32);
  g.KS = g.TP ? ceil_div(Cin * g.TP, 16) : 0;
  g.bytes = g.MT * g.KS * 1024;
  return g;
}

struct PackArgs {
  uint4* wp;
  const void* w;   // conv [Cout][Cin][Kw], transposed [Cin][Cout][Kw]
  const void* zp;  // 8-bit weights' zero point (1 or Cout values) or NULL
  int zp_dt;
  int zp_stride;
  int Cin, Cout, Kw, P, T, TP, M, KS;
  int transposed;
  int tap_major;   // convq_kernel's order: k = tap Cin + ci, bf16
  int64_t units;
};

// One 16-byte unit (eight fp16 values) a thread.
template <typename TW>
__global__ void __launch_bounds__(256) convh_pack(PackArgs A) {
  const int64_t u = blockIdx.x * int64_t{256} + threadIdx.x;
  if (u >= A.units) return;
  const int l = static_cast<int>(u % 64);
  const int s = static_cast<int>((u / 64) % A.KS);
  const int mt = static_cast<int>(u / (int64_t{64} * A.KS));
  const int m = 32 * mt + (l % 32), g = l / 32;
  const int co = m / A.P, r = m - co * A.P;
  const TW* w = static_cast<const TW*>(A.w);
  const float z = A.zp && m < A.M ? load_as_f32(A.zp, A.zp_dt, co * A.zp_stride) : 0.0f;
  h8 v;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int k = 8 * g + e;
    const int kk = 16 * s + k;
    const int ci = A.tap_major ? kk % A.Cin : s * (16 / A.TP) + k / A.TP;
    const int tp = A.tap_major ? kk / A.Cin : k % A.TP;
    const int tap = A.transposed ? r + A.P * (A.T - 1 - tp) : tp;
    float f = 0.0f;
    if (m < A.M && ci < A.Cin && tp < A.T && tap < A.Kw) {
      const int64_t idx = A.transposed ? (static_cast<int64_t>(ci) * A.Cout + co) * A.Kw + tap
                                       : (static_cast<int64_t>(co) * A.Cin + ci) * A.Kw + tap;
      f = static_cast<float>(w[idx]) - z;
    }
    if (A.tap_major) v[e] = __builtin_bit_cast(_Float16, static_cast<__bf16>(f));
    else v[e] = static_cast<_Float16>(f);
  }
  *reinterpret_cast<h8*>(A.wp + u) = v;
}

struct CArgs {
  const uint4* wp;     // packed weights
  const float* x;      // [N][Cin][L]
  float* out;          // [N][Cout][Lout]
  const float* bias;   // [Cout] or NULL
  const void* scale;   // 8-bit weights: 1 or Cout values; NULL for fp16 weights
  int scale_dt, scale_stride;
  int Cin, L, Cout, Lout, M, Nq, P, T, KS;
  int qs, ta, tm;      // x position of (q, t'): q qs + ta + t' tm
  int os, oph;         // output position of (q, r): q os + r + oph
  int wbytes;          // packed bytes (below 2^31)
};

// The power of two k with m 2^k in [2^10, 2^11) for the bits of m = max |x|
// > 0, kept within [-120, 120] so that 2^k and 2^-k are normal floats.
__device__ __forceinline__ int scale_exp(unsigned mbits) {
  const int e = static_cast<int>(mbits >> 23) - 127;  // floor(log2 m); -127 for subnormal m
  return min(120, 10 - e);
}

typedef __bf16 b8 __attribute__((ext_vector_type(8)));
constexpr float kSplitScale = 0x1p24f;

// Eight activations times kSplitScale as three bf16 parts each.
__device__ __forceinline__ void split3(const float (&v)[8], b8 (&part)[3]) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float x0 = v[e] * kSplitScale;
    part[0][e] = static_cast<__bf16>(x0);
    const float x1 = x0 - static_cast<float>(part[0][e]);
    part[1][e] = static_cast<__bf16>(x1);
    part[2][e] = static_cast<__bf16>(x1 - static_cast<float>(part[1][e]));
  }
}

// TP = 0: weights laid out for convq_kernel (tap-major bf16), for the strides
// and dilations whose window that kernel does not hold: its three products a
// weight, no scale (as fp16 operands, each weight fragment converted for two
// products, 512 -> 512 k4 over 2400 steps took 45 us; so 38; the fp16 layout 34).
template <int TP, int MI, int WK, int R>
__global__ void __launch_bounds__(kThreads) convh_kernel(CArgs A) {
  constexpr int NPO = TP ? TP : 1;
  constexpr int WN = 4 / WK, CPL = 8 / NPO, CPS = 16 / NPO;
  constexpr int BM = 32 * MI, BN = 32 * WN;
  constexpr int RED = WK > 1 ? (WK - 1) * WN * MI * 16 * 64 : 1;
  __shared__ float red[RED];       // [wk - 1][wn][register][lane]: the other waves' partials
  __shared__ int red_bad[4 * 64];  // [wave][lane]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wn = wave % WN, wk = wave / WN;
  const int ln = lane & 31, g = lane >> 5;
  // row tiles fastest: the blocks of one column range share an XCD.  The
  // tile is wave-uniform; readfirstlane says so to the compiler, which would
  // otherwise build the activations' buffer resource in vector registers
  // and wrap every load in a loop over its distinct values.
  const uint3 tile = xcd_tile();
  const int m0 = __builtin_amdgcn_readfirstlane(static_cast<int>(tile.x)) * BM;
  const int n0 = __builtin_amdgcn_readfirstlane(static_cast<int>(tile.y)) * BN;
  const int64_t b = __builtin_amdgcn_readfirstlane(static_cast<int>(tile.z));
  const int Cin = A.Cin, L = A.L, KS = A.KS;
  const int q = n0 + wn * 32 + ln;
  const int s0 = static_cast<int>(static_cast<int64_t>(KS) * wk / WK);
  const int ns = static_cast<int>(static_cast<int64_t>(KS) * (wk + 1) / WK) - s0;
  const auto xrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(A.x + b * Cin * L), 0,
                                                     Cin * L * 4, 0x00020000);
  const auto wrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint4*>(A.wp), 0, A.wbytes,
                                                     0x00020000);
  // byte offsets of this lane's TP positions in a channel row; 0x7fffffff
  // outside the signal, past the columns or past the T taps in use, and a
  // channel's offset 0x80000000 past Cin: any sum with either is past the
  // buffer (below 2^31 bytes), so the load returns 0, and no sum wraps
  uint32_t po[NPO];
#pragma unroll
  for (int t = 0; t < NPO; ++t) {
    const int p = q * A.qs + A.ta + t * A.tm;
    po[t] = q < A.Nq && t < A.T && p >= 0 && p < L ? static_cast<uint32_t>(4 * p) : 0x7fffffffu;
  }
  const int row_bytes = 4 * L;
  const uint32_t a_lane = static_cast<uint32_t>(((m0 / 32) * KS * 64 + lane) * 16);
  // per-row epilogue constants (output row offset, phase offset, scale,
  // bias), filled by the first BM threads; read after the block's barrier
  __shared__ int4 rows[BM];
  if (tid < BM) {
    const int m = m0 + tid;
    int4 rv = make_int4(-1, 0, __float_as_int(1.0f), 0);
    if (m < A.M) {
      const int co = m / A.P, r = m - co * A.P;
      rv.x = co * A.Lout;
      rv.y = r + A.oph;
      if (A.scale) rv.z = __float_as_int(load_as_f32(A.scale, A.scale_dt, co * A.scale_stride));
      if (A.bias) rv.w = __float_as_int(A.bias[co]);
    }
    rows[tid] = rv;
  }
  float bv[R][8];
  uint4 av[R][MI];
  // slice s's x values (channels s CPS + g CPL + c, each with its TP taps)
  // and weight fragments; issued whatever s (a read past the buffers
  // returns 0), so every slot's loads count the same for the waits
  auto fetch = [&](int s, float (&v)[8], uint4 (&f)[MI]) {
    uint32_t pt[NPO];
    int c_first = s * CPS + g * CPL;  // the slice's first channel of this lane
    if constexpr (TP == 0) {          // (Cin % 16 == 0: a slice lies in one tap)
      const int t = 16 * s / Cin, p = q * A.qs + A.ta + t * A.tm;
      c_first = 16 * s - t * Cin + 8 * g;
      pt[0] = q < A.Nq && t < A.T && p >= 0 && p < L ? static_cast<uint32_t>(4 * p) : 0x7fffffffu;
    } else {
#pragma unroll
      for (int t = 0; t < TP; ++t) pt[t] = po[t];
    }
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
      const int ci = c_first + c;
      const uint32_t cofs = ci < Cin ? static_cast<uint32_t>(ci * row_bytes) : 0x80000000u;
#pragma unroll
      for (int t = 0; t < NPO; ++t) {
        uint32_t off = cofs + pt[t];
        asm volatile("" : "+v"(off));  // an unconditional load
        v[c * NPO + t] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xrs, off, 0, 0));
      }
    }
    const uint32_t a_s = a_lane + static_cast<uint32_t>(s * 1024);
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) {
      uint32_t off = a_s + static_cast<uint32_t>(mi * KS * 1024);
      asm volatile("" : "+v"(off));
      const auto r = __builtin_amdgcn_raw_buffer_load_b128(wrs, off, 0, 0);
      f[mi] = make_uint4(r[0], r[1], r[2], r[3]);
    }
  };

  f16v acc[MI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[i][r] = 0.0f;
  int kcur = 0, have = 0, bad = 0;
  // one slice: the column's running scale, the split, the products
  auto mma = [&](float (&v)[8], const uint4 (&f)[MI]) {
    if constexpr (TP == 0) {  // bf16: three exact parts, as convq_kernel forms them, and no scale
      b8 part[3];
      split3(v, part);
#pragma unroll
      for (int k = 2; k >= 0; --k)
#pragma unroll
        for (int mi = 0; mi < MI; ++mi)
          acc[mi] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(b8, f[mi]), part[k], acc[mi], 0, 0, 0);
      return;
    }
    unsigned mx = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) mx = max(mx, __float_as_uint(v[e]) & 0x7fffffffu);
    const auto pr = __builtin_amdgcn_permlane32_swap(mx, mx, false, false);  // the column's other lane
    mx = max(static_cast<unsigned>(pr[0]), static_cast<unsigned>(pr[1]));
    const bool nonfinite = mx >= 0x7f800000u;
    if (nonfinite) {
      bad = 1;  // recomputed in the epilogue; no products from this slice
    } else if (mx != 0u) {
      if (!have) {
        kcur = scale_exp(mx);
        have = 1;
      } else if (static_cast<int>(mx >> 23) - 127 + kcur >= 15) {  // m 2^k >= 2^15
        const int kc = scale_exp(mx);
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[i][r] = ldexpf(acc[i][r], kc - kcur);
        kcur = kc;
      }
    }
    const float xs = nonfinite ? 0.0f : ldexpf(1.0f, kcur);
    h8 hi, lo;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float y = v[e] * xs;  // |y| < 2^15: exact
      const _Float16 hh = static_cast<_Float16>(y);
      hi[e] = hh;
      lo[e] = static_cast<_Float16>(y - static_cast<float>(hh));
    }
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) {
      const h8 a = __builtin_bit_cast(h8, f[mi]);
      acc[mi] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, hi, acc[mi], 0, 0, 0);
      acc[mi] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, lo, acc[mi], 0, 0, 0);
    }
  };
#pragma unroll
  for (int u = 0; u < R; ++u) fetch(s0 + u, bv[u], av[u]);
  // whole rounds of R slices (a slot's refill is issued whether or not its
  // slice exists: a skipped refill leaves the waits at "all loads")
  for (int i = 0; i < ns; i += R) {
#pragma unroll
    for (int u = 0; u < R; ++u) {
      if (i + u < ns) mma(bv[u], av[u]);
      fetch(s0 + i + u + R, bv[u], av[u]);
    }
  }
  const float uns = TP ? ldexpf(1.0f, -kcur) : 1.0f / kSplitScale;  // exact: a power of two
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[i][r] *= uns;
  if constexpr (WK > 1) {
    if (wk > 0) {
      float* dst = red + ((wk - 1) * WN + wn) * MI * 16 * 64 + lane;
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) dst[(i * 16 + r) * 64] = acc[i][r];
    }
    red_bad[wave * 64 + lane] = bad;
  }
  __syncthreads();  // the partials and the row constants
  if (wk > 0) return;
  if constexpr (WK > 1) {
#pragma unroll
    for (int k = 1; k < WK; ++k) {  // in wave order
      const float* src = red + ((k - 1) * WN + wn) * MI * 16 * 64 + lane;
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] += src[(i * 16 + r) * 64];
      bad |= red_bad[(k * WN + wn) * 64 + lane];
    }
  }
  if constexpr (TP == 0) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) bad |= !(fabsf(acc[i][r]) < INFINITY);
  }
  // D(i, j) of a 32x32 tile: lane j + 32 ((i / 4) % 2), register (i / 8) 4 + i % 4.
  // Stores through a buffer resource over this item's output: an offset
  // past it (a row past M, a column past Nq, a position outside [0, Lout))
  // drops the store.
  const auto ors = __builtin_amdgcn_make_buffer_rsrc(A.out + b * A.Cout * A.Lout, 0,
                                                     A.Cout * A.Lout * 4, 0x00020000);
  const int qpos = q < A.Nq ? q * A.os : INT_MIN / 2;
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int rg = 0; rg < 16; ++rg) {
      const int ml = 32 * mi + 8 * (rg / 4) + 4 * g + (rg % 4);
      const int4 rv = rows[ml];
      const int pos = qpos + rv.y;
      const bool ok = rv.x >= 0 && pos >= 0 && pos < A.Lout;
      uint32_t off = ok ? static_cast<uint32_t>(4 * (rv.x + pos)) : 0x80000000u;
      const float u = acc[mi][rg] * __int_as_float(rv.z);  // the scale (1 for fp16 weights)
      const float v = A.bias ? u + __int_as_float(rv.w) : u;
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), ors, off, 0, 0);
    }
  if (bad) {
    // a column with an infinity or a NaN: scalar fp32 products and sums over
    // the packed weights (fp16 -> fp32 exact) and the raw activations give
    // numpy's inf / NaN pattern
    const float* xb = A.x + b * Cin * L;
    const _Float16* wh = reinterpret_cast<const _Float16*>(A.wp);
    for (int i = 0; i < 16 * MI; ++i) {
      const int ml = 32 * (i / 16) + 8 * ((i % 16) / 4) + 4 * g + (i % 4);
      const int m = m0 + ml;
      const int4 rv = rows[ml];
      const int pos = qpos + rv.y;
      if (m >= A.M || pos < 0 || pos >= A.Lout) continue;
      float sum = 0.0f;
      for (int ci = 0; ci < Cin; ++ci)
        for (int t = 0; t < A.T; ++t) {
          const int p = q * A.qs + A.ta + t * A.tm;
          if (p < 0 || p >= L) continue;
          const int k = TP ? (ci % CPS) * TP + t : (t * Cin + ci) % 16;
          const int sl = TP ? ci / CPS : (t * Cin + ci) / 16;
          const int64_t unit = (static_cast<int64_t>(m / 32) * KS + sl) * 64 + (m % 32) + 32 * (k / 8);
          const _Float16 wv = wh[unit * 8 + k % 8];
          const float wf = TP ? static_cast<float>(wv) : static_cast<float>(__builtin_bit_cast(__bf16, wv));
          sum = sum + wf * xb[static_cast<int64_t>(ci) * L + p];
        }
      const float u = A.scale ? sum * __int_as_float(rv.z) : sum;
      A.out[b * A.Cout * A.Lout + rv.x + pos] = A.bias ? u + __int_as_float(rv.w) : u;
    }
  }
}

// ------------------------------------- 8-bit weights, channels in 128s
// The same implicit GEMM on the bf16 matrix cores (v_mfma_f32_32x32x16_bf16):
// an 8-bit weight less its zero point is exact in bf16, and an activation
// times 2^24 is split exactly into three bf16 parts by rounding (8 + 8 + 8
// significant bits), so three products per weight give exact fp32 products.
// The factor keeps the lower parts of the smallest floats out of bf16's
// subnormals (unscaled, activations below 2^-110 lost bits, and all but eight
// at 1e-38); the sums leave it in the epilogue.  It costs a multiplication a
// staged value (512 -> 512 k3 over 2400 steps 22.7 -> 23.0 us).  The reduction
// runs tap-major (k = t' Cin + ci): no padded taps, and an operand is eight
// channels at one time.
//
// A block owns 64 rows x 32 NI columns; its four waves take a quarter of the
// channels each and own nothing in common until they add their tiles.  A wave
// stages the time window its columns read, 32 channels at a time, in its own
// LDS (time-major, the three parts side by side, 208 bytes a row: the 32
// rows of an operand read start on distinct banks), so a value is loaded and
// split once a block instead of once a tap and 32 columns -- what bound the
// kernel above here, with ~60 VALU instructions beside four matrix
// instructions a slice.  While a chunk is multiplied the next one's values and
// weight fragments are in flight in registers.  Then each wave keeps one
// 32 x 32 tile of the 64 x 64 and adds the other waves' in wave order.
//
// An output that is not finite (an infinity or NaN in reach, a sample above
// 2^104 or a sum that 2^24 takes beyond fp32's range) is summed again with
// scalar fp32 products.
//
// Bound by each wave's chain (a chunk: window, products) at one or two waves
// a SIMD.  us, the kernel above (fp16 layout) -> this one: Conv1d 512 -> 512 k3
// over 2400 steps 32.7 -> 22.9, over 7000 76 -> 45, over 40 18.9 -> 10.3; 256 ->
// 256 k3 over 2400 15.5 -> 11.3; 512 -> 512 k7 over 7000 135 -> 87;
// ConvTranspose1d 512 -> 256 k20 s10 over 240 16.4 -> 14.0, over 700 28.9 -> 22.6.
// No further from 64 bits (2.0e-7 -> 1.9e-7 relative for the first).
constexpr int kQPitch = 208;  // bytes a staged row: three parts of 32 channels, 16 to spare
constexpr int kQRows = 64 * 16;  // bytes of the 64 rows' constants (static LDS)
constexpr int kQExchange = 4 * 3 * 16 * 64 * 4;  // bytes the waves' tiles take

template <int T, int NP, int NI>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(T == 7 && NI == 2 ? 1 : 2, 2)))
convq_kernel(CArgs A, int W) {
  extern __shared__ __align__(16) unsigned char convq_lds[];
  __shared__ int4 rows[kQRows / sizeof(int4)];  // output row offset, phase offset, scale, bias
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ln = lane & 31, g = lane >> 5;
  const uint3 tile = xcd_tile();  // row tiles fastest: a column range's blocks share an XCD
  const int m0 = __builtin_amdgcn_readfirstlane(static_cast<int>(tile.x)) * 64;
  const int n0 = __builtin_amdgcn_readfirstlane(static_cast<int>(tile.y)) * 32 * NI;
  const int64_t b = __builtin_amdgcn_readfirstlane(static_cast<int>(tile.z));
  const int Cin = A.Cin, L = A.L, C16 = Cin / 16;
  const float* xb = A.x + b * Cin * L;
  const auto xrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(xb), 0, Cin * L * 4, 0x00020000);
  const auto wrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint4*>(A.wp), 0, A.wbytes, 0x00020000);
  unsigned char* win = convq_lds + wv * W * kQPitch;
  if (tid < 64) {
    const int m = m0 + tid;
    int4 rv = make_int4(-1, 0, __float_as_int(1.0f), 0);
    if (m < A.M) {
      const int co = m / A.P, r = m - co * A.P;
      rv.x = co * A.Lout;
      rv.y = r + A.oph;
      if (A.scale) rv.z = __float_as_int(load_as_f32(A.scale, A.scale_dt, co * A.scale_stride));
      if (A.bias) rv.w = __float_as_int(A.bias[co]);
    }
    rows[tid] = rv;
  }
  // item p of a lane: eight channels (octet oct of the chunk) of staged row
  // rr, at byte offset xo of x; 0x7fffffff off the signal (loads give 0; no
  // sum with a channel's offset, below 2^31, wraps)
  uint32_t xo[NP];
  int dst[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int it = lane + 64 * p, oct = it / W, rr = it - oct * W;
    const int pos = n0 * A.qs + A.ta + rr;
    const bool ok = oct < 4;
    dst[p] = ok ? rr * kQPitch + 16 * oct : -1;
    xo[p] = ok && pos >= 0 && pos < L ? static_cast<uint32_t>(4 * pos) + static_cast<uint32_t>(32 * oct * L)
                                      : 0x7fffffffu;
  }
  const uint32_t row_bytes = static_cast<uint32_t>(4 * L);
  const int c_lo = Cin / 128 * wv, c_hi = Cin / 128 * (wv + 1);  // this wave's chunks of 32 channels
  float v[NP][8];
  auto load_x = [&](int c) {  // (past the last chunk the loads read 0 or another wave's channels)
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        uint32_t off = xo[p] + static_cast<uint32_t>(32 * c + e) * row_bytes;
        v[p][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xrs, off, 0, 0));
      }
  };
  // tap t's fragments of chunk c: k-steps 2 c and 2 c + 1 of the tap's C16,
  // row tiles m0 / 32 and the next
  const uint32_t a_lane = static_cast<uint32_t>(m0 / 32) * static_cast<uint32_t>(A.KS) * 1024u + 16u * lane;
  b8 a[T][2][2];
  auto load_a = [&](int c, auto tc) {
    constexpr int t = decltype(tc)::value;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int mi = 0; mi < 2; ++mi)
        a[t][ks][mi] = __builtin_bit_cast(
            b8, __builtin_amdgcn_raw_buffer_load_b128(
                    wrs, a_lane + static_cast<uint32_t>((mi * A.KS + t * C16 + 2 * c + ks) * 1024), 0, 0));
  };
  f16v acc[2][NI] = {};
  auto each_tap = [&](auto f) {
    [&]<int... t>(std::integer_sequence<int, t...>) { (f(std::integral_constant<int, t>{}), ...); }
    (std::make_integer_sequence<int, T>{});
  };
  // With few taps registers are left to read an operand ahead and to split
  // the next chunk's values among the last products (a SIMD has one or two
  // of these waves: nothing else fills those waits).
  constexpr bool kDeep = T <= 3 && NP <= 5;
  b8 part[NP][3];
  auto split = [&](int p) { split3(v[p], part[p]); };
  b8 x[2][NI][3];  // [step % 2][column tile][part]
  auto read_x = [&](auto step) {  // step: 2 t + ks of the chunk
    constexpr int t = decltype(step)::value / 2, ks = decltype(step)::value % 2;
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
      for (int k = 0; k < 3; ++k)
        x[ks][ni][k] = *reinterpret_cast<const b8*>(
            win + ((32 * ni + ln) * A.qs + t * A.tm) * kQPitch + 64 * k + 32 * ks + 16 * g);
  };
  auto products = [&](auto step) {
    constexpr int t = decltype(step)::value / 2, ks = decltype(step)::value % 2;
#pragma unroll
    for (int k = 2; k >= 0; --k)
#pragma unroll
      for (int mi = 0; mi < 2; ++mi)
#pragma unroll
        for (int ni = 0; ni < NI; ++ni)
          acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[t][ks][mi], x[ks][ni][k], acc[mi][ni], 0, 0, 0);
  };
  auto each_step = [&](auto f) {
    [&]<int... i>(std::integer_sequence<int, i...>) { (f(std::integral_constant<int, i>{}), ...); }
    (std::make_integer_sequence<int, 2 * T>{});
  };
  load_x(c_lo);
  each_tap([&](auto t) { load_a(c_lo, t); });
  if constexpr (kDeep)
#pragma unroll
    for (int p = 0; p < NP; ++p) split(p);
  for (int c = c_lo; c < c_hi; ++c) {
    // stage this chunk (the wave alone reads and writes its window; its LDS
    // accesses take effect in order)
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      if constexpr (!kDeep) split(p);
      if (dst[p] >= 0) {
#pragma unroll
        for (int k = 0; k < 3; ++k) *reinterpret_cast<b8*>(win + dst[p] + 64 * k) = part[p][k];
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // (sched_barrier: the scheduler would move these loads to the end of the
    // chunk, where the next one waits for them at once)
    load_x(c + 1);
    if constexpr (kDeep) read_x(std::integral_constant<int, 0>{});
    __builtin_amdgcn_sched_barrier(0);
    each_step([&](auto sc) {
      constexpr int i = decltype(sc)::value;
      if constexpr (!kDeep) read_x(sc);
      else if constexpr (i + 1 < 2 * T) read_x(std::integral_constant<int, i + 1>{});
      if constexpr (kDeep) __builtin_amdgcn_sched_barrier(0);
      products(sc);
      if constexpr (kDeep && i + 2 >= 2 * T) {
#pragma unroll
        for (int p = (i + 1 == 2 * T ? 2 : 0); p < (i + 1 == 2 * T ? NP : 2); ++p) split(p);
        // one matrix instruction, then VALU work in its shadow
#pragma unroll
        for (int k = 0; k < 6 * NI; ++k) {
          __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x2, i + 1 == 2 * T ? 12 : 8, 0);
        }
      }
      if constexpr (i % 2 == 1) load_a(c + 1, std::integral_constant<int, i / 2>{});
      if constexpr (kDeep || i % 2 == 1) __builtin_amdgcn_sched_barrier(0);
    });
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();  // every window is read
  // wave w keeps tile w = NI mi + ni; the others' go to LDS ([slot][register][lane])
  constexpr int kTiles = 2 * NI;
  float* red = reinterpret_cast<float*>(convq_lds);
  auto slot = [](int w, int q) { return NI == 2 ? w * 3 + ((q - w - 1) & 3) : w * 2 + q; };
#pragma unroll
  for (int q = 0; q < kTiles; ++q)
    if (q != wv)
#pragma unroll
      for (int r = 0; r < 16; ++r) red[(slot(wv, q) * 16 + r) * 64 + lane] = acc[q / NI][q % NI][r];
  f16v own = acc[0][0];
#pragma unroll
  for (int q = 1; q < kTiles; ++q)
    if (q == wv) own = acc[q / NI][q % NI];
  __syncthreads();
  if (wv >= kTiles) return;
  f16v sum;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    f16v part = own;
    if (w != wv) {
#pragma unroll
      for (int r = 0; r < 16; ++r) part[r] = red[(slot(w, wv) * 16 + r) * 64 + lane];
    }
    sum = w == 0 ? part : sum + part;
  }
  const int q = n0 + 32 * (wv % NI) + ln;
  const auto ors = __builtin_amdgcn_make_buffer_rsrc(A.out + b * A.Cout * A.Lout, 0,
                                                     A.Cout * A.Lout * 4, 0x00020000);
  const int qpos = q < A.Nq ? q * A.os : INT_MIN / 2;
#pragma unroll
  for (int rg = 0; rg < 16; ++rg) {
    const int ml = 32 * (wv / NI) + 8 * (rg / 4) + 4 * g + (rg % 4);
    const int4 rv = rows[ml];
    const int pos = qpos + rv.y;
    const bool ok = rv.x >= 0 && pos >= 0 && pos < A.Lout;
    float s = sum[rg] * (1.0f / kSplitScale);
    if (ok && !(fabsf(s) < INFINITY)) {
      const __bf16* wh = reinterpret_cast<const __bf16*>(A.wp);
      s = 0.0f;
      for (int ci = 0; ci < Cin; ++ci)
        for (int t = 0; t < T; ++t) {
          const int p = q * A.qs + A.ta + t * A.tm;
          if (p < 0 || p >= L) continue;
          const int k = t * Cin + ci, m = m0 + ml;
          const int64_t unit = (static_cast<int64_t>(m / 32) * A.KS + k / 16) * 64 + (m % 32) + 32 * (k % 16 / 8);
          s = s + static_cast<float>(wh[unit * 8 + k % 8]) * xb[static_cast<int64_t>(ci) * L + p];
        }
    }
    const uint32_t off = ok ? static_cast<uint32_t>(4 * (rv.x + pos)) : 0x80000000u;
    const float u = s * __int_as_float(rv.z);
    const float y = A.bias ? u + __int_as_float(rv.w) : u;
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y), ors, off, 0, 0);
  }
}

// Whether 8-bit weights of this geometry are laid out for convq_kernel: whole
// 128-channel rounds for its four waves, and not two taps of 128 channels, of
// which the fp16 layout pads none and a wave has one chunk, with nothing to
// overlap (128 -> 128 k2 over 9000 steps 11.0 us there, 11.7 here; over 17,000
// 14.3 and 17.0).  From 256 channels two taps gain more often than they lose
// (256 -> 128 stride 6 over 2400 steps 19.5 and 15.6, over 1600 13.8 and 15.0;
// 256 -> 256 over 5000 13.9 and 14.8, over 17,000 35.1 and 31.1; 512 -> 256
// stride 8 over 1000 30.3 and 23.6, over 8000 144 and 156).
static bool tap_major(const Geo& g, int w_dt) {
  return w_dt != KK_F16 && g.Cin % 128 == 0 && g.T <= 7 && !(g.T == 2 && g.Cin < 256);
}

template <int T, int NP, int NI>
static int launch_q(const CArgs& a, int W, int64_t batch) {
  const dim3 grid(static_cast<unsigned>(ceil_div(a.M, 64)), static_cast<unsigned>(ceil_div(a.Nq, 32 * NI)),
                  static_cast<unsigned>(batch));
  KK_TRY(check_xcd_grid(grid, "convq_kernel"));
  const int lds = std::max(4 * W * kQPitch, NI == 2 ? kQExchange : kQExchange * 2 / 3);
  if (lds + kQRows > 65536) KK_TRY(allow_large_lds(reinterpret_cast<const void*>(convq_kernel<T, NP, NI>)));
  KK_LAUNCH((convq_kernel<T, NP, NI>), grid, dim3(kThreads), static_cast<size_t>(lds), ctx().stream, a, W);
  return check_launch("convq_kernel");
}

// The launch shape: MI 32-row tiles a wave, WK waves a column range.
struct Shape {
  int mi, wk;
};

// 128 rows a wave when that still gives every SIMD a wave, else 64 (32 for
// at most 32 rows); then as many waves on the reduction (1, 2 or 4) as it
// takes to give every SIMD two waves, each at least three slices.
static Shape pick_shape(const CArgs& a, int64_t batch) {
  Shape s{};
  const int64_t simds = 4 * (ctx().num_cus > 0 ? ctx().num_cus : 256);
  const int64_t cols = batch * ceil_div(a.Nq, 32);
  s.mi = a.M <= 32 ? 1 : (a.M > 64 && cols * ceil_div(a.M, 128) >= simds) ? 4 : 2;
  const int64_t waves = cols * ceil_div(a.M, 32 * s.mi);
  s.wk = waves >= 2 * simds ? 1 : waves * 2 >= 2 * simds ? 2 : 4;
  while (s.wk > 1 && a.KS < 3 * s.wk) s.wk /= 2;
  return s;
}

template <int TP, int MI, int WK>
static int launch_shape(const CArgs& a, int64_t batch) {
  constexpr int BM = 32 * MI, BN = 32 * (4 / WK);
  constexpr int R = 3;  // slices in flight (six measured no faster at MI <= 2)
  const dim3 grid(static_cast<unsigned>(ceil_div(a.M, BM)), static_cast<unsigned>(ceil_div(a.Nq, BN)),
                  static_cast<unsigned>(batch));
  KK_TRY(check_xcd_grid(grid, "convh_kernel"));
  KK_LAUNCH((convh_kernel<TP, MI, WK, R>), grid, dim3(kThreads), 0, ctx().stream, a);
  return check_launch("convh_kernel");
}

template <int TP>
static int launch_tp(const CArgs& a, const Shape& s, int64_t batch) {
#define KK_CONVH_WK(MI)                                           \
  switch (s.wk) {                                                 \
    case 1: return launch_shape<TP, MI, 1>(a, batch);             \
    case 2: return launch_shape<TP, MI, 2>(a, batch);             \
    default: return launch_shape<TP, MI, 4>(a, batch);            \
  }
  if (s.mi == 1) KK_CONVH_WK(1)
  if (s.mi == 2) KK_CONVH_WK(2)
  KK_CONVH_WK(4)
#undef KK_CONVH_WK
}

// Runs convq_kernel if a block's window fits; the rule is of one to seven taps
// T, the window W of 64 columns (W32 of 32) and the blocks of 64.  Measured
// over 128 to 1024 channels, 300 to 17,000 steps, strides 1 to 4 and dilations
// 1 to 70 against the fp16 layout (1.0 = that kernel's time):
//  - 32 columns a block where 64 leave half the CUs without one (512 -> 512 k3
//    over 40 steps, 8 blocks: 14.2 us with 64, 10.1 with 32; 256 -> 256 k3 over
//    2400, 152 blocks: 11.1 either way), where 64 need more than 96 staged
//    rows, which cost more than the columns save (512 -> 512 k5 stride 2 0.46 -
//    0.55, k7 dilation 9 0.63 - 0.73; through convh_kernel<0> 0.67 - 1.03), and
//    with seven taps, whose fragments leave a SIMD one wave of 64 columns, from
//    a block a CU on (256 -> 256 over 5000 steps, 316 blocks, 0.73 against
//    0.89; over 2400, 152 blocks, 0.71 against 0.65).
//  - one tap: a window is read once, so staging pays only for few blocks (512
//    -> 512 over 9000 steps 0.67 staged, 0.65 not; 128 channels 0.90 and 0.85).
//  - wider windows: convh_kernel<0> (0.67 - 1.06; 0.98 - 1.15 with two and four
//    taps, of which the fp16 layout pads none).
template <int T>
static bool launch_q(const CArgs& a, int64_t W, int64_t batch, int* rc) {
  const int64_t cus = ctx().num_cus > 0 ? ctx().num_cus : 256;
  const int64_t W32 = W - int64_t{32} * a.qs;
  const int64_t blocks = ceil_div(a.M, 64) * ceil_div(a.Nq, 64) * batch;
  const bool narrow = blocks * 2 <= cus;
  if (W32 > 128) return false;
  const int w = static_cast<int>(std::min<int64_t>(W, 128)), w32 = static_cast<int>(W32);
  if constexpr (T == 1) {
    if (!narrow || W32 > 48) return false;
    *rc = launch_q<T, 3, 1>(a, w32, batch);
  } else if constexpr (T <= 4) {
    if (narrow && W32 <= 48) *rc = launch_q<T, 3, 1>(a, w32, batch);
    else if (narrow && W32 <= 80) *rc = launch_q<T, 5, 1>(a, w32, batch);
    else if (W <= 80) *rc = launch_q<T, 5, 2>(a, w, batch);
    else if (W <= 96) *rc = launch_q<T, 6, 2>(a, w, batch);
    else if (W32 <= 80) *rc = launch_q<T, 5, 1>(a, w32, batch);
    else if (T == 4) *rc = launch_q<4, 8, 1>(a, w32, batch);
    else return false;
  } else {
    if (!narrow && (T < 7 || blocks <= cus) && W <= 96) *rc = launch_q<T, 6, 2>(a, w, batch);
    else if (W32 <= 64) *rc = launch_q<T, 4, 1>(a, w32, batch);
    else if (W32 <= 96) *rc = launch_q<T, 6, 1>(a, w32, batch);
    else return false;
  }
  return true;
}

// tp: the taps a channel spans; 0 for tap-major weights.
static int launch(const CArgs& a, int tp, int64_t batch) {
  if (tp == 0) {
    const int64_t W = int64_t{63} * a.qs + static_cast<int64_t>(a.T - 1) * a.tm + 1;
    int rc = KK_OK;
    bool ran = false;
    switch (a.T) {
      case 1: ran = launch_q<1>(a, W, batch, &rc); break;
      case 2: ran = launch_q<2>(a, W, batch, &rc); break;
      case 3: ran = launch_q<3>(a, W, batch, &rc); break;
      case 4: ran = launch_q<4>(a, W, batch, &rc); break;
      case 5: ran = launch_q<5>(a, W, batch, &rc); break;
      case 6: ran = launch_q<6>(a, W, batch, &rc); break;
      default: ran = launch_q<7>(a, W, batch, &rc); break;
    }
    return ran ? rc : launch_tp<0>(a, pick_shape(a, batch), batch);
  }
  const Shape s = pick_shape(a, batch);
  if (tp == 2) return launch_tp<2>(a, s, batch);
  if (tp == 4) return launch_tp<4>(a, s, batch);
  return launch_tp<8>(a, s, batch);
}

// The pack of w (less its zero point) into `wp` (g.bytes, 16-byte aligned).
static int pack(const Geo& g, void* wp, const kk_tensor* w, const Dequant& dq) {
  PackArgs p{};
  p.wp = static_cast<uint4*>(wp);
  p.w = w->data;
  p.zp = dq.zp;
  p.zp_dt = dq.zp_dt;
  p.zp_stride = static_cast<int>(dq.zp_stride);
  p.Cin = static_cast<int>(g.Cin); p.Cout = static_cast<int>(g.Cout); p.Kw = static_cast<int>(g.Kw);
  p.P = static_cast<int>(g.P); p.T = static_cast<int>(g.T); p.TP = static_cast<int>(g.TP);
  p.M = static_cast<int>(g.M); p.KS = static_cast<int>(g.KS);
  p.transposed = g.transposed;
  p.tap_major = tap_major(g, w->dtype) ? 1 : 0;
  if (p.tap_major) p.KS = static_cast<int>(g.T * g.Cin / 16);  // (no more than g.KS)
  p.units = g.MT * p.KS * 64;
  const dim3 grid(static_cast<unsigned>(ceil_div(p.units, 256)));
  if (w->dtype == KK_F16) KK_LAUNCH(convh_pack<_Float16>, grid, dim3(256), 0, ctx().stream, p);
  else if (w->dtype == KK_I8) KK_LAUNCH(convh_pack<int8_t>, grid, dim3(256), 0, ctx().stream, p);
  else KK_LAUNCH(convh_pack<uint8_t>, grid, dim3(256), 0, ctx().stream, p);
  return check_launch("convh_pack");
}

// Weights the fp16 path takes: fp16 as they are; 8-bit less an 8-bit zero
// point (the difference is an integer of at most 255: exact in fp16).
static bool weights_ok(const kk_tensor* w, const Dequant& dq) {
  const bool w16 = w->dtype == KK_F16 && !dq.active;
  const bool w8 = (w->dtype == KK_I8 || w->dtype == KK_U8) &&
                  (!dq.zp || dq.zp_dt == KK_I8 || dq.zp_dt == KK_U8);
  return w16 || w8;
}

// The launch arguments of a call, or false when the fp16 path does not
// apply (more than 8 taps, or sizes beyond its 32-bit offsets and grid).
static bool make_args(CArgs* a, const Geo& g, bool taps_first, const kk_tensor* out,
                      const kk_tensor* x, const Dequant& dq, const kk_tensor* bias, int64_t stride,
                      int64_t dilation, int64_t pad0, int64_t Nq) {
  const int64_t N = x->shape[0], L = x->shape[2], Lout = out->shape[2];
  if (!g.TP || x->dtype != KK_F32 || N > 65535 || g.Cin * L * 4 >= (int64_t{1} << 31) ||
      g.Cout * Lout * 4 >= (int64_t{1} << 31) || g.bytes >= (int64_t{1} << 31) ||
      (Nq + 1) * std::max<int64_t>(stride, 1) + g.TP * dilation + pad0 >= (int64_t{1} << 29) ||
      (Nq + 1) * g.P + Lout + pad0 >= (int64_t{1} << 30) || g.M >= (int64_t{1} << 30))
    return false;
  *a = CArgs{};
  a->x = static_cast<const float*>(x->data);
  a->out = static_cast<float*>(out->data);
  a->bias = bias ? static_cast<const float*>(bias->data) : nullptr;
  a->scale = dq.scale;
  a->scale_dt = dq.scale_dt;
  a->scale_stride = static_cast<int>(dq.scale_stride);
  a->Cin = static_cast<int>(g.Cin); a->L = static_cast<int>(L);
  a->Cout = static_cast<int>(g.Cout); a->Lout = static_cast<int>(Lout);
  a->M = static_cast<int>(g.M); a->Nq = static_cast<int>(Nq); a->P = static_cast<int>(g.P);
  a->T = static_cast<int>(g.T);
  a->KS = static_cast<int>(taps_first ? g.T * g.Cin / 16 : g.KS);
  if (g.transposed) {
    a->qs = 1; a->ta = static_cast<int>(1 - g.T); a->tm = 1;
    a->os = static_cast<int>(g.P); a->oph = static_cast<int>(-pad0);
  } else {
    a->qs = static_cast<int>(stride); a->ta = static_cast<int>(-pad0); a->tm = static_cast<int>(dilation);
    a->os = 1; a->oph = 0;
  }
  // (no more than convh_pack wrote: a row tile past the last reads 0)
  a->wbytes = static_cast<int>(g.MT * a->KS * 1024);
  return true;
}

// What a packed buffer was made from (checked by every packed call).
struct PackRecord {
  const void* w;
  int64_t d0, d1, d2;
  int w_dt;
  const void* zp;
  int zp_dt;
  int transposed;
  int64_t stride;
};
static std::mutex g_pack_mu;
static std::unordered_map<const void*, PackRecord> g_packs;

static PackRecord record_of(const kk_tensor* w, const kk_tensor* w_zp, bool transposed, int64_t stride) {
  return PackRecord{w->data, w->shape[0], w->shape[1], w->shape[2], w->dtype,
                    w_zp ? w_zp->data : nullptr, w_zp ? w_zp->dtype : -1, transposed ? 1 : 0,
                    transposed ? stride : 1};
}

}  // namespace convh

using namespace convh;

void convh_forget_pack(const void* p) {
  std::lock_guard<std::mutex> lock(g_pack_mu);
  g_packs.erase(p);
}

// The fp16 matrix-core convolution of one call: true when it ran (its
// status in *rc), false when it does not apply (the caller runs the fp32
// kernels).  `packed` (checked by the caller) holds the weights laid out by
// kk_conv_pack; without it they are laid out here, in the context scratch
// (or a pooled workspace, freed after the launch in stream order).
bool convh_run(const kk_tensor* out, const kk_tensor* x, const kk_tensor* w, const Dequant& dq,
               const kk_tensor* bias, bool transposed, int64_t stride, int64_t dilation,
               int64_t pad0, int64_t Nq, const kk_tensor* packed, int* rc) {
  *rc = KK_OK;
  if (!weights_ok(w, dq) || (transposed && dilation != 1)) return false;
  const int64_t Cin = x->shape[1];
  const int64_t Cout = out->shape[1], Kw = w->shape[2];
  const Geo g = geometry(transposed, Cin, Cout, Kw, stride);
  // enough work for the matrix cores
  if (Cin < 8 || g.M * Nq * g.T * Cin < (int64_t{1} << 24)) return false;
  CArgs a;
  const bool taps_first = tap_major(g, w->dtype);
  const int tp = taps_first ? 0 : static_cast<int>(g.TP);
  if (!make_args(&a, g, taps_first, out, x, dq, bias, stride, dilation, pad0, Nq)) return false;
  if (packed) {
    a.wp = static_cast<const uint4*>(packed->data);
  } else {
    void* wp = nullptr;
    void* ws = nullptr;
    if (g.bytes <= static_cast<int64_t>(kScratchBytes)) wp = ctx().scratch;
    else if (!ctx().capturing && kk_alloc(static_cast<size_t>(g.bytes), &ws) == KK_OK) wp = ws;
    if (!wp) return false;
    *rc = pack(g, wp, w, dq);
    if (*rc == KK_OK) {
      a.wp = static_cast<const uint4*>(wp);
      *rc = launch(a, tp, x->shape[0]);
    }
    if (ws) kk_free(ws);  // stream order keeps it alive for the kernels above
    return true;
  }
  *rc = launch(a, tp, x->shape[0]);
  return true;
}

// Checks a packed buffer against the call: its size and alignment, and that
// the last kk_conv_pack into it read this w (and zero point) for this
// geometry.
int convh_check_packed(const kk_tensor* packed, const kk_tensor* w, const kk_tensor* w_zp,
                       bool transposed, int64_t stride, const char* who) {
  KK_TRY(check_tensor(packed, "packed"));
  const int64_t cin = transposed ? w->shape[0] : w->shape[1];
  const int64_t cout = transposed ? w->shape[1] : w->shape[0];
  const int64_t need = geometry(transposed, cin, cout, w->shape[2], stride).bytes;
  if (packed->dtype != KK_U8 || !is_contiguous(packed) || numel(packed) != need ||
      reinterpret_cast<uintptr_t>(packed->data) % 256 != 0)
    return set_error(KK_E_ARG, "%s: packed must be %lld contiguous, 256-byte aligned uint8 bytes",
                     who, (long long)need);
  const PackRecord want = record_of(w, w_zp, transposed, stride);
  std::lock_guard<std::mutex> lock(g_pack_mu);
  auto it = g_packs.find(packed->data);
  if (it == g_packs.end()) return set_error(KK_E_ARG, "%s: packed was not made by kk_conv_pack", who);
  const PackRecord& r = it->second;
  if (r.w != want.w || r.d0 != want.d0 || r.d1 != want.d1 || r.d2 != want.d2 || r.w_dt != want.w_dt)
    return set_error(KK_E_ARG, "%s: packed was made from another weight tensor", who);
  if (r.zp != want.zp || r.zp_dt != want.zp_dt)
    return set_error(KK_E_ARG, "%s: packed was made with another weight zero point", who);
  if (r.transposed != want.transposed || r.stride != want.stride)
    return set_error(KK_E_ARG, "%s: packed was made for another %s", who,
                     r.transposed != want.transposed ? "operation" : "stride");
  return KK_OK;
}

}  // namespace kk

using namespace kk;

extern "C" {

int kk_conv_packed_bytes(int transposed, int64_t cin, int64_t cout, int64_t k, int stride,
                         int64_t* bytes) {
  if (!bytes || cin <= 0 || cout <= 0 || k <= 0 || stride < 1)
    return set_error(KK_E_ARG, "kk_conv_packed_bytes: positive sizes, stride and an output");
  const Geo g = geometry(transposed != 0, cin, cout, k, stride);
  if (!g.TP)
    return set_error(KK_E_UNSUPPORTED, "kk_conv_packed_bytes: %lld taps a row (more than 8) are "
                     "not packed", (long long)g.T);
  *bytes = g.bytes;
  return KK_OK;
}

int kk_conv_pack(const kk_tensor* packed, const kk_tensor* w, const kk_tensor* w_zp,
                 int transposed, int stride) {
  const char* who = "kk_conv_pack";
  KK_TRY(require_ready());
  KK_TRY(check_tensor(w, "w"));
  if (w->rank != 3 || !(w->dtype == KK_F16 || w->dtype == KK_I8 || w->dtype == KK_U8) ||
      !is_contiguous(w) || numel(w) == 0 || stride < 1)
    return set_error(KK_E_ARG,
                     "%s: w must be a non-empty contiguous fp16/int8/uint8 tensor of rank 3 and "
                     "stride >= 1", who);
  const bool tr = transposed != 0;
  const int64_t cin = tr ? w->shape[0] : w->shape[1];
  const int64_t cout = tr ? w->shape[1] : w->shape[0];
  Dequant dq;
  if (w_zp) {
    if (w->dtype == KK_F16) return set_error(KK_E_ARG, "%s: an fp16 weight takes no zero point", who);
    KK_TRY(check_tensor(w_zp, "w_zp"));
    if (!(w_zp->dtype == KK_I8 || w_zp->dtype == KK_U8))
      return set_error(KK_E_ARG, "%s: w_zp must be int8/uint8", who);
    KK_TRY(zp_shift(&dq, w_zp, cout, who));
  }
  const Geo g = geometry(tr, cin, cout, w->shape[2], stride);
  if (!g.TP)
    return set_error(KK_E_UNSUPPORTED, "%s: %lld taps a row (more than 8) are not packed", who,
                     (long long)g.T);
  if (g.bytes >= (int64_t{1} << 31))
    return set_error(KK_E_UNSUPPORTED, "%s: %lld packed bytes exceed 2 GiB", who, (long long)g.bytes);
  KK_TRY(check_tensor(packed, "packed"));
  if (packed->dtype != KK_U8 || !is_contiguous(packed) || numel(packed) != g.bytes ||
      reinterpret_cast<uintptr_t>(packed->data) % 256 != 0)
    return set_error(KK_E_ARG, "%s: packed must be %lld contiguous, 256-byte aligned uint8 bytes",
                     who, (long long)g.bytes);
  {
    std::lock_guard<std::mutex> lock(g_pack_mu);
    g_packs[packed->data] = record_of(w, w_zp, tr, stride);
  }
  return pack(g, packed->data, w, dq);
}

}  // extern "C"
