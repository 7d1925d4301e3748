// Bulk dequantizers and weight quantizers (FP4 E2M1 and asymmetric INT4),
// plus the library's error-string plumbing.
//
// Compiled with -ffp-contract=off: the quantizers must reproduce the
// reference's numpy float32 arithmetic operation by operation.
#include <stdarg.h>
#include <stdio.h>

#include "mm_common.h"

static thread_local char g_err[512] = "";

void mm_set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}

extern "C" const char* mm_last_error(void) { return g_err; }

// ---------------------------------------------------------------------------
// Bulk dequant [K/8, N] -> [K, N] fp16 (kernels_core.py:747-791; bit-exact with
// src/marlin_gemm.metal:130-185).  Write-bound: 16 B out per packed word.
// V adjacent words of one word row per thread.  V = 4 (N % 4 == 0, aligned
// operands): 16-byte word loads and 8-byte stores, 512 contiguous bytes per wave
// and row, the threads numbered through all rows (a block per 1024 columns of each
// row leaves a third of the threads idle at N = 1336).  One word per thread
// (V = 1, 128 bytes per wave store) is the form any other N takes, and small
// matrices: with fewer than 256 blocks of the wide form four times the threads count
// for more (1024 x 100 2.0 against 2.4 us, 1024 x 1024 2.2 against 2.3; 2048 x 1000
// 2.8 against 2.7, 2048 x 2048 3.8 against 3.4).
// NT: the stores bypass the caches.  That is faster where a wave's rows are whole
// 128-byte lines (N % 64 == 0, W on a line); part lines are put together in the
// caches, where a destination that is used again may also still lie (48 MB of
// fp16 fit them).  us with a destination never seen before and a reused one:
//                        V = 1         V = 4         V = 4, NT
//   4096 x 14336 FP4     32.9, 23.3    29.4, 23.7    22.8, 22.6
//   4096 x 4096 FP4      11.7,  9.1    10.3,  8.2     7.4,  7.2
//   5376 x 4516 INT4     19.5, 14.1    17.1, 13.0    14.6, 14.5
//   8576 x 1336 FP4      11.3,  7.6     7.9,  7.0     7.5,  7.4
// Non-temporal loads of the words cost 1 to 4 us in each of these.
// ---------------------------------------------------------------------------
template <int V, bool INT4, bool NT = false>
__global__ void __launch_bounds__(256)
k_dequant(const uint32_t* __restrict__ B, const f16* __restrict__ S, const f16* __restrict__ Z,
          f16* __restrict__ W, int K, int N, int g) {
  typedef uint32_t wv __attribute__((ext_vector_type(V)));
  typedef f16 hv __attribute__((ext_vector_type(V)));
  int n, kp;
  if constexpr (V == 1) {
    n = blockIdx.x * 256 + threadIdx.x;
    kp = blockIdx.y;
    if (n >= N) return;
  } else {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x, per_row = (uint32_t)N / V;
    kp = (int)(i / per_row);
    n = (int)(i - kp * per_row) * V;
    if (kp >= K / 8) return;
  }
  const size_t gi = (size_t)((kp * 8) / g) * N + n;
  wv w;
  hv s, z;
  if constexpr (V == 1) {
    w[0] = B[(size_t)kp * N + n];
    s[0] = S[gi];
    if constexpr (INT4) z[0] = Z[gi];
  } else {
    w = *(const wv*)(B + (size_t)kp * N + n);
    s = *(const hv*)(S + gi);
    if constexpr (INT4) z = *(const hv*)(Z + gi);
  }
  f16x8 v[V];
#pragma unroll
  for (int j = 0; j < V; ++j) {
    const f16 sj = s[j];
    if constexpr (INT4) {
      const f16 nz = -clamp_zero(z[j]);
      v[j] = dq_u4_word(w[j], f16x2{nz, nz}, f16x2{sj, sj});
    } else {
      v[j] = dq_fp4_word(w[j], f16x2{sj, sj});
    }
    // reference guard: a non-finite scale gives +0.0
    if (!__builtin_isfinite((float)sj)) v[j] = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
  }
  f16* out = W + (size_t)kp * 8 * N + n;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    hv o;
#pragma unroll
    for (int j = 0; j < V; ++j) o[j] = v[j][i];
    if constexpr (V == 1)
      out[(size_t)i * N] = o[0];
    else if constexpr (NT)
      __builtin_nontemporal_store(o, (hv*)(out + (size_t)i * N));
    else
      *(hv*)(out + (size_t)i * N) = o;
  }
}

// ---------------------------------------------------------------------------
// FP4 quantizer, Marlin layout: metal_marlin/quantize_fp4.py:131-284 with
// quantize_to_fp4 :64-107.  One thread per (group, output column n); the input
// is W [N, K] (out_features, in_features), fp16 or fp32.
// ---------------------------------------------------------------------------
MM_DEV uint32_t e2m1_nearest(float v) {
  const float T[8] = {0.0f, 0.5f, 1.0f, 1.5f, 2.0f, 3.0f, 4.0f, 6.0f};
  // NaN: np.clip keeps it and argmin over all-NaN distances picks index 0 of
  // the negative table (NaN >= 0 is false): code 8.
  if (v != v) return 8u;
  const bool neg = !(v >= 0.0f);
  // np.clip(v, lo, hi) == minimum(maximum(v, lo), hi)
  const float c = neg ? fminf(fmaxf(v, -6.0f), 0.0f) : fminf(fmaxf(v, 0.0f), 6.0f);
  uint32_t best = 0;
  float bd = fabsf(neg ? c + T[0] : c - T[0]);
#pragma unroll
  for (int i = 1; i < 8; ++i) {
    const float d = fabsf(neg ? c + T[i] : c - T[i]);
    if (d < bd) {   // strict: ties keep the lower index, like argmin
      bd = d;
      best = i;
    }
  }
  return best + (neg ? 8u : 0u);
}

template <typename T>
MM_DEV float ld_f32(const T* p) { return (float)*p; }

template <typename T>
__global__ void __launch_bounds__(256)
k_fp4_quantize(const T* __restrict__ Wt, int N, int K, int g,
               uint32_t* __restrict__ B, f16* __restrict__ S) {
  const int n = blockIdx.x * 256 + threadIdx.x;
  const int gi = blockIdx.y;
  if (n >= N) return;
  const T* row = Wt + (size_t)n * K + (size_t)gi * g;
  // np.max and np.maximum propagate NaN (fmaxf would drop it).
  float amax = 0.0f;
  bool nan = false;
  for (int k = 0; k < g; ++k) {
    const float a = fabsf(ld_f32(row + k));
    nan |= a != a;
    amax = fmaxf(amax, a);
  }
  amax = nan ? __builtin_nanf("") : fmaxf(amax, 1e-7f);
  S[(size_t)gi * N + n] = (f16)(amax / 6.0f);
  const int wpg = g / 8;
  for (int w8 = 0; w8 < wpg; ++w8) {
    uint32_t word = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float v = ld_f32(row + 8 * w8 + i) / amax * 6.0f;
      word |= e2m1_nearest(v) << (4 * i);
    }
    B[((size_t)gi * wpg + w8) * N + n] = word;
  }
}

// ---------------------------------------------------------------------------
// Calibration-aware FP4 quantizer: the activation_ranges branch of
// quantize_fp4.py:205-256, in numpy's own arithmetic (the host derives the
// constants the way numpy does):
//   group max   np.percentile(|w|, p) ('linear': order statistics kprev and
//               knext of the group's |w|, numpy's _lerp in float32 with
//               weight gamma) when use_pct, else the absmax; a NaN in the
//               group gives NaN (numpy sorts NaN last and flags the slice);
//               then max(., f32(1e-7))
//   mode 0      group max as is (no input range)
//   mode 1      act > 1: f32(c1 * gmax) + f32(c2 * gmax), c1 = f32(1 - sf),
//               c2 = f32(sf)
//   mode 2      act <= 1: the calibrated max gmax * sqrt(act) is a float64
//               product, so the blend f32(c1 * gmax) + sf * (gmax * att) and
//               the scale's division by 6 run in float64, and the scale is the
//               float64 quotient rounded once to fp16
//   codes       nearest E2M1 of w / f32(group max) * 6, as the weight-only path
// ---------------------------------------------------------------------------
struct FqCal {
  int use_pct, kprev, knext;
  float gamma;
  int mode;
  float c1, c2;
  double sf, att;
};

// k-th smallest (0-based) of |row[0..g)| by rank counting (offline, g^2).
template <typename T>
MM_DEV float kth_abs(const T* row, int g, int k) {
  for (int i = 0; i < g; ++i) {
    const float v = fabsf(ld_f32(row + i));
    int less = 0, eq = 0;
    for (int j = 0; j < g; ++j) {
      const float a = fabsf(ld_f32(row + j));
      less += a < v;
      eq += a == v;
    }
    if (less <= k && k < less + eq) return v;
  }
  return __builtin_nanf("");
}

// fp16 of a float64 value, rounded once: round to float with the sticky bit
// kept in the last place (round-to-odd), then float -> fp16 to nearest even.
// Round-to-odd to 24 bits followed by a rounding to 11 bits is the correctly
// rounded result (the intermediate has more than 2 extra bits).
MM_DEV f16 f16_from_f64(double d) {
  float f = (float)d;
  if ((double)f != d && f == f) {
    uint32_t b = __builtin_bit_cast(uint32_t, f);
    if (fabs((double)f) > fabs(d)) b -= 1;     // back toward zero (truncation)
    f = __builtin_bit_cast(float, b | 1u);
  }
  return (f16)f;
}

template <typename T>
__global__ void __launch_bounds__(256)
k_fp4_quantize_cal(const T* __restrict__ Wt, int N, int K, int g, FqCal cal,
                   uint32_t* __restrict__ B, f16* __restrict__ S) {
  const int n = blockIdx.x * 256 + threadIdx.x;
  const int gi = blockIdx.y;
  if (n >= N) return;
  const T* row = Wt + (size_t)n * K + (size_t)gi * g;
  float amax = 0.0f;
  bool nan = false;
  for (int k = 0; k < g; ++k) {
    const float a = fabsf(ld_f32(row + k));
    nan |= a != a;
    amax = fmaxf(amax, a);
  }
  float gmw = amax;
  if (nan) {
    gmw = __builtin_nanf("");
  } else if (cal.use_pct) {
    const float a = kth_abs(row, g, cal.kprev);
    const float b = cal.knext == cal.kprev ? a : kth_abs(row, g, cal.knext);
    const float diff = b - a;
    gmw = cal.gamma >= 0.5f ? b - diff * (1.0f - cal.gamma) : a + diff * cal.gamma;
  }
  gmw = gmw != gmw ? gmw : fmaxf(gmw, 1e-7f);    // np.maximum propagates NaN
  float gmf;
  f16 scale;
  if (cal.mode == 2) {
    const double gm = (double)(cal.c1 * gmw) + cal.sf * ((double)gmw * cal.att);
    scale = f16_from_f64(gm / 6.0);
    gmf = (float)gm;
  } else {
    gmf = cal.mode == 1 ? cal.c1 * gmw + cal.c2 * gmw : gmw;
    scale = (f16)(gmf / 6.0f);
  }
  S[(size_t)gi * N + n] = scale;
  const int wpg = g / 8;
  for (int w8 = 0; w8 < wpg; ++w8) {
    uint32_t word = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float v = ld_f32(row + 8 * w8 + i) / gmf * 6.0f;
      word |= e2m1_nearest(v) << (4 * i);
    }
    B[((size_t)gi * wpg + w8) * N + n] = word;
  }
}

// ---------------------------------------------------------------------------
// Asymmetric INT4 quantizer, Marlin layout: metal_marlin.py:184-280
// (pack_u4_weights).  Input W [N, K] fp16.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
k_u4_quantize(const f16* __restrict__ Wt, int N, int K, int g,
              uint32_t* __restrict__ B, f16* __restrict__ S, f16* __restrict__ Z) {
  const int n = blockIdx.x * 256 + threadIdx.x;
  const int gi = blockIdx.y;
  if (n >= N) return;
  const f16* row = Wt + (size_t)n * K + (size_t)gi * g;
  float mn = (float)row[0], mx = (float)row[0];
  for (int k = 1; k < g; ++k) {
    const float v = (float)row[k];
    mn = fminf(mn, v);
    mx = fmaxf(mx, v);
  }
  const float s = fmaxf((mx - mn) / 15.0f, 1e-7f);
  const float z = rintf(-mn / s);
  S[(size_t)gi * N + n] = (f16)s;
  Z[(size_t)gi * N + n] = (f16)z;
  const int wpg = g / 8;
  for (int w8 = 0; w8 < wpg; ++w8) {
    uint32_t word = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float q = rintf((float)row[8 * w8 + i] / s + z);
      q = fminf(fmaxf(q, 0.0f), 15.0f);
      word |= (uint32_t)q << (4 * i);
    }
    B[((size_t)gi * wpg + w8) * N + n] = word;
  }
}

// ---------------------------------------------------------------------------
// Tiled quantizers (FP4 absmax and asymmetric INT4), same results as
// k_fp4_quantize / k_u4_quantize.  Those walk a group per thread: adjacent
// lanes sit K elements apart, so every 2-byte load is a line of its own and the
// kernel ran at 0.08 TB/s (14336 x 4096 fp16, g = 128: 1700 us).  Here a lane
// holds the 8 elements of one output word, a wave 512 consecutive k of one row
// (1 KiB of fp16, read once, kept in registers for both passes), a group's
// extremes come from the g/8 adjacent lanes that share it, and a 64 x 64-word
// tile is transposed through LDS so that the words leave as 256-byte runs of
// the Marlin layout: 36.6 us (4.0 TB/s; a large copy reaches 4.7).  What bounds
// it is arithmetic as much as memory: with a division and a search over the
// eight magnitudes per element the same tiling took 60 us.
// Takes group sizes 8 * 2^i <= 512 and 16-byte aligned weights.
// ---------------------------------------------------------------------------

// x / a, correctly rounded, for r = RN(1 / a): one Newton step on the quotient
// with an exact remainder (Markstein, "Computation of elementary functions on
// the IBM RISC System/6000 processor", 1990).  Its conditions -- no overflow or
// underflow on the way -- hold for a in [1e-7, 2^40] (both quantizers floor
// their divisor at 1e-7) and |x| that is zero or at least 2^-80; for fp16 x the
// latter always holds.  A quotient is then zero or at least 2^-120 and a
// remainder at least 2^-126, both normal; a negative x never gives -0, which
// fp4_ties_down must not get.
MM_DEV float div_by(float x, float a, float r) {
  const float q = x * r;
  return __builtin_fmaf(__builtin_fmaf(-q, a, x), r, q);
}
MM_DEV bool div_ok(float a) { return a <= 0x1p40f; }

// Moves v one step toward zero and sets its last bit: the hardware's
// round-to-even FP4 convert then sends a midpoint down, as e2m1_nearest does,
// and leaves every other |v| <= 6 (and not -0) where it was.  Checked against
// e2m1_nearest over all such floats.
MM_DEV float fp4_ties_down(float v) {
  const uint32_t u = __builtin_bit_cast(uint32_t, v);
  return __builtin_bit_cast(float, __builtin_elementwise_sub_sat(u, 1u) | 1u);
}
template <int BYTE>
MM_DEV uint32_t fp4_pair(uint32_t word, float v0, float v1) {
  return __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(word, fp4_ties_down(v0), fp4_ties_down(v1), 1.0f,
                                                  BYTE);
}

constexpr int QT_WORDS = 64;  // words (8 k) per row and block: one wave-wide load
constexpr int QT_WAVES = 4;

// QT_N: rows of W (columns of the packed matrix) per block; QT_ROWS: rows a wave
// loads together.
template <typename T, bool INT4, int QT_N, int QT_ROWS>
__global__ void __launch_bounds__(QT_WAVES * 64)
k_quantize_tile(const T* __restrict__ Wt, int N, int K, int g, uint32_t* __restrict__ B,
                f16* __restrict__ S, f16* __restrict__ Z) {
  __shared__ uint32_t words[QT_WORDS][QT_N + 1];
  __shared__ f16 sc[QT_WORDS][QT_N + 2], zp[INT4 ? QT_WORDS : 1][QT_N + 2];
  typedef T tvec __attribute__((ext_vector_type(8)));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n0 = blockIdx.x * QT_N, w0 = blockIdx.y * QT_WORDS;
  const int wpg = g >> 3;                        // lanes per group, a power of two
  const int KP = K >> 3;
  const bool live = w0 + lane < KP;              // whole groups: K % g == 0
  const int wl = live ? w0 + lane : KP - 1;
  for (int r0 = wave * QT_ROWS; r0 < QT_N; r0 += QT_WAVES * QT_ROWS) {
    tvec x[QT_ROWS];
#pragma unroll
    for (int i = 0; i < QT_ROWS; ++i)
      x[i] = *(const tvec*)(Wt + (size_t)min(n0 + r0 + i, N - 1) * K + (size_t)wl * 8);
#pragma unroll
    for (int i = 0; i < QT_ROWS; ++i) {
      uint32_t word = 0;
      float sv, zv = 0.0f;
      if constexpr (!INT4) {
        // |x| bits as integers: NaN sorts above inf, so a NaN in the group wins
        // as in np.max.
        uint32_t m = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          m = max(m, __builtin_bit_cast(uint32_t, (float)x[i][j]) & 0x7FFFFFFFu);
        for (int d = 1; d < wpg; d <<= 1) m = max(m, (uint32_t)__shfl_xor((int)m, d));
        const float a = m > 0x7F800000u ? __builtin_nanf("")
                                        : fmaxf(__builtin_bit_cast(float, m), 1e-7f);
        sv = a / 6.0f;
        bool ok = div_ok(a);
        if constexpr (sizeof(T) == 4) {
          bool tiny = false;
#pragma unroll
          for (int j = 0; j < 8; ++j)
            tiny |= fabsf((float)x[i][j]) < 0x1p-80f && (float)x[i][j] != 0.0f;
          ok = ok && !tiny;
        }
        if (ok) {
          const float r = 1.0f / a;
          float v[8];     // -0 weights come out as +0 (code 0 either way)
#pragma unroll
          for (int j = 0; j < 8; ++j) v[j] = div_by((float)x[i][j], a, r) * 6.0f;
          word = fp4_pair<0>(word, v[0], v[1]);
          word = fp4_pair<1>(word, v[2], v[3]);
          word = fp4_pair<2>(word, v[4], v[5]);
          word = fp4_pair<3>(word, v[6], v[7]);
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j) word |= e2m1_nearest((float)x[i][j] / a * 6.0f) << (4 * j);
        }
      } else {
        float mn = (float)x[i][0], mx = mn;
#pragma unroll
        for (int j = 1; j < 8; ++j) {
          mn = fminf(mn, (float)x[i][j]);
          mx = fmaxf(mx, (float)x[i][j]);
        }
        for (int d = 1; d < wpg; d <<= 1) {
          mn = fminf(mn, __shfl_xor(mn, d));
          mx = fmaxf(mx, __shfl_xor(mx, d));
        }
        sv = fmaxf((mx - mn) / 15.0f, 1e-7f);
        zv = rintf(-mn / sv);
        if (div_ok(sv)) {
          const float r = 1.0f / sv;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float q = rintf(div_by((float)x[i][j], sv, r) + zv);
            word |= (uint32_t)fminf(fmaxf(q, 0.0f), 15.0f) << (4 * j);
          }
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float q = rintf((float)x[i][j] / sv + zv);
            word |= (uint32_t)fminf(fmaxf(q, 0.0f), 15.0f) << (4 * j);
          }
        }
      }
      words[lane][r0 + i] = word;
      if ((lane & (wpg - 1)) == 0) {
        sc[lane / wpg][r0 + i] = (f16)sv;
        if constexpr (INT4) zp[lane / wpg][r0 + i] = (f16)zv;
      }
    }
  }
  __syncthreads();
  constexpr int WSTEP = QT_WAVES * 64 / QT_N;
  const int col = threadIdx.x % QT_N, n = n0 + col;
  if (n >= N) return;
  for (int w = threadIdx.x / QT_N; w < QT_WORDS && w0 + w < KP; w += WSTEP)
    B[(size_t)(w0 + w) * N + n] = words[w][col];
  for (int q = threadIdx.x / QT_N; q < QT_WORDS / wpg && w0 + q * wpg < KP; q += WSTEP) {
    const size_t at = (size_t)(w0 / wpg + q) * N + n;
    S[at] = sc[q][col];
    if constexpr (INT4) Z[at] = zp[q][col];
  }
}

// Rule of the tiled quantizers (see above); other groups and unaligned views
// take the one-thread-per-group kernels.
bool quant_tile_ok(const void* W, int g) {
  return g <= 8 * QT_WORDS && (g & (g - 1)) == 0 && ((uintptr_t)W & 15) == 0;
}

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------
static int check_dims(const char* who, int K, int N, int g) {
  MM_CHECK_ARG(K > 0 && N > 0, "%s: K=%d and N=%d must be positive", who, K, N);
  MM_CHECK_ARG(K % 8 == 0, "%s: K=%d must be divisible by 8", who, K);
  MM_CHECK_ARG(g > 0 && g % 8 == 0, "%s: group_size=%d must be a positive multiple of 8", who, g);
  MM_CHECK_ARG(K % g == 0, "%s: K=%d must be divisible by group_size=%d", who, K, g);
  return 0;
}

template <bool INT4>
static int launch_dequant(const char* who, const uint32_t* B, const uint16_t* S,
                          const uint16_t* Z, uint16_t* W, int K, int N, int g, hipStream_t st) {
  const size_t quads = (size_t)(N / 4) * (K / 8);   // of the form with four words per thread
  const bool v4 = N % 4 == 0 && quads >= 256 * 256 && quads < ((size_t)1 << 31) &&
                  ((uintptr_t)B & 15) == 0 &&
                  (((uintptr_t)S | (uintptr_t)W | (INT4 ? (uintptr_t)Z : 0)) & 7) == 0;
#define MM_LAUNCH_DEQUANT(GRID, ...)                                                             \
  hipLaunchKernelGGL((k_dequant<__VA_ARGS__>), GRID, dim3(256), 0, st, B, (const f16*)S,          \
                     (const f16*)Z, (f16*)W, K, N, g)
  const dim3 grid4((unsigned)((quads + 255) / 256));
  if (v4 && N % 64 == 0 && ((uintptr_t)W & 127) == 0)
    MM_LAUNCH_DEQUANT(grid4, 4, INT4, true);
  else if (v4)
    MM_LAUNCH_DEQUANT(grid4, 4, INT4);
  else
    MM_LAUNCH_DEQUANT(dim3(mm_cdiv(N, 256), K / 8), 1, INT4);
#undef MM_LAUNCH_DEQUANT
  MM_CHECK_LAUNCH(who);
  return 0;
}

extern "C" int mm_fp4_dequant(const uint32_t* B, const uint16_t* S, uint16_t* W, int K, int N,
                              int g, void* stream) {
  if (int rc = check_dims("mm_fp4_dequant", K, N, g)) return rc;
  return launch_dequant<false>("mm_fp4_dequant", B, S, nullptr, W, K, N, g, (hipStream_t)stream);
}

extern "C" int mm_u4_dequant(const uint32_t* B, const uint16_t* S, const uint16_t* Z, uint16_t* W,
                             int K, int N, int g, void* stream) {
  if (int rc = check_dims("mm_u4_dequant", K, N, g)) return rc;
  return launch_dequant<true>("mm_u4_dequant", B, S, Z, W, K, N, g, (hipStream_t)stream);
}

// Rows per block: a block of 64 rows works through four batches of rows in turn
// (8 to 13 us alone), which leaves most CUs idle while there are fewer of them than
// CUs; blocks of 4 rows then take one batch.  us, per-group kernel, 64 rows, 4 rows:
// INT4 33 x 1024 g = 8 2.6, 9.0, 2.4; 256 x 256 g = 32 7.3, 9.2, 2.5; FP4 (fp16)
// 1000 x 4096 g = 128 57, 12.0, 5.7; 512 x 14336 68, 12.3, 7.8; but float32
// 4096 x 4096 g = 64 161, 17.8, 19.5 (16-byte runs of output).
template <typename T, bool INT4>
static void launch_quantize_tile(const void* W, int N, int K, int g, uint32_t* B, uint16_t* S,
                                 uint16_t* Z, hipStream_t st) {
#define MM_LAUNCH_QT(QN, QR)                                                                     \
  hipLaunchKernelGGL((k_quantize_tile<T, INT4, QN, QR>),                                         \
                     dim3(mm_cdiv(N, QN), mm_cdiv(K / 8, QT_WORDS)), dim3(QT_WAVES * 64), 0, st,  \
                     (const T*)W, N, K, g, B, (f16*)S, (f16*)Z)
  if ((long)mm_cdiv(N, 64) * mm_cdiv(K / 8, QT_WORDS) < 256)
    MM_LAUNCH_QT(4, 1);
  else
    MM_LAUNCH_QT(64, 4);
#undef MM_LAUNCH_QT
}

extern "C" int mm_fp4_quantize(const void* W, int w_is_f32, int N, int K, int g, uint32_t* B,
                               uint16_t* S, void* stream) {
  if (int rc = check_dims("mm_fp4_quantize", K, N, g)) return rc;
  if (quant_tile_ok(W, g)) {
    if (w_is_f32)
      launch_quantize_tile<float, false>(W, N, K, g, B, S, nullptr, (hipStream_t)stream);
    else
      launch_quantize_tile<f16, false>(W, N, K, g, B, S, nullptr, (hipStream_t)stream);
    MM_CHECK_LAUNCH("mm_fp4_quantize");
    return 0;
  }
  dim3 grid(mm_cdiv(N, 256), K / g);
  if (w_is_f32)
    hipLaunchKernelGGL(k_fp4_quantize<float>, grid, dim3(256), 0, (hipStream_t)stream,
                       (const float*)W, N, K, g, B, (f16*)S);
  else
    hipLaunchKernelGGL(k_fp4_quantize<f16>, grid, dim3(256), 0, (hipStream_t)stream,
                       (const f16*)W, N, K, g, B, (f16*)S);
  MM_CHECK_LAUNCH("mm_fp4_quantize");
  return 0;
}

extern "C" int mm_fp4_quantize_calibrated(const void* W, int w_is_f32, int N, int K, int g,
                                          int use_pct, int kprev, int knext, float gamma,
                                          int mode, float c1, float c2, double sf, double att,
                                          uint32_t* B, uint16_t* S, void* stream) {
  if (int rc = check_dims("mm_fp4_quantize_calibrated", K, N, g)) return rc;
  MM_CHECK_ARG(!use_pct || (kprev >= 0 && kprev < g && knext >= kprev && knext < g),
               "mm_fp4_quantize_calibrated: order statistics %d, %d outside a group of %d",
               kprev, knext, g);
  MM_CHECK_ARG(mode >= 0 && mode <= 2, "mm_fp4_quantize_calibrated: mode must be 0, 1 or 2");
  const FqCal cal{use_pct != 0, kprev, knext, gamma, mode, c1, c2, sf, att};
  dim3 grid(mm_cdiv(N, 256), K / g);
  if (w_is_f32)
    hipLaunchKernelGGL(k_fp4_quantize_cal<float>, grid, dim3(256), 0, (hipStream_t)stream,
                       (const float*)W, N, K, g, cal, B, (f16*)S);
  else
    hipLaunchKernelGGL(k_fp4_quantize_cal<f16>, grid, dim3(256), 0, (hipStream_t)stream,
                       (const f16*)W, N, K, g, cal, B, (f16*)S);
  MM_CHECK_LAUNCH("mm_fp4_quantize_calibrated");
  return 0;
}

extern "C" int mm_u4_quantize(const uint16_t* W, int N, int K, int g, uint32_t* B, uint16_t* S,
                              uint16_t* Z, void* stream) {
  if (int rc = check_dims("mm_u4_quantize", K, N, g)) return rc;
  if (quant_tile_ok(W, g)) {
    launch_quantize_tile<f16, true>(W, N, K, g, B, S, Z, (hipStream_t)stream);
    MM_CHECK_LAUNCH("mm_u4_quantize");
    return 0;
  }
  dim3 grid(mm_cdiv(N, 256), K / g);
  hipLaunchKernelGGL(k_u4_quantize, grid, dim3(256), 0, (hipStream_t)stream, (const f16*)W, N,
                     K, g, B, (f16*)S, (f16*)Z);
  MM_CHECK_LAUNCH("mm_u4_quantize");
  return 0;
}
