// awk_dense.h -- DFT of one axis as a matrix product on the FP32 matrix cores.
//
// For a length n the transform is a contraction with the n x n DFT matrix.  With
// the folds e_j = x_j + x_{n-j}, o_j = x_j - x_{n-j} (e_0 = x_0) it becomes two
// real H x H products, H = n/2 + 1,
//   E_k = sum_j cos(2 pi j k / n) e_j,   O_k = sum_j sin(2 pi j k / n) o_j,
//   X_k = E_k -+ i O_k,   X_{n-k} = E_k +- i O_k,
// whose right-hand sides are real columns (real and imaginary parts of complex
// lines, or real lines).  A wave computes 32 outputs k of 32 columns with
// v_mfma_f32_32x32x2_f32; the matrix comes from a table laid out in fragment order
// (one 8-byte load per lane and step gives both the cosine and the sine).
//
// About 2 n flops per element instead of an FFT's 5 log2 n, but on a unit that is
// otherwise idle, without stages, barriers or index arithmetic, and for any n.
// It serves the lengths with no short radix plan.
//
// Rounding: sums run over 8 or 16 terms before they are folded into a second accumulator,
// so the error grows with the run and the number of folds, not with n.  Runs of 8 where
// the LDS stages round as little as runs of 16 (dense_short_runs).
#pragma once

#include "awk_fft.h"

namespace awk {

typedef float v16f __attribute__((ext_vector_type(16)));

// H <= 256: at most 8 tiles of 32 outputs.  From 7 on, the rows that the padded
// steps touch (j <= 2 ks - 1 <= n) are staged rows.
constexpr int kDenseMin = 7, kDenseMax = 511;

// tab[(tile * ks + s) * 64 + lane] = (cos, sin)(2 pi j k / n) with k = 32 tile +
// lane % 32 and j = 2 s + lane / 32; zero where j or k is past H - 1, and halved at
// j = n / 2 (whose fold e_j = 2 x_j counts it twice).
struct DenseAxis {
  const float2 *tab;
  int n, H, tiles, ks;  // ks: steps of 2 j, a multiple of 4
  int short_runs;       // sums in runs of 8 terms (else 16)
};

// Which lengths take runs of 8 terms, whose folds cost 1 to 2 % of an operator's time at
// 68^3 ... 136^3 and 3 % at 181 x 217 x 181.  The error of L^-1 against the LDS stages' (means
// over seeds, each axis): with 16 terms 1.00 ... 1.05 at 34 ... 136 and, of the longer
// lengths, at those of primes up to 19 (170, 190, 204, 238, 255: 1.01 ... 1.06), with 8
// terms 0.88 ... 1.02 and 0.98 ... 1.04.  Lengths of larger primes from 144 on (181, 217,
// 251: 0.73 ... 0.95 with 16 terms) have no need of them, and past 255 the folds of runs
// of 8 round more than they save.
inline bool dense_short_runs(int n, int largest_prime) { return n <= 143 || (n <= 255 && largest_prime <= 19); }

__device__ __forceinline__ v16f mfma32(float a, float b, v16f c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// Row (of the 32 x 32 tile) that accumulator register i of this lane holds; the
// column is lane % 32.
__device__ __forceinline__ int dense_row(int i, int lane) {
  return 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
}

// dense_tile's sums in runs of 8 G terms.
template <bool DATA_A, bool FOLD, int G>
__device__ __forceinline__ void dense_runs(const float *p, const float *q, int dp, int dq,
                                           const float2 *__restrict__ tab, int ks, v16f &E, v16f &O) {
#pragma unroll
  for (int i = 0; i < 16; ++i) E[i] = O[i] = 0.f;
  float2 t[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) t[i] = tab[i * 64];
  for (int s = 0; s < ks; s += 4 * G) {
    v16f ae, ao;
#pragma unroll
    for (int i = 0; i < 16; ++i) ae[i] = ao[i] = 0.f;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (s + 4 * g < ks) {
        float2 u[4];
        const bool more = s + 4 * g + 4 < ks;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          u[i] = t[i];
          t[i] = tab[(more ? s + 4 * g + 4 + i : i) * 64];
        }
        float a[4], b[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          a[i] = p[i * dp];
          b[i] = q[i * dq];
        }
        p += 4 * dp;
        q += 4 * dq;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float e = FOLD ? a[i] + b[i] : a[i], o = FOLD ? a[i] - b[i] : b[i];
          ae = DATA_A ? mfma32(e, u[i].x, ae) : mfma32(u[i].x, e, ae);
          ao = DATA_A ? mfma32(o, u[i].y, ao) : mfma32(u[i].y, o, ao);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      E[i] += ae[i];
      O[i] += ao[i];
    }
  }
}

// One tile: E and O summed over all j.  p / q: this lane's first values (rows j =
// lane / 32 and n - j of the staged lines, or of the two staged parts), advanced
// by dp / dq floats per step.
// DATA_A: the lines are the rows of the result and k its columns (else the lines
// are the columns).  FOLD: form e and o from the two rows (else they are given).
template <bool DATA_A, bool FOLD>
__device__ __forceinline__ void dense_tile(const float *p, const float *q, int dp, int dq,
                                           const DenseAxis &ax, int tile, int lane, v16f &E, v16f &O) {
  const float2 *tab = ax.tab + (size_t)tile * ax.ks * 64 + lane;
  if (ax.short_runs) dense_runs<DATA_A, FOLD, 1>(p, q, dp, dq, tab, ax.ks, E, O);
  else dense_runs<DATA_A, FOLD, 2>(p, q, dp, dq, tab, ax.ks, E, O);
}

// The value of the lane's neighbour (lane ^ 1): the other part of a complex column.
__device__ __forceinline__ float dense_swap(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, true));
}

// Complex lines staged as columns (rows of 32 floats, real and imaginary parts
// interleaved, row n zero): this wave's outputs X_k into A and X_{n-k} into B, k =
// 32 tile + dense_row(i).
__device__ __forceinline__ void dense_lines(const float *sm, const DenseAxis &ax, int tile, int lane,
                                            bool inv, v16f &A, v16f &B) {
  const int hi = lane >> 5, col = lane & 31;
  v16f E, O;
  dense_tile<false, true>(sm + hi * 32 + col, sm + (ax.n - hi) * 32 + col, 64, -64,
                          ax, tile, lane, E, O);
  // forward: X = E - i O: the real part takes + Im O, the imaginary part - Re O
  const float sg = ((lane & 1) != 0) != inv ? -1.f : 1.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const float w = sg * dense_swap(O[i]);
    A[i] = E[i] + w;
    B[i] = E[i] - w;
  }
}

// 16 complex columns of n rows (row stride st) into LDS, row n zero; columns past
// nvalid are zero.
__device__ __forceinline__ void dense_stage(float *sm, const float2 *__restrict__ base, size_t st, int n,
                                            int nvalid) {
  const int t = (int)threadIdx.x & 15, j0 = (int)threadIdx.x >> 4, dj = (int)blockDim.x >> 4;
  float2 *s2 = reinterpret_cast<float2 *>(sm);
  const bool ok = t < nvalid;
  for (int j = j0; j <= n; j += 8 * dj) {
    float2 v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = j + i * dj;
      v[i] = (ok && r < n) ? base[(size_t)r * st + t] : make_float2(0.f, 0.f);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = j + i * dj;
      if (r <= n) s2[r * 16 + t] = v[i];
    }
  }
}

// The same for three components (planes `plane` apart), one after the other in LDS.
__device__ __forceinline__ void dense_stage3(float *sm, const float2 *__restrict__ base, size_t plane,
                                             size_t st, int n, int nvalid) {
  const int t = (int)threadIdx.x & 15, j0 = (int)threadIdx.x >> 4, dj = (int)blockDim.x >> 4;
  float2 *s2 = reinterpret_cast<float2 *>(sm);
  const bool ok = t < nvalid;
  for (int j = j0; j <= n; j += 4 * dj) {
    float2 v[3][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = j + i * dj;
#pragma unroll
      for (int c = 0; c < 3; ++c)
        v[c][i] = (ok && r < n) ? base[c * plane + (size_t)r * st + t] : make_float2(0.f, 0.f);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = j + i * dj;
      if (r <= n) {
#pragma unroll
        for (int c = 0; c < 3; ++c) s2[(c * (n + 1) + r) * 16 + t] = v[c][i];
      }
    }
  }
}

// X_k and X_{n-k} of a tile to rows k and n - k of base (row stride st floats), the
// first nvalid complex columns.
__device__ __forceinline__ void dense_store(float *base, size_t st, const DenseAxis &ax, int tile,
                                            int lane, int nvalid, const v16f &A, const v16f &B) {
  const int col = lane & 31;
  if ((col >> 1) >= nvalid) return;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int k = 32 * tile + dense_row(i, lane);
    if (k < ax.H) {
      base[(size_t)k * st + col] = A[i];
      if (k > 0 && 2 * k != ax.n) base[(size_t)(ax.n - k) * st + col] = B[i];
    }
  }
}

}  // namespace awk
