// awk_radix.h -- two-stage transforms of any length n = ra * rb with radices up to 32
// whose prime factors are at most 13, the butterflies in registers.
//
// Stage A (radix ra, j < rb): inputs j + r rb, outputs to slots j ra + r.  Stage B
// (radix rb, j < ra): slots j + r ra times w^(r j), outputs to the same slots, which
// are the frequencies j + r ra (and the elements, for the inverse transform).  The
// radices are launch constants, so a stage is a switch over compiled butterflies:
// no per-element index arithmetic, one exchange through LDS.
#pragma once

#include "awk_fft.h"

namespace awk {

// cos and sin of 2 pi a / b at compile time (Taylor series after a reduction to
// |x| <= pi, in double).
constexpr double ct_angle(int a, int b) {
  a %= b;
  if (2 * a > b) a -= b;
  return 6.283185307179586476925286766559 * a / b;
}
constexpr double ct_cos(int a, int b) {
  const double x = ct_angle(a, b), y = x * x;
  double t = 1.0, s = 1.0;
  for (int i = 1; i < 24; ++i) {
    t *= -y / ((2 * i - 1) * (2 * i));
    s += t;
  }
  return s;
}
constexpr double ct_sin(int a, int b) {
  const double x = ct_angle(a, b), y = x * x;
  double t = x, s = x;
  for (int i = 1; i < 24; ++i) {
    t *= -y / ((2 * i) * (2 * i + 1));
    s += t;
  }
  return s;
}
template <int A, int B>
struct CtRoot {
  static constexpr float c = (float)ct_cos(A, B), s = (float)ct_sin(A, B);
};

// The first of two factors of a composite radix (R: prime): its power of two, else its
// smallest prime, which is coprime to the rest unless R is a power of one prime.
template <int R>
constexpr int ct_factor() {
  constexpr int two = R & -R;
  constexpr int f = two > 1 && two < R ? two : R == 32 ? 4 : R % 3 == 0 ? 3 : R % 5 == 0 ? 5 : R % 7 == 0 ? 7 : R;
  return f;
}
constexpr int ct_inverse(int a, int m) {  // of a modulo m, coprime
  for (int i = 1; i < m; ++i)
    if (a * i % m == 1) return i;
  return 0;
}

// The odd prime radix: outputs k and R - k share the sums of x_j + x_{R-j} against
// cosines and of x_j - x_{R-j} against sines.
template <int R, int K, int J>
__device__ __forceinline__ void prime_sums(const float2 *a, const float2 *b, float2 &c, float2 &s) {
  if constexpr (J <= (R - 1) / 2) {
    typedef CtRoot<(K * J) % R, R> W;
    c.x += W::c * a[J - 1].x;
    c.y += W::c * a[J - 1].y;
    s.x += W::s * b[J - 1].x;
    s.y += W::s * b[J - 1].y;
    prime_sums<R, K, J + 1>(a, b, c, s);
  }
}
template <int R, int K>
__device__ __forceinline__ void prime_outputs(float2 x0, const float2 *a, const float2 *b, float2 *v, bool inv) {
  if constexpr (K <= (R - 1) / 2) {
    float2 c = x0, s = make_float2(0.f, 0.f);
    prime_sums<R, K, 1>(a, b, c, s);
    const float2 w = rot(s, inv);  // -i s (forward)
    v[K] = cadd(c, w);
    v[R - K] = csub(c, w);
    prime_outputs<R, K + 1>(x0, a, b, v, inv);
  }
}

// Factors of one prime: v[n2 + B n1] -> outputs k1 + A k2: DFT_A over n1, w_R^(n2 k1), DFT_B
// over n2.
template <int R, int A, int K1, int N2>
__device__ __forceinline__ void composite_twiddle(float2 (*y)[R / A], bool inv) {
  if constexpr (K1 < A) {
    typedef CtRoot<(K1 * N2) % R, R> W;
    if constexpr (K1 * N2 != 0) y[K1][N2] = cmul(y[K1][N2], make_float2(W::c, inv ? W::s : -W::s));
    if constexpr (N2 + 1 < R / A) composite_twiddle<R, A, K1, N2 + 1>(y, inv);
    else composite_twiddle<R, A, K1 + 1, 0>(y, inv);
  }
}

template <int R>
__device__ __forceinline__ void dft_any(float2 *v, bool inv) {
  constexpr int A = ct_factor<R>(), B = R / A;
  if constexpr (R == 1) {
  } else if constexpr (R == 2 || R == 3 || R == 4 || R == 5 || R == 8 || R == 16) {
    dft<R>(v, inv);
  } else if constexpr (A == R) {
    constexpr int H = (R - 1) / 2;
    float2 a[H], b[H];
    const float2 x0 = v[0];
    float2 t = x0;
#pragma unroll
    for (int j = 1; j <= H; ++j) {
      a[j - 1] = cadd(v[j], v[R - j]);
      b[j - 1] = csub(v[j], v[R - j]);
      t = cadd(t, a[j - 1]);
    }
    v[0] = t;
    prime_outputs<R, 1>(x0, a, b, v, inv);
  } else if constexpr (ct_inverse(A, B) != 0) {
    // coprime factors (Good 1958): inputs B n1 + A n2 and outputs e1 k1 + e2 k2 (mod R), e1
    // = 1 (mod A), 0 (mod B), need no twiddles between DFT_A and DFT_B, so no roundings
    // there either.  L^-1's error against 64 bits over the LDS stages', with twiddles and
    // without: 36^3 1.11 -> 0.97, 42^3 1.04 -> 0.97, 84^3 1.04 -> 0.97, 100^3 1.05 -> 0.90;
    // times as before.
    constexpr int e1 = B * ct_inverse(B % A, A), e2 = A * ct_inverse(A, B);
    float2 y[A][B];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) {
      float2 c[A];
#pragma unroll
      for (int n1 = 0; n1 < A; ++n1) c[n1] = v[(B * n1 + A * n2) % R];
      dft_any<A>(c, inv);
#pragma unroll
      for (int k1 = 0; k1 < A; ++k1) y[k1][n2] = c[k1];
    }
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
      dft_any<B>(y[k1], inv);
#pragma unroll
      for (int k2 = 0; k2 < B; ++k2) v[(e1 * k1 + e2 * k2) % R] = y[k1][k2];
    }
  } else {
    float2 y[A][B];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) {
      float2 c[A];
#pragma unroll
      for (int n1 = 0; n1 < A; ++n1) c[n1] = v[n2 + B * n1];
      dft_any<A>(c, inv);
#pragma unroll
      for (int k1 = 0; k1 < A; ++k1) y[k1][n2] = c[k1];
    }
    composite_twiddle<R, A, 0, 0>(y, inv);
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
      dft_any<B>(y[k1], inv);
#pragma unroll
      for (int k2 = 0; k2 < B; ++k2) v[k1 + A * k2] = y[k1][k2];
    }
  }
}

template <int R>
struct Radix {
  static constexpr int value = R;
};

// f(Radix<r>()) for a supported radix r <= MAXR (1 when a length is one radix).
template <int MAXR, class F>
__device__ __forceinline__ void with_radix(int r, F f) {
#define AWK_R(R) case R: if constexpr (R <= MAXR) f(Radix<R>()); break;
  switch (r) {
    AWK_R(1) AWK_R(2) AWK_R(3) AWK_R(4) AWK_R(5) AWK_R(6) AWK_R(7) AWK_R(8) AWK_R(9) AWK_R(10) AWK_R(11)
    AWK_R(12) AWK_R(13) AWK_R(14) AWK_R(15) AWK_R(16) AWK_R(18) AWK_R(20) AWK_R(21) AWK_R(22) AWK_R(24)
    AWK_R(25) AWK_R(26) AWK_R(27) AWK_R(28) AWK_R(30) AWK_R(32)
  }
#undef AWK_R
}

inline bool radix_supported(int r) {
  if (r < 1 || r > 32) return false;
  for (int p : {17, 19, 23, 29, 31})
    if (r == p) return false;
  return true;
}

// Two radices of a length, the larger as small as possible; ra >= rb.  False if there
// are none.
inline bool radix_plan(int n, int &ra, int &rb) {
  for (int a = 1; a <= 32; ++a) {
    if (n % a || a * a < n) continue;
    if (radix_supported(a) && radix_supported(n / a)) {
      ra = a;
      rb = n / a;
      return true;
    }
  }
  return false;
}

struct RadixAxis {
  const float2 *tw;  // w^k = exp(-2 pi i k / n)
  int n, ra, rb;     // ra == 0: no plan
};

// Stage B's butterfly j in registers: the twiddles w^(r j) (before the butterfly
// forward, conjugated after it for the transposed inverse).
template <int R>
__device__ __forceinline__ void radix_twiddle(float2 *v, const float2 *__restrict__ tw, int j, bool inv) {
#pragma unroll
  for (int r = 1; r < R; ++r) v[r] = inv ? cmulc(v[r], tw[r * j]) : cmul(v[r], tw[r * j]);
}

}  // namespace awk
