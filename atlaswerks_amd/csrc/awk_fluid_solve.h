// awk_fluid_solve.h -- the per-frequency operator of the z passes.
#pragma once

#include "awk_common.h"

namespace awk {

struct SolveArgs {
  const float *cwx, *swx, *cwy, *swy, *cwz, *swz;
  const float *eig;  // 6 per frequency, or null
  float alpha, beta, gamma, scale;
  int inverse_op;  // 1: L^-1 (Cholesky), 0: L
  int divfree;
};


// Per-frequency operator: Cholesky solve of L v = b (DiffOper.cxx:1002-1083), or
// v = L b (1085-1116), or v = M b with the eigen table M = L^(+-p); then the
// divergence-free projection (948-1000) and the 1/N scale.
__device__ __forceinline__ void solve_one(const SolveArgs &s, int kx, int ky, int kz, int ny,
                                          int nxh, float2 &b0, float2 &b1, float2 &b2) {
  float2 v0, v1, v2;
  const float sx = s.swx[kx], sy = s.swy[ky], sz = s.swz[kz];
  if (s.eig) {
    const float *M = s.eig + ((size_t)(kz * ny + ky) * nxh + kx) * 6;
    const float M00 = M[0], M10 = M[1], M11 = M[2], M20 = M[3], M21 = M[4], M22 = M[5];
    v0 = make_float2(M00 * b0.x + M10 * b1.x + M20 * b2.x, M00 * b0.y + M10 * b1.y + M20 * b2.y);
    v1 = make_float2(M10 * b0.x + M11 * b1.x + M21 * b2.x, M10 * b0.y + M11 * b1.y + M21 * b2.y);
    v2 = make_float2(M20 * b0.x + M21 * b1.x + M22 * b2.x, M20 * b0.y + M21 * b1.y + M22 * b2.y);
  } else {
    const float cx = s.cwx[kx], cy = s.cwy[ky], cz = s.cwz[kz];
    const float lam = -s.alpha * (cx + cy + cz) + s.gamma;
    const float L00 = lam - s.beta * cx, L11 = lam - s.beta * cy, L22 = lam - s.beta * cz;
    const float L10 = s.beta * sx * sy, L20 = s.beta * sx * sz, L21 = s.beta * sy * sz;
    if (s.inverse_op) {
      // Same Cholesky factorisation, carried with the reciprocals g_ii = 1/G_ii
      // (rsqrt): every division of the reference becomes a multiplication.
      const float g00 = rsqrtf(L00);
      const float G10 = L10 * g00, G20 = L20 * g00;
      const float g11 = rsqrtf(L11 - G10 * G10);
      const float G21 = (L21 - G20 * G10) * g11;
      const float g22 = rsqrtf(L22 - (G20 * G20 + G21 * G21));
      float y0 = b0.x * g00, y1 = (b1.x - G10 * y0) * g11, y2 = (b2.x - G20 * y0 - G21 * y1) * g22;
      v2.x = y2 * g22; v1.x = (y1 - G21 * v2.x) * g11; v0.x = (y0 - G10 * v1.x - G20 * v2.x) * g00;
      y0 = b0.y * g00; y1 = (b1.y - G10 * y0) * g11; y2 = (b2.y - G20 * y0 - G21 * y1) * g22;
      v2.y = y2 * g22; v1.y = (y1 - G21 * v2.y) * g11; v0.y = (y0 - G10 * v1.y - G20 * v2.y) * g00;
    } else {
      v0 = make_float2(L00 * b0.x + L10 * b1.x + L20 * b2.x, L00 * b0.y + L10 * b1.y + L20 * b2.y);
      v1 = make_float2(L10 * b0.x + L11 * b1.x + L21 * b2.x, L10 * b0.y + L11 * b1.y + L21 * b2.y);
      v2 = make_float2(L20 * b0.x + L21 * b1.x + L22 * b2.x, L20 * b0.y + L21 * b1.y + L22 * b2.y);
    }
  }
  if (s.divfree && (kx | ky | kz)) {
    const float nsq = sx * sx + sy * sy + sz * sz;
    if (nsq > 0.f) {
      const float re = (v0.x * sx + v1.x * sy + v2.x * sz) / nsq;
      const float im = (v0.y * sx + v1.y * sy + v2.y * sz) / nsq;
      v0.x -= re * sx; v1.x -= re * sy; v2.x -= re * sz;
      v0.y -= im * sx; v1.y -= im * sy; v2.y -= im * sz;
    }
  }
  b0 = cscale(v0, s.scale);
  b1 = cscale(v1, s.scale);
  b2 = cscale(v2, s.scale);
}

// solve_one on one part (real or imaginary) of the three components: the operator
// is real, so the parts do not mix.
__device__ __forceinline__ void solve_part(const SolveArgs &s, int kx, int ky, int kz, int ny, int nxh,
                                           float &b0, float &b1, float &b2) {
  float2 a0 = make_float2(b0, 0.f), a1 = make_float2(b1, 0.f), a2 = make_float2(b2, 0.f);
  solve_one(s, kx, ky, kz, ny, nxh, a0, a1, a2);
  b0 = a0.x;
  b1 = a1.x;
  b2 = a2.x;
}

}  // namespace awk
