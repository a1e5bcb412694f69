// awk_fluid_any.hip -- the passes of the FluidKernelFFT operator for any axis length: two
// radices in registers (awk_radix.h), the dense product on the matrix cores
// (awk_dense.h), or LDS stages of mixed radices (chirp-z for large primes).  64, 128 and
// 256 along x, 32 to 256 along y and 128 and 256 along z have kernels of their own in
// awk_fluid.hip.
#include "awk_fluid.h"
#include "awk_radix.h"
#include "awk_fluid_solve.h"
#include "awk_fluid_x.h"

namespace awk {

// Y pass: complex FFT along y for TX kx columns of one (component, z) slab.
__global__ void __launch_bounds__(1024)
k_ypass(Axis ax, int ny, int nz, int nxh, int nxh_pad, int TX, float2 *__restrict__ spec,
        size_t plane, int inv, ReduceArgs ra, Batch bt) {
  extern __shared__ float2 sm[];
  spec += (long long)blockIdx.y * bt.spec;
  const int ntile = (nxh + TX - 1) / TX;
  const int lb = (int)xcd_block();
  if (lb >= 3 * nz * ntile) return;
  const int tile = lb % ntile, rest = lb / ntile;
  const int z = rest % nz, c = rest / nz;
  const int kx0 = tile * TX;
  float2 *base = spec + c * plane + (size_t)z * ny * nxh_pad + kx0;
  for (int w = threadIdx.x; w < TX * ny; w += blockDim.x) {
    const int t = w % TX, y = w / TX;
    sm[y * TX + t] = (kx0 + t < nxh) ? base[(size_t)y * nxh_pad + t] : make_float2(0.f, 0.f);
  }
  __syncthreads();
  lds_fft(sm, ax, TX, TX, inv != 0, sm + (size_t)ny * TX);
  for (int w = threadIdx.x; w < TX * ny; w += blockDim.x) {
    const int t = w % TX, y = w / TX;
    if (kx0 + t < nxh) base[(size_t)y * nxh_pad + t] = sm[y * TX + t];
  }
  if (ra.partials && lb == 0) {
    __syncthreads();
    batch_reduce(ra, bt);
    energy_block(ra, reinterpret_cast<double *>(sm), blockDim.x);
  }
}

// Y pass of a length with a dense plan: a wave per 32 output rows.  Bound by the
// matrix cores and the spectrum's two passes through memory together.
__global__ void __launch_bounds__(512)
k_ypass_dense(DenseAxis ax, int nz, int nxh, int nxh_pad, float2 *__restrict__ spec, size_t plane,
              int inv, ReduceArgs ra, Batch bt) {
  extern __shared__ float2 sm[];
  float *smf = reinterpret_cast<float *>(sm);
  spec += (long long)blockIdx.y * bt.spec;
  const int ntile = (nxh + 15) / 16;
  const int lb = (int)xcd_block();
  if (lb >= 3 * nz * ntile) return;
  const int tile = lb % ntile, rest = lb / ntile;
  const int z = rest % nz, c = rest / nz;
  const int kx0 = tile * 16, nvalid = min(16, nxh - kx0);
  float2 *base = spec + c * plane + (size_t)z * ax.n * nxh_pad + kx0;
  dense_stage(smf, base, (size_t)nxh_pad, ax.n, nvalid);
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  v16f A, B;
  dense_lines(smf, ax, wave, lane, inv != 0, A, B);
  dense_store(reinterpret_cast<float *>(base), 2 * (size_t)nxh_pad, ax, wave, lane, nvalid, A, B);
  if (ra.partials && lb == 0) {
    __syncthreads();
    batch_reduce(ra, bt);
    energy_block(ra, reinterpret_cast<double *>(sm), blockDim.x);
  }
}

// Z pass: forward FFT along z of 3 components x TX kx columns at one ky, the
// per-frequency solve, inverse FFT along z.
__global__ void __launch_bounds__(1024)
k_zsolve(Axis az, SolveArgs s, int ny, int nz, int nxh, int nxh_pad, int TX,
         float2 *__restrict__ spec, size_t plane, Batch bt) {
  extern __shared__ float2 sm[];
  spec += (long long)blockIdx.y * bt.spec;
  const int NL = 3 * TX;
  const int ntile = (nxh + TX - 1) / TX;
  const int lb = (int)xcd_block();
  if (lb >= ny * ntile) return;
  const int tile = lb % ntile, ky = lb / ntile;
  const int kx0 = tile * TX;
  for (int w = threadIdx.x; w < NL * nz; w += blockDim.x) {
    const int t = w % TX, rest = w / TX;
    const int c = rest % 3, z = rest / 3;
    sm[z * NL + c * TX + t] = (kx0 + t < nxh)
                                  ? spec[c * plane + ((size_t)z * ny + ky) * nxh_pad + kx0 + t]
                                  : make_float2(0.f, 0.f);
  }
  __syncthreads();
  lds_fft(sm, az, NL, NL, false, sm + (size_t)nz * NL);
  for (int w = threadIdx.x; w < TX * nz; w += blockDim.x) {
    const int t = w % TX, kz = w / TX;
    const int kx = kx0 + t;
    if (kx >= nxh) continue;
    float2 b0 = sm[kz * NL + t], b1 = sm[kz * NL + TX + t], b2 = sm[kz * NL + 2 * TX + t];
    solve_one(s, kx, ky, kz, ny, nxh, b0, b1, b2);
    sm[kz * NL + t] = b0;
    sm[kz * NL + TX + t] = b1;
    sm[kz * NL + 2 * TX + t] = b2;
  }
  __syncthreads();
  lds_fft(sm, az, NL, NL, true, sm + (size_t)nz * NL);
  for (int w = threadIdx.x; w < NL * nz; w += blockDim.x) {
    const int t = w % TX, rest = w / TX;
    const int c = rest % 3, z = rest / 3;
    if (kx0 + t < nxh) spec[c * plane + ((size_t)z * ny + ky) * nxh_pad + kx0 + t] = sm[z * NL + c * TX + t];
  }
}

// Z pass of a length with a dense plan.  A wave keeps its 32 frequencies and their
// mirrors of all three components in registers (one real or imaginary part per
// lane, on which the real operator acts separately); the components go through one
// LDS buffer in turn, forward and back.
__global__ void __launch_bounds__(512)
k_zsolve_dense(DenseAxis az, SolveArgs sa, int ny, int nxh, int nxh_pad, float2 *__restrict__ spec,
               size_t plane, Batch bt) {
  extern __shared__ float2 sm[];
  float *smf = reinterpret_cast<float *>(sm);
  spec += (long long)blockIdx.y * bt.spec;
  const int ntile = (nxh + 15) / 16;
  const int lb = (int)xcd_block();
  if (lb >= ny * ntile) return;
  const int tile = lb % ntile, ky = lb / ntile;
  const int kx0 = tile * 16, nvalid = min(16, nxh - kx0);
  const size_t zst = (size_t)ny * nxh_pad;
  float2 *base = spec + (size_t)ky * nxh_pad + kx0;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int col = lane & 31;
  v16f A[3], B[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    if (c) __syncthreads();
    dense_stage(smf, base + c * plane, zst, az.n, nvalid);
    __syncthreads();
    dense_lines(smf, az, wave, lane, false, A[c], B[c]);
  }
  const int kx = min(kx0 + (col >> 1), nxh - 1);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int k = 32 * wave + dense_row(i, lane);
    if (k < az.H) {
      float b0 = A[0][i], b1 = A[1][i], b2 = A[2][i];
      solve_part(sa, kx, ky, k, ny, nxh, b0, b1, b2);
      A[0][i] = b0; A[1][i] = b1; A[2][i] = b2;
      if (k > 0 && 2 * k != az.n) {
        b0 = B[0][i]; b1 = B[1][i]; b2 = B[2][i];
        solve_part(sa, kx, ky, az.n - k, ny, nxh, b0, b1, b2);
        B[0][i] = b0; B[1][i] = b1; B[2][i] = b2;
      }
    }
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    __syncthreads();
    dense_store(smf, 32, az, wave, lane, 16, A[c], B[c]);  // row n stays zero
    __syncthreads();
    v16f P, Q;
    dense_lines(smf, az, wave, lane, true, P, Q);
    dense_store(reinterpret_cast<float *>(base + c * plane), 2 * zst, az, wave, lane, nvalid, P, Q);
  }
}

// The same with the three components in LDS side by side and a wave per 32 frequencies
// of one component: the loads of all three in flight at once, a third of the serial
// products per wave, and the frequencies solved in pairs of parts (one factorisation
// per frequency).  For lengths whose 3 * tiles waves fit a block; 181 x 217 x 91
// frequencies 216 -> 189 us, about 57 us of it the matrix cores'.
__global__ void __launch_bounds__(1024, 5)
k_zsolve_dense3(DenseAxis az, SolveArgs sa, int ny, int nxh, int nxh_pad, float2 *__restrict__ spec,
                size_t plane, Batch bt) {
  extern __shared__ float2 sm[];
  float *smf = reinterpret_cast<float *>(sm);
  spec += (long long)blockIdx.y * bt.spec;
  const int ntile = (nxh + 15) / 16;
  const int lb = (int)xcd_block();
  if (lb >= ny * ntile) return;
  const int tile = lb % ntile, ky = lb / ntile;
  const int kx0 = tile * 16, nvalid = min(16, nxh - kx0);
  const size_t zst = (size_t)ny * nxh_pad;
  float2 *base = spec + (size_t)ky * nxh_pad + kx0;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int cs = (az.n + 1) * 32;  // floats per component
  const int c = wave % 3, w = wave / 3;
  dense_stage3(smf, base, plane, zst, az.n, nvalid);
  __syncthreads();
  v16f A, B;
  dense_lines(smf + c * cs, az, w, lane, false, A, B);
  __syncthreads();
  dense_store(smf + c * cs, 32, az, w, lane, 16, A, B);  // row n stays zero
  __syncthreads();
  for (int e = threadIdx.x; e < az.n * 16; e += blockDim.x) {
    const int t = e & 15, kz = e >> 4;
    if (t < nvalid) {
      float2 *p = sm + e;
      float2 b0 = p[0], b1 = p[cs / 2], b2 = p[cs];
      solve_one(sa, kx0 + t, ky, kz, ny, nxh, b0, b1, b2);
      p[0] = b0;
      p[cs / 2] = b1;
      p[cs] = b2;
    }
  }
  __syncthreads();
  dense_lines(smf + c * cs, az, w, lane, true, A, B);
  dense_store(reinterpret_cast<float *>(base + c * plane), 2 * zst, az, w, lane, nvalid, A, B);
}

// ------------------------------------------------------------------
// Lengths n = ra * rb (awk_radix.h).  Thread (t, j): kx column t of 16 (128-byte rows),
// butterfly j < max(ra, rb).  MAXR: the largest radix compiled in (16, or 32 for
// lengths past 16 * 16 and the like, which costs registers).

template <int MAXR>
__global__ void __launch_bounds__(16 * MAXR)
k_ypass_radix(RadixAxis ax, int nz, int nxh, int nxh_pad, float2 *__restrict__ spec, size_t plane,
              int inv, ReduceArgs ra, Batch bt) {
  extern __shared__ float2 sm[];
  spec += (long long)blockIdx.y * bt.spec;
  const int t = threadIdx.x & 15, j = threadIdx.x >> 4;
  const int ntile = (nxh + 15) / 16;
  const int lb = (int)xcd_block();
  if (lb >= 3 * nz * ntile) return;
  const int tile = lb % ntile, rest = lb / ntile;
  const int z = rest % nz, c = rest / nz;
  const bool valid = tile * 16 + t < nxh, iv = inv != 0;
  // row j + r * step of the slab: a uniform base per r and one lane offset
  char *base = reinterpret_cast<char *>(spec + c * plane + (size_t)z * ax.n * nxh_pad + tile * 16);
  const size_t rs = (size_t)nxh_pad * sizeof(float2);
  const unsigned lo = (unsigned)(j * nxh_pad + t) * (unsigned)sizeof(float2);
  auto row = [&](int r) -> float2 & { return *reinterpret_cast<float2 *>(base + (size_t)r * rs + lo); };
  const int RA = ax.ra, RB = ax.rb;
  with_radix<MAXR>(RA, [&](auto rad) {
    constexpr int R = decltype(rad)::value;
    if (j < RB) {
      float2 v[R];
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = valid ? row(r * RB) : make_float2(0.f, 0.f);
      dft_any<R>(v, iv);
#pragma unroll
      for (int r = 0; r < R; ++r) sm[(j * R + r) * 16 + t] = v[r];
    }
  });
  __syncthreads();
  with_radix<MAXR>(RB, [&](auto rad) {
    constexpr int R = decltype(rad)::value;
    if (j < RA) {
      float2 v[R];
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = sm[(j + r * RA) * 16 + t];
      radix_twiddle<R>(v, ax.tw, j, iv);
      dft_any<R>(v, iv);
      if (valid) {
#pragma unroll
        for (int r = 0; r < R; ++r) row(r * RA) = v[r];
      }
    }
  });
  if (ra.partials && lb == 0) {
    __syncthreads();
    batch_reduce(ra, bt);
    energy_block(ra, reinterpret_cast<double *>(sm), blockDim.x);
  }
}

// The three components' lines stay in LDS.  A thread's stage-B slots, its frequencies
// and the first inverse stage's slots (the forward stages transposed) are the same
// ones, so stage A and its transpose are the only exchanges along z.  CG: component
// groups of threads; 3 groups each take a component of every transform and a third of
// the frequencies (three times the loads in flight and a third of the serial chain,
// which is what small grids wait for), 1 group takes them in turn (radices above 16:
// three groups fit a block up to radix 20, which is untried).  Measured against one group: 144 x 192 x 81
// frequencies 54.6 -> 43.3 us (2.6 TB/s), 36 x 31 x 17 9.8 -> 6.7 us.
template <int MAXR, int CG>
__global__ void __launch_bounds__(16 * MAXR * CG)
k_zsolve_radix(RadixAxis az, SolveArgs sa, int ny, int nxh, int nxh_pad, float2 *__restrict__ spec,
               size_t plane, Batch bt) {
  extern __shared__ float2 sm[];
  spec += (long long)blockIdx.y * bt.spec;
  const int RA = az.ra, RB = az.rb, cs = az.n * 16;  // LDS elements per component
  // whole waves per component group
  const int gs = CG == 1 ? (int)blockDim.x : (int)blockDim.x / CG;
  const int c0 = CG == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / gs);
  const int u = (int)threadIdx.x - c0 * gs, t = u & 15, j = u >> 4;
  const int ntile = (nxh + 15) / 16;
  const int lb = (int)xcd_block();
  if (lb >= ny * ntile) return;
  const int tile = lb % ntile, ky = lb / ntile;
  const int kx = tile * 16 + t;
  const bool valid = kx < nxh;
  // row j + r of a component: a uniform base per r and one lane offset
  char *base = reinterpret_cast<char *>(spec + (size_t)ky * nxh_pad + tile * 16);
  const size_t rs = (size_t)ny * nxh_pad * sizeof(float2), ps = plane * sizeof(float2);
  const size_t lo = (size_t)j * rs + t * sizeof(float2);
  auto row = [&](int c, int r) -> float2 & {
    return *reinterpret_cast<float2 *>(base + c * ps + (size_t)r * rs + lo);
  };
  with_radix<MAXR>(RA, [&](auto rad) {
    constexpr int R = decltype(rad)::value;
    if (j < RB) {
#pragma unroll 1
      for (int c = c0; c < 3; c += CG) {
        float2 v[R];
#pragma unroll
        for (int r = 0; r < R; ++r)
          v[r] = valid ? row(c, r * RB) : make_float2(0.f, 0.f);
        dft_any<R>(v, false);
#pragma unroll
        for (int r = 0; r < R; ++r) sm[c * cs + (j * R + r) * 16 + t] = v[r];
      }
    }
  });
  __syncthreads();
  with_radix<MAXR>(RB, [&](auto rad) {
    constexpr int R = decltype(rad)::value;
#pragma unroll 1
    for (int c = j < RA ? c0 : 3; c < 3; c += CG) {
      float2 v[R];
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = sm[c * cs + (j + r * RA) * 16 + t];
      radix_twiddle<R>(v, az.tw, j, false);
      dft_any<R>(v, false);
#pragma unroll
      for (int r = 0; r < R; ++r) sm[c * cs + (j + r * RA) * 16 + t] = v[r];
    }
  });
  if (CG > 1) __syncthreads();
  if (valid && j < RA) {
#pragma unroll 2
    for (int r = c0; r < RB; r += CG) {
      float2 *p = sm + (j + r * RA) * 16 + t;
      float2 b0 = p[0], b1 = p[cs], b2 = p[2 * cs];
      solve_one(sa, kx, ky, j + r * RA, ny, nxh, b0, b1, b2);
      p[0] = b0;
      p[cs] = b1;
      p[2 * cs] = b2;
    }
  }
  if (CG > 1) __syncthreads();
  with_radix<MAXR>(RB, [&](auto rad) {
    constexpr int R = decltype(rad)::value;
#pragma unroll 1
    for (int c = j < RA ? c0 : 3; c < 3; c += CG) {
      float2 v[R];
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = sm[c * cs + (j + r * RA) * 16 + t];
      dft_any<R>(v, true);
      radix_twiddle<R>(v, az.tw, j, true);
#pragma unroll
      for (int r = 0; r < R; ++r) sm[c * cs + (j + r * RA) * 16 + t] = v[r];
    }
  });
  __syncthreads();
  with_radix<MAXR>(RA, [&](auto rad) {
    constexpr int R = decltype(rad)::value;
    if (j < RB) {
#pragma unroll 1
      for (int c = c0; c < 3; c += CG) {
        float2 v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = sm[c * cs + (j * R + r) * 16 + t];
        dft_any<R>(v, true);
        if (valid) {
#pragma unroll
          for (int r = 0; r < R; ++r) row(c, r * RB) = v[r];
        }
      }
    }
  });
}

// ------------------------------------------------------------------ host

awk_status any_setup(int lds_max) {
  // these kernels may take more than the default 64 KiB of dynamic LDS
  static bool done = false;
  if (done) return AWK_OK;
  const void *fns[] = {reinterpret_cast<const void *>(&k_xfwd<0, 0, 0>),
                       reinterpret_cast<const void *>(&k_xinv<0, 0, 0, 1>),
                       reinterpret_cast<const void *>(&k_xinv<0, 0, 0, 1, false, true>),
                       reinterpret_cast<const void *>(&k_ypass),
                       reinterpret_cast<const void *>(&k_zsolve),
                       reinterpret_cast<const void *>(&k_xfwd<0, 0, 0, XENG_DENSE>),
                       reinterpret_cast<const void *>(&k_xinv<0, 0, 0, 1, false, false, false, XENG_DENSE>),
                       reinterpret_cast<const void *>(&k_xinv<0, 0, 0, 1, false, true, false, XENG_DENSE>),
                       reinterpret_cast<const void *>(&k_ypass_dense),
                       reinterpret_cast<const void *>(&k_zsolve_dense),
                       reinterpret_cast<const void *>(&k_xfwd<0, 8, 0, XENG_RADIX32>),
                       reinterpret_cast<const void *>(&k_xinv<0, 8, 0, 1, false, false, false, XENG_RADIX32>),
                       reinterpret_cast<const void *>(&k_xinv<0, 8, 0, 1, false, true, false, XENG_RADIX32>),
                       reinterpret_cast<const void *>(&k_zsolve_dense3),
                       reinterpret_cast<const void *>(&k_zsolve_radix<16, 3>),
                       reinterpret_cast<const void *>(&k_zsolve_radix<32, 1>),
                       reinterpret_cast<const void *>(&k_ypass_radix<32>)};
  for (const void *f : fns) AWK_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lds_max));
  done = true;
  return AWK_OK;
}

#define AWK_ANY_X(K, A)                                                                          \
  AWK_LAUNCH(K, dim3(grid, bt.n), dim3(k.bd_x), k.lds_x, s, A, k.ax[0].dev(), k.xplan(), k.nx, k.ny, \
             k.nz, k.nxh, k.nxh_pad, k.rt, k.spec, k.spec_plane(), bt)

void any_xfwd(FluidKernel &k, const XFwdArgs &a, unsigned grid, hipStream_t s, const Batch &bt) {
  if (k.ax[0].radix.ra > 16) AWK_ANY_X((k_xfwd<0, 8, 0, XENG_RADIX32>), a);
  else if (k.ax[0].radix.ra) AWK_ANY_X((k_xfwd<0, 8, 0, XENG_RADIX16>), a);
  else if (k.ax[0].dense.tiles) AWK_ANY_X((k_xfwd<0, 0, 0, XENG_DENSE>), a);
  else AWK_ANY_X((k_xfwd<0, 0, 0>), a);
}

void any_xinv(FluidKernel &k, const XInvArgs &a, bool apply, unsigned grid, hipStream_t s, const Batch &bt) {
  if (k.ax[0].radix.ra > 16) {
    if (apply) AWK_ANY_X((k_xinv<0, 8, 0, 1, false, true, false, XENG_RADIX32>), a);
    else AWK_ANY_X((k_xinv<0, 8, 0, 1, false, false, false, XENG_RADIX32>), a);
  } else if (k.ax[0].radix.ra) {
    if (apply) AWK_ANY_X((k_xinv<0, 8, 0, 1, false, true, false, XENG_RADIX16>), a);
    else AWK_ANY_X((k_xinv<0, 8, 0, 1, false, false, false, XENG_RADIX16>), a);
  } else if (k.ax[0].dense.tiles) {
    if (apply) AWK_ANY_X((k_xinv<0, 0, 0, 1, false, true, false, XENG_DENSE>), a);
    else AWK_ANY_X((k_xinv<0, 0, 0, 1, false, false, false, XENG_DENSE>), a);
  } else if (apply) AWK_ANY_X((k_xinv<0, 0, 0, 1, false, true>), a);
  else AWK_ANY_X((k_xinv<0, 0, 0, 1>), a);
}
#undef AWK_ANY_X

void any_ypass(FluidKernel &k, bool inv, const ReduceArgs &ra, hipStream_t s, const Batch &bt) {
  const int ntile = (k.nxh + k.tx_y - 1) / k.tx_y;
  const unsigned grid = grid_for((long long)3 * k.nz * ntile, 1);
  const RadixAxis r = k.ax[1].radix;
#define AWK_YX(M)                                                                                \
  AWK_LAUNCH(k_ypass_radix<M>, dim3(grid, bt.n), dim3(k.bd_y), k.lds_y, s, r, k.nz, k.nxh, k.nxh_pad, k.spec, \
             k.spec_plane(), inv ? 1 : 0, ra, bt)
  if (r.ra > 16) AWK_YX(32);
  else if (r.ra) AWK_YX(16);
  else if (k.ax[1].dense.tiles)
    AWK_LAUNCH(k_ypass_dense, dim3(grid, bt.n), dim3(k.bd_y), k.lds_y, s, k.ax[1].dense, k.nz, k.nxh,
               k.nxh_pad, k.spec, k.spec_plane(), inv ? 1 : 0, ra, bt);
  else
    AWK_LAUNCH(k_ypass, dim3(grid, bt.n), dim3(k.bd_y), k.lds_y, s, k.ax[1].dev(), k.ny, k.nz, k.nxh,
               k.nxh_pad, k.tx_y, k.spec, k.spec_plane(), inv ? 1 : 0, ra, bt);
#undef AWK_YX
}

void any_zsolve(FluidKernel &k, const SolveArgs &sa, hipStream_t s, const Batch &bt) {
  const int ntile = (k.nxh + k.tx_z - 1) / k.tx_z;
  const unsigned grid = grid_for((long long)k.ny * ntile, 1);
  const RadixAxis r = k.ax[2].radix;
#define AWK_ZX(M, CG)                                                                            \
  AWK_LAUNCH((k_zsolve_radix<M, CG>), dim3(grid, bt.n), dim3(k.bd_z), k.lds_z, s, r, sa, k.ny, k.nxh, k.nxh_pad, \
             k.spec, k.spec_plane(), bt)
  if (r.ra > 16) AWK_ZX(32, 1);
  else if (r.ra) AWK_ZX(16, 3);
  else if (k.ax[2].dense.tiles && k.bd_z == 192 * k.ax[2].dense.tiles)
    AWK_LAUNCH(k_zsolve_dense3, dim3(grid, bt.n), dim3(k.bd_z), k.lds_z, s, k.ax[2].dense, sa, k.ny, k.nxh,
               k.nxh_pad, k.spec, k.spec_plane(), bt);
  else if (k.ax[2].dense.tiles)
    AWK_LAUNCH(k_zsolve_dense, dim3(grid, bt.n), dim3(k.bd_z), k.lds_z, s, k.ax[2].dense, sa, k.ny, k.nxh,
               k.nxh_pad, k.spec, k.spec_plane(), bt);
  else
    AWK_LAUNCH(k_zsolve, dim3(grid, bt.n), dim3(k.bd_z), k.lds_z, s, k.ax[2].dev(), sa, k.ny, k.nz, k.nxh,
               k.nxh_pad, k.tx_z, k.spec, k.spec_plane(), bt);
#undef AWK_ZX
}

}  // namespace awk
