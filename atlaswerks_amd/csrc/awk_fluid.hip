// awk_fluid.hip -- FluidKernelFFT: L and L^-1 of the Navier operator
//   L = -alpha*Lap - beta*grad(div) + gamma
// applied through a 3-D real FFT, on gfx950.
//
// Semantics follow DiffOper::ApplyInverseOperatorOnTheFly / ApplyOperatorOnTheFly
// (Algorithms/Common/DiffOper.cxx:747-905): scale by 1/N, forward r2c of each
// component, per-frequency 3x3 L built from the LUT of DiffOper.cxx:587-639,
// Cholesky solve (DiffOper.cxx:1002-1083) or multiply (1085-1116), c2r.
//
// Pass structure (each pass is one kernel, one HBM round trip of the spectrum):
//   X  r2c along x of row triples (x, y, z components of the same rows), two real
//      lines packed per complex line; writes the half spectrum [c][z][y][kx].
//   Y  complex FFT along y for a tile of kx columns.
//   Z  forward FFT along z for all 3 components of a kx tile, the per-frequency
//      solve (with the 1/N scale folded in), inverse FFT along z.
//   Y' inverse along y.   X' c2r along x with an epilogue (plain store, max-norm,
//      or the fused greedy hfield update).
#include <algorithm>
#include <cmath>
#include <complex>
#include <cstring>
#include <new>
#include <vector>

#include "awk_fluid.h"
#include "awk_fluid_solve.h"
#include "awk_fluid_x.h"

namespace awk {

Axis AxisPlan::dev() const {
  Axis a;
  std::memset(&a, 0, sizeof(a));
  a.tw = tw;
  a.n = n;
  a.nst = (int)rad.size();
  for (int i = 0; i < a.nst; ++i) a.rad[i] = rad[i];
  a.m = m;
  a.chirp = chirp;
  a.bhat = bhat;
  a.mtw = mtw;
  a.mst = (int)mrad.size();
  for (int i = 0; i < a.mst; ++i) a.mrad[i] = mrad[i];
  return a;
}

// Unnormalised forward DFT of a power-of-two length in double (iterative
// radix 2), for the Bluestein kernel spectrum.
static void host_fft_pow2(std::vector<std::complex<double>> &a) {
  const size_t n = a.size();
  for (size_t i = 1, j = 0; i < n; ++i) {
    size_t bit = n >> 1;
    for (; j & bit; bit >>= 1) j ^= bit;
    j ^= bit;
    if (i < j) std::swap(a[i], a[j]);
  }
  for (size_t len = 2; len <= n; len <<= 1) {
    const double ang = -2.0 * M_PI / (double)len;
    for (size_t i = 0; i < n; i += len)
      for (size_t k = 0; k < len / 2; ++k) {
        const std::complex<double> w(cos(ang * k), sin(ang * k));
        const std::complex<double> u = a[i + k], v = a[i + k + len / 2] * w;
        a[i + k] = u + v;
        a[i + k + len / 2] = u - v;
      }
  }
}

// Bluestein tables of one axis appended to the host table `tw`: the chirp
// c_j = exp(-i pi j^2 / n) (the angle from j^2 mod 2n, exact in integers), the
// spectrum of b_l = conj(c_|l|) laid cyclically over m and scaled by 1/m, and
// the m twiddles.  Returns the offsets of the three tables.
static void bluestein_tables(int n, int m, std::vector<float2> &tw, size_t off[3]) {
  off[0] = tw.size();
  std::vector<std::complex<double>> c(n), b(m, 0.0);
  for (int j = 0; j < n; ++j) {
    const long long r = ((long long)j * j) % (2LL * n);
    const double a = -M_PI * (double)r / (double)n;
    c[j] = std::complex<double>(cos(a), sin(a));
    tw.push_back(make_float2((float)c[j].real(), (float)c[j].imag()));
  }
  for (int j = 0; j < n; ++j) {
    b[j] = std::conj(c[j]);
    if (j > 0) b[m - j] = std::conj(c[j]);
  }
  host_fft_pow2(b);
  off[1] = tw.size();
  for (int k = 0; k < m; ++k)
    tw.push_back(make_float2((float)(b[k].real() / m), (float)(b[k].imag() / m)));
  off[2] = tw.size();
  for (int k = 0; k < m; ++k) {
    const double a = -2.0 * M_PI * (double)k / (double)m;
    tw.push_back(make_float2((float)cos(a), (float)sin(a)));
  }
}

static std::vector<int> factor(int n) {
  std::vector<int> r;
  int m = n;
  while (m % 16 == 0) { r.push_back(16); m /= 16; }
  if (m % 8 == 0) { r.push_back(8); m /= 8; }
  if (m % 4 == 0) { r.push_back(4); m /= 4; }
  if (m % 2 == 0) { r.push_back(2); m /= 2; }
  for (int p = 3; m > 1; p += 2)
    while (m % p == 0) { r.push_back(p); m /= p; }
  return r;
}

// ------------------------------------------------------------------ kernels



// ------------------------------------------------------------------
// Register-resident two-stage passes for N = RA * RB (RA, RB in {8, 16}).
// Thread (t, j): t = kx column within the tile (lanes, 128-B rows for TX = 16),
// j = butterfly index.  Stage 1 reads its RA inputs straight from HBM, stage 2
// gets its inputs through one LDS transpose; the outputs of the forward stage 2
// stay in registers (Z pass: for the solve and the inverse stage 1).

template <int N, int RA, int RB, int TX>
__global__ void __launch_bounds__(TX *(N / RA > N / RB ? N / RA : N / RB))
k_ypass_reg(const float2 *__restrict__ tw, int nz, int nxh, int nxh_pad, float2 *__restrict__ spec,
            size_t plane, int inv, ReduceArgs ra, Batch bt) {
  constexpr int PA = N / RA, PB = N / RB;
  __shared__ float2 sm[N * TX];
  spec += (long long)blockIdx.y * bt.spec;
  const int t = threadIdx.x % TX, j = threadIdx.x / TX;
  const int ntile = (nxh + TX - 1) / TX;
  const int lb = (int)xcd_block();
  if (lb >= 3 * nz * ntile) return;
  const int tile = lb % ntile, rest = lb / ntile;
  // inv = 0: the forward pass visits (c, z) in reverse, which pays when the x pass
  // wrote the spectrum plane by plane (its last-written planes, the likeliest still
  // held by the memory-side cache, are read first; 256^3: 78.5 -> 75.0 us,
  // measured); inv = 2: in plane order, faster after the x pass's band order
  // (79.9 -> 78.0 us).  Every block transforms its own columns, so the order
  // changes no result.
  const bool rev = inv == 0;
  const int z = rev ? nz - 1 - rest % nz : rest % nz, c = rev ? 2 - rest / nz : rest / nz;
  const int kx = tile * TX + t;
  const bool valid = kx < nxh;
  float2 *base = spec + c * plane + (size_t)z * N * nxh_pad + kx;
  const bool iv = inv == 1;
  if (j < PA) {  // stage 1: radix RA, Ns = 1, inputs y = j + r * PA
    float2 v[RA];
#pragma unroll
    for (int r = 0; r < RA; ++r) v[r] = valid ? base[(size_t)(j + r * PA) * nxh_pad] : make_float2(0.f, 0.f);
    dft<RA>(v, iv);
#pragma unroll
    for (int r = 0; r < RA; ++r) sm[(j * RA + r) * TX + t] = v[r];
  }
  __syncthreads();
  if (j < PB) {  // stage 2: radix RB, Ns = RA, inputs j + r * PB, twiddle W^(r j), outputs j + r * RA
    float2 v[RB];
#pragma unroll
    for (int r = 0; r < RB; ++r) v[r] = sm[(j + r * PB) * TX + t];
#pragma unroll
    for (int r = 1; r < RB; ++r) v[r] = iv ? cmulc(v[r], tw[r * j]) : cmul(v[r], tw[r * j]);
    dft<RB>(v, iv);
    if (valid) {
#pragma unroll
      for (int r = 0; r < RB; ++r) base[(size_t)(j + r * RA) * nxh_pad] = v[r];
    }
  }
  if (ra.partials && lb == 0) {
    __syncthreads();
    batch_reduce(ra, bt);
    energy_block(ra, reinterpret_cast<double *>(sm), TX * (PA > PB ? PA : PB));
  }
}

// The three components' z-lines stay in registers through the solve; the
// occupancy floor (3 blocks of 256 at N = 256, 4 below) makes the compiler fit
// them in 168 / 128 registers without spilling, one more resident wave per SIMD
// than it picks unasked (256^3 greedy: 111 -> 96 us).
template <int N, int RA, int RB, int TX>
__global__ void __launch_bounds__(TX *(N / RA > N / RB ? N / RA : N / RB), N >= 256 ? 3 : 4)
k_zsolve_reg(const float2 *__restrict__ tw, SolveArgs sa, int ny, int nxh, int nxh_pad,
             float2 *__restrict__ spec, size_t plane, Batch bt) {
  constexpr int PA = N / RA, PB = N / RB;  // PB = RA: threads holding the spectrum
  __shared__ float2 sm[N * TX];
  spec += (long long)blockIdx.y * bt.spec;
  const int t = threadIdx.x % TX, j = threadIdx.x / TX;
  const int ntile = (nxh + TX - 1) / TX;
  const int lb = (int)xcd_block();
  if (lb >= ny * ntile) return;
  const int tile = lb % ntile, ky = lb / ntile;
  const int kx = tile * TX + t;
  const bool valid = kx < nxh;
  const size_t zst = (size_t)ny * nxh_pad;
  float2 *base = spec + (size_t)ky * nxh_pad + kx;
  float2 X[3][RB];
  // forward: radix RA then RB; the spectrum at kz = j + r * RA lands in X[c][r]
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    if (j < PA) {
      float2 v[RA];
#pragma unroll
      for (int r = 0; r < RA; ++r)
        v[r] = valid ? base[c * plane + (size_t)(j + r * PA) * zst] : make_float2(0.f, 0.f);
      dft<RA>(v, false);
#pragma unroll
      for (int r = 0; r < RA; ++r) sm[(j * RA + r) * TX + t] = v[r];
    }
    __syncthreads();
    if (j < PB) {
#pragma unroll
      for (int r = 0; r < RB; ++r) X[c][r] = sm[(j + r * PB) * TX + t];
#pragma unroll
      for (int r = 1; r < RB; ++r) X[c][r] = cmul(X[c][r], tw[r * j]);
      dft<RB>(X[c], false);
    }
    __syncthreads();
  }
  if (j < PB && valid) {
#pragma unroll
    for (int r = 0; r < RB; ++r) solve_one(sa, kx, ky, j + r * RA, ny, nxh, X[0][r], X[1][r], X[2][r]);
  }
  // inverse: radix RB (inputs j + r * RA = the registers) then RA; outputs z = j + r * RB
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    if (j < PB) {
      dft<RB>(X[c], true);
#pragma unroll
      for (int r = 0; r < RB; ++r) sm[(j * RB + r) * TX + t] = X[c][r];
    }
    __syncthreads();
    if (j < PA) {
      float2 v[RA];
#pragma unroll
      for (int r = 0; r < RA; ++r) v[r] = sm[(j + r * PA) * TX + t];
#pragma unroll
      for (int r = 1; r < RA; ++r) v[r] = cmulc(v[r], tw[r * j]);
      dft<RA>(v, true);
      if (valid) {
#pragma unroll
        for (int r = 0; r < RA; ++r) base[c * plane + (size_t)(j + r * PA) * zst] = v[r];
      }
    }
    __syncthreads();
  }
}


// FP64 table of L^p (symmetric, 6 entries) per frequency for the eigen path
// (DiffOper::InitializeEigenLookup + PowL, DiffOper.cxx:641-745, 1176-1218).
// Jacobi rotations on the 3x3 symmetric matrix in double.
__global__ void k_eigen_table(float *__restrict__ out, int nx, int ny, int nz, int nxh, double spx,
                              double spy, double spz, double alpha, double beta, double gamma,
                              double p) {
  const size_t total = (size_t)nxh * ny * nz;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < total;
       i += (size_t)gridDim.x * blockDim.x) {
    const int kx = (int)(i % nxh);
    const int ky = (int)((i / nxh) % ny);
    const int kz = (int)(i / ((size_t)nxh * ny));
    const double PI2 = 6.283185307179586476925286766559;
    const double cx = (2.0 * cos(PI2 * kx / nx) - 2.0) / (spx * spx);
    const double cy = (2.0 * cos(PI2 * ky / ny) - 2.0) / (spy * spy);
    const double cz = (2.0 * cos(PI2 * kz / nz) - 2.0) / (spz * spz);
    const double sx = sin(PI2 * kx / nx) / spx, sy = sin(PI2 * ky / ny) / spy,
                 sz = sin(PI2 * kz / nz) / spz;
    const double lam = -alpha * (cx + cy + cz) + gamma;
    double A[3][3] = {{lam - beta * cx, beta * sx * sy, beta * sx * sz},
                      {beta * sx * sy, lam - beta * cy, beta * sy * sz},
                      {beta * sx * sz, beta * sy * sz, lam - beta * cz}};
    double Q[3][3] = {{1, 0, 0}, {0, 1, 0}, {0, 0, 1}};
    for (int sweep = 0; sweep < 32; ++sweep) {
      const double off = A[0][1] * A[0][1] + A[0][2] * A[0][2] + A[1][2] * A[1][2];
      const double dg = A[0][0] * A[0][0] + A[1][1] * A[1][1] + A[2][2] * A[2][2];
      if (off <= 1e-34 * dg) break;
      for (int pp = 0; pp < 2; ++pp)
        for (int q = pp + 1; q < 3; ++q) {
          if (A[pp][q] == 0.0) continue;
          const double th = (A[q][q] - A[pp][pp]) / (2.0 * A[pp][q]);
          const double t = (th >= 0 ? 1.0 : -1.0) / (fabs(th) + sqrt(th * th + 1.0));
          const double c = 1.0 / sqrt(t * t + 1.0), sn = t * c;
          for (int k = 0; k < 3; ++k) {
            const double akp = A[k][pp], akq = A[k][q];
            A[k][pp] = c * akp - sn * akq;
            A[k][q] = sn * akp + c * akq;
          }
          for (int k = 0; k < 3; ++k) {
            const double apk = A[pp][k], aqk = A[q][k];
            A[pp][k] = c * apk - sn * aqk;
            A[q][k] = sn * apk + c * aqk;
          }
          for (int k = 0; k < 3; ++k) {
            const double qkp = Q[k][pp], qkq = Q[k][q];
            Q[k][pp] = c * qkp - sn * qkq;
            Q[k][q] = sn * qkp + c * qkq;
          }
        }
    }
    double e[3];
    for (int j = 0; j < 3; ++j) e[j] = pow(A[j][j], p);
    double M[3][3];
    for (int r = 0; r < 3; ++r)
      for (int c = 0; c < 3; ++c)
        M[r][c] = Q[r][0] * Q[c][0] * e[0] + Q[r][1] * Q[c][1] * e[1] + Q[r][2] * Q[c][2] * e[2];
    float *o = out + i * 6;
    o[0] = (float)M[0][0];
    o[1] = (float)M[1][0];
    o[2] = (float)M[1][1];
    o[3] = (float)M[2][0];
    o[4] = (float)M[2][1];
    o[5] = (float)M[2][2];
  }
}

// ------------------------------------------------------------------ host

// LDS of the x passes: the row buffer (LS = NL + 1) plus the Bluestein work area,
// or the staged lines (with the zero row) and both parts of the frequencies.
static size_t x_lds(const AxisPlan &a, int rt) {
  if (a.dense.tiles) return (size_t)std::max(a.n + 1, 4 * a.dense.ks) * kDenseLS * sizeof(float);
  return ((size_t)a.n * (3 * rt / 2 + 1) + (size_t)a.m * (3 * rt / 2)) * sizeof(float2);
}
// LDS of the y / z passes: n lines-per-column * tx lines, plus the work area (dense:
// 16 columns of n + 1 rows).
static size_t yz_lds(const AxisPlan &a, int lines) {
  if (a.dense.tiles) return ((size_t)a.n + 1) * 16 * sizeof(float2);
  return ((size_t)a.n + (size_t)a.m) * lines * sizeof(float2);
}

// Dynamic LDS a pass block may take: gfx950's 160 KiB per workgroup, less 1 KiB
// for the kernels' static reduction arrays (the generic pass kernels are set up
// for it once; above 64 KiB a block has the CU's LDS to itself)
constexpr size_t kPassLdsMax = 160 * 1024 - 1024;

// Whether an axis is transformed as a dense product (awk_dense.h): a length with a
// prime factor above 13, whose LDS stages would be a direct DFT of that prime or a
// chirp-z transform.  L^-1 at 181 x 217 x 181 4347 -> 548 us, 251 x 241 x 239 7189 ->
// 1085, 248 x 186 x 155 2611 -> 546, 62^3 184 -> 47, 32 x 31 x 36 63 -> 25.  Over 30 lengths
// 17 ... 510 on each axis (the others 64 and 128): 1.3 ... 5 times as fast, small primes
// times 17 included (408 along x / y / z 500 / 543 / 528 -> 215 / 250 / 328 us, 510 623 /
// 646 / 644 -> 251 / 300 / 389).  Lengths of small primes are faster as radices: at 200^3
// 382 us (dense 664).
static bool use_dense(int n, const std::vector<int> &rad) {
  if (n < kDenseMin || n > kDenseMax) return false;
  for (int r : rad)
    if (r > 13 && r != 16) return true;
  return false;
}

// Whether an axis is transformed by two radices in registers (awk_radix.h): every
// length that has such a plan, up to 1024 (along z up to the 424 whose three
// components fit a block's LDS).  L^-1 against the LDS stages: 160 x 192 x 144 312 ->
// 160 us, 96^3 125 -> 59, 36^3 43 -> 26, 112^3 279 -> 78, 182^3 2199 -> 222, 240^3 931 ->
// 490, 200^3 553 -> 374, 300 x 128 x 128 317 -> 172.  Over 40 lengths 2 ... 1024 on each
// axis (the others 64 and 128): 1.02 ... 6.3 times as fast (1024 along x / y 322 / 323 ->
// 292 / 264 us), 625 along x alone 3 % slower.
static bool use_radix(int axis, int n) {
  int ra, rb;
  return n > 1 && radix_plan(n, ra, rb) && (axis < 2 || (size_t)n * 3 * 16 * sizeof(float2) <= kPassLdsMax);
}

// The fragment-order table of DenseAxis.  cos and sin of 2 pi m / n once per m.
static std::vector<float2> dense_table(int n, DenseAxis &d) {
  d.n = n;
  d.H = n / 2 + 1;
  d.tiles = (d.H + 31) / 32;
  d.ks = ((d.H + 1) / 2 + 3) / 4 * 4;
  std::vector<float2> cs(n);
  for (int m = 0; m < n; ++m) {
    const double a = 2.0 * M_PI * (double)m / (double)n;
    cs[m] = make_float2((float)cos(a), (2 * m == n || m == 0) ? 0.f : (float)sin(a));
  }
  std::vector<float2> t((size_t)d.tiles * d.ks * 64, make_float2(0.f, 0.f));
  for (int k = 0; k < d.H; ++k)
    for (int j = 0; j < d.H; ++j) {
      float2 v = cs[(int)((long long)j * k % n)];
      if (2 * j == n) v = make_float2(0.5f * v.x, 0.f);
      t[((size_t)(k / 32) * d.ks + j / 2) * 64 + (j & 1) * 32 + k % 32] = v;
    }
  return t;
}

static int pick_rt(const AxisPlan &a) {
  // the tuned RT if it fits, else the largest even RT <= 8 whose LDS fits 64 KiB
  const int want = tuning().x_rt;
  if (want > 0 && x_lds(a, want) <= 65536) return want;
  for (int rt = 8; rt >= 2; rt -= 2)  // within 64 KiB where possible (several blocks per CU)
    if (x_lds(a, rt) <= 65536) return rt;
  for (int rt = 8; rt >= 2; rt -= 2)
    if (x_lds(a, rt) <= kPassLdsMax) return rt;
  return 0;
}

static int pick_tx(const AxisPlan &a, int lines_per_col, int max_tx, int want) {
  if (want > 0 && want <= max_tx && yz_lds(a, lines_per_col * want) <= 65536) return want;
  for (int tx = max_tx; tx >= 1; tx /= 2)
    if (yz_lds(a, lines_per_col * tx) <= 65536) return tx;
  for (int tx = max_tx; tx >= 1; tx /= 2)
    if (yz_lds(a, lines_per_col * tx) <= kPassLdsMax) return tx;
  return 0;
}

static int pick_bd(int n, int nl) {
  // n * NL <= 16 * bd, bd multiple of 64, 64..1024
  int bd = (int)(((long long)n * nl + kMaxElemsPerThread - 1) / kMaxElemsPerThread);
  bd = (bd + 63) / 64 * 64;
  if (bd < 256) bd = 256;
  return bd;
}

awk_status fk_init(FluidKernel &k, int nx, int ny, int nz, const float sp[3]) {
  if (nx < 1 || ny < 1 || nz < 1) return fail(AWK_ERR_INVALID, "fluid kernel: sizes must be >= 1");
  if ((long long)nx * ny * nz > kBufMaxElems) return fail(AWK_ERR_INVALID, "fluid kernel: volume too large");
  k.nx = nx; k.ny = ny; k.nz = nz;
  k.nxh = nx / 2 + 1;
  k.nxh_pad = (k.nxh + 7) / 8 * 8;
  for (int i = 0; i < 3; ++i) k.sp[i] = sp[i];
  const int ns[3] = {nx, ny, nz};
  std::vector<float2> dense[3];
  for (int i = 0; i < 3; ++i) {
    k.ax[i].n = ns[i];
    k.ax[i].rad = factor(ns[i]);
    k.ax[i].m = 0;
    k.ax[i].mrad.clear();
    k.ax[i].dense = DenseAxis{nullptr, 0, 0, 0, 0, 0};
    k.ax[i].radix = RadixAxis{nullptr, ns[i], 0, 0};
    if (use_radix(i, ns[i])) radix_plan(ns[i], k.ax[i].radix.ra, k.ax[i].radix.rb);
    bool big = false;
    for (int r : k.ax[i].rad) big = big || r > 64;
    if (use_dense(ns[i], k.ax[i].rad)) {
      dense[i] = dense_table(ns[i], k.ax[i].dense);
      // (factor() gives primes but for powers of two)
      k.ax[i].dense.short_runs = dense_short_runs(ns[i], *std::max_element(k.ax[i].rad.begin(), k.ax[i].rad.end()));
    } else if (big) {
      // Bluestein: a power-of-two convolution of length m >= 2n - 1
      int m = 1;
      while (m < 2 * ns[i] - 1) m *= 2;
      k.ax[i].m = m;
      k.ax[i].mrad = factor(m);
    }
    if (tuning().fft_order) {  // the stages in the reverse order (a tuned plan)
      std::reverse(k.ax[i].rad.begin(), k.ax[i].rad.end());
      std::reverse(k.ax[i].mrad.begin(), k.ax[i].mrad.end());
    }
    if ((int)k.ax[i].rad.size() > kMaxStages || (int)k.ax[i].mrad.size() > 8)
      return fail(AWK_ERR_INVALID, "fluid kernel: too many FFT stages");
  }
  const DenseAxis *dx[3] = {&k.ax[0].dense, &k.ax[1].dense, &k.ax[2].dense};
  const RadixAxis *rx[3] = {&k.ax[0].radix, &k.ax[1].radix, &k.ax[2].radix};
  k.rt = rx[0]->ra ? 8 : dx[0]->tiles ? kDenseRows : pick_rt(k.ax[0]);
  k.tx_y = dx[1]->tiles || rx[1]->ra ? 16 : pick_tx(k.ax[1], 1, 16, tuning().y_tx);
  k.tx_z = dx[2]->tiles || rx[2]->ra ? 16 : pick_tx(k.ax[2], 3, 8, tuning().z_tx);
  if (!k.rt || !k.tx_y || !k.tx_z) return fail(AWK_ERR_UNSUPPORTED, "fluid kernel: axis too long for LDS staging");
  k.bd_x = rx[0]->ra ? std::max(256, (12 * rx[0]->ra + 63) / 64 * 64) : dx[0]->tiles ? std::max(256, 64 * dx[0]->tiles) : pick_bd(k.ax[0].stage_len(), 3 * k.rt / 2);
  k.bd_y = rx[1]->ra ? 16 * rx[1]->ra : dx[1]->tiles ? 64 * dx[1]->tiles : pick_bd(k.ax[1].stage_len(), k.tx_y);
  // along z a wave per tile and component (or thread group per component) where they fit a block
  const bool z3 = dx[2]->tiles ? dx[2]->tiles <= 5 : rx[2]->ra <= 16;
  k.bd_z = (z3 ? 3 : 1) * (rx[2]->ra ? (z3 ? (16 * rx[2]->ra + 63) / 64 * 64 : 16 * rx[2]->ra) : dx[2]->tiles ? 64 * dx[2]->tiles : 0);
  if (!k.bd_z) k.bd_z = pick_bd(k.ax[2].stage_len(), 3 * k.tx_z);
  if (k.bd_x > 1024 || k.bd_y > 1024 || k.bd_z > 1024)
    return fail(AWK_ERR_UNSUPPORTED, "fluid kernel: block too large");
  k.lds_x = x_lds(k.ax[0], k.rt);
  k.lds_y = std::max(yz_lds(k.ax[1], k.tx_y), (size_t)k.bd_y * sizeof(double));  // (the energy tree)
  k.lds_z = yz_lds(k.ax[2], 3 * k.tx_z) * (dx[2]->tiles && z3 ? 3 : 1);
  if (awk_status st = any_setup((int)kPassLdsMax)) return st;
  // twiddles and LUT (double -> float); the Bluestein tables follow the three
  // axes' twiddles in the same allocation
  std::vector<float2> tw((size_t)nx + ny + nz);
  size_t off = 0;
  for (int i = 0; i < 3; ++i) {
    for (int j = 0; j < ns[i]; ++j) {
      const double a = -2.0 * M_PI * (double)j / (double)ns[i];
      tw[off + j] = make_float2((float)cos(a), (float)sin(a));
    }
    off += ns[i];
  }
  size_t boff[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
  for (int i = 0; i < 3; ++i)
    if (k.ax[i].m) bluestein_tables(ns[i], k.ax[i].m, tw, boff[i]);
  size_t doff[3] = {0, 0, 0};
  for (int i = 0; i < 3; ++i) {
    doff[i] = tw.size();
    tw.insert(tw.end(), dense[i].begin(), dense[i].end());
  }
  const size_t ntw = tw.size();
  const size_t nlut = 2 * (size_t)k.nxh + 2 * (size_t)ny + 2 * (size_t)nz;
  const size_t scalars = (nlut + 3) / 4 * 4;
  std::vector<float> lut(scalars + kScalarBytes / sizeof(float), 0.f);
  {
    // DiffOper.cxx:602-625: cosW = (2cos(2 pi k/n) - 2)/sp^2, sinW = sin(2 pi k/n)/sp
    float *p = lut.data();
    const int lens[3] = {k.nxh, ny, nz};
    for (int i = 0; i < 3; ++i) {
      const double s = 2.0 * M_PI / ns[i];
      for (int j = 0; j < lens[i]; ++j) {
        p[j] = (float)((2.0 * cos(s * j) - 2.0) / ((double)sp[i] * sp[i]));
        p[lens[i] + j] = (float)(sin(s * j) / (double)sp[i]);
      }
      p += 2 * lens[i];
    }
  }
  const size_t spec_bytes = 3 * k.spec_plane() * sizeof(float2);
  AWK_HIP(dev_alloc(&k.spec, spec_bytes));
  float2 *twd = nullptr;
  AWK_HIP(dev_alloc(&twd, ntw * sizeof(float2)));
  AWK_HIP(hipMemcpy(twd, tw.data(), ntw * sizeof(float2), hipMemcpyHostToDevice));
  k.ax[0].tw = twd;
  k.ax[1].tw = twd + nx;
  k.ax[2].tw = twd + nx + ny;
  for (int i = 0; i < 3; ++i) k.ax[i].radix.tw = k.ax[i].tw;
  for (int i = 0; i < 3; ++i)
    if (k.ax[i].m) {
      k.ax[i].chirp = twd + boff[i][0];
      k.ax[i].bhat = twd + boff[i][1];
      k.ax[i].mtw = twd + boff[i][2];
    }
  for (int i = 0; i < 3; ++i)
    if (k.ax[i].dense.tiles) k.ax[i].dense.tab = twd + doff[i];
  AWK_HIP(dev_alloc(&k.lut, lut.size() * sizeof(float)));
  AWK_HIP(hipMemcpy(k.lut, lut.data(), lut.size() * sizeof(float), hipMemcpyHostToDevice));
  k.scalars = k.lut + scalars;
  k.scratch_bytes = spec_bytes + ntw * sizeof(float2) + nlut * sizeof(float);
  return AWK_OK;
}

void fk_take_blocks(FluidKernel &k, void *blocks[kFkBlocks]) {
  blocks[0] = k.spec;
  blocks[1] = const_cast<float2 *>(k.ax[0].tw);
  blocks[2] = k.lut;
  blocks[3] = k.eig;
  k.spec = nullptr;
  k.ax[0].tw = k.ax[1].tw = k.ax[2].tw = nullptr;
  k.lut = nullptr;
  k.scalars = nullptr;
  k.eig = nullptr;
}

void fk_release(FluidKernel &k) {
  void *blocks[kFkBlocks];
  fk_take_blocks(k, blocks);
  dev_free(blocks, kFkBlocks, !k.other_stream);
}

awk_status fk_prepare_eigen(FluidKernel &k, int dir, hipStream_t s) {
  if (k.eig && k.eig_dir == dir) return AWK_OK;
  const size_t nf = (size_t)k.nxh * k.ny * k.nz;
  if (!k.eig) {
    // not a kept block, which would spare the allocation that a capture refuses
    AWK_HIP(device_malloc(&k.eig, nf * 6 * sizeof(float)));
    k.scratch_bytes += nf * 6 * sizeof(float);
  }
  const double p = dir > 0 ? (double)k.lpow : -(double)k.lpow;
  unsigned grid = (unsigned)std::min<size_t>((nf + 255) / 256, 65536);
  AWK_LAUNCH(k_eigen_table, dim3(grid), dim3(256), 0, s, k.eig, k.nx, k.ny, k.nz, k.nxh,
                     (double)k.sp[0], (double)k.sp[1], (double)k.sp[2], (double)k.alpha,
                     (double)k.beta, (double)k.gamma, p);
  AWK_LAUNCH_CHECK("k_eigen_table");
  // under a capture (a relaxed one, which allows the allocation) the table is recorded and
  // not made: the next call makes it
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  AWK_HIP(hipStreamIsCapturing(s, &cap));
  k.eig_dir = cap == hipStreamCaptureStatusNone ? dir : 0;
  return AWK_OK;
}

int fk_xblocks(const FluidKernel &k) {
  return (int)grid_for((long long)k.ny * k.nz, k.rt);
}

awk_status fk_xfwd(FluidKernel &k, const XFwdArgs &a_in, hipStream_t s, int *nblocks, const Batch *b) {
  k.used_on(s);
  const Batch bt = b ? *b : Batch();
  const unsigned grid = grid_for((long long)k.ny * k.nz, k.rt);
  XFwdArgs a = a_in;
  a.band = 0;
  {
    const int bd = tuning().xfwd_band;
    const long long G = k.ny / k.rt, per = grid / kNumXcd;
    if (bd > 0 && k.ny % k.rt == 0 && G * k.nz == (long long)grid && per % G == 0 && G % bd == 0)
      a.band = bd;
  }
  const size_t lds = k.lds_x;
  const Axis ax = k.ax[0].dev();
#define AWK_XF(NC, RTC, BDC)                                                                     \
  AWK_LAUNCH((k_xfwd<NC, RTC, BDC>), dim3(grid, bt.n), dim3(BDC ? BDC : k.bd_x), lds, s, a, ax, k.xplan(), \
                     k.nx, k.ny, k.nz, k.nxh, k.nxh_pad, k.rt, k.spec, k.spec_plane(), bt)
  // block size = row length selects column mode (128^3 LDMM: 17.2 -> 16.3 us
  // against the generic 256-thread form; the spectrum is the same bit for bit)
  if (k.nx == 256) AWK_XF(256, 8, 256);
  else if (k.nx == 128) AWK_XF(128, 8, 128);
  else if (k.nx == 64) AWK_XF(64, 8, 256);
  else any_xfwd(k, a, grid, s, bt);
#undef AWK_XF
  AWK_LAUNCH_CHECK("k_xfwd");
  if (nblocks) *nblocks = (int)grid;
  return AWK_OK;
}

awk_status fk_ypass(FluidKernel &k, bool inv, hipStream_t s, const ReduceArgs *red, const Batch *b) {
  k.used_on(s);
  const Batch bt = b ? *b : Batch();
  ReduceArgs ra;
  std::memset(&ra, 0, sizeof(ra));
  if (red) ra = *red;
  const float2 *tw = k.ax[1].tw;
  const int ntile16 = (k.nxh + 15) / 16;
  const unsigned g16 = grid_for((long long)3 * k.nz * ntile16, 1);
#define AWK_YR(N, RA, RB)                                                                     \
  AWK_LAUNCH((k_ypass_reg<N, RA, RB, 16>), dim3(g16, bt.n), dim3(16 * (N / RA > N / RB ? N / RA : N / RB)), \
                     0, s, tw, k.nz, k.nxh, k.nxh_pad, k.spec, k.spec_plane(),                    \
                     inv ? 1 : tuning().yfwd_rev ? 0 : 2, ra, bt)
  if (k.ny == 256) AWK_YR(256, 16, 16);
  else if (k.ny == 128) AWK_YR(128, 16, 8);
  else if (k.ny == 64) AWK_YR(64, 8, 8);
  else if (k.ny == 32) AWK_YR(32, 8, 4);
  else any_ypass(k, inv, ra, s, bt);
#undef AWK_YR
  AWK_LAUNCH_CHECK("k_ypass");
  return AWK_OK;
}

awk_status fk_zsolve(FluidKernel &k, bool inverse_op, hipStream_t s, const Batch *b) {
  k.used_on(s);
  const Batch bt = b ? *b : Batch();
  const bool eigen = (k.flags & AWK_FK_EIGEN) || k.lpow != 1.0f;
  if (eigen) {
    awk_status st = fk_prepare_eigen(k, inverse_op ? -1 : 1, s);
    if (st) return st;
  }
  SolveArgs sa;
  sa.cwx = k.lut;
  sa.swx = k.lut + k.nxh;
  sa.cwy = k.lut + 2 * k.nxh;
  sa.swy = sa.cwy + k.ny;
  sa.cwz = sa.swy + k.ny;
  sa.swz = sa.cwz + k.nz;
  sa.eig = eigen ? k.eig : nullptr;
  sa.alpha = k.alpha;
  sa.beta = k.beta;
  sa.gamma = k.gamma;
  sa.scale = (float)(1.0 / ((double)k.nx * k.ny * k.nz));
  sa.inverse_op = inverse_op ? 1 : 0;
  sa.divfree = (k.flags & AWK_FK_DIVFREE) ? 1 : 0;
  const float2 *tw = k.ax[2].tw;
  const int ntile16 = (k.nxh + 15) / 16;
  const unsigned g16 = grid_for((long long)k.ny * ntile16, 1);
#define AWK_ZR(N, RA, RB)                                                                     \
  AWK_LAUNCH((k_zsolve_reg<N, RA, RB, 16>), dim3(g16, bt.n), dim3(16 * (N / RA > N / RB ? N / RA : N / RB)), \
                     0, s, tw, sa, k.ny, k.nxh, k.nxh_pad, k.spec, k.spec_plane(), bt)
  // 64 and below go through the two-radix kernel, whose thread groups hold one
  // component each: 11.0 -> 8.2 us at 64^3 and 8.1 -> 6.4 at 32^3; at 128 the line in
  // registers is the faster (21.3 against 23.8 us)
  if (k.nz == 256) AWK_ZR(256, 16, 16);
  else if (k.nz == 128) AWK_ZR(128, 16, 8);
  else any_zsolve(k, sa, s, bt);
#undef AWK_ZR
  AWK_LAUNCH_CHECK("k_zsolve");
  return AWK_OK;
}

awk_status fk_xinv(FluidKernel &k, const XInvArgs &a_in, hipStream_t s, int *nblocks, const Batch *b) {
  k.used_on(s);
  const Batch bt = b ? *b : Batch();
  const unsigned grid = grid_for((long long)k.ny * k.nz, k.rt);
  XInvArgs a = a_in;
  a.band = 0;
  {
    // the band block order of the composition, where whole planes of row groups
    // fill each XCD's share of the grid and the band divides a plane
    const int bd = tuning().xinv_band;
    const long long G = k.ny / k.rt, per = grid / kNumXcd;
    if (a.mode == XSTORE_COMPOSE && bd > 0 && k.ny % k.rt == 0 && G * k.nz == (long long)grid &&
        per % G == 0 && G % bd == 0)
      a.band = bd;
  }
  size_t lds = k.lds_x;
  const Axis ax = k.ax[0].dev();
#define AWK_XI3(NC, RTC, BDC, XU, PR, AP)                                                        \
  AWK_LAUNCH((k_xinv<NC, RTC, BDC, XU, PR, AP>), dim3(grid, bt.n), dim3(BDC ? BDC : k.bd_x), lds, s, a, \
                     ax, k.xplan(), k.nx, k.ny, k.nz, k.nxh, k.nxh_pad, k.rt, k.spec, k.spec_plane(), bt)
#define AWK_XIS(NC, BD, AP)                                                                      \
  AWK_LAUNCH((k_xinv<NC, 8, BD, 1, false, AP, true>), dim3(grid, bt.n), dim3(BD), lds, s, a, ax, k.xplan(), \
                     k.nx, k.ny, k.nz, k.nxh, k.nxh_pad, k.rt, k.spec, k.spec_plane(), bt)
#define AWK_XI(NC, RTC, BDC, XU)                                                                 \
  AWK_LAUNCH((k_xinv<NC, RTC, BDC, XU>), dim3(grid, bt.n), dim3(BDC ? BDC : k.bd_x), lds, s, a, ax, k.xplan(), \
                     k.nx, k.ny, k.nz, k.nxh, k.nxh_pad, k.rt, k.spec, k.spec_plane(), bt)
  const int xu = tuning().xinv_unroll;
  // xinv_pairs: waves whose points all lie inside the volume gather the
  // x-neighbour corners as 8-byte pairs (12 loads per point instead of 24; the
  // same values, so the same result)
  const bool pr = a.mode == XSTORE_COMPOSE && tuning().xinv_pairs;
  // the composition with the next iteration's deformed image (one subject per launch)
  const bool ap = a.mode == XSTORE_COMPOSE && a.i0;
  if (ap && (bt.n != 1 || !a.idef))
    return fail(AWK_ERR_INVALID, "inverse x pass: the fused apply takes one subject and an output image");
  // xinv_stage: the composition reads the field from the block's rows and their
  // neighbours staged in LDS (specialised row lengths, whole blocks in one plane).
  // Measured on the greedy step: 128^3 atlas iteration 1.52 -> 1.35 ms, but at
  // 256-long rows 0.26 -> 0.36 ms per composition (three staged rows per row read
  // through L2, with 4 blocks per CU; 0.30 ms with 512 threads of 4 points each,
  // whose FFT rounds differently), so by default rows up to 128 only.
  const int sk = tuning().xinv_stage;
  const bool stg = a.mode == XSTORE_COMPOSE && (sk == 1 || (sk == 2 && k.nx <= 128)) &&
                   k.ny % 8 == 0 && (k.nx == 256 || k.nx == 128 || k.nx == 64);
  if (stg) {
    lds = std::max(lds, (size_t)3 * (k.rt + 2) * k.nx * sizeof(float));
    if (k.nx == 256) {
      if (ap) AWK_XIS(256, 256, true);
      else AWK_XIS(256, 256, false);
    } else if (k.nx == 128) {
      if (ap) AWK_XIS(128, 256, true);
      else AWK_XIS(128, 256, false);
    } else if (ap) AWK_XIS(64, 256, true);
    else AWK_XIS(64, 256, false);
  } else if (ap) {
    if (k.nx == 256) {
      if (pr) {
        if (xu == 4) AWK_XI3(256, 8, 256, 4, true, true);
        else if (xu == 2) AWK_XI3(256, 8, 256, 2, true, true);
        else AWK_XI3(256, 8, 256, 1, true, true);
      } else if (xu == 4) AWK_XI3(256, 8, 256, 4, false, true);
      else if (xu == 2) AWK_XI3(256, 8, 256, 2, false, true);
      else AWK_XI3(256, 8, 256, 1, false, true);
    } else if (k.nx == 128) AWK_XI3(128, 8, 256, 2, false, true);
    else if (k.nx == 64) AWK_XI3(64, 8, 256, 2, false, true);
    else any_xinv(k, a, true, grid, s, bt);
  } else if (k.nx == 256) {
    if (pr) {
      if (xu == 4) AWK_XI3(256, 8, 256, 4, true, false);
      else if (xu == 2) AWK_XI3(256, 8, 256, 2, true, false);
      else AWK_XI3(256, 8, 256, 1, true, false);
    } else if (xu == 4) AWK_XI(256, 8, 256, 4);
    else if (xu == 2) AWK_XI(256, 8, 256, 2);
    else AWK_XI(256, 8, 256, 1);
  } else if (k.nx == 128) AWK_XI(128, 8, 256, 2);
  else if (k.nx == 64) AWK_XI(64, 8, 256, 2);
  else any_xinv(k, a, false, grid, s, bt);
#undef AWK_XI
#undef AWK_XI3
#undef AWK_XIS
  AWK_LAUNCH_CHECK("k_xinv");
  if (nblocks) *nblocks = (int)grid;
  return AWK_OK;
}

}  // namespace awk

using namespace awk;

extern "C" {

int awk_fft_axis_staged(int axis, int n) {
  return axis >= 0 && axis < 3 && n >= 1 && !use_radix(axis, n) && !use_dense(n, factor(n));
}

awk_status awk_fluid_kernel_create(awk_fk_t *out, int nx, int ny, int nz, float spx, float spy,
                                   float spz, float alpha, float beta, float gamma, float lpow,
                                   int flags) {
  if (!out) return fail(AWK_ERR_INVALID, "awk_fluid_kernel_create: null handle pointer");
  *out = nullptr;
  if (!(spx > 0 && spy > 0 && spz > 0)) return fail(AWK_ERR_INVALID, "awk_fluid_kernel_create: spacing must be > 0");
  awk_fluid_kernel *h = new (std::nothrow) awk_fluid_kernel();
  if (!h) return fail(AWK_ERR_ALLOC, "awk_fluid_kernel_create: host allocation failed");
  const float sp[3] = {spx, spy, spz};
  awk_status st = fk_init(h->k, nx, ny, nz, sp);
  if (st) {
    fk_release(h->k);
    delete h;
    return st;
  }
  h->k.alpha = alpha;
  h->k.beta = beta;
  h->k.gamma = gamma;
  h->k.lpow = lpow;
  h->k.flags = flags;
  *out = h;
  return AWK_OK;
}

awk_status awk_fluid_kernel_set_params(awk_fk_t h, float alpha, float beta, float gamma, float lpow,
                                       int flags) {
  if (!h) return fail(AWK_ERR_INVALID, "awk_fluid_kernel_set_params: null handle");
  FluidKernel &k = h->k;
  if (alpha != k.alpha || beta != k.beta || gamma != k.gamma || lpow != k.lpow) k.eig_dir = 0;
  k.alpha = alpha;
  k.beta = beta;
  k.gamma = gamma;
  k.lpow = lpow;
  k.flags = flags;
  return AWK_OK;
}

awk_status awk_fluid_kernel_destroy(awk_fk_t h) {
  if (!h) return AWK_OK;
  fk_release(h->k);
  delete h;
  return AWK_OK;
}

awk_status awk_fluid_kernel_scratch_bytes(awk_fk_t h, unsigned long long *bytes) {
  if (!h || !bytes) return fail(AWK_ERR_INVALID, "awk_fluid_kernel_scratch_bytes: null argument");
  *bytes = h->k.scratch_bytes;
  return AWK_OK;
}

awk_status awk_fluid_kernel_apply(awk_fk_t h, float *x, float *y, float *z, int inverse,
                                  awk_stream_t stream) {
  if (!h || !x || !y || !z) return fail(AWK_ERR_INVALID, "awk_fluid_kernel_apply: null argument");
  FluidKernel &k = h->k;
  hipStream_t s = as_stream(stream);
  XFwdArgs fa;
  std::memset(&fa, 0, sizeof(fa));
  fa.mode = XLOAD_PLAIN;
  fa.in[0] = x;
  fa.in[1] = y;
  fa.in[2] = z;
  awk_status st;
  if ((st = fk_xfwd(k, fa, s, nullptr))) return st;
  if ((st = fk_ypass(k, false, s, nullptr))) return st;
  if ((st = fk_zsolve(k, inverse != 0, s))) return st;
  if ((st = fk_ypass(k, true, s, nullptr))) return st;
  XInvArgs ia;
  std::memset(&ia, 0, sizeof(ia));
  ia.mode = XSTORE_PLAIN;
  ia.out[0] = x;
  ia.out[1] = y;
  ia.out[2] = z;
  return fk_xinv(k, ia, s, nullptr);
}

}  // extern "C"
