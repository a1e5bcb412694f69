// awk_fluid_x.h -- the x passes of the FluidKernelFFT operator (forward r2c with the
// force prologue, inverse c2r with the update epilogues), shared by the launchers of
// the specialised lengths (awk_fluid.hip) and of any length (awk_fluid_any.hip).
#pragma once

#include "awk_fluid.h"

namespace awk {

// X forward: r2c of RT spatial rows (3 components each) per block.
// Complex line layout per row pair (q = 2p, 2p+1):
//   line 3p   = (c0[2p],   c1[2p])
//   line 3p+1 = (c2[2p],   c2[2p+1])
//   line 3p+2 = (c0[2p+1], c1[2p+1])
__device__ __forceinline__ void line_targets(int line, int r0, int &rowA, int &cA, int &rowB,
                                             int &cB) {
  const int p = line / 3, e = line - 3 * p;
  const int ra = r0 + 2 * p;
  if (e == 0) { rowA = ra; cA = 0; rowB = ra; cB = 1; }
  else if (e == 1) { rowA = ra; cA = 2; rowB = ra + 1; cB = 2; }
  else { rowA = ra + 1; cA = 0; rowB = ra + 1; cB = 1; }
}

// Batched launches: subject blockIdx.y's reduction arguments.
__device__ __forceinline__ void batch_reduce(ReduceArgs &ra, const Batch &bt) {
  const long long sb = blockIdx.y;
  ra.partials += sb * bt.part;
  if (bt.scalar) {
    if (ra.energy_out) ra.energy_out += sb;
    ra.prev += sb;
    ra.have_prev += sb;
    ra.step += sb;
  }
}

// Energy bookkeeping of one greedy iteration, run by logical block 0 of the
// forward y pass (the kernel boundary after the x pass makes every partial
// visible): fixed-order FP64 sum of the x-pass block partials, then
// GreedyDeformationData::AddEnergy (GreedyDeformationData.cxx:162-184).
__device__ __forceinline__ void energy_block(const ReduceArgs &ra, double *tree, int bdim) {
  double acc = 0.0;
  acc = strided_fold(ra.partials, ra.n, (int)threadIdx.x, bdim, acc, FoldAdd());
  tree[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 512; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w && (int)threadIdx.x + w < bdim) tree[threadIdx.x] += tree[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const double e = ra.scale * tree[0];
    if (ra.energy_out) *ra.energy_out = e;
    const bool have = *ra.have_prev != 0;
    const double change = have ? e - *ra.prev : 0.0;
    unsigned f = 0;
    if (e != e || change != change) f |= AWK_FLAG_NAN_ENERGY;
    if (change > 0.0) f |= AWK_FLAG_ENERGY_INCREASE;
    raise_flags(ra.flags, f);
    if (ra.auto_reduce && change > 0.0) *ra.step = *ra.step * 0.5f;
    *ra.prev = e;
    *ra.have_prev = 1;
  }
}


// Force multiplier of the GRADMUL modes: the image i1, or an int64 fixed-point
// splat accumulator (2^-32 units), which is cleared as it is read (every voxel is
// read by exactly one thread of the x pass).  The image is read once per
// iteration: a non-temporal load, so that it does not displace in the memory-side
// cache the spectrum this pass writes and the y pass reads next.
__device__ __forceinline__ float load_mul(const XFwdArgs &a, size_t i) {
  if (a.mode == XLOAD_GRADMUL_FX) {
    const long long q = a.acc[i];
    a.acc[i] = 0;
    return splat_unq(q);
  }
  return __builtin_nontemporal_load(a.i1 + i);
}

// Column mode of the force: this thread owns column x of CR of the block's rows, q0 ..
// q0 + CR - 1, which are consecutive y at one z (yb: the block's first).  Each Idef
// value is loaded once: the column with a one-row halo in y, the two neighbouring z
// rows, and x +- 1 from the neighbouring lanes (a load only at the wave edges).  Idef
// and I1 are loaded non-temporally (the halo rows other blocks re-read come from L2):
// with the apply's hfield loads and the composition's hfield stores also streamed,
// the memory-side cache keeps this pass's spectrum for the y pass (256^3 greedy
// iteration: y pass 89 -> 78 us, whole iteration +4 %, measured).
template <int CR, class Put>
__device__ __forceinline__ void column_force(const XFwdArgs &a, int nx, int ny, int nz, int z, int yb, int q0,
                                             int x, Put put, double &ssd) {
  const int y0 = yb + q0;
  const size_t sxy = (size_t)nx * ny;
  const float *col0 = a.idef + (size_t)z * sxy + (size_t)y0 * nx + x;
  float col[CR + 2], zm[CR], zp[CR], i1v[CR], lft[CR], rgt[CR];
#pragma unroll
  for (int k = 0; k < CR + 2; ++k) {
    const int yy = y0 - 1 + k;
    col[k] = (yy >= 0 && yy < ny) ? __builtin_nontemporal_load(col0 + (ptrdiff_t)(k - 1) * nx) : 0.f;
  }
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int q = 0; q < CR; ++q) {
    zm[q] = (z > 0) ? __builtin_nontemporal_load(col0 + (ptrdiff_t)q * nx - (ptrdiff_t)sxy) : 0.f;
    zp[q] = (z < nz - 1) ? __builtin_nontemporal_load(col0 + (ptrdiff_t)q * nx + (ptrdiff_t)sxy) : 0.f;
    i1v[q] = load_mul(a, (size_t)z * sxy + (size_t)(y0 + q) * nx + x);
    lft[q] = (lane == 0 && x > 0) ? col0[(ptrdiff_t)q * nx - 1] : 0.f;
    rgt[q] = (lane == 63 && x < nx - 1) ? col0[(ptrdiff_t)q * nx + 1] : 0.f;
  }
#pragma unroll
  for (int q = 0; q < CR; ++q) {
    const float c = col[q + 1];
    const float up = __shfl_up(c, 1, 64), dn = __shfl_down(c, 1, 64);
    const float cl = (lane == 0) ? lft[q] : up;   // value at x - 1
    const float cr = (lane == 63) ? rgt[q] : dn;  // value at x + 1
    const int y = y0 + q;
    // Array3DUtils::computeGradient (Array3DUtils.txx:783-901), wrap = false
    float gx, gy, gz;
    if (nx == 1) gx = 0.f;
    else if (x > 0 && x < nx - 1) gx = div_const((cr - cl), 2.f * a.sp[0], a.r2sp[0]);
    else if (x == 0) gx = div_const((cr - c), a.sp[0], a.rsp[0]);
    else gx = div_const((c - cl), a.sp[0], a.rsp[0]);
    if (ny == 1) gy = 0.f;
    else if (y > 0 && y < ny - 1) gy = div_const((col[q + 2] - col[q]), 2.f * a.sp[1], a.r2sp[1]);
    else if (y == 0) gy = div_const((col[q + 2] - c), a.sp[1], a.rsp[1]);
    else gy = div_const((c - col[q]), a.sp[1], a.rsp[1]);
    if (nz == 1) gz = 0.f;
    else if (z > 0 && z < nz - 1) gz = div_const((zp[q] - zm[q]), 2.f * a.sp[2], a.r2sp[2]);
    else if (z == 0) gz = div_const((zp[q] - c), a.sp[2], a.rsp[2]);
    else gz = div_const((c - zm[q]), a.sp[2], a.rsp[2]);
    const float r = (a.mode == XLOAD_FORCE) ? i1v[q] - c : i1v[q];
    ssd += (double)r * (double)r;
    put(q0 + q, x, gx * r, gy * r, gz * r);
  }
}

// Which transform an x pass runs: the LDS stages; the dense product (awk_dense.h),
// whose lines are the rows' components as real lines [x][kDenseLS]; or two radices
// (awk_radix.h) of up to 16 or 32, a thread per butterfly of the 12 complex lines.
enum XEngine { XENG_STAGES = 0, XENG_DENSE = 1, XENG_RADIX16 = 2, XENG_RADIX32 = 3 };
constexpr int x_threads(int eng, int bdc) {
  return eng == XENG_DENSE || eng == XENG_RADIX32 ? 512 : eng == XENG_RADIX16 ? 256 : bdc ? bdc : 1024;
}
constexpr int kDenseLS = 33;   // floats per staged x (an odd stride: no bank conflicts along x)
constexpr int kDenseRows = 10; // rows per dense x block: 30 of the product's 32 lines

// w / n for 0 <= w < 2^16 and a launch constant n < 2^16: m = ceil(2^32 / n) (0: n = 1).
__device__ __forceinline__ int div_small(int w, unsigned m) {
  return m ? (int)__umulhi((unsigned)w, m) : w;
}

// The 12 lines of an x block (row stride LS) through two radices in LDS.
template <int MAXR, int NL, int LS>
__device__ __forceinline__ void radix_lds(float2 *sm, const RadixAxis &ax, bool inv) {
  const int line = threadIdx.x % NL, j = threadIdx.x / NL, RA = ax.ra, RB = ax.rb;
  with_radix<MAXR>(RA, [&](auto rad) {
    constexpr int R = decltype(rad)::value;
    float2 v[R];
    if (j < RB) {
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = sm[(j + r * RB) * LS + line];
      dft_any<R>(v, inv);
    }
    __syncthreads();
    if (j < RB) {
#pragma unroll
      for (int r = 0; r < R; ++r) sm[(j * R + r) * LS + line] = v[r];
    }
  });
  __syncthreads();
  with_radix<MAXR>(RB, [&](auto rad) {
    constexpr int R = decltype(rad)::value;
    if (j < RA) {
      float2 v[R];
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = sm[(j + r * RA) * LS + line];
      radix_twiddle<R>(v, ax.tw, j, inv);
      dft_any<R>(v, inv);
#pragma unroll
      for (int r = 0; r < R; ++r) sm[(j + r * RA) * LS + line] = v[r];
    }
  });
  __syncthreads();
}

// NC, RTC, BDC: compile-time length, rows per block and block size (0 = runtime).
template <int NC, int RTC, int BDC, int ENG = XENG_STAGES>
__global__ void __launch_bounds__(x_threads(ENG, BDC))
k_xfwd(XFwdArgs a, Axis ax, XPlan xp, int nx_rt, int ny, int nz, int nxh_rt, int nxh_pad, int RT_rt,
       float2 *__restrict__ spec, size_t plane, Batch bt) {
  extern __shared__ float2 sm[];
  __shared__ double red[16];
  {  // subject blockIdx.y of a batched launch
    const long long sb = blockIdx.y;
    spec += sb * bt.spec;
    if (a.idef) a.idef += sb * bt.img;
    if (a.partials) a.partials += sb * bt.part;
  }
  const int nx = NC ? NC : nx_rt, nxh = NC ? NC / 2 + 1 : nxh_rt, RT = RTC ? RTC : RT_rt;
  const int bdim = BDC ? BDC : (int)blockDim.x;
  const int NL = 3 * RT / 2, LS = NL + 1;
  const int NR = ny * nz;
  const int lb = (int)xcd_block();
  const int g = band_block(lb, a.band, ny / RT);  // the row group (its SSD partial's index)
  const int r0 = g * RT;
  if (r0 >= NR) return;
  // y and z of the block's row q: from the first row's, without a division per voxel
  const int zb = r0 / ny, yb0 = r0 - zb * ny;
  auto row_yz = [&](int q, int &y, int &z) {
    if constexpr (NC != 0) {
      y = (r0 + q) % ny;
      z = (r0 + q) / ny;
      return;
    }
    y = yb0 + q;
    z = zb;
    while (y >= ny) {
      y -= ny;
      ++z;
    }
  };
  double ssd = 0.0;
  float *smf = reinterpret_cast<float *>(sm);
  auto put = [&](int q, int x, float f0, float f1, float f2) {
    if constexpr (ENG == XENG_DENSE) {
      float *o = smf + x * kDenseLS + 3 * q;
      o[0] = f0;
      o[1] = f1;
      o[2] = f2;
      return;
    }
    const int p = q >> 1;
    if ((q & 1) == 0) {
      sm[x * LS + 3 * p] = make_float2(f0, f1);
      smf[2 * (x * LS + 3 * p + 1)] = f2;
    } else {
      sm[x * LS + 3 * p + 2] = make_float2(f0, f1);
      smf[2 * (x * LS + 3 * p + 1) + 1] = f2;
    }
  };
  bool done = false;
  if constexpr (NC != 0 && NC == BDC) {
    if (a.mode != XLOAD_PLAIN && ny % RTC == 0) {
      done = true;
      column_force<RTC>(a, NC, ny, nz, zb, yb0, 0, (int)threadIdx.x, put, ssd);
    }
  } else if constexpr (ENG != XENG_STAGES) {
    // the same for any length where the block's rows lie in one plane and its threads
    // cover a row: 256 threads take rows of up to 128 in two halves of the block's
    // rows, up to 64 (and an even half) in four quarters
    constexpr int RC = ENG == XENG_DENSE ? kDenseRows : 8;
    if (a.mode != XLOAD_PLAIN && nx <= bdim && yb0 + RC <= ny) {
      done = true;
      if (nx <= 64 && RC % 4 == 0) {
        const int h = threadIdx.x >> 6, x = threadIdx.x & 63;
        if (x < nx && h < 4) column_force<(RC + 3) / 4>(a, nx, ny, nz, zb, yb0, h * (RC / 4), x, put, ssd);
      } else if (nx <= 128) {
        const int h = threadIdx.x >> 7, x = threadIdx.x & 127;
        if (x < nx && h < 2) column_force<RC / 2>(a, nx, ny, nz, zb, yb0, h * (RC / 2), x, put, ssd);
      } else if ((int)threadIdx.x < nx) {
        column_force<RC>(a, nx, ny, nz, zb, yb0, 0, (int)threadIdx.x, put, ssd);
      }
    }
  }
  if (!done) {
#pragma unroll
  for (int w = threadIdx.x; w < RT * nx; w += bdim) {
    const int q = NC ? w / nx : div_small(w, xp.mn), x = w - q * nx;
    const int row = r0 + q;
    float f0 = 0.f, f1 = 0.f, f2 = 0.f;
    if (row < NR) {
      const size_t base = (size_t)row * nx + x;
      if (a.mode == XLOAD_PLAIN) {
        f0 = a.in[0][base];
        f1 = a.in[1][base];
        f2 = a.in[2][base];
      } else {
        // gradient of the deformed image (Array3DUtils::computeGradient, wrap=false,
        // Array3DUtils.txx:783-901), residual r = I1 - Idef and force r*grad
        // (GreedyIteratorCPU.cxx:108-117).
        int y, z;
        row_yz(q, y, z);
        const float *I = a.idef;
        const float c = I[base];
        float gx = 0.f, gy = 0.f, gz = 0.f;
        if (nx > 1) {
          if (x > 0 && x < nx - 1) gx = div_const((I[base + 1] - I[base - 1]), 2.f * a.sp[0], a.r2sp[0]);
          else if (x == 0) gx = div_const((I[base + 1] - c), a.sp[0], a.rsp[0]);
          else gx = div_const((c - I[base - 1]), a.sp[0], a.rsp[0]);
        }
        if (ny > 1) {
          if (y > 0 && y < ny - 1) gy = div_const((I[base + nx] - I[base - nx]), 2.f * a.sp[1], a.r2sp[1]);
          else if (y == 0) gy = div_const((I[base + nx] - c), a.sp[1], a.rsp[1]);
          else gy = div_const((c - I[base - nx]), a.sp[1], a.rsp[1]);
        }
        if (nz > 1) {
          const size_t s = (size_t)nx * ny;
          if (z > 0 && z < nz - 1) gz = div_const((I[base + s] - I[base - s]), 2.f * a.sp[2], a.r2sp[2]);
          else if (z == 0) gz = div_const((I[base + s] - c), a.sp[2], a.rsp[2]);
          else gz = div_const((c - I[base - s]), a.sp[2], a.rsp[2]);
        }
        const float m = load_mul(a, base);
        const float r = (a.mode == XLOAD_FORCE) ? m - c : m;
        ssd += (double)r * (double)r;
        f0 = gx * r;
        f1 = gy * r;
        f2 = gz * r;
      }
    }
    put(q, x, f0, f1, f2);
  }
  }
  if constexpr (ENG == XENG_DENSE) {
    for (int w = threadIdx.x; w < kDenseLS; w += bdim) smf[nx * kDenseLS + w] = 0.f;
    __syncthreads();
    const int lane = threadIdx.x & 63, hi = lane >> 5, col = lane & 31;
    const int tile = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    if (tile < xp.dense.tiles) {
      v16f E, O;
      dense_tile<true, true>(smf + hi * kDenseLS + col, smf + (nx - hi) * kDenseLS + col, 2 * kDenseLS,
                             -2 * kDenseLS, xp.dense, tile, lane, E, O);
      const int k = 32 * tile + col;
      if (k < nxh) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int line = dense_row(i, lane), q = line / 3, c = line - 3 * q;
          if (line < 3 * kDenseRows && r0 + q < NR)
            spec[c * plane + (size_t)(r0 + q) * nxh_pad + k] = make_float2(E[i], -O[i]);
        }
      }
    }
  } else {
  __syncthreads();
  if constexpr (ENG == XENG_RADIX16 || ENG == XENG_RADIX32)
    radix_lds<ENG == XENG_RADIX16 ? 16 : 32, 3 * RTC / 2, 3 * RTC / 2 + 1>(sm, xp.radix, false);
  else if constexpr (NC != 0) ct_fft<NC, 3 * RTC / 2, 3 * RTC / 2 + 1, BDC>(sm, ax.tw, false);
  else lds_fft(sm, ax, NL, LS, false, sm + (size_t)nx * LS);
#pragma unroll
  for (int w = threadIdx.x; w < NL * nxh; w += bdim) {
    const int line = NC ? w / nxh : div_small(w, xp.mh), k = w - line * nxh;
    const float2 Z = sm[k * LS + line];
    const float2 Zc = cconj(sm[(k ? nx - k : 0) * LS + line]);
    const float2 A = cscale(cadd(Z, Zc), 0.5f);
    const float2 d = cscale(csub(Z, Zc), 0.5f);
    const float2 B = make_float2(d.y, -d.x);
    int rowA, cA, rowB, cB;
    line_targets(line, r0, rowA, cA, rowB, cB);
    if (rowA < NR) spec[cA * plane + (size_t)rowA * nxh_pad + k] = A;
    if (rowB < NR) spec[cB * plane + (size_t)rowB * nxh_pad + k] = B;
  }
  }
  if (a.mode == XLOAD_FORCE && a.partials) {
    // deterministic block reduction of the FP64 SSD partial
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) ssd += __shfl_down(ssd, off, 64);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) red[wave] = ssd;
    __syncthreads();
    if (threadIdx.x == 0) {
      double s = 0.0;
      const int nw = (bdim + 63) >> 6;
      for (int i = 0; i < nw; ++i) s += red[i];
      a.partials[g] = s;
    }
  }
}

// X inverse: c2r of RT rows (3 components) with an epilogue.  APPLY (COMPOSE
// only): the epilogue also samples I0 at the new field (a.i0 -> a.idef), the next
// iteration's deformed image.  STG (COMPOSE only; NC, RTC, BDC set, ny % RTC == 0):
// the composition reads the current field from the block's rows and their
// neighbours staged in LDS.
template <int NC, int RTC, int BDC, int XU, bool PAIRS = false, bool APPLY = false, bool STG = false,
          int ENG = XENG_STAGES>
__global__ void __launch_bounds__(x_threads(ENG, BDC))
k_xinv(XInvArgs a, Axis ax, XPlan xp, int nx_rt, int ny, int nz, int nxh_rt, int nxh_pad, int RT_rt,
       const float2 *__restrict__ spec, size_t plane, Batch bt) {
  extern __shared__ float2 sm[];
  __shared__ float redf[16];
  {  // subject blockIdx.y of a batched launch
    const long long sb = blockIdx.y;
    spec += sb * bt.spec;
    for (int c = 0; c < 3; ++c) {
      if (a.h[c]) a.h[c] += sb * bt.field;
      if (a.hnew[c]) a.hnew[c] += sb * bt.field;
      if (a.out[c]) a.out[c] += sb * bt.field;
    }
    if (bt.scalar) a.step += sb;
    if (a.maxpart) a.maxpart += sb * (long long)gridDim.x;
  }
  const int nx = NC ? NC : nx_rt, nxh = NC ? NC / 2 + 1 : nxh_rt, RT = RTC ? RTC : RT_rt;
  const int bdim = BDC ? BDC : (int)blockDim.x;
  const int NL = 3 * RT / 2, LS = NL + 1;
  const int NR = ny * nz;
  const int lb = (int)xcd_block();
  const int g = band_block(lb, a.band, ny / RT);  // the row group
  const int r0 = g * RT;
  if (r0 >= NR) {
    // a padding block of the grid: its max partial is still read
    if ((a.mode == XSTORE_MAXNORM || a.mode == XSTORE_MAXAXPY) && threadIdx.x == 0) a.maxpart[lb] = 0.f;
    if (a.mode == XSTORE_DOT && threadIdx.x == 0) a.dotpart[lb] = 0.0;
    return;
  }
  float *smf = reinterpret_cast<float *>(sm);
  if constexpr (ENG == XENG_DENSE) {
    // x_j = sum_k w_k (cos Re X_k - sin Im X_k), w_0 = 1, else 2 (the table halves
    // the middle frequency of an even length): the parts of 30 real lines staged as
    // [k][kDenseLS], real then imaginary, rows nxh .. 2 ks - 1 zero
    const int KR = 2 * xp.dense.ks;
    float *im = smf + KR * kDenseLS;
    const int lane = threadIdx.x & 63, hi = lane >> 5, col = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), nw = bdim >> 6;
    for (int line = wave; line < 3 * kDenseRows; line += nw) {
      const int q = line / 3, c = line - 3 * q;
      const float2 *src = spec + c * plane + (size_t)(r0 + q) * nxh_pad;
      const bool ok = r0 + q < NR;
      for (int k = lane; k < KR; k += 64) {
        float2 X = (ok && k < nxh) ? src[k] : make_float2(0.f, 0.f);
        const float w = k ? 2.f : 1.f;
        // the imaginary part c2r ignores
        smf[k * kDenseLS + line] = w * X.x;
        im[k * kDenseLS + line] = (k == 0 || 2 * k == nx) ? 0.f : w * X.y;
      }
    }
    __syncthreads();
    v16f P, Q;
    if (wave < xp.dense.tiles)
      dense_tile<true, false>(smf + hi * kDenseLS + col, im + hi * kDenseLS + col, 2 * kDenseLS,
                              2 * kDenseLS, xp.dense, wave, lane, P, Q);
    __syncthreads();  // the staged frequencies are read: the lines take their place
    const int j = 32 * wave + col;
    if (wave < xp.dense.tiles && j < xp.dense.H) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int line = dense_row(i, lane);
        smf[j * kDenseLS + line] = P[i] - Q[i];
        if (j > 0 && 2 * j != nx) smf[(nx - j) * kDenseLS + line] = P[i] + Q[i];
      }
    }
    __syncthreads();
  } else {
#pragma unroll
  for (int w = threadIdx.x; w < NL * nxh; w += bdim) {
    const int line = NC ? w / nxh : div_small(w, xp.mh), k = w - line * nxh;
    int rowA, cA, rowB, cB;
    line_targets(line, r0, rowA, cA, rowB, cB);
    float2 A = rowA < NR ? spec[cA * plane + (size_t)rowA * nxh_pad + k] : make_float2(0.f, 0.f);
    float2 B = rowB < NR ? spec[cB * plane + (size_t)rowB * nxh_pad + k] : make_float2(0.f, 0.f);
    if (k == 0 || 2 * k == nx) {  // the imaginary part c2r ignores
      A.y = 0.f;
      B.y = 0.f;
    }
    sm[k * LS + line] = make_float2(A.x - B.y, A.y + B.x);               // A + iB
    if (k > 0 && nx - k >= nxh) sm[(nx - k) * LS + line] = make_float2(A.x + B.y, B.x - A.y);  // conj(A) + i conj(B)
  }
  __syncthreads();
  if constexpr (ENG == XENG_RADIX16 || ENG == XENG_RADIX32)
    radix_lds<ENG == XENG_RADIX16 ? 16 : 32, 3 * RTC / 2, 3 * RTC / 2 + 1>(sm, xp.radix, true);
  else if constexpr (NC != 0) ct_fft<NC, 3 * RTC / 2, 3 * RTC / 2 + 1, BDC>(sm, ax.tw, true);
  else lds_fft(sm, ax, NL, LS, true, sm + (size_t)nx * LS);
  }
  // the velocity at (q, x) of the block's rows
  auto vel = [&](int q, int x, float &v0, float &v1, float &v2) {
    if constexpr (ENG == XENG_DENSE) {
      const float *o = smf + x * kDenseLS + 3 * q;
      v0 = o[0];
      v1 = o[1];
      v2 = o[2];
      return;
    }
    const int p = q >> 1;
    if ((q & 1) == 0) {
      const float2 t = sm[x * LS + 3 * p];
      v0 = t.x; v1 = t.y; v2 = sm[x * LS + 3 * p + 1].x;
    } else {
      const float2 t = sm[x * LS + 3 * p + 2];
      v0 = t.x; v1 = t.y; v2 = sm[x * LS + 3 * p + 1].y;
    }
  };
  // y and z of the block's row q: from the first row's, without a division per voxel
  const int zb = r0 / ny, yb0 = r0 - zb * ny;
  auto row_yz = [&](int q, int &y, int &z) {
    if constexpr (NC != 0) {
      y = (r0 + q) % ny;
      z = (r0 + q) / ny;
      return;
    }
    y = yb0 + q;
    z = zb;
    while (y >= ny) {
      y -= ny;
      ++z;
    }
  };
  float mx = 0.f;
  double dot = 0.0;
  if (APPLY || STG || a.mode == XSTORE_COMPOSE) {
    // updateDeformation (GreedyIteratorCPU.cxx:81-95): v *= step; h <- composeHV(h, v, sp, PARTIAL_ID).
    // XU voxels per step: their 24*XU gathers are in flight together.
    const float st = *a.step;
    const Dims d{nx, ny, nz};
    // v * step / sp, with the division by the spacing taken as a reciprocal
    // multiply (exact for unit spacing)
    const float isx = 1.f / a.sp[0], isy = 1.f / a.sp[1], isz = 1.f / a.sp[2];
    const int ntot = nx * ny * nz;
    const BufLoad hx = make_buf(a.h[0], ntot), hy = make_buf(a.h[1], ntot), hz = make_buf(a.h[2], ntot);
    if constexpr (STG) {
      // The block's RT rows are y = yb .. yb + RT - 1 of plane zr.  A point whose 8
      // corners lie inside the volume, in rows yb - 1 .. yb + RT of planes zr - 1 ..
      // zr + 1 (the common case: the step moves points by less than a voxel), reads
      // them from those rows staged in LDS, one component at a time; any other
      // point gathers from memory.  The same corners and the same lerp8 as the
      // gathers, so the same results bit for bit.
      constexpr int VP = RTC * NC / BDC;  // voxels per thread
      constexpr int WR = RTC + 2;         // staged rows per plane
      const int zr = r0 / ny, yb = r0 - zr * ny;
      float px[VP], py[VP], pz[VP];
      int win[VP];  // LDS offset of corner c0 in the staged rows (-1: gather from memory)
#pragma unroll
      for (int u = 0; u < VP; ++u) {
        const int w = threadIdx.x + u * BDC;
        const int q = w / NC, x = w - q * NC;
        float v0, v1, v2;
        vel(q, x, v0, v1, v2);
        px[u] = fmaf(v0 * st, isx, (float)x);
        py[u] = fmaf(v1 * st, isy, (float)(yb + q));
        pz[u] = fmaf(v2 * st, isz, (float)zr);
        const int x0 = (int)floorf(px[u]), y0 = (int)floorf(py[u]), z0 = (int)floorf(pz[u]);
        const bool ok = x0 >= 0 && x0 < nx - 1 && y0 >= 0 && y0 < ny - 1 && z0 >= 0 && z0 < nz - 1 &&
                        y0 >= yb - 1 && y0 <= yb + RTC - 1 && z0 >= zr - 1 && z0 <= zr;
        win[u] = ok ? ((z0 - zr + 1) * WR + (y0 - yb + 1)) * NC + x0 : -1;
      }
      __syncthreads();  // every read of the transformed rows is done: sm is reused
      float hc[VP][3];
#pragma unroll
      for (int u = 0; u < VP; ++u)
        if (win[u] < 0) {
          const float3 g = trilerp3g<AWK_BG_PARTIAL_ID, BufLoad, false>(hx, hy, hz, d, px[u], py[u], pz[u]);
          hc[u][0] = g.x; hc[u][1] = g.y; hc[u][2] = g.z;
        }
      float *stg = reinterpret_cast<float *>(sm);
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        if (c) __syncthreads();  // the previous component's reads are done
        // rows outside the volume are not staged: no point in the window reads them
        const float *hs = a.h[c];
        for (int e = threadIdx.x; e < 3 * WR * (NC / 4); e += BDC) {
          const int row = e / (NC / 4), x4 = e - row * (NC / 4);
          const int zz = zr - 1 + row / WR, yy = yb - 1 + row % WR;
          if (zz >= 0 && zz < nz && yy >= 0 && yy < ny)
            *reinterpret_cast<float4 *>(stg + row * NC + 4 * x4) =
                *reinterpret_cast<const float4 *>(hs + ((size_t)zz * ny + yy) * NC + 4 * x4);
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < VP; ++u)
          if (win[u] >= 0) {
            const float *b = stg + win[u];
            const float t = px[u] - floorf(px[u]), uu = py[u] - floorf(py[u]), vv = pz[u] - floorf(pz[u]);
            hc[u][c] = lerp8(b[0], b[1], b[NC + 1], b[NC], b[WR * NC + NC], b[WR * NC + NC + 1],
                             b[WR * NC + 1], b[WR * NC], t, uu, vv);
          }
      }
#pragma unroll
      for (int u = 0; u < VP; ++u) {
        // rows r0 .. r0 + RT - 1 are contiguous in memory
        const size_t base = (size_t)r0 * NC + threadIdx.x + u * BDC;
        __builtin_nontemporal_store(hc[u][0], a.hnew[0] + base);
        __builtin_nontemporal_store(hc[u][1], a.hnew[1] + base);
        __builtin_nontemporal_store(hc[u][2], a.hnew[2] + base);
      }
      if constexpr (APPLY) {
        const BufLoad ib = make_buf(a.i0, ntot);
#pragma unroll
        for (int u = 0; u < VP; ++u) {
          const size_t base = (size_t)r0 * NC + threadIdx.x + u * BDC;
          a.idef[base] = trilerp1g<AWK_BG_VAL>(ib, d, hc[u][0], hc[u][1], hc[u][2], a.i0_bg);
        }
      }
    } else {
#pragma unroll
    for (int w0 = threadIdx.x; w0 < RT * nx; w0 += bdim * XU) {
      float px[XU], py[XU], pz[XU];
      int row_[XU], x_[XU];
#pragma unroll
      for (int u = 0; u < XU; ++u) {
        const int w = w0 + u * bdim;
        const int q = NC ? w / nx : div_small(w, xp.mn), x = w - q * nx;
        row_[u] = (w < RT * nx) ? r0 + q : NR;
        x_[u] = x;
        if (row_[u] < NR) {
          float v0, v1, v2;
          vel(q, x, v0, v1, v2);
          int y, z;
          row_yz(q, y, z);
          // explicit fma: the same rounding wherever the position is formed
          px[u] = fmaf(v0 * st, isx, (float)x);
          py[u] = fmaf(v1 * st, isy, (float)y);
          pz[u] = fmaf(v2 * st, isz, (float)z);
        }
      }
      float3 hn[XU];
#pragma unroll
      for (int u = 0; u < XU; ++u)
        if (row_[u] < NR) hn[u] = trilerp3g<AWK_BG_PARTIAL_ID, decltype(hx), PAIRS>(hx, hy, hz, d, px[u], py[u], pz[u]);
#pragma unroll
      for (int u = 0; u < XU; ++u)
        if (row_[u] < NR) {
          const size_t base = (size_t)row_[u] * nx + x_[u];
          // streamed: the next reader is the next iteration's apply (or, with
          // APPLY, the next iteration's composition gathers)
          __builtin_nontemporal_store(hn[u].x, a.hnew[0] + base);
          __builtin_nontemporal_store(hn[u].y, a.hnew[1] + base);
          __builtin_nontemporal_store(hn[u].z, a.hnew[2] + base);
        }
      if constexpr (APPLY) {
        // the next iteration's deformed image I0(hnew), from the new field still in
        // registers: the same sampling as the apply kernel on the stored field
        const BufLoad ib = make_buf(a.i0, ntot);
        float r[XU];
#pragma unroll
        for (int u = 0; u < XU; ++u)
          if (row_[u] < NR) r[u] = trilerp1g<AWK_BG_VAL>(ib, d, hn[u].x, hn[u].y, hn[u].z, a.i0_bg);
#pragma unroll
        for (int u = 0; u < XU; ++u)
          if (row_[u] < NR) a.idef[(size_t)row_[u] * nx + x_[u]] = r[u];
      }
    }
    }
  } else {
    // LDMM coefficients, in float as the reference forms them
    float cva = 0.f, cua = 0.f;
    if (a.mode == XSTORE_AXPBY) {
      const float st = *a.step;
      cva = 1.f - 2.f * st;
      cua = 2.f * st / a.sigma2;
    } else if (a.mode == XSTORE_MAXAXPY) {
      cua = -2.f / a.sigma2;
    }
#pragma unroll
    for (int w = threadIdx.x; w < RT * nx; w += bdim) {
      const int q = NC ? w / nx : div_small(w, xp.mn), x = w - q * nx;
      const int row = r0 + q;
      if (row >= NR) continue;
      float v0, v1, v2;
      vel(q, x, v0, v1, v2);
      const size_t base = (size_t)row * nx + x;
      if (a.mode == XSTORE_AXPBY) {
        // updateVelocity (LDMMIteratorCPU.cxx:175-190): v = vFac v + uFac u
        a.out[0][base] = cva * a.out[0][base] + cua * v0;
        a.out[1][base] = cva * a.out[1][base] + cua * v1;
        a.out[2][base] = cva * a.out[2][base] + cua * v2;
      } else if (a.mode == XSTORE_MAXAXPY) {
        // calcMaxDisplacement (LDMMIteratorCPU.cxx:192-212): |2 v - 2/sigma^2 u|
        const float q0 = 2.f * a.out[0][base] + cua * v0;
        const float q1 = 2.f * a.out[1][base] + cua * v1;
        const float q2 = 2.f * a.out[2][base] + cua * v2;
        mx = fmaxf(mx, sqrtf(q0 * q0 + q1 * q1 + q2 * q2));
      } else if (a.mode == XSTORE_DOT) {
        dot += (double)v0 * a.out[0][base];
        dot += (double)v1 * a.out[1][base];
        dot += (double)v2 * a.out[2][base];
      } else {
        a.out[0][base] = v0;
        a.out[1][base] = v1;
        a.out[2][base] = v2;
        if (a.mode == XSTORE_MAXNORM) mx = fmaxf(mx, sqrtf(v0 * v0 + v1 * v1 + v2 * v2));
      }
    }
  }
  // these variants only compose: without the other epilogues' code the atlas's
  // iteration is 0.4 % faster
  if constexpr (APPLY || STG) return;
  if (a.mode == XSTORE_DOT) {
    __shared__ double redd[16];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) dot += __shfl_down(dot, off, 64);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) redd[wave] = dot;
    __syncthreads();
    if (threadIdx.x == 0) {
      double t = 0.0;
      const int nw = (bdim + 63) >> 6;
      for (int i = 0; i < nw; ++i) t += redd[i];
      a.dotpart[lb] = t;
    }
  }
  if (a.mode == XSTORE_MAXNORM || a.mode == XSTORE_MAXAXPY) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_down(mx, off, 64));
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) redf[wave] = mx;
    __syncthreads();
    if (threadIdx.x == 0) {
      float m = 0.f;
      const int nw = (bdim + 63) >> 6;
      for (int i = 0; i < nw; ++i) m = fmaxf(m, redf[i]);
      a.maxpart[lb] = m;
    }
  }
}

}  // namespace awk
