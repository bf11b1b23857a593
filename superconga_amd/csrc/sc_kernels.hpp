// sc_kernels.hpp -- HIP kernels of the self-consistency iteration (gfx950).
#pragma once

#include "sc_device.hpp"
#include "sc_view.hpp"

namespace scamd {

// Order parameter and Doppler shift at sites (x, y[i]) of frame k, from the
// extended order parameter and the vector potential on the N0 grid
// (OrderParameter.h:232-269, RiccatiSolver.h:127-176,
// VectorPotential_Kernel.h:21-99, Gauges.h:25-62).
template <int R>
__device__ __forceinline__ void siteFieldRows(const GrainView &v, int k, int x, const int (&y)[R],
                                              double (&dre)[R], double (&dim)[R],
                                              double (&es)[R]) {
  const int N0 = v.N0, N1 = v.N1;
  const size_t n0 = size_t(N0) * N0;
  // (a site with no cell reads the first one: no branch, so that the loads of
  // all rows are in flight together)
  auto cells = [&](double c, double s, RotSample (&r)[R]) {
#pragma unroll
    for (int i = 0; i < R; ++i) {
      r[i] = rotatedCell(x, y[i], N1, N0, c, s);
      r[i].idx = r[i].valid ? r[i].idx : 0;
    }
  };
  RotSample r[R];
  cells(double(global(v.opCos)[k]), double(global(v.opSin)[k]), r);
#pragma unroll
  for (int i = 0; i < R; ++i) dre[i] = dim[i] = es[i] = 0.0;
  for (int c = 0; c < v.Nc; ++c) {
    const double b = global(v.basis)[c * v.Na + k];
    const double *p = v.extDelta + size_t(c) * 2 * n0;
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const double re = bilinear(p, N0, r[i]), im = bilinear(p + n0, N0, r[i]);
      if (r[i].valid) {
        dre[i] += b * re;
        dim[i] += b * im;
      }
    }
  }
  if (v.useField) {
    double ax[R], ay[R];
#pragma unroll
    for (int i = 0; i < R; ++i) ax[i] = ay[i] = 0.0;
    if (v.useInduced) {
      cells(double(global(v.aCos)[k]), double(global(v.aSin)[k]), r);
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const double a0 = bilinear(v.A, N0, r[i]), a1 = bilinear(v.A + n0, N0, r[i]);
        ax[i] = r[i].valid ? a0 * v.lambdaInv2 : 0.0;
        ay[i] = r[i].valid ? a1 * v.lambdaInv2 : 0.0;
      }
    }
    const double off = -0.5 * double(N1 - 1);
    const double c = global(v.saCos)[k], s = global(v.saSin)[k];
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const double px0 = (double(x) + off) * v.h, py0 = (double(y[i]) + off) * v.h;
      const double px = px0 * c - py0 * s, py = px0 * s + py0 * c;
      double ex, ey;
      if (v.gauge == 0) {
        ex = 0.0;
        ey = px * v.fluxDensity;
      } else if (v.gauge == 1) {
        const double f = 0.5 * v.fluxDensity;
        ex = -py * f;
        ey = px * f;
      } else {
        const double r2 = fmax(px * px + py * py, 1e-7);
        const double f = v.fluxDensity * v.area / (2.0 * M_PI * r2);
        ex = -py * f;
        ey = px * f;
      }
      es[i] = double(v.charge) *
              (global(v.vFx)[k] * (ax[i] + ex) + global(v.vFy)[k] * (ay[i] + ey));
    }
  }
}
__device__ __forceinline__ void siteFields(const GrainView &v, int k, int x, int y, double &dre,
                                           double &dim, double &es) {
  const int ys[1] = {y};
  double re[1], im[1], e[1];
  siteFieldRows<1>(v, k, x, ys, re, im, e);
  dre = re[0];
  dim = im[0];
  es = e[0];
}

// The sweep's work counters (sc_view.hpp).
__global__ void resetCounter(int *c) {
  c[0] = 0;
  c[1] = 0;
  c[kAgainCount] = 0;
}

// The site fields a sweep reads, for the tiles of frames [k0, ...): each
// block covers one tile (16 adjacent columns of one frame and the rows a
// sweep may read there), 16 columns x 16 rows per pass, so that the writes
// of a row of the tile are contiguous.  F is planar [3][frames][N1^2] with
// plane stride `plane`; frame k is at (k - k0) * N1^2.
// A thread takes two of its rows at a time: their taps wait for memory together
// (octagon of 930 sites a side, 128 angles: 1.69 ms one by one, 1.42 by two, 1.51
// by four, which spill).
constexpr int kFieldRows = 2;
__device__ __forceinline__ void fieldsTile(const GrainView &v, const int *tl, int k0,
                                           long long plane, double *Fout) {
  const GlobalPtr<const int> tg = global(tl);
  const int k = tg[0], x = tg[1] + int(threadIdx.x & 15), y0 = tg[2], y1 = tg[3];
  const GlobalPtr<double> F = global(Fout);
  const int N1 = v.N1;
  if (x >= N1) return;
  const size_t base = size_t(k - k0) * N1 * N1 + x;
  for (int y = y0 + int(threadIdx.x >> 4); y <= y1; y += 16 * kFieldRows) {
    int ys[kFieldRows];
    double re[kFieldRows], im[kFieldRows], es[kFieldRows];
#pragma unroll
    for (int i = 0; i < kFieldRows; ++i) ys[i] = min(y + 16 * i, y1);
    siteFieldRows<kFieldRows>(v, k, x, ys, re, im, es);
#pragma unroll
    for (int i = 0; i < kFieldRows; ++i) {
      if (y + 16 * i > y1) break;
      const size_t at = base + size_t(ys[i]) * N1;
      F[at] = re[i];
      F[plane + at] = im[i];
      F[2 * plane + at] = es[i];
    }
  }
}
__global__ void fieldsKernel(GrainView v, const int *tiles, int numTiles, int k0,
                             long long plane, double *F) {
  const long long tile = xcdBlock(numTiles);
  if (tile < 0) return;
  fieldsTile(v, tiles + 4 * size_t(tile), k0, plane, F);
}
// The site fields of several grains in one launch (a batch): grain j of the
// job list (view grainOf[j]) owns the blocks [tileStart[j], tileStart[j+1])
// of the numTiles in total, one tile each, every frame of the grain.
__global__ void fieldsBatchKernel(const GrainView *__restrict__ views,
                                  const int *__restrict__ grainOf,
                                  const int *__restrict__ tileStart, int numJobs, int numTiles) {
  const long long b = xcdBlock(numTiles);
  if (b < 0) return;
  int lo = 0, hi = numJobs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (tileStart[mid] <= b) lo = mid;
    else hi = mid - 1;
  }
  const GrainView &v = views[grainOf[lo]];
  // the view's site-field buffer is the grain's own, written here and read
  // by the sweep that follows
  fieldsTile(v, v.fieldTiles + 4 * (b - tileStart[lo]), 0, v.fieldPlane,
             const_cast<double *>(v.fields));
}

// Homogeneous coherence functions at the exit crossings of one direction
// (RiccatiSolverConfined.h:400-468, 673-767): one thread per (crossing,
// energy); crossing i lies in column col[i] = k * N1 + x at row y[i].  For
// gamma the out storage takes gamma, for gamma~ it takes gamma~.
__global__ void initialOutKernel(GrainView v, const int *col, const int *yOf,
                                 long long nOut, int tilde, double *bOut) {
  const long long tid = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  const int Ne = v.Ne;
  if (tid >= nOut * Ne) return;
  const long long i = tid / Ne;
  const int e = int(tid - i * Ne);
  const int c = col[i];
  const int k = c / v.N1, x = c - k * v.N1, y = yOf[i];
  double dre, dim, es;
  siteFields(v, k, x, y, dre, dim, es);
  Cx<double> ga, gt;
  const double ere = v.energyRe ? v.energyRe[e] : 0.0;
  homogeneous(Cx<double>{dre, dim}, Cx<double>{ere + es, v.energy[e]}, ga, gt);
  const Cx<double> b = tilde ? gt : ga;
  bOut[tid] = b.re;
  bOut[nOut * Ne + tid] = b.im;
}

// Extension of values outwards from the boundary
// (geometry/domain_ops.h:11-57): target <- mean of its listed sources, for
// `planes` values per site.  A target index t addresses block t / siteStride
// and site t % siteStride; value q of a site lives at
// base + (block - blockBase) * blockStride + site * siteScale + q * planeStride.
__global__ void extendKernel(double *base, const int *target, const int *offset,
                             const int *source, int numTargets, int planes,
                             long long planeStride, long long siteStride,
                             long long blockStride, long long siteScale,
                             long long blockBase) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= numTargets) return;
  const long long tg = target[t];
  const long long blk = tg / siteStride;
  const long long site = tg - blk * siteStride;
  double *p0 = base + (blk - blockBase) * blockStride;
  const int o0 = offset[t], o1 = offset[t + 1];
  const double inv = double(o1 - o0);
  for (int q = 0; q < planes; ++q) {
    double *p = p0 + q * planeStride;
    double val = 0.0;
    for (int o = o0; o < o1; ++o) {
      const long long s = source[o] - blk * siteStride;
      val = (o == o0) ? p[s * siteScale] : val + p[s * siteScale];
    }
    p[site * siteScale] = val / inv;
  }
}

// The contribution of frame k to the angle sums of reference site (x, y):
// the bilinear back-rotation of the frame's four Green-function planes,
// weighted by the basis functions and the angle weight (gatherKernel and
// gatherRangeKernel share it so that both add the same terms in the same
// order).
__device__ __forceinline__ void gatherAngle(const GrainView &v, int k, int x, int y,
                                            double (&dre)[4], double (&dim)[4], double &jx,
                                            double &jy, double &fe) {
  const int N0 = v.N0, N1 = v.N1, Na = v.Na, Nc = v.Nc;
  const size_t n1 = size_t(N1) * N1;
  const RotSample r = rotatedCell(x, y, N0, N1, double(v.bkCos[k]), double(v.bkSin[k]));
  if (!r.valid) return;
  // four values per site: taps (x, y), (x+1, y), (x, y+1), (x+1, y+1)
  const double2 *Gk = reinterpret_cast<const double2 *>(v.G + size_t(k) * n1 * 4);
  const size_t i00 = size_t(r.idx) * 2, i10 = i00 + 2, i01 = i00 + size_t(N1) * 2,
               i11 = i01 + 2;
  const double2 a00 = Gk[i00], b00 = Gk[i00 + 1];
  const double2 a10 = Gk[i10], b10 = Gk[i10 + 1];
  const double2 a01 = Gk[i01], b01 = Gk[i01 + 1];
  const double2 a11 = Gk[i11], b11 = Gk[i11 + 1];
  double gre, gim, gj, gf;
  {
#pragma clang fp contract(off)
    const double wx0 = 1.0 - r.fx, wx1 = r.fx, wy0 = 1.0 - r.fy, wy1 = r.fy;
    gre = wy0 * (wx0 * a00.x + wx1 * a10.x) + wy1 * (wx0 * a01.x + wx1 * a11.x);
    gim = wy0 * (wx0 * a00.y + wx1 * a10.y) + wy1 * (wx0 * a01.y + wx1 * a11.y);
    gj = wy0 * (wx0 * b00.x + wx1 * b10.x) + wy1 * (wx0 * b01.x + wx1 * b11.x);
    gf = wy0 * (wx0 * b00.y + wx1 * b10.y) + wy1 * (wx0 * b01.y + wx1 * b11.y);
  }
  const double w = v.weight[k];
  for (int c = 0; c < Nc && c < 4; ++c) {
    const double b = v.basis[c * Na + k];
    dre[c] += (gre * b) * w;
    dim[c] += (gim * b) * w;
  }
  jx += (v.vFx[k] * w) * gj;
  jy += (v.vFy[k] * w) * gj;
  fe += w * gf;
}

// The gap equation's, the current's and the free-energy density's final
// scaling of the angle sums of one site.
__device__ __forceinline__ void gatherStore(const GrainView &v, int site,
                                            const double (&dre)[4], const double (&dim)[4],
                                            double jx, double jy, double fe,
                                            const double *coupling, double currentFactor,
                                            double *deltaOut, double *currentOut,
                                            double *energyDensity) {
  const size_t n0 = size_t(v.N0) * v.N0;
  for (int c = 0; c < v.Nc && c < 4; ++c) {
    deltaOut[size_t(c) * 2 * n0 + site] = dre[c] * coupling[c];
    deltaOut[size_t(c) * 2 * n0 + n0 + site] = dim[c] * coupling[c];
  }
  currentOut[site] = jx * currentFactor;
  currentOut[n0 + site] = jy * currentFactor;
  energyDensity[site] = fe;
}

// Back-rotation of the Green functions of every frame to the reference grid
// and the angle integration (ComputeOrderParameter.h:174-262,
// ComputeCurrent.h:142-222, ComputeFreeEnergy.h:260-279), one thread per
// inside site of the reference grain.
__global__ void gatherKernel(GrainView v, const int *sites, int numSites,
                             const double *coupling, double currentFactor,
                             double *deltaOut, double *currentOut,
                             double *energyDensity) {
  const long long blk = xcdBlock((numSites + blockDim.x - 1) / blockDim.x);
  if (blk < 0) return;
  const int t = int(blk * blockDim.x + threadIdx.x);
  if (t >= numSites) return;
  const int N0 = v.N0;
  const int site = sites[t];
  const int x = site % N0, y = site / N0;
  double dre[4] = {0, 0, 0, 0}, dim[4] = {0, 0, 0, 0};
  double jx = 0.0, jy = 0.0, fe = 0.0;
  for (int k = 0; k < v.Na; ++k) gatherAngle(v, k, x, y, dre, dim, jx, jy, fe);
  gatherStore(v, site, dre, dim, jx, jy, fe, coupling, currentFactor, deltaOut, currentOut,
              energyDensity);
}

// The angle sums of frames [k0, k1) added to running sums, one thread per
// inside site: acc holds, per inside site t, Re and Im of every component's
// sum, then jx, jy and the free-energy density (at acc[q * numSites + t]).
// Called for consecutive ranges from k0 = 0 it adds the same terms in the
// same order as gatherKernel.
__global__ void gatherRangeKernel(GrainView v, const int *sites, int numSites, int k0, int k1,
                                  double *acc) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= numSites) return;
  const int N0 = v.N0, Nc = v.Nc;
  const int site = sites[t];
  const int x = site % N0, y = site / N0;
  const size_t ns = size_t(numSites);
  double dre[4] = {0, 0, 0, 0}, dim[4] = {0, 0, 0, 0};
  for (int c = 0; c < Nc && c < 4; ++c) {
    dre[c] = acc[size_t(2 * c) * ns + t];
    dim[c] = acc[size_t(2 * c + 1) * ns + t];
  }
  double jx = acc[size_t(2 * Nc) * ns + t], jy = acc[size_t(2 * Nc + 1) * ns + t];
  double fe = acc[size_t(2 * Nc + 2) * ns + t];
  for (int k = k0; k < k1; ++k) gatherAngle(v, k, x, y, dre, dim, jx, jy, fe);
  for (int c = 0; c < Nc && c < 4; ++c) {
    acc[size_t(2 * c) * ns + t] = dre[c];
    acc[size_t(2 * c + 1) * ns + t] = dim[c];
  }
  acc[size_t(2 * Nc) * ns + t] = jx;
  acc[size_t(2 * Nc + 1) * ns + t] = jy;
  acc[size_t(2 * Nc + 2) * ns + t] = fe;
}

// The final scaling of the running sums of gatherRangeKernel.
__global__ void gatherFinishKernel(GrainView v, const int *sites, int numSites,
                                   const double *acc, const double *coupling,
                                   double currentFactor, double *deltaOut, double *currentOut,
                                   double *energyDensity) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= numSites) return;
  const int Nc = v.Nc;
  const size_t ns = size_t(numSites);
  double dre[4] = {0, 0, 0, 0}, dim[4] = {0, 0, 0, 0};
  for (int c = 0; c < Nc && c < 4; ++c) {
    dre[c] = acc[size_t(2 * c) * ns + t];
    dim[c] = acc[size_t(2 * c + 1) * ns + t];
  }
  gatherStore(v, sites[t], dre, dim, acc[size_t(2 * Nc) * ns + t],
              acc[size_t(2 * Nc + 1) * ns + t], acc[size_t(2 * Nc + 2) * ns + t], coupling,
              currentFactor, deltaOut, currentOut, energyDensity);
}

// Specular boundary condition as a precomputed stencil per entry crossing
// (BoundaryConditionSpecular.h:108-358), one thread per (crossing, energy).
// The previous in-values feed the residual statistics
// (ComputeResidual.h:54-106): per block sums of |d|, |old|, d^2, old^2 and
// maxima of |d|, |old|.
__global__ void boundaryKernel(double *bin, const double *bout, long long nIn,
                               long long nOut, int Ne, const int *offset,
                               const int *src, const double *w,
                               const double *wsum, double *partials) {
  const long long tid = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  double s[6] = {0, 0, 0, 0, 0, 0};
  const long long total = nIn * Ne;
  if (tid < total) {
    const long long i = tid / Ne;
    const int e = int(tid - i * Ne);
    double re = 0.0, im = 0.0;
    for (int o = offset[i]; o < offset[i + 1]; ++o) {
      const size_t si = size_t(src[o]) * Ne + e;
      re += bout[si] * w[o];
      im += bout[size_t(nOut) * Ne + si] * w[o];
    }
    const double ws = wsum[i];
    const double nre = ws > 0.0 ? re / ws : 0.0;
    const double nim = ws > 0.0 ? im / ws : 0.0;
    const double ore = bin[tid], oim = bin[total + tid];
    bin[tid] = nre;
    bin[total + tid] = nim;
    const double d1 = ore - nre, d2 = oim - nim;
    s[0] = fabs(d1) + fabs(d2);
    s[1] = fabs(ore) + fabs(oim);
    s[2] = d1 * d1 + d2 * d2;
    s[3] = ore * ore + oim * oim;
    s[4] = fmax(fabs(d1), fabs(d2));
    s[5] = fmax(fabs(ore), fabs(oim));
  }
  __shared__ double sh[6][256];
  for (int q = 0; q < 6; ++q) sh[q][threadIdx.x] = s[q];
  __syncthreads();
  for (int m = blockDim.x / 2; m > 0; m >>= 1) {
    if (threadIdx.x < m)
      for (int q = 0; q < 6; ++q)
        sh[q][threadIdx.x] = q < 4 ? sh[q][threadIdx.x] + sh[q][threadIdx.x + m]
                                   : fmax(sh[q][threadIdx.x], sh[q][threadIdx.x + m]);
    __syncthreads();
  }
  if (threadIdx.x == 0)
    for (int q = 0; q < 6; ++q) partials[size_t(blockIdx.x) * 6 + q] = sh[q][0];
}

// Residual statistics of old/new arrays (ComputeResidual.h:54-106), same six
// per-block quantities as boundaryKernel.
__global__ void statsKernel(const double *oldv, const double *newv, long long n,
                            double *partials) {
  double s[6] = {0, 0, 0, 0, 0, 0};
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const double o = oldv[i];
    const double d = o - (newv ? newv[i] : 0.0);
    s[0] += fabs(d);
    s[1] += fabs(o);
    s[2] += d * d;
    s[3] += o * o;
    s[4] = fmax(s[4], fabs(d));
    s[5] = fmax(s[5], fabs(o));
  }
  __shared__ double sh[6][256];
  for (int q = 0; q < 6; ++q) sh[q][threadIdx.x] = s[q];
  __syncthreads();
  for (int m = blockDim.x / 2; m > 0; m >>= 1) {
    if (threadIdx.x < m)
      for (int q = 0; q < 6; ++q)
        sh[q][threadIdx.x] = q < 4 ? sh[q][threadIdx.x] + sh[q][threadIdx.x + m]
                                   : fmax(sh[q][threadIdx.x], sh[q][threadIdx.x + m]);
    __syncthreads();
  }
  if (threadIdx.x == 0)
    for (int q = 0; q < 6; ++q) partials[size_t(blockIdx.x) * 6 + q] = sh[q][0];
}

// Generic block sums: partial[b] = sum_i f(i) with f selected by `op`:
// 0: a[i]; 1: a[i]*b[i]; 2: a[i]^2 masked by mask[i] (mask may be null).
__global__ void sumKernel(const double *a, const double *b, const uint8_t *mask,
                          long long n, int op, double *partials) {
  double s = 0.0;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    if (mask && !mask[i]) continue;
    const double x = a[i];
    s += op == 0 ? x : (op == 1 ? x * b[i] : x * x);
  }
  __shared__ double sh[256];
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int m = blockDim.x / 2; m > 0; m >>= 1) {
    if (threadIdx.x < m) sh[threadIdx.x] += sh[threadIdx.x + m];
    __syncthreads();
  }
  if (threadIdx.x == 0) partials[blockIdx.x] = sh[0];
}

// B = dAy/dx - dAx/dy with one-sided differences at the edges
// (GridFunctions_GPU.h:326-353); writes B^2.
__global__ void curlSquareKernel(const double *A, int N, double invH, double *out) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= N * N) return;
  const int x = t % N, y = t / N;
  const size_t n = size_t(N) * N;
  const int xn = min(x + 1, N - 1), xp = max(x - 1, 0);
  const int yn = min(y + 1, N - 1), yp = max(y - 1, 0);
  const double dAy = (A[n + size_t(y) * N + xn] - A[n + size_t(y) * N + xp]) / double(xn - xp);
  const double dAx = (A[size_t(yn) * N + x] - A[size_t(yp) * N + x]) / double(yn - yp);
  const double b = (dAy - dAx) * invH;
  out[t] = b * b;
}

// ---------------- elementwise kernels of the accelerators ----------------
// x += (g - x) * s  (Picard.h:133-138)
__global__ void picardKernel(double *x, const double *g, long long n, double s) {
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i < n) x[i] += (g[i] - x[i]) * s;
}
// d = g - x
__global__ void diffKernel(double *d, const double *g, const double *x, long long n) {
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i < n) d[i] = g[i] - x[i];
}
// x = sum_i (X_i + D_i s) w_i over the history (Anderson.h:336-355)
// x = sum_q w_q (X_q + s D_q) (Anderson.h:329-352); the history pointers and
// weights travel in the kernel arguments.
constexpr int kMaxHistory = 16;
struct AndersonTerms {
  const double *X[kMaxHistory];
  const double *D[kMaxHistory];
  double w[kMaxHistory];
};
__global__ void andersonCombine(double *x, AndersonTerms t, int m, long long n, double s) {
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= n) return;
  double acc = 0.0;
  for (int q = 0; q < m; ++q) acc += (t.X[q][i] + t.D[q][i] * s) * t.w[q];
  x[i] = acc;
}
// running mean and step per field (CongAcc.h:271-297); the per-field step
// and inertia travel by value (at most 4 order-parameter components and the
// vector potential: 10 fields)
constexpr int kMaxFields = 16;
struct FieldCoefficients {
  double step[kMaxFields];
  double inertia[kMaxFields];
};
__global__ void congaccKernel(double *x, double *mean, const double *d, FieldCoefficients c,
                              long long fieldSize, long long n) {
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int f = int(i / fieldSize);
  const double m = mean[i] * c.inertia[f] + d[i] * (1.0 - c.inertia[f]);
  mean[i] = m;
  x[i] += c.step[f] * m;
}
// x += d * s (BarzilaiBorwein.h:237-240)
__global__ void axpyKernel(double *x, const double *d, long long n, double s) {
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i < n) x[i] += d[i] * s;
}
// y = a * base + sum_q c_q v_q (base may alias y; no v_q may alias y)
constexpr int kMaxCombine = 2 * kMaxHistory + 4;
struct CombineTerms {
  const double *v[kMaxCombine];
  double c[kMaxCombine];
};
__global__ void combineTermsKernel(double *y, const double *base, double a, CombineTerms t,
                                   int m, long long n) {
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= n) return;
  double acc = base ? a * base[i] : 0.0;
  for (int q = 0; q < m; ++q) acc += t.c[q] * t.v[q][i];
  y[i] = acc;
}
// mean = (sum of the block partials, in block order) / count: one block loads
// them side by side and one thread adds them from LDS (loaded one by one, each
// waiting for memory, 1024 partials took 56 us; 9 us so).
__global__ __launch_bounds__(256) void finishMeanKernel(const double *partials, long long blocks,
                                                        double count, double *mean) {
  __shared__ double sh[1024];
  double s = 0.0;
  for (long long b0 = 0; b0 < blocks; b0 += 1024) {
    const int n = int(blocks - b0 < 1024 ? blocks - b0 : 1024);
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += 256) sh[i] = partials[b0 + i];
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll 16
      for (int i = 0; i < n; ++i) s += sh[i];
    }
  }
  if (threadIdx.x == 0) *mean = s / count;
}

// Dot products of one vector with up to kMaxDots others in one pass over it:
// partials[block * m + i] = block-partial of sum a * b_i.
constexpr int kMaxDots = 16;
struct DotOperands {
  const double *b[kMaxDots];
};
__global__ __launch_bounds__(256) void multiDotKernel(const double *a, DotOperands b,
                                                      int m, long long n,
                                                      double *partials) {
  double s[kMaxDots];
#pragma unroll
  for (int i = 0; i < kMaxDots; ++i) s[i] = 0.0;
  for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < n;
       e += (long long)gridDim.x * blockDim.x) {
    const double x = a[e];
#pragma unroll
    for (int i = 0; i < kMaxDots; ++i)
      if (i < m) s[i] += x * b.b[i][e];
  }
  __shared__ double sh[256];
  for (int i = 0; i < m; ++i) {
    sh[threadIdx.x] = s[i];
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1) {
      if (threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
      __syncthreads();
    }
    if (threadIdx.x == 0) partials[size_t(blockIdx.x) * m + i] = sh[0];
    __syncthreads();
  }
}
// The same over several groups in one launch: block b belongs to the group
// g with blockStart[g] <= b < blockStart[g + 1] and writes its partials at
// offset[g] + (b - blockStart[g]) * m[g].
constexpr int kMaxDotGroups = 8;
struct DotGroupTable {
  const double *a[kMaxDotGroups];
  const double *b[kMaxDotGroups][kMaxDots];
  int m[kMaxDotGroups];
  long long n[kMaxDotGroups];
  long long offset[kMaxDotGroups];
  int blockStart[kMaxDotGroups + 1];
  int numGroups;
};
__global__ __launch_bounds__(256) void multiDotGroupsKernel(DotGroupTable t, double *partials) {
  int g = 0;
  while (g + 1 < t.numGroups && int(blockIdx.x) >= t.blockStart[g + 1]) ++g;
  const int blk = int(blockIdx.x) - t.blockStart[g];
  const int nb = t.blockStart[g + 1] - t.blockStart[g];
  const int m = t.m[g];
  const long long n = t.n[g];
  const double *a = t.a[g];
  double s[kMaxDots];
#pragma unroll
  for (int i = 0; i < kMaxDots; ++i) s[i] = 0.0;
  for (long long e = blk * (long long)blockDim.x + threadIdx.x; e < n;
       e += (long long)nb * blockDim.x) {
    const double x = a[e];
#pragma unroll
    for (int i = 0; i < kMaxDots; ++i)
      if (i < m) s[i] += x * t.b[g][i][e];
  }
  __shared__ double sh[256];
  for (int i = 0; i < m; ++i) {
    sh[threadIdx.x] = s[i];
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1) {
      if (threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
      __syncthreads();
    }
    if (threadIdx.x == 0) partials[t.offset[g] + size_t(blk) * m + i] = sh[0];
    __syncthreads();
  }
}
// heavy ball (Polyak.h:216-240)
__global__ void polyakKernel(double *x, double *vel, const double *g,
                             long long n, double s, double drag) {
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double d = g[i] - x[i];
  const double u = vel[i] * (1.0 - drag) + d * s;
  vel[i] = u;
  x[i] += u;
}
// zero the sites outside the reference grain
__global__ void maskKernel(double *p, const uint8_t *dom, long long n0, int planes) {
  const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (i >= n0 * planes) return;
  if (!dom[i % n0]) p[i] = 0.0;
}

} // namespace scamd
