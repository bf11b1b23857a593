// sc_sweep.hpp -- the Riccati sweep kernels (gfx950), instantiated by
// sc_sweep_fp64.hip and sc_sweep_mixed.hip.
#pragma once

#include "sc_device.hpp"
#include "sc_engine.hpp"
#include "sc_util.hpp"
#include "sc_view.hpp"

#include <algorithm>

namespace scamd {

// One step for one energy: Matsubara energies (i omega) or, with KEL,
// real-frequency energies E + i delta.
template <bool KEL, bool WHOLE, typename T>
__device__ __forceinline__ Cx<T> stepE(const StepSite<T> &p, T ser, T sej, Cx<T> y0, int &neg) {
  if constexpr (KEL) return stepEnergy<WHOLE>(p, ser, sej, y0, neg);
  else return stepEnergy<WHOLE>(p, ser, y0, neg);
}

// Sums over the energy groups of a column (lanes c, c + cols, ...) into its
// group-0 lane: a butterfly when the groups fill the wavefront, else a tree.
__device__ __forceinline__ void sumGroups(double (&q)[4], int gp, int cols, int g, int lane) {
  if (gp * cols == 64) {
    for (int m = cols; m < 64; m <<= 1) {
#pragma unroll
      for (int i = 0; i < 4; ++i) q[i] += __shfl_xor(q[i], m);
    }
    return;
  }
  int top = 1;
  while (2 * top < gp) top *= 2;
  if (gp > 1)
    for (int m = top; m > 0; m >>= 1) {
      const bool add = g + m < gp;
      const int src = add ? lane + m * cols : lane;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const double o = __shfl(q[i], src);
        q[i] += add ? o : 0.0;
      }
    }
}

// lo holds a's lower and b's lower 32 lanes, hi a's upper and b's upper ones
// (permlane32_swap); with 16: even and odd rows of 16 lanes alike.  The sum
// lo + hi reduces a in the lower lanes (even rows) and b in the upper ones
// (odd rows): one swap for two sums.
__device__ __forceinline__ double pairSum32(double a, double b) {
  const unsigned long long ua = __builtin_bit_cast(unsigned long long, a),
                           ub = __builtin_bit_cast(unsigned long long, b);
  const auto l = __builtin_amdgcn_permlane32_swap(unsigned(ua), unsigned(ub), false, false);
  const auto h = __builtin_amdgcn_permlane32_swap(unsigned(ua >> 32), unsigned(ub >> 32), false,
                                                  false);
  const unsigned long long x = (unsigned long long)h[0] << 32 | l[0],
                           y = (unsigned long long)h[1] << 32 | l[1];
  return __builtin_bit_cast(double, x) + __builtin_bit_cast(double, y);
}
__device__ __forceinline__ double pairSum16(double a, double b) {
  const unsigned long long ua = __builtin_bit_cast(unsigned long long, a),
                           ub = __builtin_bit_cast(unsigned long long, b);
  const auto l = __builtin_amdgcn_permlane16_swap(unsigned(ua), unsigned(ub), false, false);
  const auto h = __builtin_amdgcn_permlane16_swap(unsigned(ua >> 32), unsigned(ub >> 32), false,
                                                  false);
  const unsigned long long x = (unsigned long long)h[0] << 32 | l[0],
                           y = (unsigned long long)h[1] << 32 | l[1];
  return __builtin_bit_cast(double, x) + __builtin_bit_cast(double, y);
}

__device__ __forceinline__ StepSite<double> apart(StepSite<double> p) {
  opaque(p.a4.re);
  opaque(p.a4.im);
  opaque(p.seir);
  opaque(p.kh);
  opaqueScalar(p.root);
  return p;
}
__device__ __forceinline__ StepSite<float> apart(StepSite<float> p) {
  opaque(p.a4.re);
  opaque(p.a4.im);
  opaque(p.sei);
  p.a = {0.25f * p.a4.re, 0.25f * p.a4.im};
  p.sD = {-p.a4.re, p.a4.im};
  opaqueScalar(p.one);
  return p;
}
// only what the energies form of the constant apart; the constant of q
__device__ __forceinline__ StepSite<double> fresh(StepSite<double> p) {
  opaqueScalar(p.root);
  return p;
}
__device__ __forceinline__ StepSite<float> fresh(StepSite<float> p) {
  opaqueScalar(p.one);
  return p;
}
__device__ __forceinline__ StepSite<double> alike(StepSite<double> p, const StepSite<double> &q) {
  p.root = q.root;
  return p;
}
__device__ __forceinline__ StepSite<float> alike(StepSite<float> p, const StepSite<float> &q) {
  p.one = q.one;
  return p;
}
// the step of gamma~ (-conj(D)) where p is that of gamma, and the other way
__device__ __forceinline__ StepSite<double> tilde(StepSite<double> p) {
  p.a4.im = -p.a4.im;
  return p;
}
__device__ __forceinline__ StepSite<float> tilde(StepSite<float> p) {
  p.a.im = -p.a.im;
  p.a4.im = -p.a4.im;
  p.sD.im = -p.sD.im;
  return p;
}

// One row of a column: the site fields and the label.
struct SiteRow {
  double re, im, es;
  int lab;
};

// The Riccati sweep.  A workgroup of two wavefronts handles an item: `cols`
// adjacent columns of one frame, each carried by `groups` lanes holding EL
// Ozaki energies each (lane = group * cols + column; the 64 - groups * cols
// lanes past the last group and the columns past ncols repeat their neighbours
// and write nothing).  One wavefront integrates gamma~ from the top of the item
// downwards, the other gamma from the bottom upwards (`up`).  In the first half
// each keeps every second site of its own in the slot's scratch; where they
// meet they wait for each other, and in the second half each takes the sites of
// the other one from there, those in between by the same step again, and forms
// the energy-summed Green functions at every inside site.  Boundary in-values
// are read and out-values written as in RiccatiSolverConfined.h:129-312.
//
// What bounds it: kept at every site, gamma~ made 81 of the 95 GB an FP64
// sweep of 5.06e9 steps moved, 4.5 TB/s against the 4.7 TB/s of a large copy.
// A step costs 42 FP64 instructions against 32 bytes of scratch, so half of the
// steps taken once more is cheaper than keeping them: 25% more steps for 43%
// fewer bytes.  It is then bound by the issue of those instructions.
// Two wavefronts and half the rows each, instead of one that goes down and up
// again, halve the chain of steps that bounds a small grain, and the length of
// an item at the end of the queue.
//
// Both halves take two sites at a time.  In the interior of the grain (no
// lane at a crossing, the great majority) the pair runs without a branch;
// otherwise its sites are taken one by one with everything that a crossing
// asks for.  The rows of the next pair are loaded while a pair is taken.
// Every path through a pair issues its loads before its stores, so that the
// wait for the former leaves the latter in flight.
//
// What the next crossing of a lane's column needs waits in the lane's LDS
// (the in-values) and registers (the distances): read at the crossing, they
// would cost the wavefront a memory latency at each of its columns' ends.
//
// Lanes outside the grain (label 0) go on stepping with the fields they
// find: their values are finite, are written nowhere, and a trajectory that
// (re)enters starts from its boundary value or from zero.
//
// Returns false where a step's discriminant left the right half plane and
// WHOLE is not set: the item is then to be swept again with it (its outputs
// are written whole again).  That takes a step h |Re e| of order one, a Doppler
// shift of the order of the inverse lattice spacing.
template <typename T, int EL, bool KEL, bool WHOLE>
__device__ __forceinline__ bool sweepItem(const SweepArgs &a, const GrainView &v,
                                          const SweepItemDev &it, Cx<T> *scr, Cx<T> *lds,
                                          bool up) {
  const unsigned lane = threadIdx.x & 63;
  const int cols = v.cols;
  const int gp = v.groups; // lanes per column
  const int g = int(lane) / cols;
  const int c = int(lane) - g * cols;
  const int N1 = v.N1, Ne = v.Ne;
  const size_t n1 = size_t(N1) * N1;
  const T h = T(v.h);
  const int k = it.angle;
  const bool real = c < it.ncols && g < gp; // a lane of the item's own columns
  const unsigned x = unsigned(it.x0 + min(c, it.ncols - 1));
  const int e0 = min(g, gp - 1) * EL;
  T ser[EL], sej[EL];
#pragma unroll
  for (int j = 0; j < EL; ++j) {
    // energies past the last repeat it with no weight
    const int e = min(e0 + j, Ne - 1);
    ser[j] = -h * T(global(v.energy)[e]);
    sej[j] = KEL ? h * T(global(v.energyRe)[e]) : T(0);
  }
  const int len = it.yhi - it.ylo + 1;
  const size_t col = size_t(k) * N1 + x;
  const GlobalPtr<const double> fRe = global(v.fields + size_t(k - v.fieldBase) * n1);
  const GlobalPtr<const double> fIm = fRe + v.fieldPlane, fEs = fIm + v.fieldPlane;
  const GlobalPtr<const int8_t> lab = global(v.labels + size_t(k) * n1);
  // row of the site `at` steps from the wavefront's own end
  auto rowOf = [&](int at) { return up ? it.ylo + at : it.yhi - at; };
  auto loadRow = [&](int at) {
    const size_t o = size_t(rowOf(min(max(at, 0), len - 1))) * N1;
    unsigned xo = x; // a 32-bit offset to the row's scalar address
    opaque(xo);
    SiteRow r;
    r.re = (fRe + o)[xo];
    r.im = (fIm + o)[xo];
    r.es = (fEs + o)[xo];
    r.lab = (lab + o)[xo];
    return r;
  };
  // Delta for gamma, -conj(Delta) for gamma~
  const T sign = up ? T(1) : T(-1);
  // labels of the sites where the own trajectory enters and leaves
  const int entryLabel = up ? 2 : 3, exitLabel = up ? 3 : 2;
  // rows of the first half: the own ones and the other wavefront's, which
  // keep the upper half's sites first
  const int down = (len + 1) / 2, own = up ? len - down : down, other = len - own;
  Cx<T> *const ownScr = scr + (up ? size_t(down) * EL * 64 : 0);
  Cx<T> *const otherScr = scr + (up ? 0 : size_t(down) * EL * 64);
  // what is kept: the even sites (counted from the end they started from),
  // then the odd ones that start from a boundary value
  const int ownOdd = (own + 1) / 2, otherOdd = (other + 1) / 2;
  auto keep = [](Cx<T> *p, int row, int j) { return p + (size_t(row) * EL + j) * 64; };
  // whether any lane of a pair needs more than a plain step: a crossing, or a
  // change between outside and inside from the site before on
  auto crossing = [](int lp, int l0, int l1) {
    return (l0 | l1) >= 2 || (lp != 0) != (l0 != 0) || (l0 != 0) != (l1 != 0);
  };
  int neg = 0;
  // the next in-value of a lane into its LDS (energies past the last, and the
  // crossing past the last, read what follows: the storage is padded)
  auto fetchEntry = [&](int ci, GlobalPtr<const double> bin, long long nIn) {
    const GlobalPtr<const double> re = bin + (size_t(ci) * Ne + e0), im = re + size_t(nIn) * Ne;
#pragma unroll
    for (int j = 0; j < EL; ++j) lds[j * 64 + lane] = Cx<T>{T(re[j]), T(im[j])};
  };
  // the same inside a pass, for columns that are entered again: one energy
  // after the other, for its registers
  auto fetchAgain = [&](int ci, GlobalPtr<const double> bin, long long nIn) {
    const GlobalPtr<const double> re = bin + (size_t(ci) * Ne + e0), im = re + size_t(nIn) * Ne;
#pragma unroll
    for (int j = 0; j < EL; ++j) {
      lds[j * 64 + lane] = Cx<T>{T(re[j]), T(im[j])};
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // the step into a site that may be an entry (from the in-value over the
  // crossing's distance), the first of the item or the first inside (from
  // zero), or plain
  auto enter = [&](bool entry, bool first, int lp, Cx<T> D, T es, Cx<T> dPrev, T esPrev, T dist,
                   Cx<T>(&coh)[EL]) {
    const T part = entry ? dist : first ? T(0.5) : T(1);
    const bool whole = entry || first;
    const StepSite<T> ps =
        stepSite(whole ? D : Cx<T>{(dPrev.re + D.re) * T(0.5), (dPrev.im + D.im) * T(0.5)},
                 whole ? es : (esPrev + es) * T(0.5), part * h);
    if (first || lp == 0) {
#pragma unroll
      for (int j = 0; j < EL; ++j) coh[j] = {T(0), T(0)};
    }
    if (entry) {
#pragma unroll
      for (int j = 0; j < EL; ++j) coh[j] = lds[j * 64 + lane];
    }
#pragma unroll
    for (int j = 0; j < EL; ++j) {
      coh[j] = stepE<KEL, WHOLE>(ps, ser[j] * part, sej[j] * part, coh[j], neg);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // the out-values of an exit
  auto leave = [&](Cx<T> D, T es, T dr, int ci, GlobalPtr<double> bout, long long nOut,
                   const Cx<T>(&coh)[EL]) {
    const StepSite<T> pe = fresh(stepSite(D, es, dr * h));
    const GlobalPtr<double> re = bout + (size_t(ci) * Ne + e0), im = re + size_t(nOut) * Ne;
#pragma unroll
    for (int j = 0; j < EL; ++j) {
      const Cx<T> bv = stepE<KEL, WHOLE>(pe, ser[j] * dr, sej[j] * dr, coh[j], neg);
      if (real && e0 + j < Ne) {
        re[j] = double(bv.re);
        im[j] = double(bv.im);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // next entry and exit of the lane's column (-1: it has none)
  int in = global(up ? v.idxInG : v.idxInGt)[col], out = global(up ? v.idxOutG : v.idxOutGt)[col];
  const GlobalPtr<const double> distIn = global(up ? v.distInG : v.distInGt),
                                distOut = global(up ? v.distOutG : v.distOutGt);
  const GlobalPtr<const double> bIn = global(up ? v.bInG : v.bInGt);
  const GlobalPtr<double> bOut = global(up ? v.bOutG : v.bOutGt);
  const long long nIn = up ? v.nInG : v.nInGt, nOut = up ? v.nOutG : v.nOutGt;
  T dIn = T(distIn[max(in, 0)]), dOut = T(distOut[max(out, 0)]);
  fetchEntry(max(in, 0), bIn, nIn);
  // what a site with a crossing asks for: the step into it and, at an exit,
  // the out-values
  auto cross = [&](bool first, int lc, int lq, Cx<T> D, T es, Cx<T> dp, T ep, Cx<T>(&coh)[EL]) {
    enter(lc == entryLabel, first, lq, D, es, dp, ep, dIn, coh);
    if (lc == entryLabel) {
      ++in;
      dIn = T(distIn[in]);
      if (it.reentered) fetchAgain(in, bIn, nIn);
    }
    if (lc == exitLabel) {
      leave(D, es, dOut, out, bOut, nOut, coh);
      ++out;
      dOut = T(distOut[out]);
    }
  };
  Cx<T> coh[EL];
#pragma unroll
  for (int j = 0; j < EL; ++j) coh[j] = {T(0), T(0)};
  Cx<T> dPrev = {T(0), T(0)};
  T esPrev = T(0);
  int lp = 0;

  // ---------------- first half: keep every second site ----------------
  {
    // a burn-in sweep keeps nothing: all its lanes store into one element
    const unsigned at = a.burnin ? 0u : lane;
    SiteRow n0 = loadRow(0), n1r = loadRow(1);
    for (int t = 0; t < own; t += 2) {
      const SiteRow r0 = n0, r1 = n1r;
      n0 = loadRow(t + 2);
      n1r = loadRow(t + 3);
      const bool both = t + 1 < own;
      const Cx<T> D0 = {T(r0.re) * sign, T(r0.im)}, D1 = {T(r1.re) * sign, T(r1.im)};
      const T es0 = T(r0.es), es1 = T(r1.es);
      const int row = a.burnin ? 0 : t / 2;
      if (both && t > 0 && !__any(crossing(lp, r0.lab, r1.lab))) {
        const StepSite<T> p0 = fresh(stepSite(
            Cx<T>{(dPrev.re + D0.re) * T(0.5), (dPrev.im + D0.im) * T(0.5)}, (esPrev + es0) * T(0.5), h));
        const StepSite<T> p1 = fresh(stepSite(
            Cx<T>{(D0.re + D1.re) * T(0.5), (D0.im + D1.im) * T(0.5)}, (es0 + es1) * T(0.5), h));
#pragma unroll
        for (int j = 0; j < EL; ++j) {
          coh[j] = stepE<KEL, WHOLE>(p0, ser[j], sej[j], coh[j], neg);
          storeStream(keep(ownScr, row, j) + at, coh[j]);
        }
#pragma unroll
        for (int j = 0; j < EL; ++j) coh[j] = stepE<KEL, WHOLE>(p1, ser[j], sej[j], coh[j], neg);
      } else {
        const int n = both ? 2 : 1;
#pragma unroll 1
        for (int i = 0; i < n; ++i) {
          const int lc = i ? r1.lab : r0.lab;
          cross(t + i == 0, lc, i ? r0.lab : lp, i ? D1 : D0, i ? es1 : es0, i ? D0 : dPrev,
                i ? es0 : esPrev, coh);
          if (i == 0 || __any(lc == entryLabel)) {
            const int rw = a.burnin ? 0 : (i ? ownOdd + t / 2 : t / 2);
#pragma unroll
            for (int j = 0; j < EL; ++j) storeStream(keep(ownScr, rw, j) + at, coh[j]);
          }
        }
      }
      dPrev = both ? D1 : D0;
      esPrev = both ? es1 : es0;
      lp = both ? r1.lab : r0.lab;
    }
  }
  // the other wavefront's sites are complete and visible
  __syncthreads();

  // ---------------- second half: Green functions ----------------
  if (other > 0) {
    // twice the residues, in LDS: read at each use (volatile), they leave 2 EL
    // registers to the rest
    const LdsPtr<volatile T> res2 =
        (LdsPtr<volatile T>)(reinterpret_cast<T *>(lds + EL * 64) + lane);
    if constexpr (!KEL) {
#pragma unroll
      for (int j = 0; j < EL; ++j)
        res2[j * 64] = e0 + j < Ne ? T(2.0 * global(v.residue)[min(e0 + j, Ne - 1)]) : T(0);
    }
    // sites are counted as the other wavefront counts them, from its end: the
    // own next one is other - 1; the lowest kept one
    const int top = (other - 1) & ~1;
    // lanes with no record to write store into the scratch of that site: it
    // is read (by this wavefront alone) before the first store and never again
    Cx<T> *const sink = keep(otherScr, top / 2, 0);
    const bool quarter = gp == 4 && cols == 16;
    const int comp = quarter ? ((g & 1) << 1 | g >> 1) : 0; // after pairSum32, pairSum16
    double *const Gk = v.G + size_t(k - v.angleBase) * n1 * (KEL ? size_t(Ne) : 4);

    // Green functions of site y (GreensFunctionStatic.h:125-157,
    // LocalGreens.h:32-70, ComputeFreeEnergy.h:95-160).  Per energy, with
    // p = gamma gamma~, F = 2 i / (1 + p), u = gamma~ - gamma, w = gamma + gamma~:
    //   f + f~* = F u [real part], -F w [imag part],
    //   Re g = Im((1 - p) / (1 + p)) = -2 Im p / |1 + p|^2
    //   Re i(D* gamma - D gamma~) summed as D.re Su + D.im Sw with
    //   Su = sum r Im u, Sw = sum r Re w.
    // (p and w are symmetric in the two; u is formed as the other one's minus
    // the own, and its sums change sign where the own is gamma~).
    // A Keldysh sweep stores the spectral weight of every energy
    // (ComputeLDOS.h:126-151 with LocalGreens.h:32-45), -Im(i X) with
    // X = -(1 - p) / (1 + p), i.e. (1 - |p|^2) / |1 + p|^2.
    struct Green {
      double dr = 0.0, di = 0.0, j = 0.0, su = 0.0, sw = 0.0;
    };
    auto addGreen = [&](Green &q, int j, Cx<T> mine, Cx<T> its) {
      const Cx<T> p = mine * its;
      const T pr = T(1) + p.re;
      const T rd = rcpT(pr * pr + p.im * p.im);
      const Cx<T> u = its - mine, w = mine + its;
      const double r = double(res2[j * 64]);
      const T X = p.im * u.re - pr * u.im, Y = p.im * w.im + pr * w.re;
      q.dr += r * double(rd * X);
      q.di -= r * double(rd * Y);
      q.j -= r * double(rd * p.im);
      q.su += r * double(u.im);
      q.sw += r * double(w.re);
    };
    auto putGreen = [&](const Green &q, const SiteRow &f, int y) {
      const bool record = !a.burnin && f.lab > 0 && real;
      double *const site = Gk + (size_t(y) * N1 + x) * 4;
      const double sg = up ? 1.0 : -1.0;
      double s[4] = {sg * q.dr, q.di, q.j, 0.5 * (f.re * (sg * q.su) + f.im * q.sw)};
      if (quarter) {
        const double r = pairSum16(pairSum32(s[0], s[1]), pairSum32(s[2], s[3]));
        double *const dst = record ? site + comp : reinterpret_cast<double *>(sink);
        *global(dst) = r;
      } else {
        sumGroups(s, gp, cols, g, int(lane));
        typedef typename VecOf<double>::type D2;
        D2 *const dst = record && g == 0 ? reinterpret_cast<D2 *>(site) : reinterpret_cast<D2 *>(sink);
        const GlobalPtr<D2> o = global(dst);
        o[0] = D2{s[0], s[1]};
        o[1] = D2{s[2], s[3]};
      }
    };
    // An even energy's weight waits for the next one's where both fit one
    // 16-byte store (EL and Ne even): half the stores, each to a line of its
    // own per lane.
    double held = 0.0;
    const bool twos = EL % 2 == 0 && Ne % 2 == 0;
    auto putWeight = [&](int j, Cx<T> ga, Cx<T> gt, const SiteRow &f, int y) {
      const Cx<T> p = ga * gt;
      const T pr = T(1) + p.re;
      const T wgt = (T(1) - (p.re * p.re + p.im * p.im)) * rcpT(pr * pr + p.im * p.im);
      const bool record = !a.burnin && f.lab > 0 && real && e0 + j < Ne;
      double *const dst = record ? Gk + (size_t(y) * N1 + x) * Ne + e0 + j
                                 : reinterpret_cast<double *>(sink);
      if (!twos) {
        *global(dst) = double(wgt);
      } else if (j % 2 == 0) {
        held = double(wgt);
      } else {
        typedef typename VecOf<double>::type D2;
        *global(reinterpret_cast<D2 *>(record ? dst - 1 : dst)) = D2{held, double(wgt)};
      }
    };

    // the other one's even site t of a pair; each energy's next one is loaded
    // into its registers after their last use
    Cx<T> ck[EL];
    auto loadKept = [&](int t, int j) {
      ck[j] = loadStream(keep(otherScr, a.burnin ? 0 : max(t, 0) / 2, j) + lane);
    };
    // site t is the own site len - 1 - t; the pair of top is (top + 1, top)
    SiteRow r0 = loadRow(len - 2 - top), r1 = loadRow(len - 1 - top);
#pragma unroll
    for (int j = 0; j < EL; ++j) loadKept(top, j);
    for (int t = top; t >= 0; t -= 2) {
      const bool both = t + 1 < other; // site t + 1, then site t
      const int at1 = len - 1 - t, at0 = at1 - 1, y1 = rowOf(at1), y0 = rowOf(at0);
      const Cx<T> D0 = {T(r0.re) * sign, T(r0.im)}, D1 = {T(r1.re) * sign, T(r1.im)};
      const T es0 = T(r0.es), es1 = T(r1.es);
      // the own step from site t + 1 to t
      auto pairStep = [&] {
        return stepSite(Cx<T>{(D0.re + D1.re) * T(0.5), (D0.im + D1.im) * T(0.5)},
                        (es0 + es1) * T(0.5), h);
      };
      SiteRow n0, n1r;
      if (both && at0 > 0 && !__any(crossing(lp, r0.lab, r1.lab))) {
        // and the other one's from t to t + 1
        const StepSite<T> p1 = pairStep(), pt = fresh(tilde(p1));
        const StepSite<T> p0 = alike(stepSite(
            Cx<T>{(dPrev.re + D0.re) * T(0.5), (dPrev.im + D0.im) * T(0.5)}, (esPrev + es0) * T(0.5), h), pt);
        Green q0, q1;
#pragma unroll
        for (int j = 0; j < EL; ++j) {
          const Cx<T> its = stepE<KEL, WHOLE>(pt, ser[j], sej[j], ck[j], neg);
          coh[j] = stepE<KEL, WHOLE>(p0, ser[j], sej[j], coh[j], neg);
          if constexpr (KEL) putWeight(j, coh[j], its, r0, y0);
          else addGreen(q0, j, coh[j], its);
        }
        if constexpr (!KEL) putGreen(q0, r0, y0);
        n0 = loadRow(at0 + 2);
        n1r = loadRow(at1 + 2);
        const StepSite<T> pe = apart(p1);
#pragma unroll
        for (int j = 0; j < EL; ++j) {
          coh[j] = stepE<KEL, WHOLE>(pe, ser[j], sej[j], coh[j], neg);
          if constexpr (KEL) putWeight(j, coh[j], ck[j], r1, y1);
          else addGreen(q1, j, coh[j], ck[j]);
          loadKept(t - 2, j);
        }
        if constexpr (!KEL) putGreen(q1, r1, y1);
      } else {
#pragma unroll 1
        for (int i = both ? 0 : 1; i < 2; ++i) {
          const int lc = i ? r1.lab : r0.lab;
          const bool after = i && both;
          cross((i ? at1 : at0) == 0, lc, after ? r0.lab : lp, i ? D1 : D0, i ? es1 : es0,
                after ? D0 : dPrev, after ? es0 : esPrev, coh);
          SiteRow f;
          f.re = i ? r1.re : r0.re;
          f.im = i ? r1.im : r0.im;
          f.lab = lc;
          f.es = 0.0;
          const int y = i ? y1 : y0;
          // the other one's odd site: kept where any lane of it enters there
          // (and the own one leaves), else the step from the even site (from
          // zero where that is outside)
          const bool kept = i == 0 && __any(lc == exitLabel);
          const bool zero = r1.lab == 0;
          const StepSite<T> po = apart(tilde(pairStep()));
          Green q;
#pragma unroll
          for (int j = 0; j < EL; ++j) {
            Cx<T> its = ck[j];
            int from = __builtin_amdgcn_readfirstlane(i ? 2 : kept ? 1 : 0);
            opaqueScalar(from); // one energy after the other
            if (from == 1)
              its = loadStream(keep(otherScr, a.burnin ? 0 : otherOdd + t / 2, j) + lane);
            else if (from == 0)
              its = stepE<KEL, WHOLE>(po, ser[j], sej[j], zero ? Cx<T>{T(0), T(0)} : its, neg);
            if constexpr (KEL) putWeight(j, coh[j], its, f, y);
            else addGreen(q, j, coh[j], its);
            opaque(q.dr);
            opaque(q.di);
            opaque(q.j);
            opaque(q.su);
            opaque(q.sw);
            __builtin_amdgcn_sched_barrier(0);
          }
          if constexpr (!KEL) putGreen(q, f, y);
        }
        n0 = loadRow(at0 + 2);
        n1r = loadRow(at1 + 2);
#pragma unroll
        for (int j = 0; j < EL; ++j) loadKept(t - 2, j);
      }
      dPrev = D1;
      esPrev = es1;
      lp = r1.lab;
      r0 = n0;
      r1 = n1r;
    }
  }
  return WHOLE || !__any(neg < 0);
}

// What a workgroup keeps in LDS: per wavefront the entry values and the
// residues, then the item in hand and whether each wavefront asks to sweep it
// again.
template <typename T, int EL> struct SweepLds {
  Cx<T> of[2][EL * 64 + EL * 32];
  int item, again[2];
};

// Persistent workgroups pulling items from the work counter.  The second
// launch bound asks the compiler for a register budget that leaves room for
// WAVES wavefronts per SIMD.
// The views and items come as restrict-qualified parameters as well: the
// sweep never writes them, and with that known the compiler reads them with
// scalar loads once per item (in SGPRs, uniform across the wavefront) and
// reaches the arrays they point at with global (not flat) loads, instead of
// reloading each field after every store the sweep makes.
template <typename T, int EL, int WAVES, bool KEL>
__global__ __launch_bounds__(128, WAVES) void sweepKernel(SweepArgs a,
                                                           const GrainView *__restrict__ views,
                                                           const SweepItemDev *__restrict__ items) {
  Cx<T> *scr = reinterpret_cast<Cx<T> *>(a.scratch) + size_t(blockIdx.x) * a.slotStride;
  __shared__ SweepLds<T, EL> lds;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int last = -1;;) {
    if (wave == 0) {
      // every lane takes part in the fetch (lane 0 adds one, the others
      // zero): no branch on the lane index surrounds it, so the compiler
      // cannot merge it with a lane-0 branch of the item into a loop that
      // some lanes re-enter without lane 0.  Lane 0's old value is the item.
      lds.item = __builtin_amdgcn_readfirstlane(atomicAdd(a.counter, threadIdx.x == 0 ? 1 : 0));
    }
    // the item is known, and the last one done (its scratch is free again)
    __syncthreads();
    const int item = __builtin_amdgcn_readfirstlane(lds.item);
    if (wave == 0 && last >= 0 && (lds.again[0] | lds.again[1])) {
      // noted for sweepAgainKernel (every lane stores the same number)
      const int at = __builtin_amdgcn_readfirstlane(
          atomicAdd(a.counter + kAgainCount, threadIdx.x == 0 ? 1 : 0));
      a.counter[kAgainList + at] = last;
    }
    if (item >= a.numItems) break;
    const SweepItemDev it = items[item];
    lds.again[wave] =
        sweepItem<T, EL, KEL, false>(a, views[it.grain], it, scr, lds.of[wave], wave != 0) ? 0 : 1;
    last = item;
  }
}

// The items that sweepKernel noted, by the root of any discriminant (none, as
// a rule).  A kernel of its own: with both in one, the second copy's registers
// made the first one spill.
template <typename T, int EL, bool KEL>
__global__ __launch_bounds__(128, 1) void sweepAgainKernel(SweepArgs a,
                                                           const GrainView *__restrict__ views,
                                                           const SweepItemDev *__restrict__ items) {
  Cx<T> *scr = reinterpret_cast<Cx<T> *>(a.scratch) + size_t(blockIdx.x) * a.slotStride;
  __shared__ SweepLds<T, EL> lds;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int count = __builtin_amdgcn_readfirstlane(a.counter[kAgainCount]);
  if (count == 0) return;
  for (;;) {
    if (wave == 0)
      lds.item =
          __builtin_amdgcn_readfirstlane(atomicAdd(a.counter + 1, threadIdx.x == 0 ? 1 : 0));
    __syncthreads();
    const int n = __builtin_amdgcn_readfirstlane(lds.item);
    if (n >= count) break;
    const SweepItemDev it = items[__builtin_amdgcn_readfirstlane(a.counter[kAgainList + n])];
    sweepItem<T, EL, KEL, true>(a, views[it.grain], it, scr, lds.of[wave], wave != 0);
  }
}

// Launches the variant (energies per lane, wavefronts per SIMD) of one
// arithmetic; false where it is not compiled.
template <typename T>
bool launchSweepOf(int el, int waves, const SweepArgs &a, int slots, hipStream_t stream,
                   bool keldysh) {
  // slots are wavefronts, two to a workgroup; the second kernel runs one
  // wavefront per SIMD
  const int groups = slots / 2, again = std::min(groups, kSweepAgainSlots / 2);
#define SC_LAUNCH(E, W)                                                              \
  if (el == E && waves == W) {                                                       \
    sweepKernel<T, E, W, KEL><<<groups, 128, 0, stream>>>(a, a.views, a.items);        \
    SC_HIP(hipGetLastError());                                                       \
    sweepAgainKernel<T, E, KEL><<<again, 128, 0, stream>>>(a, a.views, a.items);      \
    SC_HIP(hipGetLastError());                                                       \
    return true;                                                                     \
  }
  if (keldysh) {
    constexpr bool KEL = true;
    SC_KELDYSH_VARIANTS(SC_LAUNCH)
  } else {
    constexpr bool KEL = false;
    SC_SWEEP_VARIANTS(SC_LAUNCH)
  }
#undef SC_LAUNCH
  return false;
}

} // namespace scamd
