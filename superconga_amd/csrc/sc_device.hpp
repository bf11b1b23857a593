// sc_device.hpp -- device arithmetic shared by the kernels (gfx950).
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>
#include <limits>

namespace scamd {

// Complex value aligned to its full size so that it moves as one vector
// access.
template <typename T> struct alignas(2 * sizeof(T)) Cx {
  T re, im;
};

template <typename T> __device__ __forceinline__ Cx<T> cx(T r, T i) {
  return Cx<T>{r, i};
}
template <typename T> __device__ __forceinline__ Cx<T> operator+(Cx<T> a, Cx<T> b) {
  return {a.re + b.re, a.im + b.im};
}
template <typename T> __device__ __forceinline__ Cx<T> operator-(Cx<T> a, Cx<T> b) {
  return {a.re - b.re, a.im - b.im};
}
template <typename T> __device__ __forceinline__ Cx<T> operator*(Cx<T> a, Cx<T> b) {
  return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
template <typename T> __device__ __forceinline__ Cx<T> scale(Cx<T> a, T s) {
  return {a.re * s, a.im * s};
}

// Device pointers that reach a kernel inside a struct are generic: accesses
// through them compile to flat_* instructions, which also count against the
// LDS/scalar wait counter, so each wait for a lane shuffle or a scalar load
// would also wait for them.  Every buffer the kernels address lives in global
// memory; through global() the accesses are global_* instructions.
template <typename T> using GlobalPtr = __attribute__((address_space(1))) T *;
template <typename T> __device__ __forceinline__ GlobalPtr<T> global(T *p) {
  return (GlobalPtr<T>)p;
}

template <typename T> using LdsPtr = __attribute__((address_space(3))) T *;

// Streaming access to the sweep scratch: every element is written once and
// read once, so the accesses carry the non-temporal hint and leave the cache
// to the grids the sweep samples.
template <typename T> struct VecOf;
template <> struct VecOf<double> { typedef double type __attribute__((ext_vector_type(2))); };
template <> struct VecOf<float> { typedef float type __attribute__((ext_vector_type(2))); };
template <typename T> __device__ __forceinline__ void storeStream(Cx<T> *p, Cx<T> v) {
  typedef typename VecOf<T>::type V;
  V w;
  w.x = v.re;
  w.y = v.im;
  __builtin_nontemporal_store(w, reinterpret_cast<V *>(p));
}
template <typename T> __device__ __forceinline__ Cx<T> loadStream(const Cx<T> *p) {
  typedef typename VecOf<T>::type V;
  const V w = __builtin_nontemporal_load(reinterpret_cast<const V *>(p));
  return Cx<T>{w.x, w.y};
}

// Reciprocal, reciprocal square root and square root.  FP32: the hardware
// v_rcp_f32 / v_rsq_f32 (1 ulp).  FP64: the hardware v_rcp_f64 / v_rsq_f64
// estimate (largest relative error measured over 2^-6 to 2^6: 4.6e-8 and
// 5.3e-8) refined by one third-order step, whose error is of the order of the
// cube of the estimate's (1e-22): 3 and 5 instructions to the last bits
// (1.1e-16 and 1.4e-16 measured), against 4 and 7 for two Newton steps.
__device__ __forceinline__ float fmaT(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double fmaT(double a, double b, double c) { return fma(a, b, c); }
__device__ __forceinline__ float rcpT(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ float rsqT(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ __forceinline__ float sqrtT(float x) { return x * __builtin_amdgcn_rsqf(x); }
__device__ __forceinline__ double rcpT(double x) {
  const double r = __builtin_amdgcn_rcp(x);
  const double e = fma(-x, r, 1.0);
  return fma(r, fma(e, e, e), r); // r (1 + e + e^2)
}
__device__ __forceinline__ double rsqT(double x) {
  const double r = __builtin_amdgcn_rsq(x);
  const double e = fma(-(x * r), r, 1.0);
  return fma(r * e, fma(e, 0.375, 0.5), r); // r (1 + e/2 + 3 e^2 / 8)
}
// sqrt(x) of a positive x: the step of rsqT applied to x r
__device__ __forceinline__ double sqrtT(double x) {
  const double r = __builtin_amdgcn_rsq(x);
  const double g = x * r;
  const double e = fma(-g, r, 1.0);
  return fma(g * e, fma(e, 0.375, 0.5), g);
}
// Kept for the host-visible unit checks and the bulk solution.
__device__ __forceinline__ double drcp(double x) { return rcpT(x); }
__device__ __forceinline__ float drcp(float x) { return rcpT(x); }

// sqrt(2) times the principal complex square root (Kahan's formulation): with
// u = |x| + |z|, sqrt(2 z) = (sqrt(u), y / sqrt(u)) for x >= 0 and
// (|y| / sqrt(u), copysign(sqrt(u), y)) otherwise; both parts come from one
// reciprocal square root of u.
// |z|^2 is held at or above the smallest normal number, so z = 0 gives a
// root of order 1e-77 (1e-10 in FP32) instead of 0 -- negligible beside the
// O(1) terms it is added to -- with no branch and no select: the square roots
// of a lane's energies stay in one basic block and their latencies overlap.
template <typename T> __device__ __forceinline__ Cx<T> csqrt2(Cx<T> z) {
#pragma clang fp contract(off)
  const T n = fmaT(z.re, z.re, fmaT(z.im, z.im, std::numeric_limits<T>::min()));
  const T u = fabs(z.re) + sqrtT(n);
  const T r = rsqT(u);
  const T t = u * r;
  const T q = z.im * r;
  const bool right = z.re >= T(0);
  return {right ? t : fabs(q), right ? q : copysign(t, z.im)};
}
template <typename T> __device__ __forceinline__ Cx<T> csqrt(Cx<T> z) {
  return scale(csqrt2(z), T(0.70710678118654752440));
}

// A value the compiler knows nothing about and, being volatile, forms anew each
// time it is reached.  Without it the loop invariants of every energy (and the
// expressions that two steps have in common) are formed once and held: the
// pass needs some 60 registers more and spills.
template <typename T> __device__ __forceinline__ void opaque(T &x) { asm volatile("" : "+v"(x)); }
template <typename T> __device__ __forceinline__ void opaqueScalar(T &x) {
  asm volatile("" : "+s"(x));
}

// The sign of every x seen so far: negative once one was.
__device__ __forceinline__ void noteSign(int &neg, float x) { neg |= __float_as_int(x); }
__device__ __forceinline__ void noteSign(int &neg, double x) { neg |= __double2hiint(x); }

// The root of a step's discriminant.  WHOLE: of any z.  Else of z with
// z.re >= 0, two multiplies without the 7 instructions of the selects, and neg
// turns negative where that does not hold: the caller takes the steps again.
template <bool WHOLE, typename T>
__device__ __forceinline__ Cx<T> stepRoot2(Cx<T> z, int &neg) {
#pragma clang fp contract(off)
  if constexpr (WHOLE) return csqrt2(z);
  noteSign(neg, z.re);
  const T n = fmaT(z.re, z.re, fmaT(z.im, z.im, std::numeric_limits<T>::min()));
  const T u = z.re + sqrtT(n);
  const T r = rsqT(u);
  return {u * r, z.im * r};
}

// a / b through the reciprocal of |b|^2 (|b| is of order one here).
template <typename T> __device__ __forceinline__ Cx<T> cdiv(Cx<T> a, Cx<T> b) {
  const T r = rcpT(b.re * b.re + b.im * b.im);
  return {(a.re * b.re + a.im * b.im) * r, (a.im * b.re - a.re * b.im) * r};
}

// One implicit-midpoint step of the Riccati equation (RiccatiSolutions.h:65-94):
// y solves a (y + y0)^2 + (s e - 1) y + (s e + 1) y0 + s D = 0 with s = i h and
// a = s conj(D) / 4.  In FP32 it is the quadratic's root taken whole: with
// b = 2 a y0 + s e - 1, c = (a y0 + s e + 1) y0 + s D,
//   y = 2 c / (-b + sqrt(b^2 - 4 a c)).
// In FP64, with disc = b^2 - 4 a c = (s e - 1)^2 + h^2 |D|^2 - 8 a y0, where only
// the last term depends on y0, and R = sqrt(disc), the same root as an increment:
//   y = y0 + 2 (y0 w + s D) / (2 - w),   w = s e + 1 - R,
// 42 add/multiply instructions instead of 63; 1 - R is exact in floating point,
// and the error is that of the root taken whole (1e-15 of y) or below.
// FP32 keeps the root: an increment form of 32 instructions is 20 times closer
// to FP64 (1e-7 of y after 600 steps of h = 0.05, against 2e-6 of the root, whose
// rounding of 1 - s e acts alike at every step), but the FP32 solution moves by
// what it gains: by 2e-4 of the current after two runs of an accelerated solve.
// The quantities that only depend on the site (D, the energy shift Re e and
// h) are formed once per site and shared by every Ozaki energy.
// The FP64 arithmetic is written with explicit fused multiply-adds, so that
// every place that takes the same step (a sweep, a segment integrated again
// from a checkpoint, the adjoint) rounds alike.
template <typename T> struct StepSite;

// FP64: everything but w is scaled so that the quotient needs no factor, disc
// by 1/2.
template <> struct StepSite<double> {
  Cx<double> a4; // 4 a = i h conj(D); s D = (-a4.re, a4.im)
  double sei;    // Im(s e) = h Re e
  double seir;   // sqrt(2) sei
  double kh;     // (h^2 |D|^2 - sei^2) / 2
  double root;   // sqrt(1/2)
  __device__ __forceinline__ Cx<double> a() const { return {0.25 * a4.re, 0.25 * a4.im}; }
  __device__ __forceinline__ Cx<double> sD() const { return {-a4.re, a4.im}; }
};
__device__ __forceinline__ StepSite<double> stepSite(Cx<double> D, double shift, double h) {
#pragma clang fp contract(off)
  StepSite<double> p;
  p.a4 = {h * D.im, h * D.re};
  p.sei = h * shift;
  p.seir = 1.41421356237309504880 * p.sei;
  p.kh = 0.5 * fma(p.a4.re, p.a4.re, fma(p.a4.im, p.a4.im, -(p.sei * p.sei)));
  p.root = 0.70710678118654752440;
  return p;
}
// ser = Re(s e) = -h Im e (the Matsubara part).
template <bool WHOLE>
__device__ __forceinline__ Cx<double> stepEnergy(const StepSite<double> &p, double ser,
                                                 Cx<double> y0, int &neg) {
#pragma clang fp contract(off)
  const double b = fma(p.root, ser, -p.root); // (Re(s e) - 1) / sqrt(2)
  const Cx<double> z = {fma(p.a4.im, y0.im, fma(-p.a4.re, y0.re, fma(b, b, p.kh))),
                        fma(-p.a4.im, y0.re, fma(-p.a4.re, y0.im, p.seir * b))};
  const Cx<double> R = stepRoot2<WHOLE>(z, neg);
  const Cx<double> w = {(1.0 - R.re) + ser, p.sei - R.im};
  const Cx<double> c = {fma(w.re, y0.re, fma(-w.im, y0.im, -p.a4.re)),
                        fma(w.re, y0.im, fma(w.im, y0.re, p.a4.im))};
  const Cx<double> q = {fma(-0.5, w.re, 1.0), 0.5 * w.im}; // conj(1 - w / 2)
  const double r = rcpT(fma(q.re, q.re, q.im * q.im));
  return {fma(fma(c.re, q.re, -(c.im * q.im)), r, y0.re),
          fma(fma(c.im, q.re, c.re * q.im), r, y0.im)};
}

template <> struct StepSite<float> {
  Cx<float> a;  // s conj(D) / 4
  Cx<float> a4; // 4 a
  Cx<float> sD; // s D = (-4 a.re, 4 a.im)
  float sei;    // Im(s e) = h Re e
  float one;
};
__device__ __forceinline__ StepSite<float> stepSite(Cx<float> D, float shift, float h) {
  StepSite<float> p;
  p.a4 = {h * D.im, h * D.re};
  p.a = {0.25f * p.a4.re, 0.25f * p.a4.im};
  p.sD = {-p.a4.re, p.a4.im};
  p.sei = h * shift;
  p.one = 1.f;
  return p;
}
// The principal root with Kahan's selects: of any discriminant, WHOLE or not.
__device__ __forceinline__ Cx<float> rootOfStep(Cx<float> z) {
  const float n = fmax(z.re * z.re + z.im * z.im, std::numeric_limits<float>::min());
  const float m = n * rsqT(n);
  const float u = 0.5f * (fabs(z.re) + m);
  const float r = rsqT(u);
  const float t = u * r;
  const float q = (0.5f * z.im) * r;
  const bool right = z.re >= 0.f;
  return {right ? t : fabs(q), right ? q : copysign(t, z.im)};
}
template <bool WHOLE>
__device__ __forceinline__ Cx<float> stepEnergy(const StepSite<float> &p, float ser, Cx<float> y0,
                                                int &) {
  const Cx<float> ay = p.a * y0;
  const Cx<float> b = {2.f * ay.re + (ser - p.one), 2.f * ay.im + p.sei};
  const Cx<float> t = {ay.re + (ser + p.one), ay.im + p.sei};
  const Cx<float> c = t * y0 + p.sD;
  const Cx<float> ac4 = p.a4 * c;
  const Cx<float> disc = {b.re * b.re - b.im * b.im - ac4.re, 2.f * b.re * b.im - ac4.im};
  const Cx<float> sq = rootOfStep(disc);
  return cdiv(c + c, sq - b);
}

// Real-frequency energies eps = E + i delta: sej = h E joins the site's
// Im(s e) (the Doppler shift enters the same way).
template <bool WHOLE>
__device__ __forceinline__ Cx<double> stepEnergy(const StepSite<double> &p, double ser, double sej,
                                                 Cx<double> y0, int &neg) {
  StepSite<double> e = p;
  e.sei = p.sei + sej;
  e.seir = 1.41421356237309504880 * e.sei;
  e.kh = fma(0.5 * (p.sei - e.sei), p.sei + e.sei, p.kh);
  return stepEnergy<WHOLE>(e, ser, y0, neg);
}
template <bool WHOLE>
__device__ __forceinline__ Cx<float> stepEnergy(const StepSite<float> &p, float ser, float sej,
                                                Cx<float> y0, int &neg) {
  StepSite<float> e = p;
  e.sei = p.sei + sej;
  return stepEnergy<WHOLE>(e, ser, y0, neg);
}
// a step from any y0
template <typename T>
__device__ __forceinline__ Cx<T> stepEnergy(const StepSite<T> &p, T ser, Cx<T> y0) {
  int neg = 0;
  return stepEnergy<true>(p, ser, y0, neg);
}

// Workgroups are dispatched round robin over the eight XCDs, each with its
// own L2.  A grid of 8 * ceil(n / 8) blocks read through this mapping gives
// every XCD a contiguous range of the n logical blocks (spatially coherent
// sites or tiles share their L2 lines); -1 for the padding blocks.
constexpr int kNumXcd = 8;
__device__ __forceinline__ long long xcdBlock(long long nLogical) {
  const long long per = (nLogical + kNumXcd - 1) / kNumXcd;
  const long long b = blockIdx.x;
  const long long l = (b % kNumXcd) * per + b / kNumXcd;
  return l < nLogical ? l : -1;
}
inline unsigned xcdGrid(long long nLogical) {
  return static_cast<unsigned>(((nLogical + kNumXcd - 1) / kNumXcd) * kNumXcd);
}

template <typename T>
__device__ __forceinline__ Cx<T> riccatiStep(Cx<T> D, Cx<T> e, Cx<T> y0, T h) {
  return stepEnergy(stepSite(D, e.re, h), -h * e.im, y0);
}

// Homogeneous (bulk) solutions (RiccatiSolutions.h:36-54).
template <typename T>
__device__ __forceinline__ void homogeneous(Cx<T> D, Cx<T> e, Cx<T> &g, Cx<T> &gt) {
  const Cx<T> e2 = e * e;
  const Cx<T> om = csqrt(Cx<T>{D.re * D.re + D.im * D.im - e2.re, T(0) - e2.im});
  const Cx<T> den = {e.re - om.im, e.im + om.re}; // e + i Omega
  const Cx<T> inv = cdiv(Cx<T>{T(1), T(0)}, den);
  g = Cx<T>{-(D.re * inv.re - D.im * inv.im), -(D.re * inv.im + D.im * inv.re)};
  gt = Cx<T>{D.re * inv.re + D.im * inv.im, D.re * inv.im - D.im * inv.re};
}

// Bilinear sample of a planar N x N grid at the rotated position of a site of
// a grid of side M (insertRotatedGrid, GridFunctions_GPU.h:436-489).  The
// coordinate arithmetic is kept free of contractions so that the integer
// cell decisions are taken on the same rounded values on every platform.
struct RotSample {
  int idx;      // Yi * N + Xi
  double fx, fy;
  bool valid;
};
__device__ __forceinline__ RotSample rotatedCell(int x, int y, int M, int N,
                                                 double c, double s) {
#pragma clang fp contract(off)
  const double xt = (N - M) / 2.0;
  const double sh = (N - 1) / 2.0;
  const double X = x + xt - sh;
  const double Y = y + xt - sh;
  const double Xr = X * c - Y * s + sh;
  const double Yr = X * s + Y * c + sh;
  const int Xi = static_cast<int>(Xr);
  const int Yi = static_cast<int>(Yr);
  RotSample r;
  r.valid = (Xi >= 0) && (Xi + 1 < N) && (Yi >= 0) && (Yi + 1 < N);
  r.fx = Xr - static_cast<double>(Xi);
  r.fy = Yr - static_cast<double>(Yi);
  r.idx = Yi * N + Xi;
  return r;
}
__device__ __forceinline__ double bilinear(const double *__restrict__ grid, int N,
                                           const RotSample &r) {
#pragma clang fp contract(off)
  // two neighbours in one 16-byte load, of 8-byte alignment
  typedef double Two __attribute__((ext_vector_type(2), aligned(8)));
  const GlobalPtr<const double> p = global(grid) + r.idx;
  const Two lo = *(GlobalPtr<const Two>)p, hi = *(GlobalPtr<const Two>)(p + N);
  const double a = (1.0 - r.fx) * lo.x + r.fx * lo.y;
  const double b = (1.0 - r.fx) * hi.x + r.fx * hi.y;
  return (1.0 - r.fy) * a + r.fy * b;
}

} // namespace scamd
