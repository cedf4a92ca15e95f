// Parts the one-sweep steps share (step3d.hip, step2d.hip).
#pragma once

#include "kernel_common.h"

namespace gmes_engine {

#define GMES_CONST __attribute__((address_space(4)))
// uniform reads of data no kernel writes meanwhile: scalar loads
template <class V>
__device__ __forceinline__ V cld(const V* p) {
  return *(const GMES_CONST V*)(uintptr_t)p;
}

// Block -> job of a batched launch, by scalar loads; the job in constant memory.
template <class J>
__device__ __forceinline__ const GMES_CONST J* step_job(const J* jobs, int njobs, int64_t b) {
  int lo = 0, hi = njobs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (cld(&jobs[mid].block0) <= b) lo = mid;
    else hi = mid - 1;
  }
  return (const GMES_CONST J*)(uintptr_t)(jobs + lo);
}

// Division by a cell size or a CPML kappa.  EXACT: every divisor of the sim
// is a power of two (kappa: 1), so multiplying by the reciprocal rounds the
// same real number and gives the quotient's bits.
template <bool EXACT, class T, class R>
__device__ __forceinline__ T by_size(T x, R d, R inv_d) {
  if constexpr (EXACT) return vscl(inv_d, x);
  else return vdiv(x, d);
}
template <bool EXACT, class T, class R>
__device__ __forceinline__ T by_kappa(T x, R k) {
  if constexpr (EXACT) return x;
  else return vdiv(x, k);
}

// Absorber row of one axis: CPML b, c, kappa (FP32: 1/kappa); UPML c1..c6.
template <class R, int PML>
struct Rows {
  R v[PML == 2 ? 6 : 3];
};

__device__ __forceinline__ float vneg(float a) { return -a; }
__device__ __forceinline__ double vneg(double a) { return -a; }
template <class R>
__device__ __forceinline__ cplx<R> vneg(cplx<R> a) {
  return {-a.re, -a.im};
}
template <class T>
__device__ __forceinline__ T vsel(bool c, T a, T b) {
  if constexpr (is_cplx<T>::value) return {c ? a.re : b.re, c ? a.im : b.im};
  else return c ? a : b;
}

// New value of one component, with the formulas and operand order of
// update_value (kernels.hip).  plain: Dielectric; cpml: CPML with rows r1, r2
// of the curl axes, old words o1, o2 and new ones n1, n2 (of a lane that is
// no CPML cell, `is` false, the Dielectric value all the same: where both
// words are dead the two agree in finite values but zeros' signs, and an
// infinite difference times c = 0 is NaN); upml: rows r1, r2 of the curl axes
// and r0 of the own one.
template <bool E, bool X, class T, class R>
__device__ __forceinline__ T plain_value(R c, T f, T D1, T D2, R d1, R i1, R d2, R i2) {
  if constexpr (std::is_same<R, float>::value) {
    const T a = vscl(i1, D1), b = vscl(i2, D2);
    return E ? fma_(c, vsub(a, b), f) : fma_(c, vsub(b, a), f);
  } else {
    const T a = by_size<X>(D1, d1, i1), b = by_size<X>(D2, d2, i2);
    return vadd(f, vscl(c, E ? vsub(a, b) : vsub(b, a)));
  }
}

template <bool E, bool X, class T, class R>
__device__ __forceinline__ T cpml_value(R c, T f, T D1, T D2, R d1, R i1, R d2, R i2, const Rows<R, 1>& r1,
                                        const Rows<R, 1>& r2, T o1, T o2, T& n1, T& n2, bool is = true) {
  if constexpr (std::is_same<R, float>::value) {
    const T a = vscl(i1, D1), b = vscl(i2, D2);
    n1 = fma_(r1.v[1], a, vscl(r1.v[0], o1));
    n2 = fma_(r2.v[1], b, vscl(r2.v[0], o2));
    const T t = vsub(vadd(fma_(-r2.v[2], b, vscl(r1.v[2], a)), n1), n2);
    return fma_(c, vsel(is, E ? t : vneg(t), E ? vsub(a, b) : vsub(b, a)), f);
  } else {
    const T a = by_size<X>(D1, d1, i1), b = by_size<X>(D2, d2, i2);
    n1 = vadd(vscl(r1.v[0], o1), by_size<X>(vscl(r1.v[1], D1), d1, i1));
    n2 = vadd(vscl(r2.v[0], o2), by_size<X>(vscl(r2.v[1], D2), d2, i2));
    const T t = vsub(vadd(vsub(by_kappa<X>(a, r1.v[2]), by_kappa<X>(b, r2.v[2])), n1), n2);
    return vadd(f, vscl(c, vsel(is, E ? t : vneg(t), E ? vsub(a, b) : vsub(b, a))));
  }
}

// The same where both curl axes are dead: the words are +0, or NaN where the
// difference is not finite.
__device__ __forceinline__ float plus_zero(float a, float b) { return __builtin_fmaf(0.0f, a, b); }
__device__ __forceinline__ double plus_zero(double a, double b) { return __builtin_fma(0.0, a, b); }
template <class R>
__device__ __forceinline__ cplx<R> plus_zero(cplx<R> a, cplx<R> b) {
  return {plus_zero(a.re, b.re), plus_zero(a.im, b.im)};
}
template <bool E, bool X, class T, class R>
__device__ __forceinline__ T dead_value(R c, T f, T D1, T D2, R d1, R i1, R d2, R i2, bool is) {
  constexpr bool F = std::is_same<R, float>::value;
  T a, b;
  if constexpr (F) {
    a = vscl(i1, D1);
    b = vscl(i2, D2);
  } else {
    a = by_size<X>(D1, d1, i1);
    b = by_size<X>(D2, d2, i2);
  }
  const T d = vsub(a, b), t = vadd(plus_zero(F ? b : D2, plus_zero(F ? a : D1, d)), T{});
  const T u = vsel(is, E ? t : vneg(t), E ? d : vsub(b, a));
  if constexpr (F) return fma_(c, u, f);
  else return vadd(f, vscl(c, u));
}

// c: dt / eps; q: 1 / eps (FP32) or eps (FP64)
template <bool E, bool X, class T, class R>
__device__ __forceinline__ T upml_value(R q, T f, T D1, T D2, R d1, R i1, R d2, R i2, const Rows<R, 2>& r1,
                                        const Rows<R, 2>& r2, const Rows<R, 2>& r0, T o, T& n) {
  if constexpr (std::is_same<R, float>::value) {
    const T cu = vsub(vscl(i1, D1), vscl(i2, D2));
    n = E ? fma_(r1.v[1], cu, vscl(r1.v[0], o)) : fma_(-r1.v[1], cu, vscl(r1.v[0], o));
    return fma_(r2.v[3] * q, fma_(-r0.v[5], o, vscl(r0.v[4], n)), vscl(r2.v[2], f));
  } else {
    const T cu = vsub(by_size<X>(D1, d1, i1), by_size<X>(D2, d2, i2));
    n = E ? vadd(vscl(r1.v[0], o), vscl(r1.v[1], cu)) : vsub(vscl(r1.v[0], o), vscl(r1.v[1], cu));
    return vadd(vscl(r2.v[2], f), vdiv(vscl(r2.v[3], vsub(vscl(r0.v[4], n), vscl(r0.v[5], o))), q));
  }
}

template <class R>
__device__ __forceinline__ cplx<R> phase_of(const GMES_CONST cplx<R>& p) {
  return {p.re, p.im};
}
// x times the phase (real fields: x)
template <class T>
__device__ __forceinline__ T phased(const GMES_CONST cplx<typename real_of<T>::type>& p, T x) {
  if constexpr (is_cplx<T>::value) return cmul(phase_of(p), x);
  else return x;
}

// Dummy and Const cells and cells with a point source: a handful per sim.
// f is the cell's old value, v its updated one.
template <class T>
__device__ __forceinline__ T step_rare(const StepRare* q, const double* waves, int64_t wave_n, int64_t row, T f, T v) {
  using R = typename real_of<T>::type;
  const int keep = gld(&q->keep), wave = gld(&q->wave);
  if (keep == 1) v = f;
  if (keep == 2) v = make_val<T>((R)gld(&q->re), (R)gld(&q->im));
  if (wave >= 0) {
    const double* w = waves + (wave * wave_n + row) * 2;
    const T wv = make_val<T>((R)gld(w), (R)gld(w + 1));
    v = gld(&q->kind) == GMES_SRC_SET ? wv : vsub(v, wv);
  }
  return v;
}

}  // namespace gmes_engine
