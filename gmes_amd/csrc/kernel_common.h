// Device helpers shared by the kernel files: real and complex arithmetic,
// global-memory accessors, curl operands and the E ghost images.
#pragma once

#include "engine_kernels.h"

namespace gmes_engine {

// ---------------------------------------------------------------- arithmetic
template <class R> __device__ __forceinline__ R vadd(R a, R b) { return a + b; }
template <class R> __device__ __forceinline__ R vsub(R a, R b) { return a - b; }
template <class R> __device__ __forceinline__ R vscl(R s, R a) { return s * a; }
template <class R> __device__ __forceinline__ R vdiv(R a, R d) { return a / d; }
template <class R> __device__ __forceinline__ cplx<R> vadd(cplx<R> a, cplx<R> b) { return {a.re + b.re, a.im + b.im}; }
template <class R> __device__ __forceinline__ cplx<R> vsub(cplx<R> a, cplx<R> b) { return {a.re - b.re, a.im - b.im}; }
template <class R> __device__ __forceinline__ cplx<R> vscl(R s, cplx<R> a) { return {s * a.re, s * a.im}; }
template <class R> __device__ __forceinline__ cplx<R> vdiv(cplx<R> a, R d) { return {a.re / d, a.im / d}; }
template <class R> __device__ __forceinline__ cplx<R> cmul(cplx<R> a, cplx<R> b) {
  return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
template <class T> __device__ __forceinline__ T vzero() { return T{}; }

// Global-memory accessors.  A device allocation reached through a pointer
// read from memory (a batch job table) is not known to be global: plain
// accesses through it become generic (flat) instructions, which also wait
// on LDS traffic.  These access it through an address-space-1 pointer.
#define GMES_GLOBAL __attribute__((address_space(1)))
template <class T>
__device__ __forceinline__ T gld(const T* p) {
  return *(const GMES_GLOBAL T*)p;
}
template <class T>
__device__ __forceinline__ void gst(T* p, T v) {
  *(GMES_GLOBAL T*)p = v;
}
// complex words and records move as native vectors (a class-typed copy
// would take a generic pointer again)
template <class R>
using vec2_t = R __attribute__((ext_vector_type(2)));
template <class R>
__device__ __forceinline__ cplx<R> gld(const cplx<R>* p) {
  const vec2_t<R> v = *(const GMES_GLOBAL vec2_t<R>*)p;
  return {v.x, v.y};
}
template <class R>
__device__ __forceinline__ void gst(cplx<R>* p, cplx<R> v) {
  *(GMES_GLOBAL vec2_t<R>*)p = vec2_t<R>{v.re, v.im};
}
template <class R>
__device__ __forceinline__ DevRec<R> load_rec(const DevRec<R>* p) {
  constexpr int n = sizeof(DevRec<R>) / 16;
  union {
    DevRec<R> r;
    i4_t v[n];
  } u;
#pragma unroll
  for (int c = 0; c < n; ++c) u.v[c] = ((const GMES_GLOBAL i4_t*)p)[c];
  return u.r;
}

// Streaming accesses: field words and material ids are touched once per
// launch, so they are loaded and stored non-temporally (no reuse to keep
// in L2).  GMES_NT=0 builds the plain form.
#ifndef GMES_NT
#define GMES_NT 1
#endif
template <class R> __device__ __forceinline__ R ld_nt(const R* p) {
#if GMES_NT
  return __builtin_nontemporal_load((const __attribute__((address_space(1))) R*)p);
#else
  return *(const __attribute__((address_space(1))) R*)p;
#endif
}
template <class R> __device__ __forceinline__ cplx<R> ld_nt(const cplx<R>* p) {
  return {ld_nt(&p->re), ld_nt(&p->im)};
}
template <class R> __device__ __forceinline__ void st_nt(R* p, R v) {
#if GMES_NT
  __builtin_nontemporal_store(v, (__attribute__((address_space(1))) R*)p);
#else
  *(__attribute__((address_space(1))) R*)p = v;
#endif
}
template <class R> __device__ __forceinline__ void st_nt(cplx<R>* p, cplx<R> v) {
  st_nt(&p->re, v.re);
  st_nt(&p->im, v.im);
}
template <class R> __device__ __forceinline__ R re_of(R a) { return a; }
template <class R> __device__ __forceinline__ R re_of(cplx<R> a) { return a.re; }
template <class R> __device__ __forceinline__ R im_of(R) { return R(0); }
template <class R> __device__ __forceinline__ R im_of(cplx<R> a) { return a.im; }
template <class T> __device__ __forceinline__ T make_val(typename real_of<T>::type re, typename real_of<T>::type im);
template <> __device__ __forceinline__ float make_val<float>(float re, float) { return re; }
template <> __device__ __forceinline__ double make_val<double>(double re, double) { return re; }
template <> __device__ __forceinline__ cplx<float> make_val<cplx<float>>(float re, float im) { return {re, im}; }
template <> __device__ __forceinline__ cplx<double> make_val<cplx<double>>(double re, double im) { return {re, im}; }


template <class T>
__device__ __forceinline__ T ld(const FieldArgs<T>& a, int c, int i, int j, int k) {
  // an inactive component is (1,1,1) and reads as zero (src/cpp23_support.hh:52-74)
  if (!(a.active & (1u << c))) return vzero<T>();
  return gld(a.f[c] + didx(a, c, i, j, k));
}

// Curl differences D1, D2 of component C at (i,j,k): src/pw_dielectric.hh
// :118-119 (Ex) :157-158 (Ey) :197-198 (Ez) :292-293 (Hx) :331-332 (Hy) :370-371 (Hz)
template <int C, class T>
__device__ __forceinline__ void curl_terms(const FieldArgs<T>& a, int i, int j, int k, T& D1, T& D2) {
  if constexpr (C == 0) {
    D1 = vsub(ld(a, 5, i + 1, j + 1, k), ld(a, 5, i + 1, j, k));
    D2 = vsub(ld(a, 4, i + 1, j, k + 1), ld(a, 4, i + 1, j, k));
  } else if constexpr (C == 1) {
    D1 = vsub(ld(a, 3, i, j + 1, k + 1), ld(a, 3, i, j + 1, k));
    D2 = vsub(ld(a, 5, i + 1, j + 1, k), ld(a, 5, i, j + 1, k));
  } else if constexpr (C == 2) {
    D1 = vsub(ld(a, 4, i + 1, j, k + 1), ld(a, 4, i, j, k + 1));
    D2 = vsub(ld(a, 3, i, j + 1, k + 1), ld(a, 3, i, j, k + 1));
  } else if constexpr (C == 3) {
    D1 = vsub(ld(a, 2, i, j, k - 1), ld(a, 2, i, j - 1, k - 1));
    D2 = vsub(ld(a, 1, i, j - 1, k), ld(a, 1, i, j - 1, k - 1));
  } else if constexpr (C == 4) {
    D1 = vsub(ld(a, 0, i - 1, j, k), ld(a, 0, i - 1, j, k - 1));
    D2 = vsub(ld(a, 2, i, j, k - 1), ld(a, 2, i - 1, j, k - 1));
  } else {
    D1 = vsub(ld(a, 1, i, j - 1, k), ld(a, 1, i - 1, j - 1, k));
    D2 = vsub(ld(a, 0, i - 1, j, k), ld(a, 0, i - 1, j - 1, k));
  }
}

template <int C> struct Ax;
template <> struct Ax<0> { static constexpr int a1 = 1, a2 = 2, a0 = 0; };
template <> struct Ax<1> { static constexpr int a1 = 2, a2 = 0, a0 = 1; };
template <> struct Ax<2> { static constexpr int a1 = 0, a2 = 1, a0 = 2; };
template <> struct Ax<3> { static constexpr int a1 = 1, a2 = 2, a0 = 0; };
template <> struct Ax<4> { static constexpr int a1 = 2, a2 = 0, a0 = 1; };
template <> struct Ax<5> { static constexpr int a1 = 0, a2 = 1, a0 = 2; };

__device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ cplx<float> fma_(float a, cplx<float> b, cplx<float> c) {
  return {__builtin_fmaf(a, b.re, c.re), __builtin_fmaf(a, b.im, c.im)};
}

// Periodic / Bloch ghost planes of E written by the thread that owns the
// source cell (the copy k_ghost<E> makes, fused into the E update when
// nothing else writes or reads the planes involved before that copy would
// run).  x is the cell's new value; ix its storage index.  Same phase
// products and corner order as k_ghost: ph1 * x on the a1 ghost plane,
// ph2 * x on the a2 plane, ph2 * (ph1 * x) on the corner line.
template <class T>
__device__ __forceinline__ T ghost_phase(const cplx<typename real_of<T>::type>& ph, T x) {
  if constexpr (is_cplx<T>::value) return cmul(ph, x);
  else return x;
}

template <class T>
__device__ __forceinline__ void fused_ghost(const MainArgs<T>& m, int C, T* __restrict__ F, const int ix[3], T x) {
  const int a1 = m.gax[C][0], a2 = m.gax[C][1];
  const int* sh = m.fa.s[C];
  const int dst1 = sh[a1] - 1, dst2 = sh[a2] - 1;
  const bool on1 = ix[a1] == 0, on2 = ix[a2] == 0;
  if (!on1 && !on2) return;
  int g[3] = {ix[0], ix[1], ix[2]};
  T x1 = x;
  if (on1) {
    x1 = ghost_phase<T>(m.gph[C][0], x);
    g[a1] = dst1;
    gst(F + didx(m.fa, C, g[0], g[1], g[2]), x1);
    g[a1] = 0;
  }
  if (on2) {
    g[a2] = dst2;
    gst(F + didx(m.fa, C, g[0], g[1], g[2]), ghost_phase<T>(m.gph[C][1], x));
    if (on1) {
      g[a1] = dst1;
      gst(F + didx(m.fa, C, g[0], g[1], g[2]), ghost_phase<T>(m.gph[C][1], x1));
    }
  }
}

// Dispersive (ADE) cells: the new value of cell q of a list of n cells from
// its old value e_now and the curl cu() = D1/d1 - D2/d2, which the two-kernel
// step's lists load when the state words are on their way back (before them,
// the Drude list of 160^3 FP64 took 82 us for 76).  State words are read
// from st and the new ones written to so (the same array, or the other set
// of a one-sweep step; `keep` false: not at all).  a: the record's
// coefficients, P1 and P2 its pole counts.
//
// Drude and Lorentz poles: src/pw_drude.hh:90-101,145-150; src/pw_lorentz.hh:96-107,150-156
template <class T, class Cu>
__device__ __forceinline__ T ade_drude_value(const typename real_of<T>::type* a, int P, const T* st, T* so, int n,
                                             int q, bool keep, T e_now, Cu cu) {
  const auto* cc = a + 3 * P;
  T sum = vzero<T>();
  for (int p = 0; p < P; ++p) {
    const T q_old = ld_nt(st + p * n + q);
    const T q_now = ld_nt(st + (P + p) * n + q);
    const T q_new = vadd(vadd(vscl(gld(a + 3 * p), q_old), vscl(gld(a + 3 * p + 1), q_now)), vscl(gld(a + 3 * p + 2), e_now));
    if (keep) {
      st_nt(so + p * n + q, q_now);
      st_nt(so + (P + p) * n + q, q_new);
    }
    sum = vadd(sum, vsub(q_new, q_now));
  }
  const T c = cu();
  return vadd(vadd(vscl(gld(cc), c), vscl(gld(cc + 1), sum)), vscl(gld(cc + 2), e_now));
}

// Drude-critical-points, ADE form: src/pw_dcp.hh:105-167,200-225
// words: 0 e_old | 1..D q_old | D+1..2D q_now | 2D+1.. p_old | 2D+C+1.. p_now
template <class T, class Cu>
__device__ __forceinline__ T ade_dcp_value(const typename real_of<T>::type* a, int D, int NC, const T* st, T* so,
                                           int n, int q, bool keep, T e_now, Cu cu) {
  using R = typename real_of<T>::type;
  const R* b = a + 3 * D;
  const R* cc = b + 5 * NC;
  const T e_old = gld(st + q);
  T ds = vzero<T>(), cs = vzero<T>();
  for (int p = 0; p < D; ++p)
    ds = vadd(ds, vsub(vscl(R(1) - gld(a + 3 * p + 1), gld(st + (1 + D + p) * n + q)),
                       vscl(gld(a + 3 * p), gld(st + (1 + p) * n + q))));
  for (int p = 0; p < NC; ++p)
    cs = vadd(cs, vsub(vscl(R(1) - gld(b + 5 * p + 1), gld(st + (1 + 2 * D + NC + p) * n + q)),
                       vscl(gld(b + 5 * p), gld(st + (1 + 2 * D + p) * n + q))));
  const T c = cu();
  const T e_new = vadd(vadd(vadd(vscl(gld(cc), c), vscl(gld(cc + 1), vadd(ds, cs))), vscl(gld(cc + 2), e_old)),
                       vscl(gld(cc + 3), e_now));
  if (!keep) return e_new;
  const T mix = vadd(vadd(e_old, vscl(R(2), e_now)), e_new);
  for (int p = 0; p < D; ++p) {
    const T qo = gld(st + (1 + p) * n + q), qn = gld(st + (1 + D + p) * n + q);
    const T qq = vadd(vadd(vscl(gld(a + 3 * p), qo), vscl(gld(a + 3 * p + 1), qn)), vscl(gld(a + 3 * p + 2), mix));
    st_nt(so + (1 + p) * n + q, qn);
    st_nt(so + (1 + D + p) * n + q, qq);
  }
  for (int p = 0; p < NC; ++p) {
    const T po = gld(st + (1 + 2 * D + p) * n + q), pn = gld(st + (1 + 2 * D + NC + p) * n + q);
    const T pp = vadd(vadd(vadd(vadd(vscl(gld(b + 5 * p), po), vscl(gld(b + 5 * p + 1), pn)),
                                vscl(gld(b + 5 * p + 2), e_old)),
                           vscl(gld(b + 5 * p + 3), e_now)),
                      vscl(gld(b + 5 * p + 4), e_new));
    st_nt(so + (1 + 2 * D + p) * n + q, pn);
    st_nt(so + (1 + 2 * D + NC + p) * n + q, pp);
  }
  st_nt(so + q, e_now);
  return e_new;
}

// Drude-critical-points, PLRC/RC form: src/pw_dcp.hh:467-518,564-586.
// State words are complex for any field type: psi_dp (re part = psi_dp_re,
// im part = psi_dp_im), psi_cp_re, psi_cp_im.
template <class T, class Cu>
__device__ __forceinline__ T ade_plrc_value(const typename real_of<T>::type* a, int D, int NC,
                                            const cplx<typename real_of<T>::type>* st,
                                            cplx<typename real_of<T>::type>* so, int n, int q, bool keep, T fv, Cu cu) {
  using R = typename real_of<T>::type;
  using Z = cplx<R>;
  const R* b = a + 3 * D;
  const R* cc = b + 6 * NC;
  const Z e_now = {re_of(fv), im_of(fv)};
  R sdr = R(0), sdi = R(0);
  for (int p = 0; p < D; ++p) {
    const Z v = gld(st + p * n + q);
    sdr = sdr + v.re;
    sdi = sdi + v.im;
  }
  Z scr = {R(0), R(0)}, sci = {R(0), R(0)};
  for (int p = 0; p < NC; ++p) scr = vadd(scr, gld(st + (D + p) * n + q));
  for (int p = 0; p < NC; ++p) sci = vadd(sci, gld(st + (D + NC + p) * n + q));
  const Z psi = {sdr + scr.re, sdi + sci.re};  // .real() of the imaginary-part sum
  Z e_new;
  const T c = cu();
  if constexpr (is_cplx<T>::value) {
    e_new = vadd(vadd(vscl(gld(cc), Z{c.re, c.im}), vscl(gld(cc + 1), e_now)), vscl(gld(cc + 2), psi));
  } else {
    e_new.re = (gld(cc) * c + gld(cc + 1) * e_now.re) + gld(cc + 2) * psi.re;
    e_new.im = gld(cc + 1) * e_now.im + gld(cc + 2) * psi.im;
  }
  if (keep) {
    for (int p = 0; p < D; ++p) {
      Z v = gld(st + p * n + q);
      v.re = (gld(a + 3 * p) * e_new.re + gld(a + 3 * p + 1) * e_now.re) + gld(a + 3 * p + 2) * v.re;
      v.im = (gld(a + 3 * p) * e_new.im + gld(a + 3 * p + 1) * e_now.im) + gld(a + 3 * p + 2) * v.im;
      gst(so + p * n + q, v);
    }
    for (int p = 0; p < NC; ++p) {
      const Z b0 = {gld(b + 6 * p), gld(b + 6 * p + 1)}, b1 = {gld(b + 6 * p + 2), gld(b + 6 * p + 3)},
              b2 = {gld(b + 6 * p + 4), gld(b + 6 * p + 5)};
      const Z vr = gld(st + (D + p) * n + q), vi = gld(st + (D + NC + p) * n + q);
      gst(so + (D + p) * n + q, vadd(vadd(vscl(e_new.re, b0), vscl(e_now.re, b1)), cmul(b2, vr)));
      gst(so + (D + NC + p) * n + q, vadd(vadd(vscl(e_new.im, b0), vscl(e_now.im, b1)), cmul(b2, vi)));
    }
  }
  return make_val<T>(e_new.re, e_new.im);
}

template <class T, class Cu>
__device__ __forceinline__ T ade_value(int cls, const typename real_of<T>::type* a, int P1, int P2, const void* st,
                                       void* so, int n, int q, bool keep, T e_now, Cu cu) {
  using Z = cplx<typename real_of<T>::type>;
  if (cls == GMES_CLS_DRUDE)
    return ade_drude_value<T>(a, P1, static_cast<const T*>(st), static_cast<T*>(so), n, q, keep, e_now, cu);
  if (cls == GMES_CLS_DCP_ADE)
    return ade_dcp_value<T>(a, P1, P2, static_cast<const T*>(st), static_cast<T*>(so), n, q, keep, e_now, cu);
  return ade_plrc_value<T>(a, P1, P2, static_cast<const Z*>(st), static_cast<Z*>(so), n, q, keep, e_now, cu);
}

// Batched launches: block -> job by binary search on the jobs' first
// blocks (uniform across a block).
template <class J>
__device__ __forceinline__ int find_job(const J* jobs, int njobs, int64_t b) {
  int lo = 0, hi = njobs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (jobs[mid].block0 <= b) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

}  // namespace gmes_engine
