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
