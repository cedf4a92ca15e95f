// One-sweep 1-D step: a whole leapfrog step of a TEM line in one launch.
//
// The lines are short (hundreds of cells), so a step is its launches: ghosts,
// E, source, ghosts, H took 17.5 us a step (801 cells, FP64), 23 us for the
// auxiliary grid of a total-field box; one launch takes 4.7.  As in 2-D the step reads one set of
// buffers and writes another; a thread owns a cell, a block's last thread is a
// rim.  Everything that does not depend on a cell's record (field operands,
// absorber words and rows) is loaded with its id, so the chain of loads is the
// id, the record, and a dispersive cell's state.
//
// GMES_TYPE: 0 float, 1 double, 2 complex float, 3 complex double.
#include "step_common.h"

namespace gmes_engine {

#if GMES_TYPE == 0
typedef float step1_t;
#elif GMES_TYPE == 1
typedef double step1_t;
#elif GMES_TYPE == 2
typedef cplx<float> step1_t;
#else
typedef cplx<double> step1_t;
#endif

template <class T>
using Step1Ptr = const GMES_CONST Step1Args<T>*;

template <class T, int PML, int F>
struct Step1Ops {
  using R = typename real_of<T>::type;
  T f, s;
  R r[3][PML == 1 ? 3 : 2];  // rows along the first curl axis, the second, the own one
  DevRec<R> rec;
};

// Operands of field F (0 E, 1 H) at cell q.
template <class T, int PML, int F>
__device__ __forceinline__ void step1_load(Step1Ptr<T> m, int q, Step1Ops<T, PML, F>& l) {
  const unsigned e = (unsigned)(q * m->st[F]);
  const uint16_t id = gld(m->ids[F] + e);
  l.f = gld(m->fi[F] + e);
  constexpr int line = F == 0 ? 1 : 0;  // which curl axis is the line's
  if constexpr (PML != 0) {
    l.s = gld(m->si[F] + e);
    constexpr int w = PML == 1 ? 3 : 6;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      if (PML == 1 && a == 2) continue;  // CPML: no row of the own axis
      const auto* p = m->row[F][a] + (a == line ? q * w : 0) + (PML == 2 ? 2 * a : 0);
#pragma unroll
      for (int v = 0; v < (PML == 1 ? 3 : 2); ++v) l.r[a][v] = gld(p + v);
    }
  }
  l.rec = load_rec(m->recs + id);
}

// New value of the cell from the difference D along the line.
template <class T, int PML, int F>
__device__ __forceinline__ T step1_value(Step1Ptr<T> m, int q, const Step1Ops<T, PML, F>& l, T D, bool keep) {
  using R = typename real_of<T>::type;
  constexpr bool E = F == 0;
  // axes: 0 e, 1 h, 2 the line.  E: curl axes h, line; H: line, e
  constexpr int a1 = E ? 1 : 2, a2 = E ? 2 : 0;
  const T D1 = E ? T{} : D, D2 = E ? D : T{};
  const int cls = l.rec.cls;
  const unsigned e = (unsigned)(q * m->st[F]);
  if (cls == GMES_CLS_DUMMY) return l.f;
  if (cls == GMES_CLS_CONST) return make_val<T>(l.rec.val_re, l.rec.val_im);
  if constexpr (PML == 1) {
    if (cls == GMES_CLS_CPML) {
      Rows<R, 1> r1, r2;
#pragma unroll
      for (int v = 0; v < 3; ++v) {
        r1.v[v] = l.r[0][v];
        r2.v[v] = l.r[1][v];
      }
      T n1, n2;
      const T v = cpml_value<E, false>(l.rec.c0, l.f, D1, D2, m->d[a1], m->inv_d[a1], m->d[a2], m->inv_d[a2], r1, r2,
                                       E ? T{} : l.s, E ? l.s : T{}, n1, n2);
      // live words only (psi_live, kernels.hip): with c = 0 the word is +0
      if (keep && (E ? r2 : r1).v[1] != R(0)) gst(m->so[F] + e, E ? n2 : n1);
      return v;
    }
  } else if constexpr (PML == 2) {
    if (cls == GMES_CLS_UPML) {
      Rows<R, 2> r1, r2, r0;
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        r1.v[v] = l.r[0][v];
        r2.v[2 + v] = l.r[1][v];
        r0.v[4 + v] = l.r[2][v];
      }
      const R c = std::is_same<R, float>::value ? l.rec.inv_eps : l.rec.eps_mu;
      T n;
      const T v = upml_value<E, false>(c, l.f, D1, D2, m->d[a1], m->inv_d[a1], m->d[a2], m->inv_d[a2], r1, r2, r0, l.s, n);
      if (keep) gst(m->so[F] + e, n);
      return v;
    }
  }
  if (E && cls >= GMES_CLS_DRUDE) {
    const T curl = vsub(vdiv(D1, m->d[a1]), vdiv(D2, m->d[a2]));
    const auto cu = [curl] { return curl; };
    const int k = cls - GMES_CLS_DRUDE;
    return ade_value<T>(cls, m->coef + l.rec.coef_off, l.rec.n1, l.rec.n2, k == 0 ? m->ade_in[0] : k == 1 ? m->ade_in[1] : m->ade_in[2],
                        k == 0 ? m->ade_out[0] : k == 1 ? m->ade_out[1] : m->ade_out[2],
                        k == 0 ? m->ade_n[0] : k == 1 ? m->ade_n[1] : m->ade_n[2], gld(m->adeq + e), keep, l.f, cu);
  }
  return plain_value<E, false>(l.rec.c0, l.f, D1, D2, m->d[a1], m->inv_d[a1], m->d[a2], m->inv_d[a2]);
}

template <class T>
__device__ __forceinline__ T step1_sources(Step1Ptr<T> m, int F, int q, int64_t row, int64_t wave_n, T v) {
  using R = typename real_of<T>::type;
  for (int s = 0; s < m->nsrc; ++s)
    if (m->src[s].c == F && m->src[s].q == q) {
      const double* w = m->waves + (m->src[s].wave * wave_n + row) * 2;
      const T wv = make_val<T>((R)gld(w), (R)gld(w + 1));
      v = m->src[s].kind == GMES_SRC_SET ? wv : vsub(v, wv);
    }
  return v;
}

template <class T, int PML>
__device__ __forceinline__ void step1d_tile(Step1Ptr<T> m, int blk, T* eb) {
  using R = typename real_of<T>::type;
  const int t = threadIdx.x, q0 = blk * (kStep1Threads - 1), q = q0 + t, n = m->n;
  const bool used = q <= n, own = q < n && t < kStep1Threads - 1;
  const int qe = q >= n ? 0 : q;
  int64_t row = 0, wave_n = 0;
  if (m->nsrc || blk == 0) {
    const int64_t clk = m->ctl->clk[m->par];
    row = clk - m->ctl->wave_step0;
    wave_n = m->ctl->wave_n;
    if (blk == 0 && t == 0) {  // the step's tick
      m->ctl->clk[1 - m->par] = clk + 1;
      m->ctl->clock = clk + 1;
    }
  }
  Step1Ops<T, PML, 0> le{};
  Step1Ops<T, PML, 1> lh{};
  T hm{}, e{};
  if (used) {
    step1_load<T, PML, 0>(m, qe, le);
    step1_load<T, PML, 1>(m, qe, lh);
    hm = gld(m->fi[1] + (unsigned)((qe ? qe - 1 : n - 1) * m->st[1]));
    const cplx<R> ph{m->ph[1][1].re, m->ph[1][1].im};
    if (qe == 0) hm = ghost_phase<T>(ph, hm);
    e = step1_value<T, PML, 0>(m, qe, le, vsub(lh.f, hm), own);
    e = step1_sources<T>(m, 0, qe, row, wave_n, e);
  }
  eb[t] = e;
  __syncthreads();
  if (!own) return;
  const cplx<R> pc0{m->ph[0][0].re, m->ph[0][0].im}, pl0{m->ph[0][1].re, m->ph[0][1].im}, pc1{m->ph[1][0].re, m->ph[1][0].im},
      pl1{m->ph[1][1].re, m->ph[1][1].im};
  T ep = eb[t + 1];
  if (q == n - 1) ep = ghost_phase<T>(pl0, ep);
  T h = step1_value<T, PML, 1>(m, q, lh, vsub(ep, e), true);
  h = step1_sources<T>(m, 1, q, row, wave_n, h);
  T* const pe = m->fo[0] + (int64_t)q * m->st[0];
  T* const ph = m->fo[1] + (int64_t)q * m->st[1];
  gst(pe, e);
  gst(ph, h);
  if (m->ghosts) {  // E's images from the new values, H's from the old ones
    const T ec = ghost_phase<T>(pc0, e);
    if (m->gc[0]) gst(pe + m->gc[0], ec);
    if (q == 0) {
      gst(pe + (int64_t)n * m->st[0], ghost_phase<T>(pl0, e));
      if (m->gc[0]) gst(pe + (int64_t)n * m->st[0] + m->gc[0], ghost_phase<T>(pl0, ec));
    }
    if (m->gc[1]) gst(ph + m->gc[1], ghost_phase<T>(pc1, lh.f));
    if (q == n - 1) {
      const T hl = ghost_phase<T>(pl1, lh.f);
      gst(ph - (int64_t)n * m->st[1], hl);
      if (m->gc[1]) gst(ph - (int64_t)n * m->st[1] + m->gc[1], ghost_phase<T>(pc1, hl));
    }
  }
}

template <class T, int PML>
__global__ void __launch_bounds__(kStep1Threads) k_step1d(Step1Args<T>) {
  __shared__ T eb[kStep1Threads];
  step1d_tile<T, PML>((Step1Ptr<T>)__builtin_amdgcn_kernarg_segment_ptr(), (int)blockIdx.x, eb);
}

template <class T>
__global__ void __launch_bounds__(kStep1Threads) k_step1d_batch(const Step1Job<T>* jobs, int njobs) {
  __shared__ T eb[kStep1Threads];
  const GMES_CONST Step1Job<T>* J = step_job(jobs, njobs, (int64_t)blockIdx.x);
  const int blk = (int)((int64_t)blockIdx.x - J->block0);
  if (J->a.absorber == 0) step1d_tile<T, 0>(&J->a, blk, eb);
  else if (J->a.absorber == 1) step1d_tile<T, 1>(&J->a, blk, eb);
  else step1d_tile<T, 2>(&J->a, blk, eb);
}

template <class T>
void launch_step1d_batch(const Step1Job<T>* jobs, int njobs, int64_t nblocks, hipStream_t st) {
  if (njobs) hipLaunchKernelGGL((k_step1d_batch<T>), dim3((unsigned)nblocks), dim3(kStep1Threads), 0, st, jobs, njobs);
}
template void launch_step1d_batch<step1_t>(const Step1Job<step1_t>*, int, int64_t, hipStream_t);

template <class T>
void launch_step1d(const Step1Args<T>& m, hipStream_t st) {
  const dim3 grid((m.n + kStep1Threads - 2) / (kStep1Threads - 1)), block(kStep1Threads);
  if (m.absorber == 0) hipLaunchKernelGGL((k_step1d<T, 0>), grid, block, 0, st, m);
  else if (m.absorber == 1) hipLaunchKernelGGL((k_step1d<T, 1>), grid, block, 0, st, m);
  else hipLaunchKernelGGL((k_step1d<T, 2>), grid, block, 0, st, m);
}
template void launch_step1d<step1_t>(const Step1Args<step1_t>&, hipStream_t);

}  // namespace gmes_engine
