// What a one-sweep 3-D step leaves out (see FixArgs): dispersive media and
// sources on many cells (the faces of a total-field box), whose E changes
// after its update and before H reads it.
//
// The sweep updates every cell as if there were none: a dispersive cell keeps
// its E.  k_fix_e then updates the dispersive cells from the old H, and applies
// the E sources; k_fix_h computes the H cells next to those again, from the old
// H and the new E, and applies the H sources.  The absorber state of such an H
// cell would have advanced twice: sims that have one take the two-kernel step.
// While the lists are a small part of the cells, each launch is bound by its
// start and the latency of its few dependent loads (4 to 6 us; the two-kernel
// step has one launch per dispersive class and component, two for sources, two
// for ghosts); where media fill much of the grid they move most of E and H a
// second time (complex FP32 384 x 384 x 192 with 12 % dispersive cells: 0.35 and
// 0.29 ms beside the sweep's 0.785), and sims with more take the two-kernel step
// (sweep_list_limit).  Per step, two-kernel step first: complex FP32 192 x 192 x 128,
// dispersive objects and a plane wave, 252 -> 180 us (137 of them the sweep,
// k_fix_h 24, k_fix_e 11); 112^3 slab with a plane wave and a flux plane 105 ->
// 76 (46, 11, 5); FP32 96^3 CPML box with dispersive objects 64 -> 36.
//
// GMES_TYPE: 0 float, 1 double, 2 complex float.
#include "step_common.h"

namespace gmes_engine {

#if GMES_TYPE == 0
typedef float fix_t;
#elif GMES_TYPE == 1
typedef double fix_t;
#else
typedef cplx<float> fix_t;
#endif

template <class T>
using FixPtr = const GMES_CONST FixArgs<T>*;

// Value of an array of one component at thread coordinates x moved by s along
// axis a, wrapped with the ghost phase.
template <class T, class R>
__device__ __forceinline__ T moved(const T* f, int pi, int p, const GMES_CONST int* n, const int x[3], int a, int s,
                                   const GMES_CONST cplx<R>& ph) {
  int y[3] = {x[0], x[1], x[2]};
  bool wrap = false;
#pragma unroll
  for (int q = 0; q < 3; ++q)
    if (q == a) {
      y[q] += s;
      if (y[q] < 0) { y[q] = n[q] - 1; wrap = true; }
      if (y[q] >= n[q]) { y[q] = 0; wrap = true; }
    }
  const T v = gld(f + y[0] * pi + y[1] * p + y[2]);
  return wrap ? phased<T>(ph, v) : v;
}

// The operations of a source group on value v (src_group, kernels.hip).
template <class T>
__device__ __forceinline__ T fix_source(FixPtr<T> m, const SrcGroup& grp, T v) {
  using R = typename real_of<T>::type;
  const int64_t row = (m->ctl->clock - 1) - m->ctl->wave_step0;
  for (int o = grp.begin; o < grp.end; ++o) {
    const DevSrcOp<R> op = m->ops[o];
    if (op.kind == GMES_SRC_SET || op.kind == GMES_SRC_SUB) {
      const double* w = m->waves + (op.wave * m->ctl->wave_n + row) * 2;
      const T wv = make_val<T>((R)w[0], (R)w[1]);
      v = op.kind == GMES_SRC_SET ? wv : vsub(v, wv);
    } else {
      const T* aux = static_cast<const T*>(m->aux[op.aux][op.aux_comp]);
      T a0 = gld(aux + op.i0), a1 = gld(aux + op.i1);
      if (op.wave >= 0) {
        const R env = (R)m->waves[(op.wave * m->ctl->wave_n + row) * 2];
        a0 = vscl(env, a0);
        a1 = vscl(env, a1);
      }
      const T inc = vadd(vscl(op.r0, a0), vscl(op.r1, a1));
      v = op.kind == GMES_SRC_AUX_ADD ? vadd(v, vscl(op.k, inc)) : vsub(v, vscl(op.k, inc));
    }
  }
  return v;
}

template <class T>
__device__ __forceinline__ void fix_e(FixPtr<T> m, int b) {
  using R = typename real_of<T>::type;
  if (b >= m->first_src) {
    const int g = (b - m->first_src) * kFixBlock + (int)threadIdx.x;
    if (g >= m->nge) return;
    const SrcGroup grp = m->groups[g];
    T* F = m->base[grp.comp] + grp.cell;
    gst(F, fix_source<T>(m, grp, gld(F)));
    return;
  }
  int l = m->nade - 1;
  while (l > 0 && b < m->ade[l].first) --l;
  const int q = (b - m->ade[l].first) * kFixBlock + (int)threadIdx.x;
  if (q >= m->ade[l].n) return;
  const int c = m->ade[l].comp, a1 = c == 2 ? 0 : c + 1, a2 = c == 0 ? 2 : c - 1;
  const int flat = gld(m->ade[l].cell + q), r = flat / m->ade[l].s2, i = r / m->ade[l].s1;
  const int x[3] = {i, r - i * m->ade[l].s1, flat - r * m->ade[l].s2};
  const DevRec<R>* rec = m->recs + gld(m->ade[l].rec + q);
  const int e = x[0] * m->pe[c] + x[1] * m->re[c] + x[2];
  const T e_now = gld(m->ei[c] + e);
  const T h2 = gld(m->hi[a2] + x[0] * m->ph[a2] + x[1] * m->rh[a2] + x[2]);
  const T h1 = gld(m->hi[a1] + x[0] * m->ph[a1] + x[1] * m->rh[a1] + x[2]);
  const T D1 = vsub(h2, moved<T, R>(m->hi[a2], m->ph[a2], m->rh[a2], m->n, x, a1, -1, m->phh[a2][a1]));
  const T D2 = vsub(h1, moved<T, R>(m->hi[a1], m->ph[a1], m->rh[a1], m->n, x, a2, -1, m->phh[a1][a2]));
  const T curl = vsub(vdiv(D1, m->d[a1]), vdiv(D2, m->d[a2]));
  const auto cu = [curl] { return curl; };
  gst(m->eo[c] + e, ade_value<T>(m->ade[l].cls, m->coef + gld(&rec->coef_off), gld(&rec->n1), gld(&rec->n2),
                                m->ade[l].state, m->ade[l].state, m->ade[l].n, q, true, e_now, cu));
}

template <class T>
__device__ __forceinline__ void fix_h(FixPtr<T> m, int b) {
  using R = typename real_of<T>::type;
  const int c = b >= m->item_blk[2] ? 2 : b >= m->item_blk[1] ? 1 : 0;
  const int q = (b - m->item_blk[c]) * kFixBlock + (int)threadIdx.x;
  if (q >= m->nitem[c]) return;
  const int a1 = c == 2 ? 0 : c + 1, a2 = c == 0 ? 2 : c - 1;
  const int cell = gld(&m->items[m->first_item[c] + q].cell), grp = gld(&m->items[m->first_item[c] + q].grp);
  const int r = cell / m->n[2], i = r / m->n[1];
  const int x[3] = {i, r - i * m->n[1], cell - r * m->n[2]};
  const int h = x[0] * m->ph[c] + x[1] * m->rh[c] + x[2];
  const DevRec<R>* rec = m->recs + gld(m->hid[c] + h);
  const T old = gld(m->hi[c] + h);
  const T* const e2 = m->eo[a2];
  const T* const e1 = m->eo[a1];
  const T E2 = gld(e2 + x[0] * m->pe[a2] + x[1] * m->re[a2] + x[2]), E1 = gld(e1 + x[0] * m->pe[a1] + x[1] * m->re[a1] + x[2]);
  const T D1 = vsub(moved<T, R>(e2, m->pe[a2], m->re[a2], m->n, x, a1, 1, m->phe[a2][a1]), E2);
  const T D2 = vsub(moved<T, R>(e1, m->pe[a1], m->re[a1], m->n, x, a2, 1, m->phe[a1][a2]), E1);
  const int cls = gld(&rec->cls);
  T v;
  if (cls == GMES_CLS_DUMMY) {
    v = old;
  } else if (cls == GMES_CLS_CONST) {
    v = make_val<T>(gld(&rec->val_re), gld(&rec->val_im));
  } else {  // Dielectric, or CPML at dead coordinates
    const Rows<R, 1> dead{{R(0), R(0), R(1)}};
    T w1, w2;
    v = cpml_value<false, false>(gld(&rec->c0), old, D1, D2, m->d[a1], m->inv_d[a1], m->d[a2], m->inv_d[a2], dead, dead,
                                 T{}, T{}, w1, w2, cls == GMES_CLS_CPML);
  }
  if (grp >= 0) v = fix_source<T>(m, m->groups[grp], v);
  gst(m->ho[c] + h, v);
}

template <class T>
__global__ void __launch_bounds__(kFixBlock) k_fix_e(FixArgs<T>) {
  fix_e<T>((FixPtr<T>)__builtin_amdgcn_kernarg_segment_ptr(), (int)blockIdx.x);
}
template <class T>
__global__ void __launch_bounds__(kFixBlock) k_fix_h(FixArgs<T>) {
  fix_h<T>((FixPtr<T>)__builtin_amdgcn_kernarg_segment_ptr(), (int)blockIdx.x);
}
template <class T, bool E>
__global__ void __launch_bounds__(kFixBlock) k_fix_batch(const FixJob<T>* jobs, int njobs) {
  const GMES_CONST FixJob<T>* J = step_job(jobs, njobs, (int64_t)blockIdx.x);
  const int b = (int)((int64_t)blockIdx.x - J->block0);
  if constexpr (E) fix_e<T>(&J->a, b);
  else fix_h<T>(&J->a, b);
}

template <class T>
void launch_fix_batch(bool electric, const FixJob<T>* jobs, int njobs, int64_t nblocks, hipStream_t st) {
  if (!njobs || !nblocks) return;
  const dim3 grid((unsigned)nblocks), block(kFixBlock);
  if (electric) hipLaunchKernelGGL((k_fix_batch<T, true>), grid, block, 0, st, jobs, njobs);
  else hipLaunchKernelGGL((k_fix_batch<T, false>), grid, block, 0, st, jobs, njobs);
}
template void launch_fix_batch<fix_t>(bool, const FixJob<fix_t>*, int, int64_t, hipStream_t);

template <class T>
void launch_fix_e(const FixArgs<T>& a, hipStream_t st) {
  if (a.eblocks) hipLaunchKernelGGL((k_fix_e<T>), dim3(a.eblocks), dim3(kFixBlock), 0, st, a);
}
template <class T>
void launch_fix_h(const FixArgs<T>& a, hipStream_t st) {
  if (a.hblocks) hipLaunchKernelGGL((k_fix_h<T>), dim3(a.hblocks), dim3(kFixBlock), 0, st, a);
}
template void launch_fix_e<fix_t>(const FixArgs<fix_t>&, hipStream_t);
template void launch_fix_h<fix_t>(const FixArgs<fix_t>&, hipStream_t);

#if GMES_TYPE == 0
// Marks the H cells that read E component c of cell x: of the two others, the
// one at x and the one before along the third axis.
__device__ __forceinline__ void mark_readers(const FixBuild& b, int c, const int x[3]) {
  for (int h = 0; h < 3; ++h) {
    if (h == c) continue;
    const int a = 3 - c - h;  // H component h differs E component c along it
    for (int s = 0; s < 2; ++s) {
      int y[3] = {x[0], x[1], x[2]};
      y[a] = s ? (y[a] ? y[a] - 1 : b.n[a] - 1) : y[a];
      b.mark[h * b.cells + ((int64_t)y[0] * b.n[1] + y[1]) * b.n[2] + y[2]] = 1;
    }
  }
}

__global__ void __launch_bounds__(256) k_fix_mark_ade(FixBuild b) {
  const int q = blockIdx.x * 256 + threadIdx.x;
  if (q >= b.ade_n) return;
  const int flat = b.ade_cell[q], r = flat / b.s2, i = r / b.s1;
  const int x[3] = {i, r - i * b.s1, flat - r * b.s2};
  mark_readers(b, b.comp, x);
}

// thread coordinates of a group's cell
__device__ __forceinline__ void group_cell(const FixBuild& b, const SrcGroup& g, int x[3]) {
  const int e = (int)(g.cell - b.base[g.comp]);
  x[0] = e / b.pi[g.comp];
  const int r = e - x[0] * b.pi[g.comp];
  x[1] = r / b.p[g.comp];
  x[2] = r - x[1] * b.p[g.comp];
  if (g.comp >= 3)
    for (int a = 0; a < 3; ++a) x[a] -= a != g.comp - 3;
}

__global__ void __launch_bounds__(256) k_fix_mark_src(FixBuild b) {
  const int q = blockIdx.x * 256 + threadIdx.x;
  if (q >= b.ngroups) return;
  const SrcGroup g = b.groups[q];
  int x[3];
  group_cell(b, g, x);
  if (g.comp < 3) mark_readers(b, g.comp, x);
  else b.mark[(g.comp - 3) * b.cells + ((int64_t)x[0] * b.n[1] + x[1]) * b.n[2] + x[2]] = 1;
}

__global__ void __launch_bounds__(256) k_fix_count(FixBuild b) {
  __shared__ int n;
  if (threadIdx.x == 0) n = 0;
  __syncthreads();
  const int c = blockIdx.y;
  int mine = 0;
  for (int s = 0; s < kFixMark / 256; ++s) {
    const int64_t q = (int64_t)blockIdx.x * kFixMark + s * 256 + threadIdx.x;
    if (q < b.cells && b.mark[c * b.cells + q]) ++mine;
  }
  atomicAdd(&n, mine);
  __syncthreads();
  if (threadIdx.x == 0) b.count[c * b.nblk + blockIdx.x] = n;
}

// one wave per block of kFixMark cells: items in the order of the cells
__global__ void __launch_bounds__(64) k_fix_fill(FixBuild b) {
  const int c = blockIdx.y, lane = threadIdx.x;
  int at = b.count[c * b.nblk + blockIdx.x];
  for (int s = 0; s < kFixMark / 64; ++s) {
    const int64_t q = (int64_t)blockIdx.x * kFixMark + s * 64 + lane;
    const bool on = q < b.cells && b.mark[c * b.cells + q];
    const unsigned long long all = __ballot(on);
    if (on) {
      b.items[at + __popcll(all & ((1ull << lane) - 1ull))] = FixItem{(int32_t)q, -1};
      const int r = (int)(q / b.n[2]);
      const int x[3] = {r / b.n[1], r % b.n[1], (int)(q - (int64_t)r * b.n[2])};
      const int cls = b.cls[b.hid[c][x[0] * b.pi[3 + c] + x[1] * b.p[3 + c] + x[2]]];
      bool live = cls == GMES_CLS_UPML;
      for (int a = 0; a < 3 && cls == GMES_CLS_CPML; ++a)
        if (a != c) live = live || x[a] < (b.run_h[a] & 0xFFFF) || x[a] >= (b.run_h[a] >> 16);
      if (live) *b.bad = 1;
    }
    at += __popcll(all);
  }
}

// the group of each H source, into its item
__global__ void __launch_bounds__(256) k_fix_groups(FixBuild b) {
  const int q = b.nge + blockIdx.x * 256 + threadIdx.x;
  if (q >= b.ngroups) return;
  const SrcGroup g = b.groups[q];
  int x[3];
  group_cell(b, g, x);
  const int c = g.comp - 3, cell = (int)(((int64_t)x[0] * b.n[1] + x[1]) * b.n[2] + x[2]);
  int lo = b.first_item[c], hi = lo + b.nitem[c] - 1;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (b.items[mid].cell < cell) lo = mid + 1;
    else hi = mid;
  }
  b.items[lo].grp = q;
}

void launch_fix_mark_ade(const FixBuild& b, hipStream_t st) {
  hipLaunchKernelGGL(k_fix_mark_ade, dim3((b.ade_n + 255) / 256), dim3(256), 0, st, b);
}
void launch_fix_mark_src(const FixBuild& b, hipStream_t st) {
  hipLaunchKernelGGL(k_fix_mark_src, dim3((b.ngroups + 255) / 256), dim3(256), 0, st, b);
}
void launch_fix_count(const FixBuild& b, hipStream_t st) {
  hipLaunchKernelGGL(k_fix_count, dim3(b.nblk, 3), dim3(256), 0, st, b);
}
void launch_fix_fill(const FixBuild& b, hipStream_t st) {
  hipLaunchKernelGGL(k_fix_fill, dim3(b.nblk, 3), dim3(64), 0, st, b);
  if (b.ngroups > b.nge)
    hipLaunchKernelGGL(k_fix_groups, dim3((b.ngroups - b.nge + 255) / 256), dim3(256), 0, st, b);
}
#endif

}  // namespace gmes_engine
