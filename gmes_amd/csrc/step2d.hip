// One-sweep 2-D step: a whole leapfrog step of a collapsed-z mode (TMz, TEz)
// in one kernel.
//
// The two-kernel step needs four launches (ghosts, E, source, H) and one
// more per dispersive class and component; a small sim's step is those
// launches (200^2 FP64: 4.1 us each), a large one's the second pass over
// the fields.  Here the fields are read from one set of buffers and written
// to another (see step3d.hip), so one launch does it all: 6 words per cell.
// Measured per step, before and after: TMz 200^2 FP64 CPML 16.6 -> 5.7 us,
// TEz 517 x 389 FP32 UPML with dispersive rods 38.9 -> 13, Bloch TMz 96^2
// complex FP64 13.7 -> 4.6, TMz 2048^2 FP32 CPML 89 -> 30 (3.6 TB/s).  Small
// sims: one launch and the latency of its two or three rows.  Large ones: the
// scalar and vector instructions of a row (with every pointer read where it is
// used, 180 scalar instructions a row, 2048^2 took 37 us; held to 64
// registers for two more waves a SIMD it spills, 40 us).
//
// A block owns a stretch of columns (j) and marches over rows (i), a thread
// per column, with the operands of the next two rows on their way.  In row
// q it puts its H into LDS, updates E(q) with the H of the column before
// and of the row before, puts that into LDS for the next row, and updates
// H(q - 1) with E(q) and the E of the next column at q - 1; one barrier a
// row.  A block's last row is a rim, whose E it computes for the H of the
// row below.  Rows that fit a block wrap inside it; longer ones have two
// more lanes, one computing E in the column after the stretch, one loading
// H in the column before.  Dispersive cells read their state from one set
// of arrays and write another, so rims can compute them too.
//
// GMES_TYPE: 0 float, 1 double, 2 complex float, 3 complex double.
#include "step_common.h"

namespace gmes_engine {

#if GMES_TYPE == 0
typedef float step2_t;
#elif GMES_TYPE == 1
typedef double step2_t;
#elif GMES_TYPE == 2
typedef cplx<float> step2_t;
#else
typedef cplx<double> step2_t;
#endif

template <class T>
using Step2Ptr = const GMES_CONST Step2Args<T>*;
// arguments are read where they are used (see StepPtr)
template <class T>
__device__ __forceinline__ Step2Ptr<T> fresh2(Step2Ptr<T> p) {
  asm("" : "+s"(p));
  return p;
}

// Operands of a row, loaded two rows ahead.
template <class T, int PML>
struct Step2Ops {
  T f[3];
  T s[PML == 0 ? 1 : 4];  // CPML: E x, y words, H x, y words; UPML: the components'
  unsigned id;
};

// Update of the component along C; y holds its row along y (a register
// copy), x and z rows are the same for the whole block.
template <bool E, int C, bool X, class T, class R>
__device__ __forceinline__ T step2_cpml(Step2Ptr<T> m, R c, T f, T D1, T D2, int q, const R* y, T ox, T oy, T& nx,
                                        T& ny) {
  constexpr int a1 = (C + 1) % 3, a2 = (C + 2) % 3;
  Rows<R, 1> r[3];
#pragma unroll
  for (int v = 0; v < 3; ++v) {
    if (a1 == 0 || a2 == 0) r[0].v[v] = cld(m->row[C][0] + q * 3 + v);
    r[1].v[v] = y[v];
    if (a1 == 2 || a2 == 2) r[2].v[v] = cld(m->row[C][2] + v);
  }
  const T o[3] = {ox, oy, T{}};
  T n1, n2;
  const T v = cpml_value<E, X>(c, f, D1, D2, m->d[a1], m->inv_d[a1], m->d[a2], m->inv_d[a2], r[a1], r[a2], o[a1],
                               o[a2], n1, n2);
  if (a1 == 0) nx = n1;
  if (a2 == 0) nx = n2;
  if (a1 == 1) ny = n1;
  if (a2 == 1) ny = n2;
  return v;
}

template <bool E, int C, bool X, class T, class R>
__device__ __forceinline__ T step2_upml(Step2Ptr<T> m, R c, T f, T D1, T D2, int q, const R* y, T o, T& n) {
  constexpr int a1 = (C + 1) % 3, a2 = (C + 2) % 3;
  Rows<R, 2> r[3];
  // of each axis the pair its place needs: c1, c2 of a1, c3, c4 of a2, c5, c6 of the own
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int p = a == a1 ? 0 : a == a2 ? 2 : 4;
#pragma unroll
    for (int v = 0; v < 2; ++v)
      r[a].v[p + v] = a == 0 ? cld(m->row[C][0] + q * 6 + p + v) : a == 1 ? y[v] : cld(m->row[C][2] + p + v);
  }
  return upml_value<E, X>(c, f, D1, D2, m->d[a1], m->inv_d[a1], m->d[a2], m->inv_d[a2], r[a1], r[a2], r[C], o, n);
}

// Element at byte offset o of an array (uniform base, 32-bit lane offset).
template <class T>
__device__ __forceinline__ T at(const T* p, unsigned o) {
  return gld(reinterpret_cast<const T*>(reinterpret_cast<const char*>(p) + o));
}
template <class T>
__device__ __forceinline__ void put(T* p, unsigned o, T v) {
  st_nt(reinterpret_cast<T*>(reinterpret_cast<char*>(p) + o), v);
}

template <class T, bool TM, int PML, bool ADE, bool X>
__device__ __forceinline__ void step2d_tile(Step2Ptr<T> mp, unsigned blk, char* lds) {
  using R = typename real_of<T>::type;
  constexpr unsigned S = sizeof(T);
  Step2Ptr<T> m = fresh2<T>(mp);
  const int t = threadIdx.x, nt = (int)blockDim.x;
  Step2Ent<R>* const et = reinterpret_cast<Step2Ent<R>*>(lds);
  {
    static_assert(sizeof(Step2Ent<R>) % 16 == 0, "entries move as 16-byte words");
    constexpr int kq = sizeof(Step2Ent<R>) / 16;
    i4_t* dst = reinterpret_cast<i4_t*>(et);
    const i4_t* src = reinterpret_cast<const i4_t*>(m->tab);
    for (int e = t; e < m->nent * kq; e += nt) dst[e] = gld(src + e);
  }
  T* const xb = reinterpret_cast<T*>(et + m->nent);  // [2][nt] H for the next column
  T* const eb = xb + 2 * nt;                         // [2][nt] E for the column before
  // each XCD a contiguous run of tiles: neighbours share rim lines in its L2
  const unsigned per = ((unsigned)m->nblk + 7u) / 8u;
  const unsigned b = (blk & 7u) * per + (blk >> 3);
  if ((blk >> 3) >= per || b >= (unsigned)m->nblk) return;
  const int nx = m->n[0], ny = m->n[1], whole = m->whole;
  const int c = (int)(b / (unsigned)m->nj), tile = (int)(b - (unsigned)c * (unsigned)m->nj);
  const int i0 = c * m->ch, i1 = min(i0 + m->ch, nx);
  const int j0 = tile * m->w, w = min(m->w, ny - j0);
  const bool own = t < w;
  const int j = own ? j0 + t : (t == w + 1 ? (j0 ? j0 - 1 : ny - 1) : (j0 + w == ny ? 0 : j0 + w));
  const int tl = t ? t - 1 : (whole ? w - 1 : w + 1);             // lane of the column before
  const int tr = (whole && t == w - 1) ? 0 : min(t + 1, nt - 1);  // and of the one after
  const bool used = t < (whole ? w : w + 2);

  // the component whose H the next column reads, the one the next row reads
  // (TMz: Hx, Hy; TEz: Hz, Hz), and the E whose column and row they read
  constexpr int HJ = TM ? 0 : 2, HI = TM ? 1 : 2, EJ = TM ? 2 : 0, EI = TM ? 2 : 1;
  // CPML words along x and y: E's (TMz: Ez, Ez; TEz: Ey, Ex), H's (Hy, Hx; Hz, Hz)
  constexpr int EX = TM ? 2 : 1, EY = TM ? 2 : 0, HX = TM ? 1 : 2, HY = TM ? 0 : 2;
  constexpr int C0 = TM ? 2 : 0, C1 = TM ? 0 : 2;  // first E, first H component

  // The addresses of the march stay in scalar registers; what only absorber,
  // special, source and ghost cells need is read where they need it.
  const T* const f0 = m->fi[0];
  const T* const f1 = m->fi[1];
  const T* const f2 = m->fi[2];
  T* const w0 = m->fo[0];
  T* const w1 = m->fo[1];
  T* const w2 = m->fo[2];
  const uint16_t* const ids = m->ids;
  const R d0 = m->d[0], d1 = m->d[1], d2 = m->d[2], v0 = m->inv_d[0], v1 = m->inv_d[1], v2 = m->inv_d[2];
  const unsigned pi = (unsigned)m->pi;
  const int ghosts = m->ghosts;
  const int nsrc = m->nsrc;
  bool sources = false;  // a source in the block's rows
  for (int s = 0; s < nsrc; ++s)
    sources = sources || (m->src[s].i >= i0 && m->src[s].i <= i1) || (i1 == nx && m->src[s].i == 0);

  // absorber: live words by coordinate, rows along y
  bool lye = false, lyh = false;
  int rune = 0, runh = 0;          // runs along x
  R ye[2][3] = {}, yh[2][3] = {};  // UPML: pairs of the first and second E (H) component
  auto live = [](int run, int x) { return x < (run & 0xFFFF) || x >= (run >> 16); };
  if constexpr (PML == 1) {
    rune = m->run[EX][0];
    runh = m->run[HX][0];
    lye = live(m->run[EY][1], j);
    lyh = live(m->run[HY][1], j);
#pragma unroll
    for (int v = 0; v < 3; ++v) {
      ye[0][v] = gld(m->row[EY][1] + j * 3 + v);
      yh[0][v] = gld(m->row[HY][1] + j * 3 + v);
    }
  } else if constexpr (PML == 2) {
    rune = m->run[0][0];
    lye = live(m->run[0][1], j);
    // the pair of axis y: c1, c2 for an x-directed component, c3, c4 for z, c5, c6 for y
    auto pair = [&](int cc) { return cc == 0 ? 0 : cc == 2 ? 2 : 4; };
#pragma unroll
    for (int v = 0; v < 2; ++v) {
      ye[0][v] = gld(m->row[C0][1] + j * 6 + pair(C0) + v);
      yh[0][v] = gld(m->row[C1][1] + j * 6 + pair(C1) + v);
      if constexpr (TM) yh[1][v] = gld(m->row[1][1] + j * 6 + pair(1) + v);
      else ye[1][v] = gld(m->row[1][1] + j * 6 + pair(1) + v);
    }
  }
  const bool wave_live = PML != 0 && __any(lye || lyh);

  // (past the last row, and in idle lanes, the operands are left undefined:
  // keeping the old ones instead would move registers, behind a wait)
  auto load = [&](int q) {
    Step2Ops<T, PML> l;
    const int qe = q == nx ? 0 : q;
    const unsigned e = (unsigned)qe * pi + (unsigned)j, o = e * S;
    if (used && q <= i1) {
      l.f[0] = at(f0, o);
      l.f[1] = at(f1, o);
      l.f[2] = at(f2, o);
      l.id = at(ids, e * 2u);
    }
    if constexpr (PML != 0) {
#pragma unroll
      for (int a = 0; a < 4; ++a) l.s[a] = T{};
      const bool xe = live(rune, qe), xh = PML == 1 && live(runh, qe);
      if (q <= i1 && (wave_live || xe || xh)) {
        const Step2Ptr<T> m = fresh2<T>(mp);
        if constexpr (PML == 1) {
          if (used && xe) l.s[0] = at(m->si[EX][0], o);
          if (used && lye) l.s[1] = at(m->si[EY][1], o);
          if (own && q < i1) {
            if (xh) l.s[2] = at(m->si[HX][0], o);
            if (lyh) l.s[3] = at(m->si[HY][1], o);
          }
        } else {
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            const bool electric = TM ? a == 2 : a != 2;
            if (used && (lye || xe) && (electric || (own && q < i1))) l.s[a] = at(m->si[a][0], o);
          }
        }
      }
    }
    return l;
  };

  int64_t row = 0, wave_n = 0;
  if (nsrc || blk == 0) {
    const int64_t clk = cld(&m->ctl->clk[m->par]);
    row = clk - cld(&m->ctl->wave_step0);
    wave_n = cld(&m->ctl->wave_n);
    if (blk == 0 && t == 0) {  // the step's tick
      m->ctl->clk[1 - m->par] = clk + 1;
      m->ctl->clock = clk + 1;
    }
  }

  Step2Ops<T, PML> l0 = load(i0);
  T hi_prev = T{};  // the H of the row before that E reads
  if (used) hi_prev = at(HI == 1 ? f1 : f2, ((unsigned)(i0 ? i0 - 1 : nx - 1) * pi + (unsigned)j) * S);
  Step2Ops<T, PML> l1 = load(i0 + 1);

  // values of the row before: new E, old H and their entry and absorber words
  T pe[3]{}, ph[3]{}, ps[4]{};
  unsigned pid = 0;
  Step2Ent<R> pen{};

  // Dummy, Const and dispersive cells
  auto special = [&](int cc, bool electric, unsigned id, int qe, T f, T D1, T D2, T v) -> T {
    const Step2Ptr<T> m = fresh2<T>(mp);
    const Step2Cell* x = m->cells + id * 3 + cc;
    const int kind = gld(&x->kind);
    if (kind == 1) v = f;
    if (kind == 2) v = make_val<T>((R)gld(&x->re), (R)gld(&x->im));
    if constexpr (ADE) {
      if (electric && kind == 3) {
        const DevRec<R>* rec = m->recs + gld(&x->rec);
        const int cls = gld(&rec->cls), s = cls - GMES_CLS_DRUDE;
        const int q = gld(m->adeq[cc] + ((unsigned)qe * pi + (unsigned)j));
        const int a1 = cc == 2 ? 0 : cc + 1, a2 = cc == 0 ? 2 : cc - 1;
        const T curl = vsub(vdiv(D1, m->d[a1]), vdiv(D2, m->d[a2]));
        const auto cu = [curl] { return curl; };
        const bool keep = own && qe >= i0 && qe < i1;
        const R* a = m->coef + gld(&rec->coef_off);
        const int p1 = gld(&rec->n1), p2 = gld(&rec->n2);
        using Z = cplx<R>;
        if (s == 0)
          v = ade_drude_value<T>(a, p1, static_cast<const T*>(m->ade_in[cc][0]), static_cast<T*>(m->ade_out[cc][0]),
                                 m->ade_n[cc][0], q, keep, f, cu);
        else if (s == 1)
          v = ade_dcp_value<T>(a, p1, p2, static_cast<const T*>(m->ade_in[cc][1]),
                               static_cast<T*>(m->ade_out[cc][1]), m->ade_n[cc][1], q, keep, f, cu);
        else
          v = ade_plrc_value<T>(a, p1, p2, static_cast<const Z*>(m->ade_in[cc][2]),
                                static_cast<Z*>(m->ade_out[cc][2]), m->ade_n[cc][2], q, keep, f, cu);
      }
    }
    return v;
  };
  auto sourced = [&](int cc, int qe, T v) -> T {
    const Step2Ptr<T> m = fresh2<T>(mp);
    for (int s = 0; s < nsrc; ++s) {
      if (m->src[s].c != cc || m->src[s].i != qe) continue;
      if (m->src[s].j == j) {
        const double* w = m->waves + (m->src[s].wave * wave_n + row) * 2;
        const T wv = make_val<T>((R)gld(w), (R)gld(w + 1));
        v = m->src[s].kind == GMES_SRC_SET ? wv : vsub(v, wv);
      }
    }
    return v;
  };
  // the ghost images of the cell at p: value v; order a1, a2 of the copies,
  // d: from the cell to its image along an axis (0: not on its source plane)
  auto ghost = [&](int cc, T* p, int64_t d1, int64_t d2, T v) {
    const Step2Ptr<T> m = fresh2<T>(mp);
    const int a1 = cc == 2 ? 0 : cc + 1, a2 = cc == 0 ? 2 : cc - 1;
    const cplx<R> q1{m->ph[cc][a1].re, m->ph[cc][a1].im}, q2{m->ph[cc][a2].re, m->ph[cc][a2].im};
    const T v1 = ghost_phase<T>(q1, v);
    if (d1) gst(p + d1, v1);
    if (d2) gst(p + d2, ghost_phase<T>(q2, v));
    if (d1 && d2) gst(p + d1 + d2, ghost_phase<T>(q2, v1));
  };
  // ghost images of row q: E's from the new values, H's from the old ones
  auto ghost_row = [&](int q, const T (&ne)[3], const T (&oh)[3]) {
    const Step2Ptr<T> m = fresh2<T>(mp);
    const int64_t e = (int64_t)q * pi + j;
#pragma unroll
    for (int C = 0; C < 3; ++C) {
      const bool electric = TM ? C == 2 : C != 2;
      const int64_t gx = electric ? (q == 0 ? (int64_t)nx * pi : 0) : (q == nx - 1 ? -(int64_t)nx * pi : 0);
      const int64_t gy = electric ? (j == 0 ? ny : 0) : (j == ny - 1 ? -ny : 0), gz = m->pk[C];
      const T v = electric ? ne[C] : oh[C];
      T* const p = (C == 0 ? w0 : C == 1 ? w1 : w2) + e;
      if (C == 0) ghost(0, p, gy, gz, v);
      else if (C == 1) ghost(1, p, gz, gx, v);
      else ghost(2, p, gx, gy, v);
    }
  };

  // The operands of a row make way for those of the row after the next, early
  // (for more time on their way) or once the row is done with them: replaced
  // early, in other registers, they have to be moved, and waited for, at the end
  // of every other row.  With UPML words or dispersive cells late is better (TEz
  // 517 x 389 FP32 UPML with dispersive rods 13.3 -> 12.4 us, 1000 x 2000 53 ->
  // 47) and with wider words a little (2048^2 FP64 CPML 57 -> 55); else early
  // (1200^2 FP32 CPML 14.2 against 14.7).
  constexpr bool LATE = PML == 2 || ADE || S > 4;
  auto body = [&](int q, int par, Step2Ops<T, PML>& next) {
    const Step2Ops<T, PML> l = next;
    const int qe = q == nx ? 0 : q;
    xb[par * nt + t] = l.f[HJ];
    __syncthreads();
    if (!LATE) next = load(q + 2);
    T hj = xb[par * nt + tl], hi = hi_prev;
    if constexpr (is_cplx<T>::value) {
      const Step2Ptr<T> m = fresh2<T>(mp);
      if (j == 0) hj = phased<T>(m->ph[HJ][1], hj);
      if (qe == 0) hi = phased<T>(m->ph[HI][0], hi);
    }
    const Step2Ent<R> en = et[used ? l.id : 0u];
    const T dhj = vsub(l.f[HJ], hj), dhi = vsub(l.f[HI], hi);
    T ne[3] = {};
    T n[4] = {};  // new absorber words: CPML E x, y, H x, y; UPML the components'
    if constexpr (TM) {
      ne[2] = plain_value<true, X>(en.c[2], l.f[2], dhi, dhj, d0, v0, d1, v1);
    } else {
      ne[0] = plain_value<true, X>(en.c[0], l.f[0], dhj, T{}, d1, v1, d2, v2);
      ne[1] = plain_value<true, X>(en.c[1], l.f[1], T{}, dhi, d2, v2, d0, v0);
    }
    const bool stores = own && q < i1;
    if (used && (en.meta & (TM ? 0x30u : 0x0Fu))) {
      const Step2Ptr<T> m = fresh2<T>(mp);
      const unsigned o = ((unsigned)qe * pi + (unsigned)j) * S;
#pragma unroll
      for (int C = 0; C < 3; ++C) {
        if (TM ? C != 2 : C == 2) continue;
        const T D1 = C == 0 ? dhj : C == 1 ? T{} : dhi, D2 = C == 0 ? T{} : C == 1 ? dhi : dhj;
        const unsigned kind = (en.meta >> (2 * C)) & 3u;
        if constexpr (PML == 1) {
          if (kind == 1u) {
            if (C == 0) ne[0] = step2_cpml<true, 0, X, T, R>(m, en.c[0], l.f[0], D1, D2, qe, ye[0], l.s[0], l.s[1], n[0], n[1]);
            else if (C == 1) ne[1] = step2_cpml<true, 1, X, T, R>(m, en.c[1], l.f[1], D1, D2, qe, ye[0], l.s[0], l.s[1], n[0], n[1]);
            else ne[2] = step2_cpml<true, 2, X, T, R>(m, en.c[2], l.f[2], D1, D2, qe, ye[0], l.s[0], l.s[1], n[0], n[1]);
            if (stores) {
              if (C == EX && live(rune, qe)) put(m->so[EX][0], o, n[0]);
              if (C == EY && lye) put(m->so[EY][1], o, n[1]);
            }
          }
        } else if constexpr (PML == 2) {
          if (kind == 1u) {
            if (C == 0) ne[0] = step2_upml<true, 0, X, T, R>(m, en.c[0], l.f[0], D1, D2, qe, ye[0], l.s[0], n[0]);
            else if (C == 1) ne[1] = step2_upml<true, 1, X, T, R>(m, en.c[1], l.f[1], D1, D2, qe, ye[1], l.s[1], n[1]);
            else ne[2] = step2_upml<true, 2, X, T, R>(m, en.c[2], l.f[2], D1, D2, qe, ye[0], l.s[2], n[2]);
            if (stores) put(m->so[C][0], o, n[C]);
          }
        }
        if (kind == 2u) ne[C] = special(C, true, l.id, qe, l.f[C], D1, D2, ne[C]);
      }
    }
    if (sources) {
      if constexpr (TM) {
        ne[2] = sourced(2, qe, ne[2]);
      } else {
        ne[0] = sourced(0, qe, ne[0]);
        ne[1] = sourced(1, qe, ne[1]);
      }
    }
    eb[par * nt + t] = ne[EJ];
    if (own) {
      if (q < i1) {
        const unsigned o = ((unsigned)q * pi + (unsigned)j) * S;
        if constexpr (TM) {
          put(w2, o, ne[2]);
        } else {
          put(w0, o, ne[0]);
          put(w1, o, ne[1]);
        }
        if (ghosts) ghost_row(q, ne, l.f);
      }
      if (q > i0) {  // H of the row before
        const int qh = q - 1;
        T ej = eb[(par ^ 1) * nt + tr], ei = ne[EI];
        if constexpr (is_cplx<T>::value) {
          const Step2Ptr<T> m = fresh2<T>(mp);
          if (j == ny - 1) ej = phased<T>(m->ph[EJ][1], ej);
          if (q == nx) ei = phased<T>(m->ph[EI][0], ei);
        }
        const T dj = vsub(ej, pe[EJ]), di = vsub(ei, pe[EI]);
        const unsigned o = ((unsigned)qh * pi + (unsigned)j) * S;
        T nh[3] = {};
        if constexpr (TM) {
          nh[0] = plain_value<false, X>(pen.c[0], ph[0], dj, T{}, d1, v1, d2, v2);
          nh[1] = plain_value<false, X>(pen.c[1], ph[1], T{}, di, d2, v2, d0, v0);
        } else {
          nh[2] = plain_value<false, X>(pen.c[2], ph[2], di, dj, d0, v0, d1, v1);
        }
        if (pen.meta & (TM ? 0x0Fu : 0x30u)) {
          const Step2Ptr<T> m = fresh2<T>(mp);
#pragma unroll
          for (int C = 0; C < 3; ++C) {
            if (TM ? C == 2 : C != 2) continue;
            const T D1 = C == 0 ? dj : C == 1 ? T{} : di, D2 = C == 0 ? T{} : C == 1 ? di : dj;
            const unsigned kind = (pen.meta >> (2 * C)) & 3u;
            if constexpr (PML == 1) {
              if (kind == 1u) {
                if (C == 0) nh[0] = step2_cpml<false, 0, X, T, R>(m, pen.c[0], ph[0], D1, D2, qh, yh[0], ps[2], ps[3], n[2], n[3]);
                else if (C == 1) nh[1] = step2_cpml<false, 1, X, T, R>(m, pen.c[1], ph[1], D1, D2, qh, yh[0], ps[2], ps[3], n[2], n[3]);
                else nh[2] = step2_cpml<false, 2, X, T, R>(m, pen.c[2], ph[2], D1, D2, qh, yh[0], ps[2], ps[3], n[2], n[3]);
                if (C == HX && live(runh, qh)) put(m->so[HX][0], o, n[2]);
                if (C == HY && lyh) put(m->so[HY][1], o, n[3]);
              }
            } else if constexpr (PML == 2) {
              if (kind == 1u) {
                if (C == 0) nh[0] = step2_upml<false, 0, X, T, R>(m, pen.c[0], ph[0], D1, D2, qh, yh[0], ps[0], n[0]);
                else if (C == 1) nh[1] = step2_upml<false, 1, X, T, R>(m, pen.c[1], ph[1], D1, D2, qh, yh[1], ps[1], n[1]);
                else nh[2] = step2_upml<false, 2, X, T, R>(m, pen.c[2], ph[2], D1, D2, qh, yh[0], ps[2], n[2]);
                put(m->so[C][0], o, n[C]);
              }
            }
            if (kind == 2u) nh[C] = special(C, false, pid, qh, ph[C], D1, D2, nh[C]);
          }
        }
        if (sources) {
          if constexpr (TM) {
            nh[0] = sourced(0, qh, nh[0]);
            nh[1] = sourced(1, qh, nh[1]);
          } else {
            nh[2] = sourced(2, qh, nh[2]);
          }
        }
        if constexpr (TM) {
          put(w0, o, nh[0]);
          put(w1, o, nh[1]);
        } else {
          put(w2, o, nh[2]);
        }
      }
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      pe[a] = ne[a];
      ph[a] = l.f[a];
    }
    if constexpr (PML != 0) {
#pragma unroll
      for (int a = 0; a < 4; ++a) ps[a] = l.s[a];
    }
    hi_prev = l.f[HI];
    pid = l.id;
    pen = en;
    if (LATE) next = load(q + 2);
  };
  int q = i0;
  for (; q < i1; q += 2) {
    body(__builtin_amdgcn_readfirstlane(q), 0, l0);
    body(__builtin_amdgcn_readfirstlane(q + 1), 1, l1);
  }
  if (q == i1) body(__builtin_amdgcn_readfirstlane(q), 0, l0);
}

template <class T, bool TM, int PML, bool ADE, bool X>
__global__ void __launch_bounds__(kStep2Threads<T>) k_step2d(Step2Args<T>) {
  extern __shared__ __attribute__((aligned(16))) char step2_lds_mem[];
  step2d_tile<T, TM, PML, ADE, X>((Step2Ptr<T>)__builtin_amdgcn_kernarg_segment_ptr(), blockIdx.x, step2_lds_mem);
}

// Every member in one launch, by its mode and absorber.
template <class T>
__global__ void __launch_bounds__(kStep2BatchThreads) k_step2d_batch(const Step2Job<T>* jobs, int njobs) {
  extern __shared__ __attribute__((aligned(16))) char step2_lds_mem[];
  const GMES_CONST Step2Job<T>* J = step_job(jobs, njobs, (int64_t)blockIdx.x);
  const Step2Ptr<T> m = &J->a;
  const unsigned blk = (unsigned)((int64_t)blockIdx.x - J->block0);
  const int kind = J->tm * 3 + J->absorber;
  if (kind == 0) step2d_tile<T, false, 0, true, false>(m, blk, step2_lds_mem);
  else if (kind == 1) step2d_tile<T, false, 1, true, false>(m, blk, step2_lds_mem);
  else if (kind == 2) step2d_tile<T, false, 2, true, false>(m, blk, step2_lds_mem);
  else if (kind == 3) step2d_tile<T, true, 0, true, false>(m, blk, step2_lds_mem);
  else if (kind == 4) step2d_tile<T, true, 1, true, false>(m, blk, step2_lds_mem);
  else step2d_tile<T, true, 2, true, false>(m, blk, step2_lds_mem);
}

template <class T>
void launch_step2d_batch(const Step2Job<T>* jobs, int njobs, int64_t nblocks, size_t lds, hipStream_t st) {
  if (njobs)
    hipLaunchKernelGGL((k_step2d_batch<T>), dim3((unsigned)nblocks), dim3(kStep2BatchThreads), (unsigned)lds, st, jobs, njobs);
}
template void launch_step2d_batch<step2_t>(const Step2Job<step2_t>*, int, int64_t, size_t, hipStream_t);

template <class T, bool TM, int PML, bool ADE>
static void launch_step2d_x(const Step2Args<T>& m, hipStream_t st) {
  const dim3 grid(((unsigned)m.nblk + 7u) / 8u * 8u), block(step2_threads(m.w, m.whole));
  const unsigned lds = (unsigned)step2_lds<T>((int)block.x, m.nent);
  if constexpr (sizeof(typename real_of<T>::type) == 8) {
    if (m.exact) {
      hipLaunchKernelGGL((k_step2d<T, TM, PML, ADE, true>), grid, block, lds, st, m);
      return;
    }
  }
  hipLaunchKernelGGL((k_step2d<T, TM, PML, ADE, false>), grid, block, lds, st, m);
}

template <class T>
void launch_step2d(const Step2Args<T>& m, bool tm, int absorber, bool ade, hipStream_t st) {
#define GMES_STEP2(TM, P, A) \
  if (tm == TM && absorber == P && ade == A) return launch_step2d_x<T, TM, P, A>(m, st);
  GMES_STEP2(false, 0, false) GMES_STEP2(false, 1, false) GMES_STEP2(false, 2, false)
  GMES_STEP2(true, 0, false) GMES_STEP2(true, 1, false) GMES_STEP2(true, 2, false)
  GMES_STEP2(false, 0, true) GMES_STEP2(false, 1, true) GMES_STEP2(false, 2, true)
  GMES_STEP2(true, 0, true) GMES_STEP2(true, 1, true) GMES_STEP2(true, 2, true)
#undef GMES_STEP2
}

template void launch_step2d<step2_t>(const Step2Args<step2_t>&, bool, int, bool, hipStream_t);

}  // namespace gmes_engine
