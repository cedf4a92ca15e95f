// One-sweep 3-D step: E and H of a leapfrog step in one kernel.
//
// The two-kernel step (kernels.hip) moves 18 field words per cell: six read
// and three written by each half step, and both halves already run at the
// rate of a device copy.  One sweep needs 12.  A block takes whole (j, k)
// rows -- `rows` of them, the last a rim whose E it computes again for the
// H of the row below -- and marches along i, keeping the E of the plane
// before in registers and LDS.  Because E is needed by blocks other than
// its owner, and H of a neighbour is read after that neighbour may have
// advanced, the step reads one set of buffers and writes another.
//
// Per thread (j, k) and plane q of the march:
//   1. wait for the operands of plane q, barrier
//   2. issue the loads of plane q + 1: FP32 fields straight into LDS, the
//      absorber's z words into registers; issue the x and y words of plane q
//   3. store the results of the plane before
//   4. E(q) from LDS neighbours, into the other half of LDS for plane q + 1
//   5. H(q - 1) from E(q - 1) and E(q)
// Neighbours come from LDS, not from overlapping global loads: with those
// the L1 request rate bounds the kernel (256^3 FP32 without an absorber:
// 228 us against 180 us, which is the rate of a copy of the same bytes).
// Rows are whole so that the periodic wrap along k stays inside the block.
//
// A CPML cell and a Dielectric one beside it run the same instructions and differ
// in the last operand, chosen by class (171 x 150 x 139 FP64 143 us without the
// choice, 147 with it): where both words are dead the two values agree but where a
// difference is not finite, and in zeros' signs.
//
// Blocks differ in the absorber words they hold: a body with none, with CPML
// words along z (every row has those at both ends), along x and z, along y and
// z, with all, with UPML.  The words of a body are loaded a plane ahead,
// except in the body with all of them (blocks at the edges; every block of a
// small sim), which loads those along x and y in the plane that uses them:
// ahead they cost 98 registers and one block per CU in FP32.
//
// Measured per step, two-kernel step first: FP32 256^3 CPML 344 -> 248 us (one
// body for all blocks 293), 181 x 203 x 225 UPML 210 -> 168, 96^3 CPML 39 ->
// 26, 64^3 UPML 24 -> 11; FP64 CPML 171 x 150 x 139 189 -> 147, 64^3 31 -> 17;
// complex FP32 with z layers 192 x 192 x 128 190 -> 138, 112^3 72 -> 46.  What
// bounds it: without an absorber the bytes (256^3 FP32 188 us, 4.3 TB/s); with
// one the latency of a plane, 1 to 2 us, of which a CU has few in flight (24
// waves in FP32, 12 to 16 with 8-byte words, by their registers: held to 128
// registers the 8-byte bodies with all words spill, 171 x 150 x 139 320 us).
//
// Ghost planes: operands wrap by index (with the Bloch phase), and the
// owners of source-plane cells write the ghost images of both types with
// the values and products of the separate copies (k_ghost): E's from the
// new E, H's from the old H, as the copies at the two places of a step
// leave them.
#include "step_common.h"

namespace gmes_engine {

// Buffer accesses: a resource (base, size) per array, the plane as scalar
// offset, the lane's place in the plane as vector offset.  One scalar offset
// serves every array of a stagger, so an access costs no address arithmetic
// (with 64-bit pointers the march spent 236 scalar instructions a plane, and
// a CU's one scalar unit was the bound).
__device__ float raw_load_f32(i4_t r, int v, int s, int aux) __asm("llvm.amdgcn.raw.buffer.load.f32");
__device__ vec2_t<float> raw_load_v2f32(i4_t r, int v, int s, int aux) __asm("llvm.amdgcn.raw.buffer.load.v2f32");
__device__ void raw_store_f32(float x, i4_t r, int v, int s, int aux) __asm("llvm.amdgcn.raw.buffer.store.f32");
__device__ void raw_store_v2f32(vec2_t<float> x, i4_t r, int v, int s, int aux) __asm("llvm.amdgcn.raw.buffer.store.v2f32");
__device__ short raw_load_i16(i4_t r, int v, int s, int aux) __asm("llvm.amdgcn.raw.buffer.load.i16");
__device__ int raw_load_i32(i4_t r, int v, int s, int aux) __asm("llvm.amdgcn.raw.buffer.load.i32");

constexpr int kAuxNt = 2;  // non-temporal

// One dword per active lane from memory straight into LDS, at lds (bytes
// from the block's base, below 64 KiB) + 4 * lane: no register holds it in
// flight.  The compiler does not see these loads; the march waits for them
// (vmcnt) before the barrier that opens their plane.
__device__ __forceinline__ void lds_load(i4_t r, unsigned v, unsigned s, unsigned lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds"
               :
               : "s"(lds), "v"(v), "s"(r), "s"(s)
               : "memory", "m0");
}
__device__ __forceinline__ void lds_load_nt(i4_t r, unsigned v, unsigned s, unsigned lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen nt lds"
               :
               : "s"(lds), "v"(v), "s"(r), "s"(s)
               : "memory", "m0");
}

template <class T>
__device__ __forceinline__ T bld(const GMES_CONST i4_t& r, unsigned v, unsigned s, int aux = 0) {
  if constexpr (std::is_same<T, float>::value) {
    return raw_load_f32(r, (int)v, (int)s, aux);
  } else {
    const vec2_t<float> x = raw_load_v2f32(r, (int)v, (int)s, aux);
    return __builtin_bit_cast(T, x);
  }
}
template <class T>
__device__ __forceinline__ void bst(const GMES_CONST i4_t& r, unsigned v, unsigned s, T x) {
  if constexpr (std::is_same<T, float>::value) raw_store_f32(x, r, (int)v, (int)s, kAuxNt);
  else raw_store_v2f32(__builtin_bit_cast(vec2_t<float>, x), r, (int)v, (int)s, kAuxNt);
}

// Absorber rows of one axis: CPML b, c, kappa (FP32: 1/kappa); UPML c1..c4
// of the row two components share, c5, c6 of the third's.  Those of the
// block's j and k live in LDS: held in registers for the whole march they
// cost 12 (CPML) to 24 (UPML) of them, twice that in FP64.
template <int PML> struct RowStride { static constexpr int v = PML == 2 ? 8 : 4; };
// A CPML coordinate without live state: c = 0, kappa = 1, and b multiplies a
// word that is +0.
template <class R, int PML>
__device__ __forceinline__ void stage_row(R* dst, const R* shared, const R* own, int xs, int xo, bool live) {
  if constexpr (PML != 2) {
    dst[0] = live ? gld(shared + xs * 3) : R(0);
    dst[1] = live ? gld(shared + xs * 3 + 1) : R(0);
    dst[2] = live ? gld(shared + xs * 3 + 2) : R(1);
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q) dst[q] = gld(shared + xs * 6 + q);
    dst[4] = gld(own + xo * 6 + 4);
    dst[5] = gld(own + xo * 6 + 5);
  }
}

template <class R, int PML>
__device__ __forceinline__ Rows<R, PML == 2 ? 2 : 1> lds_row(const R* p) {
  Rows<R, PML == 2 ? 2 : 1> r;
#pragma unroll
  for (int q = 0; q < (PML == 2 ? 6 : 3); ++q) r.v[q] = p[q];
  return r;
}

// the row of a CPML coordinate without live state
template <class R, int PML>
__device__ __forceinline__ Rows<R, PML == 2 ? 2 : 1> dead_row() {
  Rows<R, PML == 2 ? 2 : 1> r{};
  r.v[2] = R(1);
  return r;
}

// a row along x, the same for the whole block
template <class R, int PML>
__device__ __forceinline__ Rows<R, PML == 2 ? 2 : 1> x_row(const R* shared, const R* own, int xs, int xo, bool live) {
  Rows<R, PML == 2 ? 2 : 1> r;
  if constexpr (PML != 2) {
    r.v[0] = live ? cld(shared + xs * 3) : R(0);
    r.v[1] = live ? cld(shared + xs * 3 + 1) : R(0);
    r.v[2] = live ? cld(shared + xs * 3 + 2) : R(1);
  } else if constexpr (PML == 2) {
#pragma unroll
    for (int q = 0; q < 6; ++q) r.v[q] = q < 4 ? cld(shared + xs * 6 + q) : cld(own + xo * 6 + q);
  }
  return r;
}

// The arguments stay in constant memory (the kernel's own argument block, or
// a job of a batch) and are read where they are used, through a pointer the
// compiler cannot see through: hoisted out of the march their ~60 pointers
// overflowed the scalar registers, and every access went through a lane of
// a spill register (400 v_readlane in the CPML kernel).
template <class T>
using StepPtr = const GMES_CONST Step3Args<T>*;
template <class T>
__device__ __forceinline__ StepPtr<T> fresh(StepPtr<T> p) {
  asm("" : "+s"(p));
  return p;
}
// The operands a thread loads for one plane, a plane ahead.
template <class T, int PML>
struct StepOps {
  T hx, hy, hz;  // its own H cells (the H neighbours on the + side of its E)
  T e0, e1, e2;  // old E
  T hxj, hzj;    // H one row below: the block's first row only
  // absorber words of E at this plane, of H one plane before.  CPML: the
  // two that live along z, which every row has at both ends; those along x
  // and y are read where they are used, by the few planes and rows that
  // have them (all twelve ahead took 98 registers and one block per CU).
  T s[PML == 2 ? 3 : PML >= kPmlXZ ? 4 : 2], g[PML == 2 ? 3 : PML >= kPmlXZ ? 4 : 2];
  uint32_t id;
};

// Rectangle rc and its block rb of a launch's block.  Consecutive blocks go to
// consecutive XCDs: each XCD gets a contiguous run of a rectangle's tiles, so
// that the rim rows two blocks share meet in one L2 (256^3 without an
// absorber: 189 to 180 us).
template <class T>
__device__ __forceinline__ bool step3d_block(StepPtr<T> m, unsigned blk, int& rc, unsigned& rb) {
  const int slot = (int)(blk >> 3);
  rc = m->nrect - 1;
  while (rc > 0 && slot < m->rect[rc].first) --rc;
  rb = (blk & 7u) * (unsigned)m->rect[rc].per + (unsigned)(slot - m->rect[rc].first);
  return rb < (unsigned)m->rect[rc].nblk && slot - m->rect[rc].first < m->rect[rc].per;
}

// X: see by_size (FP64 only)
template <class T, int PML, bool X>
__device__ __forceinline__ void step3d_tile(StepPtr<T> mp, unsigned blk, char* lds) {
  using R = typename real_of<T>::type;
  StepPtr<T> m = fresh<T>(mp);
  constexpr unsigned S = sizeof(T);
  const int t = threadIdx.x;
  const int nx = m->n[0], ny = m->n[1], nz = m->n[2];
  // 4-byte words: operands of a plane arrive in LDS by themselves (lds_load);
  // per parity of the plane hx, hz (each after the row below the block's
  // first), hy and old Ex, Ey, Ez, then the exchange of new E.  8-byte words
  // arrive in registers and H is put there.
  constexpr bool DMA = sizeof(T) == 4;
  // CPML; with live words along x, along y
  constexpr bool CP = PML != 0 && PML != 2, LX = PML == 1 || PML == kPmlXZ, LY = PML == 1 || PML == kPmlYZ;
  const int nt = (int)blockDim.x, NT = nt;
  T* const xb = reinterpret_cast<T*>(lds);  // DMA: [2][3 NT] new E after the operands; else [2][hx, hy, hz, ex, ey, ez][NT]
  const int slot = DMA ? 2 * nz + 6 * nt : 6 * NT;   // words of a parity's operands
  T* const eb = DMA ? xb + 2 * slot : xb + 3 * NT;   // new E: + parity * eslot + component * est
  const int eslot = DMA ? 3 * nt : 6 * NT, est = DMA ? nt : NT;
  StepEnt<R>* const et = reinterpret_cast<StepEnt<R>*>(xb + (DMA ? (2 * (2 * nz + 9 * nt) + 3) / 4 * 4 : 12 * NT));
  {
    constexpr int kq = sizeof(StepEnt<R>) / 16;
    i4_t* dst = reinterpret_cast<i4_t*>(et);
    const i4_t* src = static_cast<const i4_t*>(m->tab);
    for (int e = t; e < (m->net + m->nht) * kq; e += (int)blockDim.x) dst[e] = gld(src + e);
  }
  int rc;
  unsigned rb;
  if (!step3d_block<T>(m, blk, rc, rb)) return;
  const unsigned rnj = (unsigned)m->rect[rc].nj;
  const int c = (int)(rb / rnj), tile = (int)(rb - (unsigned)c * rnj);
  const int i0 = m->rect[rc].i0 + c * m->rect[rc].ch, i1 = min(i0 + m->rect[rc].ch, m->rect[rc].i1);
  const int j0 = m->rect[rc].j0 + tile * (m->rows - 1), jw = min(m->rows - 1, m->rect[rc].j1 - j0);  // own rows
  // lanes past the last row repeat a row of the block and store nothing
  const int tr = (int)((unsigned)t / (unsigned)nz), k = t - tr * nz;
  const int tj = min(tr, jw);
  const int j = j0 + tj == ny ? 0 : j0 + tj;
  const bool own = tr < jw;
  const bool edge = tj == 0;
  const unsigned W0 = (unsigned)m->W0 * S, W2 = (unsigned)m->W2 * S;  // bytes of a row
  const unsigned PX = (unsigned)(ny + 1) * W0, PY = (unsigned)ny * W0, PZ = (unsigned)(ny + 1) * W2;  // of a plane
  const unsigned b0 = (unsigned)j * W0 + (unsigned)k * S, b2 = (unsigned)j * W2 + (unsigned)k * S;
  const int jm = j ? j - 1 : ny - 1;  // row of the H below, one row up
  const unsigned bj0 = (unsigned)jm * W0 + (unsigned)k * S, bj2 = (unsigned)jm * W2 + (unsigned)k * S;
  const unsigned PI = (unsigned)ny * W0 / S * (unsigned)m->idw;  // ids: rows at the pitch of Ex
  const int tm = k ? t - 1 : t + nz - 1, tp = k == nz - 1 ? t + 1 - nz : t + 1;

  // absorber rows of the block: E along y, H along y, E along z, H along z
  using RowT = Rows<R, PML == 2 ? 2 : 1>;
  constexpr int rs = RowStride<PML>::v;
  bool ly = false, lz = false, lyh = false, lzh = false;  // live state along y, z (CPML); outside the box (UPML)
  R* const rows_y = reinterpret_cast<R*>(et + m->net + m->nht);
  R* const rows_yh = rows_y + m->rows * rs;
  R* const rows_z = rows_yh + m->rows * rs;
  R* const rows_zh = rows_z + nz * rs;
  bool wave_live = false;  // some lane of the wave has live state along y or z
  if constexpr (PML != 0) {
    auto live = [](int run, int x) { return x < (run & 0xFFFF) || x >= (run >> 16); };
    ly = live(m->run_e[1], j);
    lz = live(m->run_e[2], k);
    lyh = live(m->run_h[1], j + 1);
    lzh = live(m->run_h[2], k + 1);
    if (CP && !LY) ly = lyh = false;
    wave_live = __any(ly || lz || lyh || lzh);
    if ((!CP || LY) && k == 0 && tr == tj) {
      stage_row<R, PML>(rows_y + tj * rs, m->re[1], m->oe[1], j, j, ly);
      stage_row<R, PML>(rows_yh + tj * rs, m->rh[1], m->oh[1], j + 1, j, lyh);
    }
    if (tr == 0) {
      stage_row<R, PML>(rows_z + k * rs, m->re[2], m->oe[2], k, k, lz);
      stage_row<R, PML>(rows_zh + k * rs, m->rh[2], m->oh[2], k + 1, k, lzh);
    }
  }
  const int run_e = m->run_e[0], run_h = m->run_h[0];
  auto xlive_e = [&](int x) { return x < (run_e & 0xFFFF) || x >= (run_e >> 16); };
  auto xlive_h = [&](int x) { return x < (run_h & 0xFFFF) || x >= (run_h >> 16); };
  // live state along x: E at plane q; H at x = q (Hy, Hz of plane q - 1;
  // UPML: any of its three)
  auto x_of_e = [&](int q) { return (LX || PML == 2) && xlive_e(q == nx ? 0 : q); };
  auto x_of_h = [&](int q) { return (LX || PML == 2) && (xlive_h(q) || (PML == 2 && xlive_h(q - 1))); };
  const bool out_e = ly || lz, out_h = ly || lz || lyh || lzh;  // UPML: outside the box whatever x

  const unsigned wave0 = (unsigned)__builtin_amdgcn_readfirstlane(t) * 4u;  // LDS bytes before the wave's lanes
  // step q of the march: operands of E at plane q (nx: plane 0) and, past
  // the first, the absorber words of H at plane q - 1
  auto load = [&](int q, StepOps<T, PML>& l) {
    const StepPtr<T> m = fresh<T>(mp);
    const unsigned qe = q == nx ? 0u : (unsigned)q;
    const unsigned ox = qe * PX, oy = qe * PY, oz = qe * PZ;
    const unsigned hx = ox + W0 + S, hy = oy + PY + S, hz = oz + PZ + W2;
    if constexpr (DMA) {
      const unsigned o = (unsigned)((q & 1) * slot) * 4u + wave0, n4 = (unsigned)nz * 4u, t4 = (unsigned)nt * 4u;
      const i4_t h0 = m->hi[0], h2 = m->hi[2];
      lds_load(h0, b0, hx, o + n4);
      lds_load(h2, b2, hz, o + 2 * n4 + t4);
      if (tr == 0) {
        lds_load(h0, bj0, hx, o);
        lds_load(h2, bj2, hz, o + n4 + t4);
      }
      lds_load(m->hi[1], b0, hy, o + 2 * n4 + 2 * t4);
      lds_load_nt(m->ei[0], b0, ox, o + 2 * n4 + 3 * t4);
      lds_load_nt(m->ei[1], b0, oy, o + 2 * n4 + 4 * t4);
      lds_load_nt(m->ei[2], b2, oz, o + 2 * n4 + 5 * t4);
    } else {
      if (edge) {
        l.hxj = bld<T>(m->hi[0], bj0, hx);
        l.hzj = bld<T>(m->hi[2], bj2, hz);
      }
      l.hx = bld<T>(m->hi[0], b0, hx);
      l.hy = bld<T>(m->hi[1], b0, hy);
      l.hz = bld<T>(m->hi[2], b2, hz);
      l.e0 = bld<T>(m->ei[0], b0, ox, kAuxNt);
      l.e1 = bld<T>(m->ei[1], b0, oy, kAuxNt);
      l.e2 = bld<T>(m->ei[2], b2, oz, kAuxNt);
    }
    if (m->idw == 2) l.id = (uint16_t)raw_load_i16(m->ids, (int)(b0 / S * 2u), (int)(qe * PI), kAuxNt);
    else l.id = (uint32_t)raw_load_i32(m->ids, (int)(b0 / S * 4u), (int)(qe * PI), kAuxNt);
    if constexpr (PML != 0) {
      const bool lx = x_of_e(q), lxh = x_of_h(q);
#pragma unroll
      for (int c = 0; c < (int)(sizeof(l.s) / sizeof(T)); ++c) l.s[c] = l.g[c] = T{};
      if (wave_live || lx || lxh) {
        const StepPtr<T> m = fresh<T>(mp);
        const unsigned px = (unsigned)(q - 1) * PX + W0 + S, py = (unsigned)q * PY + S, pz = (unsigned)q * PZ + W2;
        if constexpr (CP) {
          if (lz) {
            l.s[0] = bld<T>(m->si[0], b0, ox + m->ds[0]);
            l.s[1] = bld<T>(m->si[1], b0, oy);
          }
          if (q > i0 && lzh && own) {
            l.g[0] = bld<T>(m->sh[0], b0, px + m->ds[3]);
            l.g[1] = bld<T>(m->sh[1], b0, py);
          }
          if constexpr (PML == kPmlXZ) {
            if (lx) {
              l.s[2] = bld<T>(m->si[1], b0, oy + m->ds[1]);
              l.s[3] = bld<T>(m->si[2], b2, oz);
            }
            if (lxh && q > i0 && own) {
              l.g[2] = bld<T>(m->sh[1], b0, py + m->ds[4]);
              l.g[3] = bld<T>(m->sh[2], b2, pz);
            }
          } else if constexpr (PML == kPmlYZ) {
            if (ly) {
              l.s[2] = bld<T>(m->si[0], b0, ox);
              l.s[3] = bld<T>(m->si[2], b2, oz + m->ds[2]);
            }
            if (lyh && q > i0 && own) {
              l.g[2] = bld<T>(m->sh[0], b0, px);
              l.g[3] = bld<T>(m->sh[2], b2, pz + m->ds[5]);
            }
          }
        } else {
          if (out_e || lx) {
            l.s[0] = bld<T>(m->si[0], b0, ox);
            l.s[1] = bld<T>(m->si[1], b0, oy);
            l.s[2] = bld<T>(m->si[2], b2, oz);
          }
          if (q > i0 && own && (out_h || lxh)) {
            l.g[0] = bld<T>(m->sh[0], b0, px);
            l.g[1] = bld<T>(m->sh[1], b0, py);
            l.g[2] = bld<T>(m->sh[2], b2, pz);
          }
        }
      }
    }
  };

  int64_t row = 0, wave_n = 0;
  if (m->waves || blk == 0) {
    const int64_t clk = cld(&m->ctl->clk[m->par]);
    row = clk - cld(&m->ctl->wave_step0);
    wave_n = cld(&m->ctl->wave_n);
    if (blk == 0 && t == 0) {  // the step's tick
      m->ctl->clk[1 - m->par] = clk + 1;
      m->ctl->clock = clk + 1;
    }
  }

  StepOps<T, PML> ahead{};
  load(i0, ahead);
  const unsigned ip = (unsigned)(i0 ? i0 : nx);
  // E of the plane before and the old H beside it (Hy, Hz: also the H on the
  // - x side of this plane's E); new H of the plane before that
  T ex{}, ey{}, ez{}, hx{}, hy = bld<T>(m->hi[1], b0, ip * PY + S), hz = bld<T>(m->hi[2], b2, ip * PZ + W2);
  T nhx{}, nhy{}, nhz{};
  T n[3][CP ? 2 : 1] = {}, r[3][CP ? 2 : 1] = {};  // their new absorber words
  uint32_t hid = 0, meta_e = 0, meta_h = 0;  // UPML: which components those words belong to
  const double* const waves = m->waves;
  const StepRare* const rare = m->rare;
  const int net = m->net, ghosts = m->ghosts;

  // E of plane p (absorber words along x: lx) to memory
  auto store_e = [&](int p) {
    const StepPtr<T> m = fresh<T>(mp);
    const unsigned ox = (unsigned)p * PX, oy = (unsigned)p * PY, oz = (unsigned)p * PZ;
    bst<T>(m->eo[0], b0, ox, ex);
    bst<T>(m->eo[1], b0, oy, ey);
    bst<T>(m->eo[2], b2, oz, ez);
    if constexpr (PML != 0) {
      const bool lx = x_of_e(p);
      if (wave_live || lx) {
        if constexpr (CP) {
          if (ly) {
            bst<T>(m->so[0], b0, ox, n[0][0]);
            bst<T>(m->so[2], b2, oz + m->ds[2], n[2][1]);
          }
          if (lz) {
            bst<T>(m->so[0], b0, ox + m->ds[0], n[0][1]);
            bst<T>(m->so[1], b0, oy, n[1][0]);
          }
          if (lx) {
            bst<T>(m->so[1], b0, oy + m->ds[1], n[1][1]);
            bst<T>(m->so[2], b2, oz, n[2][0]);
          }
        } else {
          if (meta_e & 2u) bst<T>(m->so[0], b0, ox, n[0][0]);
          if (meta_e & 4u) bst<T>(m->so[1], b0, oy, n[1][0]);
          if (meta_e & 8u) bst<T>(m->so[2], b2, oz, n[2][0]);
        }
      }
    }
  };
  auto store_h = [&](int p) {  // the H cells of plane p
    const StepPtr<T> m = fresh<T>(mp);
    const unsigned ox = (unsigned)p * PX + W0 + S, oy = (unsigned)(p + 1) * PY + S, oz = (unsigned)(p + 1) * PZ + W2;
    bst<T>(m->ho[0], b0, ox, nhx);
    bst<T>(m->ho[1], b0, oy, nhy);
    bst<T>(m->ho[2], b2, oz, nhz);
    if constexpr (PML != 0) {
      const bool lxh = x_of_h(p + 1);
      if (wave_live || lxh) {
        if constexpr (CP) {
          if (lyh) {
            bst<T>(m->sh[0], b0, ox, r[0][0]);
            bst<T>(m->sh[2], b2, oz + m->ds[5], r[2][1]);
          }
          if (lzh) {
            bst<T>(m->sh[0], b0, ox + m->ds[3], r[0][1]);
            bst<T>(m->sh[1], b0, oy, r[1][0]);
          }
          if (lxh) {
            bst<T>(m->sh[1], b0, oy + m->ds[4], r[1][1]);
            bst<T>(m->sh[2], b2, oz, r[2][0]);
          }
        } else {
          if (meta_h & 2u) bst<T>(m->sh[0], b0, ox, r[0][0]);
          if (meta_h & 4u) bst<T>(m->sh[1], b0, oy, r[1][0]);
          if (meta_h & 8u) bst<T>(m->sh[2], b2, oz, r[2][0]);
        }
      }
    }
  };

  // Results are stored one step late, behind the loads of the next plane, which
  // are on their way before them.  (The wait for loads into LDS is for stores too:
  // one counter, in order.)
  for (int qv = i0; qv <= i1; ++qv) {
    const int q = __builtin_amdgcn_readfirstlane(qv);
    // CPML words along x and y, where there are any, for E at this plane and
    // H one plane before
    T s00{}, s21{}, s11{}, s20{}, g00{}, g21{}, g11{}, g20{};
    if constexpr (PML == 1) {
      const StepPtr<T> m = fresh<T>(mp);
      const unsigned qe = q == nx ? 0u : (unsigned)q;
      const unsigned ox = qe * PX, oy = qe * PY, oz = qe * PZ;
      const unsigned px = (unsigned)(q - 1) * PX + W0 + S, py = (unsigned)q * PY + S, pz = (unsigned)q * PZ + W2;
      if (ly) {
        s00 = bld<T>(m->si[0], b0, ox);
        s21 = bld<T>(m->si[2], b2, oz + m->ds[2]);
      }
      if (lyh && q > i0 && own) {
        g00 = bld<T>(m->sh[0], b0, px);
        g21 = bld<T>(m->sh[2], b2, pz + m->ds[5]);
      }
      if (x_of_e(q)) {
        s11 = bld<T>(m->si[1], b0, oy + m->ds[1]);
        s20 = bld<T>(m->si[2], b2, oz);
      }
      if (x_of_h(q) && q > i0 && own) {
        g11 = bld<T>(m->sh[1], b0, py + m->ds[4]);
        g20 = bld<T>(m->sh[2], b2, pz);
      }
    }
    StepOps<T, PML> l = ahead;
    if constexpr (PML == kPmlXZ) {
      s11 = l.s[2];
      s20 = l.s[3];
      g11 = l.g[2];
      g20 = l.g[3];
    } else if constexpr (PML == kPmlYZ) {
      s00 = l.s[2];
      s21 = l.s[3];
      g00 = l.g[2];
      g21 = l.g[3];
    }
    const T* const ob = xb + (q & 1) * slot;
    T* const we = eb + (q & 1) * eslot;
    const T* const re = eb + (1 - (q & 1)) * eslot;
    if constexpr (DMA) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    } else {
      T* const wb = xb + (q & 1) * slot;
      wb[t] = l.hx;
      wb[NT + t] = l.hy;
      wb[2 * NT + t] = l.hz;
    }
    __syncthreads();
    if (q < i1) load(q + 1, ahead);
    if (own) {
      if (q > i0) store_e(q - 1);
      if (q > i0 + 1) store_h(q - 2);
    }
    const bool wrap = q == nx;
    const int qe = wrap ? 0 : q;
    const bool lx = x_of_e(q), lxh = x_of_h(q), pml = PML != 0 && (wave_live || lx || lxh);
    T hyp = hy, hzp = hz;
    if constexpr (is_cplx<T>::value) {
      if (qe == 0) {
        const StepPtr<T> m = fresh<T>(mp);
        hyp = phased<T>(m->ph[1][0], hyp);
        hzp = phased<T>(m->ph[2][0], hzp);
      }
    }
    T hxj, hzj, hxk, hyk;
    if constexpr (DMA) {
      const T* const o = ob + t;
      hxj = o[0];  // the row below: the block's own, or the one loaded before its first
      l.hx = o[nz];
      hxk = ob[nz + tm];
      hzj = o[nz + nt];
      l.hz = o[2 * nz + nt];
      l.hy = o[2 * nz + 2 * nt];
      hyk = ob[2 * nz + 2 * nt + tm];
      l.e0 = o[2 * nz + 3 * nt];
      l.e1 = o[2 * nz + 4 * nt];
      l.e2 = o[2 * nz + 5 * nt];
    } else {
      hxj = l.hxj;
      hzj = l.hzj;
      if (!edge) {
        hxj = ob[t - nz];
        hzj = ob[2 * NT + t - nz];
      }
      hxk = ob[tm];
      hyk = ob[NT + tm];
    }
    const StepPtr<T> m = fresh<T>(mp);
    if constexpr (is_cplx<T>::value) {
      if (j == 0) {
        hxj = phased<T>(m->ph[0][1], hxj);
        hzj = phased<T>(m->ph[2][1], hzj);
      }
      if (k == 0) {
        hxk = phased<T>(m->ph[0][2], hxk);
        hyk = phased<T>(m->ph[1][2], hyk);
      }
    }
    const unsigned eid = l.id & ((1u << m->eb) - 1u);
    const StepEnt<R> en = et[eid];
    const R d0 = m->d[0], d1 = m->d[1], d2 = m->d[2], v0 = m->inv_d[0], v1 = m->inv_d[1], v2 = m->inv_d[2];
    // a wave without live words, but with CPML cells, takes their formula too
    // (with words of 0): its value is not the Dielectric one where a difference
    // is infinite
    T nex, ney, nez;
    auto plain_e = [&]() {
      nex = plain_value<true, X>(en.c[0], l.e0, vsub(l.hz, hzj), vsub(l.hy, hyk), d1, v1, d2, v2);
      ney = plain_value<true, X>(en.c[1], l.e1, vsub(l.hx, hxk), vsub(l.hz, hzp), d2, v2, d0, v0);
      nez = plain_value<true, X>(en.c[2], l.e2, vsub(l.hy, hyp), vsub(l.hx, hxj), d0, v0, d1, v1);
    };
    if constexpr (PML == 0) {
      plain_e();
    } else if (!pml && !(CP && __any(en.meta & kStepAbsorberCells))) {
      plain_e();
      meta_e = 0;
    } else {
      const RowT rx = CP && !LX ? dead_row<R, PML>() : x_row<R, PML>(m->re[0], m->oe[0], qe, qe, lx),
                  ry = CP && !LY ? dead_row<R, PML>() : lds_row<R, PML>(rows_y + tj * rs),
                 rz = lds_row<R, PML>(rows_z + k * rs);
      if constexpr (CP) {
        nex = cpml_value<true, X>(en.c[0], l.e0, vsub(l.hz, hzj), vsub(l.hy, hyk), d1, v1, d2, v2, ry, rz, s00, l.s[0],
                                  n[0][0], n[0][1], en.meta & 2u);
        ney = cpml_value<true, X>(en.c[1], l.e1, vsub(l.hx, hxk), vsub(l.hz, hzp), d2, v2, d0, v0, rz, rx, l.s[1], s11,
                                  n[1][0], n[1][1], en.meta & 4u);
        if constexpr (!LX && !LY) nez = dead_value<true, X>(en.c[2], l.e2, vsub(l.hy, hyp), vsub(l.hx, hxj), d0, v0, d1, v1, en.meta & 8u);
        else nez = cpml_value<true, X>(en.c[2], l.e2, vsub(l.hy, hyp), vsub(l.hx, hxj), d0, v0, d1, v1, rx, ry, s20, s21,
                                  n[2][0], n[2][1], en.meta & 8u);
      } else {
        plain_e();
        meta_e = en.meta;
        if (en.meta & 2u)
          nex = upml_value<true, X>(en.c[0], l.e0, vsub(l.hz, hzj), vsub(l.hy, hyk), d1, v1, d2, v2, ry, rz, rx,
                                    l.s[0], n[0][0]);
        if (en.meta & 4u)
          ney = upml_value<true, X>(en.c[1], l.e1, vsub(l.hx, hxk), vsub(l.hz, hzp), d2, v2, d0, v0, rz, rx, ry,
                                    l.s[1], n[1][0]);
        if (en.meta & 8u)
          nez = upml_value<true, X>(en.c[2], l.e2, vsub(l.hy, hyp), vsub(l.hx, hxj), d0, v0, d1, v1, rx, ry, rz,
                                    l.s[2], n[2][0]);
      }
    }
    if (en.meta & kStepRareCell) {
      const StepRare* x = rare + eid * 3;
      nex = step_rare<T>(x, waves, wave_n, row, l.e0, nex);
      ney = step_rare<T>(x + 1, waves, wave_n, row, l.e1, ney);
      nez = step_rare<T>(x + 2, waves, wave_n, row, l.e2, nez);
    }
    we[t] = nex;
    we[est + t] = ney;
    we[2 * est + t] = nez;
    if (ghosts && own && q < i1) {
      // ghost images: E's from the new values, H's from the old ones
      const unsigned ox = (unsigned)q * PX, oy = (unsigned)q * PY, oz = (unsigned)q * PZ;
      if (k == 0) {
        const StepPtr<T> m = fresh<T>(mp);
        const unsigned last = b0 + (unsigned)nz * S;
        bst<T>(m->eo[0], last, ox, phased<T>(m->pe[0][2], nex));
        const T y1 = phased<T>(m->pe[1][2], ney);
        bst<T>(m->eo[1], last, oy, y1);
        bst<T>(m->ho[0], b0 + W0, ox, hxk);
        bst<T>(m->ho[1], b0, oy + PY, hyk);
        if (q == 0) {
          bst<T>(m->eo[1], last, (unsigned)nx * PY, phased<T>(m->pe[1][0], y1));
          const T y = bld<T>(m->hi[1], last, (unsigned)nx * PY);
          bst<T>(m->ho[1], b0, 0, phased<T>(m->ph[1][0], phased<T>(m->ph[1][2], y)));
        }
      }
      if (j == 0) {
        const StepPtr<T> m = fresh<T>(mp);
        const unsigned r0 = (unsigned)k * S;
        const T x1 = phased<T>(m->pe[0][1], nex);
        bst<T>(m->eo[0], r0, ox + PX - W0, x1);
        bst<T>(m->eo[2], r0, oz + PZ - W2, phased<T>(m->pe[2][1], nez));
        bst<T>(m->ho[0], r0 + S, ox, hxj);
        bst<T>(m->ho[2], r0, oz + PZ, hzj);
        if (k == 0) {
          const unsigned last = (unsigned)nz * S;
          bst<T>(m->eo[0], last, ox + PX - W0, phased<T>(m->pe[0][2], x1));
          const T x = bld<T>(m->hi[0], last, ox + PX - W0);
          bst<T>(m->ho[0], 0, ox, phased<T>(m->ph[0][2], phased<T>(m->ph[0][1], x)));
        }
      }
      if (q == 0) {
        const StepPtr<T> m = fresh<T>(mp);
        bst<T>(m->eo[1], b0, (unsigned)nx * PY, phased<T>(m->pe[1][0], ney));
        const T z1 = phased<T>(m->pe[2][0], nez);
        bst<T>(m->eo[2], b2, (unsigned)nx * PZ, z1);
        bst<T>(m->ho[1], b0 + S, 0, hyp);
        bst<T>(m->ho[2], b2 + W2, 0, hzp);
        if (j == 0) {
          const unsigned r0 = (unsigned)k * S, o = (unsigned)nx * PZ + PZ - W2;
          bst<T>(m->eo[2], r0, o, phased<T>(m->pe[2][1], z1));
          const T z = bld<T>(m->hi[2], r0, o);
          bst<T>(m->ho[2], r0, 0, phased<T>(m->ph[2][1], phased<T>(m->ph[2][0], z)));
        }
      }
    }
    if (q > i0 && own) {
      T exj = re[t + nz], ezj = re[2 * est + t + nz];
      T exk = re[tp], eyk = re[est + tp];
      T eyi = ney, ezi = nez;
      const StepPtr<T> m = fresh<T>(mp);
      if constexpr (is_cplx<T>::value) {
        if (j == ny - 1) {
          exj = phased<T>(m->pe[0][1], exj);
          ezj = phased<T>(m->pe[2][1], ezj);
        }
        if (k == nz - 1) {
          exk = phased<T>(m->pe[0][2], exk);
          eyk = phased<T>(m->pe[1][2], eyk);
        }
        if (wrap) {
          eyi = phased<T>(m->pe[1][0], eyi);
          ezi = phased<T>(m->pe[2][0], ezi);
        }
      }
      const StepEnt<R> eh = et[net + hid];
      const R d0 = m->d[0], d1 = m->d[1], d2 = m->d[2], v0 = m->inv_d[0], v1 = m->inv_d[1], v2 = m->inv_d[2];
      auto plain_h = [&]() {
        nhx = plain_value<false, X>(eh.c[0], hx, vsub(ezj, ez), vsub(eyk, ey), d1, v1, d2, v2);
        nhy = plain_value<false, X>(eh.c[1], hy, vsub(exk, ex), vsub(ezi, ez), d2, v2, d0, v0);
        nhz = plain_value<false, X>(eh.c[2], hz, vsub(eyi, ey), vsub(exj, ex), d0, v0, d1, v1);
      };
      if constexpr (PML == 0) {
        plain_h();
      } else if (!pml && !(CP && __any(eh.meta & kStepAbsorberCells))) {
        plain_h();
        meta_h = 0;
      } else {
        const RowT rx = CP && !LX ? dead_row<R, PML>() : x_row<R, PML>(m->rh[0], m->oh[0], q, q - 1, lxh),
                    ry = CP && !LY ? dead_row<R, PML>() : lds_row<R, PML>(rows_yh + tj * rs),
                   rz = lds_row<R, PML>(rows_zh + k * rs);
        if constexpr (CP) {
          nhx = cpml_value<false, X>(eh.c[0], hx, vsub(ezj, ez), vsub(eyk, ey), d1, v1, d2, v2, ry, rz, g00, l.g[0],
                                     r[0][0], r[0][1], eh.meta & 2u);
          nhy = cpml_value<false, X>(eh.c[1], hy, vsub(exk, ex), vsub(ezi, ez), d2, v2, d0, v0, rz, rx, l.g[1], g11,
                                     r[1][0], r[1][1], eh.meta & 4u);
          if constexpr (!LX && !LY) nhz = dead_value<false, X>(eh.c[2], hz, vsub(eyi, ey), vsub(exj, ex), d0, v0, d1, v1, eh.meta & 8u);
          else nhz = cpml_value<false, X>(eh.c[2], hz, vsub(eyi, ey), vsub(exj, ex), d0, v0, d1, v1, rx, ry, g20, g21,
                                     r[2][0], r[2][1], eh.meta & 8u);
        } else {
          plain_h();
          meta_h = eh.meta;
          if (eh.meta & 2u)
            nhx = upml_value<false, X>(eh.c[0], hx, vsub(ezj, ez), vsub(eyk, ey), d1, v1, d2, v2, ry, rz, rx, l.g[0],
                                       r[0][0]);
          if (eh.meta & 4u)
            nhy = upml_value<false, X>(eh.c[1], hy, vsub(exk, ex), vsub(ezi, ez), d2, v2, d0, v0, rz, rx, ry, l.g[1],
                                       r[1][0]);
          if (eh.meta & 8u)
            nhz = upml_value<false, X>(eh.c[2], hz, vsub(eyi, ey), vsub(exj, ex), d0, v0, d1, v1, rx, ry, rz, l.g[2],
                                       r[2][0]);
        }
      }
      if (eh.meta & kStepRareCell) {
        const StepRare* x = rare + (net + hid) * 3;
        nhx = step_rare<T>(x, waves, wave_n, row, hx, nhx);
        nhy = step_rare<T>(x + 1, waves, wave_n, row, hy, nhy);
        nhz = step_rare<T>(x + 2, waves, wave_n, row, hz, nhz);
      }
    }
    ex = nex;
    ey = ney;
    ez = nez;
    hx = l.hx;
    hy = l.hy;
    hz = l.hz;
    hid = l.id >> m->eb;
  }
  if (own) store_h(i1 - 1);
}

template <class T, int PML> struct StepWaves { static constexpr int v = PML == 0 || PML == kPmlZ ? 4 : 3; };
template <int PML> struct StepWaves<float, PML> { static constexpr int v = PML ? 6 : 8; };

template <class T, int PML, bool X>
__global__ void __launch_bounds__(step3_max_threads<T>(PML)) __attribute__((amdgpu_waves_per_eu(StepWaves<T, PML>::v))) k_step3d(Step3Args<T>) {
  extern __shared__ __attribute__((aligned(16))) char step_lds[];
  const StepPtr<T> m = (StepPtr<T>)__builtin_amdgcn_kernarg_segment_ptr();
  if constexpr (PML == kPmlMixed) {
    int rc;
    unsigned rb;
    (void)step3d_block<T>(m, blockIdx.x, rc, rb);
    const int kind = m->rect[rc].kind;
    if (kind == kPmlZ) step3d_tile<T, kPmlZ, X>(m, blockIdx.x, step_lds);
    else if (kind == kPmlXZ) step3d_tile<T, kPmlXZ, X>(m, blockIdx.x, step_lds);
    else if (kind == kPmlYZ) step3d_tile<T, kPmlYZ, X>(m, blockIdx.x, step_lds);
    else step3d_tile<T, 1, X>(m, blockIdx.x, step_lds);
  } else {
    step3d_tile<T, PML, X>(m, blockIdx.x, step_lds);
  }
}

__global__ void __launch_bounds__(256) k_step_ids(StepIdArgs a) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t r = t / a.n[2];
  if (r >= (int64_t)a.n[0] * a.n[1]) return;
  const int k = (int)(t - r * a.n[2]), i = (int)(r / a.n[1]), j = (int)(r - (int64_t)i * a.n[1]);
  uint32_t v = 0;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if (h >= a.types) continue;
    uint16_t id[3];
#pragma unroll
    for (int c = 0; c < 3; ++c)
      id[c] = gld(a.ids[3 * h + c] + a.first[3 * h + c] + i * a.plane[3 * h + c] + j * a.row[3 * h + c] + k);
    const uint64_t key = step_key(id[0], id[1], id[2]);
    uint32_t at = step_hash(key, a.mask[h]);
    for (uint32_t n = 0; n <= a.mask[h]; ++n) {  // every cell's triple is in the table
      const uint64_t got = gld(&a.tab[h][at].key);
      if (got == key) {
        v |= (uint32_t)gld(&a.tab[h][at].id) << (h ? a.shift : 0);
        break;
      }
      at = (at + 1) & a.mask[h];
    }
  }
  if (a.out16) gst(a.out16 + (int64_t)r * a.pitch + k, (uint16_t)v);
  else gst(a.out + (int64_t)r * a.pitch + k, v);
}

void launch_step_ids(const StepIdArgs& a, hipStream_t st) {
  const int64_t n = (int64_t)a.n[0] * a.n[1] * a.n[2];
  hipLaunchKernelGGL(k_step_ids, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a);
}

__global__ void __launch_bounds__(256) k_list_places(PlaceArgs a) {
  const int q = blockIdx.x * 256 + threadIdx.x;
  if (q >= a.n) return;
  const int x = a.cell[q], k = x % a.s2, r = x / a.s2, j = r % a.s1, i = r / a.s1;
  a.out[i * a.pi + j * a.p + k * a.pk] = q;
}

void launch_list_places(const PlaceArgs& a, hipStream_t st) {
  hipLaunchKernelGGL(k_list_places, dim3((unsigned)(a.n + 255) / 256), dim3(256), 0, st, a);
}

__global__ void k_clock_copy(Ctl* ctl) { ctl->clk[0] = ctl->clk[1] = ctl->clock; }

void launch_clock_copy(Ctl* ctl, hipStream_t st) { hipLaunchKernelGGL(k_clock_copy, dim3(1), dim3(1), 0, st, ctl); }

// Every block of every member, by its own kind; blocks of one size.  LEAN: see
// step3_batch_threads (in the kernel of all kinds, complex FP32 slabs with z
// layers run at 12 waves a CU, and no faster than two batched launches).  us
// per step, two launches each for E and H before: 8 2-D and 6 3-D FP32 members
// of 128 to 640 and 64 to 160 cells a side 329 -> 259 (3-D 243 -> 216); 8
// complex FP32 slabs of 64 to 206 with plane waves 970 -> 855; 4 FP64 CPML
// boxes of 64 to 128 274 -> 187.
template <class T, bool X, bool LEAN>
__global__ void __launch_bounds__(step3_batch_threads<T>(LEAN))
    __attribute__((amdgpu_waves_per_eu(StepWaves<T, LEAN ? kPmlZ : kPmlMixed>::v))) k_step3d_batch(const Step3Job<T>* jobs, int njobs) {
  extern __shared__ __attribute__((aligned(16))) char step_lds[];
  const GMES_CONST Step3Job<T>* J = step_job(jobs, njobs, (int64_t)blockIdx.x);
  const StepPtr<T> m = &J->a;
  const unsigned blk = (unsigned)((int64_t)blockIdx.x - J->block0);
  int rc;
  unsigned rb;
  (void)step3d_block<T>(m, blk, rc, rb);
  const int kind = m->rect[rc].kind;
  if constexpr (LEAN) {
    if (kind == kPmlZ) step3d_tile<T, kPmlZ, X>(m, blk, step_lds);
    else step3d_tile<T, kPmlNone, X>(m, blk, step_lds);
  } else {
    if (kind == kPmlZ) step3d_tile<T, kPmlZ, X>(m, blk, step_lds);
    else if (kind == kPmlXZ) step3d_tile<T, kPmlXZ, X>(m, blk, step_lds);
    else if (kind == kPmlYZ) step3d_tile<T, kPmlYZ, X>(m, blk, step_lds);
    else if (kind == kPmlXYZ) step3d_tile<T, kPmlXYZ, X>(m, blk, step_lds);
    else step3d_tile<T, kUpml, X>(m, blk, step_lds);
  }
}

template <class T>
void launch_step3d_batch(const Step3Job<T>* jobs, int njobs, int64_t nblocks, bool exact, bool lean, size_t lds,
                         hipStream_t st) {
  if (!njobs) return;
  const dim3 grid((unsigned)nblocks), block(step3_batch_threads<T>(lean));
#define GMES_BATCH3(X)                                                                                          \
  {                                                                                                             \
    if (lean) hipLaunchKernelGGL((k_step3d_batch<T, X, true>), grid, block, (unsigned)lds, st, jobs, njobs);    \
    else hipLaunchKernelGGL((k_step3d_batch<T, X, false>), grid, block, (unsigned)lds, st, jobs, njobs);        \
  }
  if constexpr (std::is_same<T, double>::value) {
    if (exact) {
      GMES_BATCH3(true)
      return;
    }
  }
  GMES_BATCH3(false)
#undef GMES_BATCH3
}
template void launch_step3d_batch<float>(const Step3Job<float>*, int, int64_t, bool, bool, size_t, hipStream_t);
template void launch_step3d_batch<double>(const Step3Job<double>*, int, int64_t, bool, bool, size_t, hipStream_t);
template void launch_step3d_batch<cplx<float>>(const Step3Job<cplx<float>>*, int, int64_t, bool, bool, size_t, hipStream_t);

template <class T>
void launch_step3d(const Step3Args<T>& m, int absorber, int nthreads, hipStream_t st) {
  const dim3 grid(8u * (unsigned)m.slots), block(nthreads);
  const unsigned lds = (unsigned)step3_lds<T>(nthreads, m.net + m.nht, m.rows, m.n[2], absorber);
#define GMES_STEP(X)                                                                              \
  {                                                                                               \
    if (absorber == 0) hipLaunchKernelGGL((k_step3d<T, 0, X>), grid, block, lds, st, m);          \
    else if (absorber == 1) hipLaunchKernelGGL((k_step3d<T, 1, X>), grid, block, lds, st, m);     \
    else if (absorber == kPmlZ) hipLaunchKernelGGL((k_step3d<T, kPmlZ, X>), grid, block, lds, st, m);     \
    else if (absorber == kPmlMixed) hipLaunchKernelGGL((k_step3d<T, kPmlMixed, X>), grid, block, lds, st, m);     \
    else hipLaunchKernelGGL((k_step3d<T, 2, X>), grid, block, lds, st, m);                        \
  }
  if constexpr (std::is_same<T, double>::value) {
    if (m.exact) {
      GMES_STEP(true)
      return;
    }
  }
  GMES_STEP(false)
#undef GMES_STEP
}

template void launch_step3d<float>(const Step3Args<float>&, int, int, hipStream_t);
template void launch_step3d<double>(const Step3Args<double>&, int, int, hipStream_t);
template void launch_step3d<cplx<float>>(const Step3Args<cplx<float>>&, int, int, hipStream_t);

}  // namespace gmes_engine
