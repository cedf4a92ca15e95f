// Kernel argument blocks and launchers shared by kernels.hip and engine.hip.
#pragma once

#include "engine_internal.h"

namespace gmes_engine {

typedef int i4_t __attribute__((ext_vector_type(4)));

constexpr int kDm2Max = 8;    // transitions per DM2 cell held in registers
constexpr int kRecLds = 128;  // records staged in LDS by the 3-D main kernel

// Per-sim control block in device memory: everything a step reads that
// changes between steps, so one captured step graph can be replayed.
struct Ctl {
  int64_t clock;       // steps started (thread 0 of the first kernel of a step adds 1)
  int64_t wave_step0;  // absolute step of waveform row 0
  int64_t wave_n;      // rows per waveform
  int64_t probe_base;  // absolute step of probe slot 0
  int64_t dft_step0;   // absolute step of DFT weight row 0
  int64_t dft_n;       // rows of DFT weights
  int32_t err;         // deferred device error (1 NaN, 2 no convergence)
  int32_t pad_;
  int64_t clk[2];      // the clock as the one-sweep steps pass it on (StepArgs::par)
};

constexpr int kPad = 32;  // elements before row 0 of every device array

// Device layout of a component: logical (i,j,k) of a component with shape
// (s0,s1,s2) lives at element kPad + (i*s1 + j)*p + k - koff.  The row
// pitch p is s2 rounded up to 32 elements when s2 >= 32 (else s2), and
// koff = 1 for Hx and Hy on a padded layout, so that the first updated
// cell of every row (k = 0 for E and Hz, k = 1 for Hx, Hy) starts a
// 128-byte line.  3-D sims with rows under 256 cells keep p = s2 and
// koff = 0 (gmes_sim::packed).  Collapsed-z 2-D modes (TMz, TEz) keep each z
// plane of a component in one piece: element kPad + i*pi + j + k*pk - koff,
// with rows along j padded the same way (koff = 1 for Hx and Hz, updated
// from j = 1).  With k fastest, every second element of Hx, Hy (TMz) or Ex,
// Ey (TEz) is a ghost, and the launches move twice the bytes they use.
// Material ids and CPML/UPML state use the same layout.
template <class T>
struct FieldArgs {
  T* f[6];
  int s[6][3];
  int pi[6], p[6], pk[6];  // strides along i, j, k
  int koff[6];
  unsigned active;
};

template <class T>
__host__ __device__ __forceinline__ int didx(const FieldArgs<T>& a, int c, int i, int j, int k) {
  return kPad + i * a.pi[c] + j * a.p[c] + k * a.pk[c] - a.koff[c];
}

template <class T>
struct MainArgs {
  using R = typename real_of<T>::type;
  FieldArgs<T> fa;
  const uint16_t* ids[6];
  const DevRec<R>* recs;
  const R* prof;
  const int64_t* prof_off;
  void* pml[6];
  int dsize[6];  // device elements per component (offset of the 2nd CPML word)
  R d[3];
  R inv_d[3];
  int nrec;
  int n[3];  // nx, ny, nz
  // 1: the 3-D E kernel writes the E ghost planes itself (fused_ghost)
  int fuse;
  int gax[3][2];      // transverse axes a1, a2 of Ex, Ey, Ez
  cplx<R> gph[3][2];  // ghost phase along a1, a2
  const uint8_t* ids8[6];  // the ids as bytes (real-FP32 3-D sims), when narrow
  int narrow;
  // generic kernels: 1 when every row has at most 2 elements (kext); each
  // thread then covers a whole row (bx = 1)
  int kloop, kext;
  // real-FP32 3-D kernels: components with CPML state (bit c), and per axis
  // the coordinate run (lo | hi << 16) where every CPML profile's c is zero
  unsigned cpml_mask;
  int prun[3];
  int po0[6][3];  // offsets of profile set 0's rows (component, axis) in the pool
  // real-FP32 3-D kernels with CPML state in all three components of the
  // field type: pp = 1 when, per axis, the two components that read a
  // profile along it have identical set-0 rows; pprow[a] is then the pool
  // offset of one of them, and the kernels load the row of each axis with
  // the cell's other operands (lanes outside the zero-c run of that axis)
  int pp;
  int pprow[3];
  // real-FP32 3-D kernels: components whose UPML state word is loaded with
  // the other operands (bit c), and a box (per axis lo | hi << 16) that
  // holds no UPML cell of those components
  unsigned upml_mask;
  int ubox[3];
  // real-FP32 3-D kernels whose three components of the field type all
  // carry prefetched UPML state: ur = 1 when, per axis, the two components
  // that read it as a curl axis have identical set-0 rows; urs[a] is then
  // the pool offset of that row and uro[a] that of the owning component's
  // row, and the kernels load both with the cell's other operands (lanes
  // outside ubox)
  int ur;
  int urs[3], uro[3];
  // 2-D modes with a collapsed z axis (TMz): 1 when the E kernel writes the
  // z ghost plane (k = 0) of Hx and Hy, which no E update reads, in place
  // of that part of the H ghost copy; hzph: the copy's phase along z for
  // Hx and Hy; hyxph: Hy's phase along x (its corner line)
  int hzg;
  cplx<R> hzph[2];
  cplx<R> hyxph;
};

// ---- one-sweep steps
// A whole leapfrog step of one sim in one kernel (step3d.hip): the
// fields are read from one set of buffers (fi) and written to another (fo),
// so E can be computed again where a neighbouring block needs it and H
// follows from it at once.  A cell's three E components (and the three H
// components the same thread owns) share one table entry.
// Dummy, Const and source cells are flagged (StepRare has the details).
constexpr uint32_t kStepRareCell = 1, kStepAbsorberCells = 14;  // CPML, UPML: bit 1 + t for component t
template <class R>
struct alignas(16) StepEnt {
  R c[3];         // dt/eps; UPML cells: 1/eps (FP32) or eps (FP64)
  uint32_t meta;  // kStepRareCell | 2 << t per absorber component
};

// Absorbers of a one-sweep step: none, CPML with state along x, y and z, UPML,
// CPML with state along z only, a launch with blocks of several kinds, CPML
// along x and z, along y and z.
constexpr int kPmlNone = 0, kPmlXYZ = 1, kUpml = 2, kPmlZ = 3, kPmlMixed = 4, kPmlXZ = 5, kPmlYZ = 6;
// cells [i0, i1) x [j0, j1) of a launch: ch planes per block, nj tiles along
// j, nblk blocks; per: blocks of it per XCD, first: those of the rectangles before
struct StepRect {
  int i0, i1, j0, j1, ch, nj, nblk, per, first, kind;
};

template <class T>
struct Step3Args {
  using R = typename real_of<T>::type;
  // buffer resources (base address, bytes): each starts at the array's
  // logical element (0, 0, 0)
  i4_t ei[3], hi[3];  // old E, H
  i4_t eo[3], ho[3];  // new E, H
  i4_t si[3], so[3];  // E absorber state, read and written
  i4_t sh[3];         // H absorber state (in place: only its owner touches a word)
  i4_t ids;           // [i][j][k] table entries of the E and H cells of thread (i, j, k): E | H << eb,
  int eb, idw;        // in words of idw bytes (2 when both fit, else 4 and eb = 16)
  int W0, W2;      // row pitch of Ex, Ey, Hx, Hy and of Ez, Hz
  int n[3];
  const void* tab;      // StepEnt<R>[net + nht]: E entries, then H entries
  const StepRare* rare;  // [3 * (net + nht)]
  int net, nht;
  unsigned ds[6];  // CPML: bytes from the first word of a component's state to the second
  R d[3], inv_d[3];
  const R* re[3];  // absorber rows of E along x, y, z (CPML: b, c, kappa; UPML: c1..c6 of the shared row)
  const R* rh[3];  // the same of H
  const R* oe[3];  // UPML: rows of the component whose own axis it is
  const R* oh[3];
  int run_e[3], run_h[3];  // CPML: per axis the coordinates lo | hi << 16 without live state; UPML: the UPML-free box
  cplx<R> pe[3][3];  // ghost phase of E component c along axis a
  cplx<R> ph[3][3];  // of H
  int rows;        // (j) rows per block, the last one a rim
  int nrect, slots;  // rectangles, blocks per XCD
  StepRect rect[9];
  const double* waves;
  Ctl* ctl;
  int par;
  int exact;       // FP64: every division is by a power of two
  int ghosts;      // write the ghost planes: the last step of a call, unless a monitor reads them
};
// Cells a one-sweep 3-D step leaves to two launches after it (stepfix.hip):
// dispersive E cells and E cells with sources that do not fit its table, then
// the H cells whose curl reads those, and H cells with such sources.
constexpr int kFixBlock = 256, kFixMark = 1024;
struct FixItem {
  int32_t cell;  // thread (i * ny + j) * nz + k
  int32_t grp;   // source group, -1: none
};
template <class T>
struct FixArgs {
  using R = typename real_of<T>::type;
  // by direction, at thread (0, 0, 0)'s cell
  const T* ei[3];  // old E, H
  const T* hi[3];
  T* eo[3];        // new ones
  T* ho[3];
  T* base[6];      // new arrays from element 0 (source groups)
  int pe[3], re[3], ph[3], rh[3];  // strides along i and j of E, H
  int n[3];
  cplx<R> phe[3][3], phh[3][3];    // ghost phases of component c along axis a
  R d[3], inv_d[3];
  const DevRec<R>* recs;
  const R* coef;
  const uint16_t* hid[3];
  struct { const int32_t* cell; const uint16_t* rec; void* state; int n, comp, cls, first, s1, s2; } ade[9];
  int nade;
  const SrcGroup* groups;  // E's, then H's
  int nge, first_src;      // E groups, their first block
  const DevSrcOp<R>* ops;
  const double* waves;
  const void* aux[8][6];   // current fields of the auxiliary grids
  Ctl* ctl;
  const FixItem* items;
  int nitem[3], first_item[3], item_blk[3];  // of Hx, Hy, Hz; first item, first block
  int eblocks, hblocks;
};
template <class T> void launch_fix_e(const FixArgs<T>& a, hipStream_t st);
template <class T> void launch_fix_h(const FixArgs<T>& a, hipStream_t st);
// Marks the H cells of the lists (phase 0: dispersive cells and E groups, the
// H cells that read them; H groups, themselves), counts them per kFixMark
// cells, writes the items, and their groups.
struct FixBuild {
  int n[3];
  int64_t cells;           // n[0] * n[1] * n[2]
  uint8_t* mark;           // [3][cells]
  int32_t* count;          // [3][blocks]: marked cells, then their first item
  int nblk;
  FixItem* items;
  int nitem[3], first_item[3];
  const int32_t* ade_cell; // one list
  int ade_n, comp, s1, s2;
  const SrcGroup* groups;
  int ngroups, nge;
  int64_t base[6];         // element of logical (0, 0, 0)
  int pi[6], p[6];
  const uint16_t* hid[3];  // at thread (0, 0, 0)
  const int32_t* cls;      // class of each record
  int run_h[3];            // thread coordinates without live CPML state
  int* bad;                // an absorber cell with live state is among them
};
void launch_fix_mark_ade(const FixBuild& b, hipStream_t st);
void launch_fix_mark_src(const FixBuild& b, hipStream_t st);
void launch_fix_count(const FixBuild& b, hipStream_t st);
void launch_fix_fill(const FixBuild& b, hipStream_t st);

// The same for a collapsed-z 2-D mode (TMz: Ez, Hx, Hy; TEz: Ex, Ey, Hz).
// Arrays are indexed by the direction of the component; thread (i, j) owns
// one cell of each, at element off + i * pi + j of its arrays.
constexpr int kStep2Src = 16;
struct Step2Cell {
  int32_t kind;  // 0 the update of its entry, 1 Dummy, 2 Const, 3 dispersive
  int32_t rec;   // dispersive: its record
  double re, im; // Const value
};
template <class R>
struct Step2Ent {
  R c[3];         // dt/eps; UPML: 1/eps (FP32) or eps (FP64)
  uint32_t meta;  // 2 bits a component: 0 Dielectric, 1 absorber, 2 see Step2Cell
};
template <class T>
struct Step2Args {
  using R = typename real_of<T>::type;
  const T* fi[3];       // old fields, at thread (0, 0)'s cells
  T* fo[3];             // new ones
  // absorber words: CPML [x word, y word] of E and of H, UPML the component's
  const T* si[3][2];
  T* so[3][2];          // (H: the same arrays, only the owner touches a word)
  int pi;               // stride along i, of every array
  int64_t pk[3];        // from the updated z plane to its ghost plane (0: none)
  const uint16_t* ids;  // [i * pi + j] entries
  int n[2];
  const Step2Ent<R>* tab;
  const Step2Cell* cells;  // [3 * entry + direction]
  int nent;
  R d[3], inv_d[3];
  const R* row[3][3];   // absorber rows of component c along axis a, at thread (0, 0)'s coordinate
  int run[3][2];        // CPML: thread coordinates lo | hi << 16 without live state, x and y; UPML: [0] the UPML-free box
  cplx<R> ph[3][3];     // ghost phase of component c along axis a
  const DevRec<R>* recs;
  const R* coef;
  const int32_t* adeq[3];  // place of a dispersive cell in its list, at thread (0, 0)'s cell
  const void* ade_in[3][3];
  void* ade_out[3][3];
  int ade_n[3][3];
  int nsrc;
  struct { int c, i, j, wave, kind; } src[kStep2Src];
  int w;                // columns a block owns; n[1] when whole (neighbours wrap inside the block)
  int whole;
  int ch;               // rows per block
  int nj, nblk;
  const double* waves;
  Ctl* ctl;
  int par;
  int exact;
  int ghosts;
};
// threads of a block at most: 8-byte and wider words need more than 64 registers
template <class T> constexpr int kStep2Threads = sizeof(T) == 4 ? 1024 : 512;
// threads of a block: its columns and, unless rows are whole, two rim lanes
inline int step2_threads(int w, int whole) { return ((whole ? w : w + 2) + 63) / 64 * 64; }
template <class T>
inline size_t step2_lds(int nthreads, int nent) {
  return (size_t)nent * sizeof(Step2Ent<typename real_of<T>::type>) + 4 * (size_t)nthreads * sizeof(T);
}

// The same for a 1-D line (TEM modes; also the auxiliary grids of total-field
// boxes): component e of E, h = e + 1 of H, along axis e + 2 (mod 3).
template <class T>
struct Step1Args {
  using R = typename real_of<T>::type;
  const T* fi[2];   // old E, H at cell 0
  T* fo[2];
  const T* si[2];   // absorber words: CPML along the line, UPML the component's
  T* so[2];
  int st[2];        // element strides along the line
  int64_t gc[2];    // from a cell to its ghost image along the collapsed axis
  const uint16_t* ids[2];
  int n;
  const DevRec<R>* recs;
  const R* coef;
  const R* row[2][3];  // absorber rows of E, H: first curl axis, second, own; the line's at cell 0
  cplx<R> ph[2][2];    // ghost phase along the collapsed axis, along the line
  R d[3], inv_d[3];    // of axes e, h, the line
  const int32_t* adeq;
  const void* ade_in[3];
  void* ade_out[3];
  int ade_n[3];
  int nsrc;
  struct { int c, q, wave, kind; } src[kStep2Src];
  const double* waves;
  Ctl* ctl;
  int par, ghosts, absorber;
};
constexpr int kStep1Threads = 256;
template <class T>
void launch_step1d(const Step1Args<T>& m, hipStream_t st);

// Batched one-sweep launches: job tables as those below.  3-D and 2-D jobs start
// at a multiple of 8 blocks (their blocks go round the XCDs).
template <class T> struct Step3Job { Step3Args<T> a; int64_t block0; };
template <class T> struct Step2Job { Step2Args<T> a; int tm, absorber; int64_t block0; };
template <class T> struct Step1Job { Step1Args<T> a; int64_t block0; };
template <class T> struct FixJob { FixArgs<T> a; int64_t block0; };
constexpr int kStep2BatchThreads = 256;
// lean: jobs without CPML words along x and y and without UPML, whose 8-byte
// bodies fit 128 registers
template <class T> constexpr int step3_batch_threads(bool lean) { return sizeof(T) == 8 && lean ? 1024 : 768; }
template <class T>
void launch_step3d_batch(const Step3Job<T>* jobs, int njobs, int64_t nblocks, bool exact, bool lean, size_t lds,
                         hipStream_t st);
template <class T>
void launch_step2d_batch(const Step2Job<T>* jobs, int njobs, int64_t nblocks, size_t lds, hipStream_t st);
template <class T>
void launch_step1d_batch(const Step1Job<T>* jobs, int njobs, int64_t nblocks, hipStream_t st);
template <class T>
void launch_fix_batch(bool electric, const FixJob<T>* jobs, int njobs, int64_t nblocks, hipStream_t st);

// The entry ids of a sim, looked up from its material ids on the device.
struct StepKey {
  uint64_t key, id;  // key ~0: empty slot
};
__host__ __device__ inline uint64_t step_key(uint16_t a, uint16_t b, uint16_t c) {
  return a | (uint64_t)b << 16 | (uint64_t)c << 32;
}
__host__ __device__ inline uint32_t step_hash(uint64_t key, uint32_t mask) {
  return (uint32_t)((key * 0x9E3779B97F4A7C15ull) >> 40) & mask;
}
struct StepIdArgs {
  const uint16_t* ids[6];
  int64_t first[6], plane[6], row[6];  // element of thread (0, 0, 0), strides along i and j
  const StepKey* tab[2];               // E, H; open addressing, at most a quarter full
  uint32_t mask[2];
  int n[3];
  int pitch;       // of out's rows
  int types;       // 1: one triple per cell (2-D modes), 2: E | H << shift
  int shift;
  uint32_t* out;   // or, when out16
  uint16_t* out16;
};
void launch_step_ids(const StepIdArgs& a, hipStream_t st);
// out[element of cell[q]] = q, for the cells of a list
struct PlaceArgs {
  const int32_t* cell;
  int n, s1, s2, pi, p, pk;
  int32_t* out;  // at element (0, 0, 0)
};
void launch_list_places(const PlaceArgs& a, hipStream_t st);
// threads of a block at most: with 8-byte words the kernels of a full
// absorber need 150 to 172 registers, three waves a SIMD
constexpr int kStepMaxThreads = 1024;
template <class T>
constexpr int step3_max_threads(int absorber) {
  return sizeof(T) == 8 && absorber != kPmlNone && absorber != kPmlZ ? 768 : kStepMaxThreads;
}
// bytes of LDS of a block: exchange buffers, entries, absorber rows
template <class T>
inline size_t step3_lds(int nthreads, int nent, int rows, int nz, int absorber) {
  using R = typename real_of<T>::type;
  const size_t stride = absorber == kUpml ? 8 : absorber ? 4 : 0;
  const size_t exchange = sizeof(T) == 4 ? (2 * (2 * (size_t)nz + 9 * (size_t)nthreads) + 3) / 4 * 4 * sizeof(T)
                                         : (size_t)12 * nthreads * sizeof(T);
  return exchange + (size_t)nent * sizeof(StepEnt<R>) +
         2 * (size_t)(rows + nz) * stride * sizeof(R);
}

template <class T>
struct AdeArgs {
  using R = typename real_of<T>::type;
  FieldArgs<T> fa;
  const int32_t* cell;
  const uint16_t* rec;
  void* state;
  int n;
  const DevRec<R>* recs;
  const R* coef;
  R d[3];
  R dt;
  Ctl* ctl;
};

template <class T>
struct SrcArgs {
  using R = typename real_of<T>::type;
  FieldArgs<T> fa;
  const SrcGroup* groups;
  int ngroups;
  const DevSrcOp<R>* ops;
  const double* waves;
  void* const* aux;
  Ctl* ctl;
};

template <class T>
struct ProbeArgs {
  FieldArgs<T> fa;
  const int64_t* cells;
  const int32_t* comps;
  int n;
  int types;  // 0: H, 1: E, 2: both
  double* buf;
  int64_t cap;
  Ctl* ctl;
};

template <class T>
struct GhostArgs {
  using R = typename real_of<T>::type;
  FieldArgs<T> fa;
  int ncomp;
  int comp[3];
  int ax[3][3];      // a1, a2, own axis
  int64_t count[3];  // ghost points per component
  cplx<R> ph[3][2];  // phase of the copy along a1, a2
  int tick;
  Ctl* ctl;
  int64_t skip[3];   // leading points of a component's copy left out (written elsewhere)
};

// Batched-launch job tables: one entry per member sim; block0 is the
// member's first block in the launch (entries sorted by block0).
// 3-D and collapsed-z members run flat blocks of 256 consecutive points,
// so rows that are not a multiple of a tile width leave no lanes idle:
// 3-D, gx blocks per i plane over its row-major (j, k) points; collapsed
// z, gx blocks over the row-major (i, j) plane whose rows are bx long.
// Other members run bx x (256/bx) tiles, gx along k and gy along j per
// plane.
template <class T>
struct MainJob {
  MainArgs<T> m;
  int bx;
  int gx, gy;
  int pad_;
  int64_t block0;
};

template <class T>
struct SrcJob {
  SrcArgs<T> a;
  int64_t block0;
};

template <class T>
struct GhostJob {
  GhostArgs<T> g;
  int64_t block0;
};

// Running-DFT monitor of one component over a box of storage indices:
// acc[f][cell] += w[row][f][E or H] * F(cell) in FP64, on steps that are
// multiples of decim.
template <class T>
struct DftJob {
  T* f;
  int pi, p, pk, koff, comp;
  int lo[3], n[3];
  int nfreq, decim, electric;
  int64_t ncells;
  double* acc;      // [nfreq][ncells][re, im]
  const double* w;  // [row][nfreq][2: E, H][re, im]
  Ctl* ctl;
  int64_t block0;
};

template <class T>
struct AdeJob {
  AdeArgs<T> a;
  int comp;
  int pad_;
  int64_t block0;
};

// Sum of |F|^2 over a box of storage indices of one component, in FP64
// and in a fixed order: pass 1 reduces kSqBlockCells cells per block into
// partial[block]; pass 2 (one block) reduces the partials into
// partial[nblocks].  The same box gives the same bits whatever buffer
// holds the partials.
constexpr int kSqBlockCells = 2048;  // 256 threads x 8 cells
template <class T>
struct SqBox {
  const T* f;    // element 0 of the device array
  int pi, p, pk, koff;
  int lo[3], n[3];
  int ncells;    // < 2^31 (a component holds < 2^31 elements)
};
inline int64_t sq_blocks(int64_t ncells) { return (ncells + kSqBlockCells - 1) / kSqBlockCells; }
template <class T>
void launch_sum_sq(const SqBox<T>& b, double* partial, hipStream_t st);

// Elements of esize bytes of a component between the host's dense (i, j, k)
// order and its device layout (field reads and writes): dev points at the
// element of (0, 0, 0).
struct LayoutArgs {
  int64_t total;
  int n1, n2;      // extents along j, k
  int pi, p, pk;
};
void launch_layout_copy(bool to_device, void* dense, void* dev, const LayoutArgs& a, int esize, hipStream_t st);
// out[x] = (uint8_t)ids[x]
void launch_narrow_ids(const uint16_t* ids, uint8_t* out, int64_t n, hipStream_t st);
template <class T>
void launch_main(bool electric, const MainArgs<T>& m, int ext[3], int bx, int by, hipStream_t st);
// flat blocks over packed rows (3-D; see k_main3d_flat)
template <class T>
void launch_main3d_flat(bool electric, const MainArgs<T>& m, hipStream_t st);
// collapsed-z 2-D kernels: i rows per thread (1 measured fastest of 1, 2
// and 4 at 4096^2; 1.4x the generic kernel in FP32)
constexpr int k2zRows = 1;
// kinds of batched main launch
// kBatch3dLds / kBatch2zLds: 3-D / collapsed-z jobs whose record tables
// all fit the LDS staging (RecStage::use_lds for 256-thread blocks)
// kBatch3dPP: real-FP32 3-D jobs whose records fit the LDS staging and
// whose CPML profile rows the kernel loads with the other operands
// (MainArgs::pp); kBatch3dUR: the same for UPML rows (MainArgs::ur)
constexpr int kBatchGeneric = 0, kBatch3d = 1, kBatch2z = 2, kBatch3dLds = 3, kBatch2zLds = 4, kBatch3dPP = 5,
              kBatch3dUR = 6;
template <class T>
void launch_main_batch(bool electric, int kind, const MainJob<T>* jobs, int njobs, int64_t nblocks,
                       hipStream_t st);
template <class T>
void launch_src_batch(const SrcJob<T>* jobs, int njobs, int64_t nblocks, hipStream_t st);
template <class T>
void launch_ade_batch(int cls, const AdeJob<T>* jobs, int njobs, int64_t nblocks, hipStream_t st);
template <class T>
void launch_dft_batch(const DftJob<T>* jobs, int njobs, int64_t nblocks, hipStream_t st);
template <class T>
void launch_ghost_batch(const GhostJob<T>* jobs, int njobs, int64_t nblocks, int tick, hipStream_t st);
template <class T>
void launch_main2z(bool electric, const MainArgs<T>& m, int ext[3], hipStream_t st);
template <class T>
void launch_main3d(bool electric, const MainArgs<T>& m, int bx, int by, int ichunk, hipStream_t st);
template <class T>
void launch_step3d(const Step3Args<T>& m, int absorber, int nthreads, hipStream_t st);
template <class T>
void launch_step2d(const Step2Args<T>& m, bool tm, int absorber, bool ade, hipStream_t st);
// clk[0] = clk[1] = clock: before the first one-sweep step after others
void launch_clock_copy(Ctl* ctl, hipStream_t st);
template <class T>
void launch_ade(int cls, int c, const AdeArgs<T>& m, hipStream_t st);
template <class T>
void launch_src(const SrcArgs<T>& m, hipStream_t st);
template <class T>
void launch_probe(const ProbeArgs<T>& m, hipStream_t st);
template <class T>
void launch_ghost(const GhostArgs<T>& m, int64_t total, hipStream_t st);

}  // namespace gmes_engine
