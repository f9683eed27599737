// libimx: one launch per RK stage on the fused FP32/FP64 handles, for trsk10's
// methods (HTC or HC), alone, with APVM or with diffusion, and for pxt16's (HTC).
//
// The three passes of imx_swm.hip (fast_tri, fast_cell, fast_edge) hand q,
// phi and the two Coriolis partials of every edge through memory and wait
// for each other three times per stage. Here a block takes a stretch of the
// Hilbert-ordered cells and evaluates the whole stage for the edges and
// cells it owns out of LDS:
//   local cells   own cells, then the far ends of their owned edges (C: all
//                 cells whose Bernoulli potential and Coriolis partials the
//                 own edges need), then the rest of the rings of C (L)
//   P0  u, u l and the dual length of every edge owned by a local cell, and
//       h of every local cell, to LDS
//   P1  PV of every triangle around a cell of C
//   P2  fast_cell's work for every cell of C; RK update of h on own cells
//   P3  fast_edge's work and the RK update of u on own edges
// APVM adds the Perot velocity at every cell of L and grad q at the triangles
// around C, between P1 and P2; for these the block also holds the rings of L
// and the PV of every triangle around a cell of L, and takes the weights from
// tables in its own order.
// pxt16 replaces the Coriolis partials by two Perot vectors of every cell of
// C, which P3 reads; diffusion adds K zeta at the triangles and its jump at
// the own edges.
// Nothing but the new state and the accumulators is written. Cells and
// triangles on the rim are evaluated by every block that needs them (1.2 to
// 1.4 times the work of the mesh), with the same expressions on the same
// inputs, so a result does not depend on how the mesh is cut into blocks.
//
// Measured (us per RK4 step, three passes -> this; 16-step graphs on both
// sides would take 6 off the first figures): glevel 5 FP32 43 -> 19.7, glevel
// 7 78 -> 43.5, FP64 105 -> 68, glevel 8 191 -> 110.6, FP64 380 -> 211,
// glevel 9 948 -> 516. The three passes moved 252 MB per stage at glevel 8;
// this moves 181 (FETCH_SIZE x 2 + WRITE_SIZE) at 6.6 TB/s, against 7.8 for a
// copy that stays in the last-level cache. What bounds it there: the vector
// units are busy 47 % of the time (686 instructions a wave), memory most of
// the rest. What was worth most: every load issued before the first barrier
// (with each phase loading its own tables a glevel-8 stage took 45 us instead
// of 32), then fewer vector instructions (32 -> 27.6).
//
// APVM, four passes -> this: glevel 5 FP32 64 -> 24.3, glevel 7 126 -> 77,
// FP64 204 -> 165, glevel 8 459 -> 285, FP64 839 -> 686, glevel 9 1858 -> 1124.
// The passes read three-component weights as four words and wrote the
// velocities, gradients and partials; this moves 371 MB per stage at glevel 8
// (about 330 of it tables, 1.45 times the mesh's for the rim) at 5.1 TB/s, a
// large copy's rate: the tables no longer fit the last-level cache.
// pxt16, three passes -> this: glevel 5 FP32 52 -> 19.7, glevel 7 105 -> 56.6,
// FP64 159 -> 87, glevel 8 378 -> 158, FP64 659 -> 377. Diffusion: 53 -> 21.7,
// 89 -> 48.9, 124 -> 74, 223 -> 119, 488 -> 236.
//
// Blocks are cut greedily along the curve so that |C| fills the block's
// threads and |L| its LDS. Ids inside a block are 10-bit, which packs the
// topology of a cell into 16 bytes; lengths are stored once per edge, in FP32 as
// 1 / l and l~, and the kinetic-energy and vorticity coefficients are formed
// from them. The momentum tendency is multiplied by 1 / l: an error of that
// factor is the same in every step and adds up over a run. With l stored, rounded
// to FP32 and then inverted (a second rounding), h' at glevel 4 after 48 steps
// was 2.39e-7 off (trsk10, ten seeds; HC 4.53e-7) where the three passes, which
// read 1 / l, are 2.14e-7 off (3.84e-7); with 1 / l stored it is 2.04e-7
// (3.83e-7). The lengths, which the other terms take, bear the second rounding
// without effect. Three reciprocals a thread more: 1 % at glevel 5, less from 6
// on; a table of 1 / l beside l took 3 % at glevels 7 to 9.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <memory>
#include <new>
#include <string>
#include <thread>
#include <type_traits>
#include <vector>

#include "imx_device.h"

#define MX IMX_MAXNB
#define NXCD 8
#define HTR_GUARD (1.1920928955078125e-07 / 100000.0)
// local ids are 10-bit
#define LID 1023
// topology half word of a cell slot: neighbour | OWN (the cell owns the edge)
// | K (which of its owner's edges, 2 bits) | signs of the Coriolis term and,
// in the top bit, of the flux
#define SB_OWN 10
#define SB_K 11
#define SB_TNR 14
#define SB_TTG 15
// fourth topology word: owner of triangle j (0 cell, 1 nb_j, 2 nb_j+1; 2
// bits at 2j), k of triangle j (bit 12+j), hexagon (bit 18)
#define SW_KT 12
#define SW_HEX 18
#define SW_FZ 19  // sign of the tangential diffusion at edge j (bit 19 + j)

// bits of the handle's cell words (imx_swm.hip)
#define BA_TTG 3
#define BA_TNR 9
#define BA_OWN 15
#define BA_FZ 21
#define BB_TSEL 12
#define BB_KT 24
#define OTH_MASK 0x3FFFFFFF
#define OTH_V2 30

namespace imx {

template <typename T>
struct alignas(2 * sizeof(T)) Pair {
  T x, y;
};
template <typename T>
struct alignas(4 * sizeof(T)) Quad {
  T x, y, z, w;
};
template <typename T>
struct Tri {
  T x, y, z;
};

// caps of a block of nt threads: local cells (and at most nt past the own
// ones, at most nt in C), cells of L, triangles, triangles around C
static constexpr int kPlain = 0, kApvm = 1, kPerot = 2, kDiff = 3;  // stage_build's schemes
static constexpr int cap_a(int nt) { return nt + nt / 2 + 64; }
static constexpr int cap_l(int nt, bool ap) { return ap ? nt + nt / 4 + 64 : nt; }
static constexpr int cap_t(int nt, bool ap) { return ap ? 3 * nt : 2 * nt + nt / 2 + 64; }
static constexpr int cap_g(int nt) { return 2 * nt + nt / 4 + 32; }

//
// Which cells, triangles and edges a block holds follows from the mesh, the
// block's threads and whether it holds APVM's wider ring: the cut, made on the
// host. What the handle's tables say of them (signs, weights, the Coriolis
// parameter) is filled in by stage_fill, again whenever those tables change.
struct Stage {
  int nt = 0, nblk = 0, remap = 1;
  int scheme = kPlain;
  bool wide = false;  // the cut holds APVM's ring
  Alloc A, O;         // the cut and the plain scheme's values; an option's
  int4 *head = nullptr;      // [nblk] first own cell, own cells | |L| << 16, |C| | triangles around C << 16,
                             // local cells | triangles << 16
  int32_t *halo = nullptr;   // [nblk][nt] cells of the local ids past the own ones
  uint4 *topo = nullptr;     // [nblk][cap_l]
  void *cw = nullptr;        // [nblk][2][nt] Quad: kite fractions 0-3; 4, 5, 1 / sum l l~, with diffusion K / A;
                             // pxt16: PV weights of the earlier triangle at edges 0-3; 4, 5
  void *eld = nullptr;       // [NE] Pair: 1 / length (FP64: length), dual length
  uint16_t *oth = nullptr;   // [NE] local id of the edge's other cell | it is v1 << 10; 0xFFFF dummy
  uint32_t *tv = nullptr;    // [nblk][cap_t] vertices a, b (10 bits each), edge bits (9), curl signs (3)
  uint16_t *tslot = nullptr; // [nblk][cap_t] local slot 2 owner + k
  void *tk = nullptr;        // [nblk][cap_t] Quad: kite weights, 1 / (A_t a)
  void *tf = nullptr;        // [nblk][cap_t] Coriolis parameter
  void *wc = nullptr;        // APVM, pxt16: [nblk][6][cap_l] Tri: Perot weights of a cell's velocity
  void *wt = nullptr;        // APVM: [nblk][3][cap_g] Tri: those of grad q at a triangle
  ushort4 *tn = nullptr;     // APVM: [nblk][cap_g] local slots of the triangles across and its own
  void *en = nullptr;        // pxt16: [NE] Tri: normal of the Coriolis term
  void *tkt = nullptr;       // diffusion: [nblk][cap_t] coefficient at triangles
};

template <typename T>
struct StageArgs {
  const int4 *head;
  const int32_t *halo;
  const uint4 *topo;
  const Quad<T> *cw;
  const Pair<T> *eld;
  const uint16_t *oth;
  const uint32_t *tv;
  const uint16_t *tslot;
  const Quad<T> *tk;
  const T *tf;
  const double *iaa;
  const T *hs, *us, *h0, *u0, *gb, *dte;
  const double *dtc;
  T *hout, *uout, *acch, *accu, *q, *du_out;
  double *dh_out;
  int *flag;
  double href, ca, cb;  // the stage's step and its weight in the sum (ensembles: per cell)
  T grav, inv_a, cat, cbt;
  int nblk, remap, use_pv, flin, zero_mom;
  int whole;  // the third stage: its state is a whole step away
};
// the operands of the options, which the plain scheme's kernel does not take:
// with them its arguments are a cache line longer and a glevel-6 step 1.3 %
// slower
template <typename T>
struct StageOpts : StageArgs<T> {
  const Tri<T> *wc, *wt, *en;
  const T *tkt;
  const ushort4 *tn;
  T pvsdt;
};

// Compensated summation: c gathers the exact rounding errors of s (Knuth's
// two-sum, which needs no branch on the larger operand).
__device__ __forceinline__ void two_sum(double &s, double &c, double x) {
  const double t = s + x;
  const double y = t - s;
  c += (s - (t - y)) + (x - y);
  s = t;
}

__device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }
// x with its sign changed when bit 31 of m is set (the other bits are 0)
__device__ __forceinline__ float flip(float x, uint32_t m) { return __uint_as_float(__float_as_uint(x) ^ m); }
__device__ __forceinline__ double flip(double x, uint32_t m) {
  return __longlong_as_double(__double_as_longlong(x) ^ ((long long)m << 32));
}
// 1/x to about an ulp: the hardware's estimate and Newton steps
__device__ __forceinline__ float recip(float x) {
  const float r = __builtin_amdgcn_rcpf(x);
  return __builtin_fmaf(__builtin_fmaf(-x, r, 1.0f), r, r);
}
__device__ __forceinline__ double recip(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
  return __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
}
// l, 1 / l and l / l~ of the stored length: 1 / l in FP32; in FP64 l, whose reciprocal
// is as good as a stored one and which three edges a thread fewer then need
// (glevel 7: 68.4 us a step, with 1 / l stored 69.1)
__device__ __forceinline__ float length(float s) { return recip(s); }
__device__ __forceinline__ float inverse_length(float s) { return s; }
__device__ __forceinline__ float length_ratio(float s, float dl) { return recip(s * dl); }
__device__ __forceinline__ double length(double s) { return s; }
__device__ __forceinline__ double inverse_length(double s) { return recip(s); }
__device__ __forceinline__ double length_ratio(double s, double dl) { return s * recip(dl); }
template <typename T>
__device__ __forceinline__ T stored_length(double l) {
  return sizeof(T) == 4 ? (T)(1.0 / l) : (T)l;
}
// element i of a table, by a 32-bit byte offset (tables are under 4 GiB; see
// stage_build): one scalar base and one vector register for the address
template <typename X>
__device__ __forceinline__ X at(const X *p, uint32_t i) {
  return *(const X *)((const char *)p + (uint32_t)(i * (uint32_t)sizeof(X)));
}
template <typename X>
__device__ __forceinline__ void put(X *p, uint32_t i, X v) {
  *(X *)((char *)p + (uint32_t)(i * (uint32_t)sizeof(X))) = v;
}

// MODE: 0 the first RK stage, 1 the second and third, 2 the last, 3 a
// tendency. SCHEME: trsk10's methods (kPlain), with APVM or diffusion, or
// pxt16's (kPerot).
template <typename T, int NT, int MODE, int SCHEME, class Args>
__global__ __launch_bounds__(NT, SCHEME == kApvm && NT == 512 ? 4 : 1) void fast_stage(const Args a) {
  constexpr bool AP = SCHEME == kApvm, PX = SCHEME == kPerot, DF = SCHEME == kDiff;
  constexpr int LC = cap_a(NT), CL = cap_l(NT, AP), TC = cap_t(NT, AP), GC = cap_g(NT);
  constexpr int NR = (TC + NT - 1) / NT, NG = (GC + NT - 1) / NT;
  __shared__ T sU[3 * LC], sD[3 * LC], sA[3 * LC];  // u, dual length, u l
  __shared__ T sH[LC], sQ[2 * LC], sPhi[NT], sPP[6 * NT];
  __shared__ Tri<T> sV[AP ? CL : 1], sG[AP ? 2 * CL : 1];  // Perot velocity at cells, grad q at triangles
  T *sP = sPP, *sPo = sPP + 3 * NT;  // partials of the own edges' owners and other cells
  Tri<T> *sAB = reinterpret_cast<Tri<T> *>(sPP);  // pxt16: Perot vectors of u h, u h q at the cells of C
  __shared__ T sE[PX || DF ? 3 * NT : 1];  // own edges: PV (pxt16), the jump of K zeta (diffusion)
  __shared__ T sZ[DF ? 2 * LC : 1];        // K zeta
  int b = blockIdx.x;
  if (a.remap) b = (b % NXCD) * (gridDim.x / NXCD) + b / NXCD;
  if (b >= a.nblk) return;
  const int tid = threadIdx.x;
  // Every load of the stage is issued before the first barrier, in two
  // generations: the block's tables, which need nothing, and the state,
  // whose places the first ones give; the phases then run out of registers
  // and LDS. Lanes past a list read its last entry instead of branching
  // around the load.
  const int32_t *halo = a.halo + (size_t)b * NT;
  const int hcell = at(halo, tid);
  const uint4 *topo = a.topo + (size_t)b * CL;
  const uint4 tp = at(topo, tid);
  const Quad<T> *cw = a.cw + (size_t)b * 2 * NT;
  const Quad<T> w0 = at(cw, tid), w1 = at(cw + NT, tid);
  const int4 hd = a.head[b];
  const int own0 = hd.x, nown = hd.y & 0xFFFF, nL = hd.y >> 16, nC = hd.z & 0xFFFF, nG = hd.z >> 16;
  const int nTri = hd.w >> 16, nh = (hd.w & 0xFFFF) - nown;
  const T href = (T)a.href;
  const int oc = min(tid, nown - 1);

  const T hh = at(a.hs, hcell);
  T hu[3];
  Pair<T> hl[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    hu[k] = at(a.us, 3 * hcell + k);
    hl[k] = at(a.eld, 3 * hcell + k);
  }
  const T ho = at(a.hs + own0, oc);
  T eu[3];
  Pair<T> el[3];
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    const int e = min(tid + r * NT, 3 * nown - 1);
    eu[r] = at(a.us + 3 * (size_t)own0, e);
    el[r] = at(a.eld + 3 * (size_t)own0, e);
  }
  // the state first: P0 waits for it alone
  __builtin_amdgcn_sched_barrier(0);
  uint32_t tv[NR];
  int tsl[NR];
  Quad<T> tk[NR];
  T tf[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const int t = min(tid + r * NT, nTri - 1);
    tv[r] = at(a.tv + (size_t)b * TC, t);
    tsl[r] = at(a.tslot + (size_t)b * TC, t);
    tk[r] = at(a.tk + (size_t)b * TC, t);
    tf[r] = at(a.tf + (size_t)b * TC, t);
  }
  uint4 tpl;
  T tkt[NR];
  if constexpr (DF)
#pragma unroll
    for (int r = 0; r < NR; ++r) tkt[r] = at(a.tkt + (size_t)b * TC, min(tid + r * NT, nTri - 1));
  Tri<T> wc[AP ? 2 : 1][MX];
  if constexpr (PX)
#pragma unroll
    for (int j = 0; j < MX; ++j) wc[0][j] = at(a.wc + (size_t)b * MX * CL + j * CL, tid);
  if constexpr (AP) {
    const Tri<T> *w = a.wc + (size_t)b * MX * CL;
    const int i = min(tid + NT, CL - 1);
    tpl = at(topo, i);
#pragma unroll
    for (int j = 0; j < MX; ++j) {
      wc[0][j] = at(w + j * CL, tid);
      wc[1][j] = at(w + j * CL, i);
    }
  }
  // the RK operands of the own cells and edges
  __builtin_amdgcn_sched_barrier(0);
  const double iaa = at(a.iaa + own0, oc);
  T y0 = (T)0, ac = (T)0, v0[3], av[3];
  uint32_t ow[3];
  Tri<T> en[3];
  if (MODE != 3) y0 = at(a.h0 + own0, oc);
  if (MODE == 1 || MODE == 2) ac = at((const T *)a.acch + own0, oc);
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    const int e = min(tid + r * NT, 3 * nown - 1);
    ow[r] = at(a.oth + 3 * (size_t)own0, e);
    if constexpr (PX) en[r] = at(a.en + 3 * (size_t)own0, e);
    if (MODE != 3) v0[r] = at(a.u0 + 3 * (size_t)own0, e);
    if (MODE == 1 || MODE == 2) av[r] = at((const T *)a.accu + 3 * (size_t)own0, e);
  }
  __builtin_amdgcn_sched_barrier(0);

  // P0: the local state to LDS
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    // used here, so the load is not moved into the branch below
    asm volatile("" : "+v"(eu[r]), "+v"(el[r].x), "+v"(el[r].y));
    const int i = tid + r * NT;
    if (i < 3 * nown) {
      sU[i] = eu[r];
      sD[i] = el[r].y;
      sA[i] = eu[r] * length(el[r].x);
    }
  }
  if (tid < nown) sH[tid] = ho;
  if (tid < nh) {
    const int lc = nown + tid;
    sH[lc] = hh;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      sU[3 * lc + k] = hu[k];
      sD[3 * lc + k] = hl[k].y;
      sA[3 * lc + k] = hu[k] * length(hl[k].x);
    }
  }
  ushort4 tn[NG];
  Tri<T> wt[NG][3];
  if constexpr (AP) {
#pragma unroll
    for (int r = 0; r < NG; ++r) {
      const int t = min(tid + r * NT, nG - 1);
      tn[r] = at(a.tn + (size_t)b * GC, t);
#pragma unroll
      for (int m = 0; m < 3; ++m) wt[r][m] = at(a.wt + ((size_t)b * 3 + m) * GC, t);
    }
  }
  __syncthreads();

  if constexpr (AP) {
    // Perot velocity at the cells of L (a pentagon's padded slot has a zero
    // weight)
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int i = tid + r * NT;
      if (i >= nL) continue;
      const uint4 t4 = r ? tpl : tp;
      const uint32_t wj[3] = {t4.x, t4.y, t4.z};
      Tri<T> v{(T)0, (T)0, (T)0};
#pragma unroll
      for (int j = 0; j < MX; ++j) {
        const uint32_t f = j % 2 ? wj[j / 2] >> 16 : wj[j / 2];
        const T u = sU[3 * ((f >> SB_OWN) & 1 ? i : (int)(f & LID)) + ((f >> SB_K) & 3)];
        v.x = fma_(wc[r][j].x, u, v.x);
        v.y = fma_(wc[r][j].y, u, v.y);
        v.z = fma_(wc[r][j].z, u, v.z);
      }
      sV[i] = v;
    }
  }
  // P1: PV at triangles
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    if (tid + r * NT >= nTri) continue;
    const uint32_t v = tv[r];
    const int sl = tsl[r];
    const Quad<T> k = tk[r];
    T eta = tf[r];
    const int o = sl >> 1, va = v & LID, vb = (v >> 10) & LID;
    const int eb = v >> 20;
    const int e0 = 3 * ((eb & 1) ? o : va) + ((eb >> 1) & 3);
    const int e1 = 3 * (((eb >> 3) & 1) ? va : vb) + ((eb >> 4) & 3);
    const int e2 = 3 * (((eb >> 6) & 1) ? vb : o) + ((eb >> 7) & 3);
    if (DF || !a.flin) {
      T z = flip(sA[e0], (v << 2) & 0x80000000u);
      z += flip(sA[e1], (v << 1) & 0x80000000u);
      z += flip(sA[e2], v & 0x80000000u);
      if (!a.flin) eta = fma_(z, k.w, eta);
      if constexpr (DF) sZ[sl] = tkt[r] * (z * k.w);
    }
    T hsum = k.x * sH[o];
    hsum = fma_(k.y, sH[va], hsum);
    hsum = fma_(k.z, sH[vb], hsum);
    const T ht = href + hsum;
    T qq = (T)0;
    if (a.use_pv) {
      if (fabs((double)ht) < HTR_GUARD) a.flag[0] = 1;
      else qq = eta / ht;
    }
    sQ[sl] = qq;
    // the field a caller may read: the last stage's, or a tendency's
    if (MODE >= 2 && o < nown) put(a.q + 2 * (size_t)own0, sl, qq);
  }
  __syncthreads();

  if constexpr (AP) {
    // grad q at the triangles around C
#pragma unroll
    for (int r = 0; r < NG; ++r) {
      if (tid + r * NT >= nG) continue;
      const T qt = sQ[tn[r].w];
      const T d[3] = {sQ[tn[r].x] - qt, sQ[tn[r].y] - qt, sQ[tn[r].z] - qt};
      Tri<T> g{(T)0, (T)0, (T)0};
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        g.x = fma_(wt[r][m].x, d[m], g.x);
        g.y = fma_(wt[r][m].y, d[m], g.y);
        g.z = fma_(wt[r][m].z, d[m], g.z);
      }
      sG[tn[r].w] = g;
    }
    __syncthreads();
  }

  // P2: cells
  if (tid < nC) {
    const uint32_t wj[3] = {tp.x, tp.y, tp.z};
    const bool hex = (tp.w >> SW_HEX) & 1;
    int nb[MX], ed[MX];
    uint32_t f[MX];
#pragma unroll
    for (int j = 0; j < MX; ++j) {
      // the slot's half word in the upper half: signs by plain masks
      f[j] = j % 2 ? wj[j / 2] : wj[j / 2] << 16;
      nb[j] = (f[j] >> 16) & LID;
      ed[j] = 3 * (((f[j] >> (16 + SB_OWN)) & 1) ? tid : nb[j]) + ((f[j] >> (16 + SB_K)) & 3);
    }
    const T hc = sH[tid];
    double dv = 0.0, dvc = 0.0;
    T ke = (T)0;
    T G[MX];  // mass flux; pxt16: u h
    Tri<T> v{(T)0, (T)0, (T)0};
    double du = 0.0;
#pragma unroll
    for (int j = 0; j < MX; ++j) {
      const bool valid = (j < MX - 1) || hex;
      const T u = sU[ed[j]], dl = sD[ed[j]];
      // both cells of an edge form the same product, so the mass flux
      // cancels exactly between them
      const double he = fma_(0.5, (double)hc + (double)sH[nb[j]], a.href);
      double g = (double)flip(u, f[j] & 0x80000000u) * he * (double)dl;
      if (!valid) g = 0.0;
      if (j == 0) dv = g;
      else two_sum(dv, dvc, g);
      if constexpr (PX) {
        // perhx: the kinetic energy of the Perot velocity (a pentagon's
        // padded slot has a zero weight)
        G[j] = u * (T)he;
        v.x = fma_(wc[0][j].x, u, v.x);
        v.y = fma_(wc[0][j].y, u, v.y);
        v.z = fma_(wc[0][j].z, u, v.z);
      } else {
        G[j] = (T)g;
        ke = fma_(valid ? sA[ed[j]] : (T)0, u * dl, ke);
      }
      if constexpr (DF) du += valid ? (double)flip(u, f[j] & 0x80000000u) * (double)dl : 0.0;
    }
    T K = PX ? (v.x * v.x + v.y * v.y + v.z * v.z) / (T)2 : ke * w1.z;
    // the normal part of the diffusion: grad(K div u) folds into the potential
    if constexpr (DF) K -= (T)(du * (double)w1.w);
    T qt[MX];
    int ts[MX];
#pragma unroll
    for (int j = 0; j < MX; ++j) {
      const int sel = (tp.w >> (2 * j)) & 3;
      const int to = (sel == 0) ? tid : (sel == 1) ? nb[j] : nb[(j + 1) % MX];
      ts[j] = 2 * to + ((tp.w >> (SW_KT + j)) & 1);
      qt[j] = sQ[ts[j]];
    }
    // a pentagon's padded slot may name a triangle that is not local
    if (!hex) qt[MX - 1] = (T)0;
    if (a.gb) K += at(a.gb, tid < nown ? own0 + tid : halo[tid - nown]);
    sPhi[tid] = fma_(a.grav, hc, K) * a.inv_a;
    if (tid < nown) {
      const double dh = -(dv + dvc) * iaa;
      // the step over the stage's share of it (1, 2 halves) and over 6 or 3
      double ca = a.ca, cb = a.cb;
      if (a.dtc) {
        const double dt = at(a.dtc + own0, tid);
        ca = a.whole ? dt : 0.5 * dt;
        cb = MODE == 1 ? dt / 3.0 : dt / 6.0;
      }
      if (MODE == 3) {
        put(a.dh_out + own0, tid, dh);
      } else if (MODE < 2) {
        put(a.hout + own0, tid, (T)((double)y0 + ca * dh));
        put(a.acch + own0, tid, MODE == 0 ? (T)(cb * dh) : (T)((double)ac + cb * dh));
      } else {
        put(a.hout + own0, tid, (T)((double)y0 + ((double)ac + cb * dh)));
      }
    }
    // PV at the cell's edges: edge j lies between ring triangles j-1 and j
    T qe[MX];
    const T ql = hex ? qt[MX - 1] : qt[MX - 2];
    if constexpr (PX) {
      const T w[MX] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y};
#pragma unroll
      for (int j = 0; j < MX; ++j) qe[j] = w[j] * (j ? qt[j - 1] : ql) + ((T)1 - w[j]) * qt[j];
    } else {
      qe[0] = (T)0.5 * (ql + qt[0]);
#pragma unroll
      for (int j = 1; j < MX; ++j) qe[j] = (T)0.5 * (qt[j - 1] + qt[j]);
    }
    if constexpr (AP) {
      // q_e -= pvspar dt (grad q(t_{j-1}) + grad q(t_j)) . (v(c) + v(nb_j))
      if (!hex) ts[MX - 1] = ts[MX - 2];  // the ring's last triangle, and in place of the pad
      const Tri<T> vs = sV[tid];
      Tri<T> gp = sG[ts[MX - 1]];
#pragma unroll
      for (int j = 0; j < MX; ++j) {
        const Tri<T> g = sG[ts[j]], v = sV[nb[j]];
        qe[j] -= a.pvsdt * ((gp.x + g.x) * (vs.x + v.x) + (gp.y + g.y) * (vs.y + v.y) + (gp.z + g.z) * (vs.z + v.z));
        gp = g;
      }
      if (!hex) qe[MX - 1] = (T)0;
    }
    if constexpr (PX) {
      // pered: the Perot reconstruction here of uh (q_e + q_l) / 2 for an edge
      // l is (q_l A + B) / 2 with A = P(uh) and B = P(uh q); P3 takes both
      // cells' A and B with q_l
      Tri<T> A{(T)0, (T)0, (T)0}, B{(T)0, (T)0, (T)0};
#pragma unroll
      for (int j = 0; j < MX; ++j) {
        const T uq = G[j] * qe[j];
        A.x = fma_(wc[0][j].x, G[j], A.x);
        A.y = fma_(wc[0][j].y, G[j], A.y);
        A.z = fma_(wc[0][j].z, G[j], A.z);
        B.x = fma_(wc[0][j].x, uq, B.x);
        B.y = fma_(wc[0][j].y, uq, B.y);
        B.z = fma_(wc[0][j].z, uq, B.z);
        if (tid < nown && ((f[j] >> (16 + SB_OWN)) & 1) && (j < MX - 1 || hex)) sE[ed[j]] = qe[j];
      }
      sAB[tid] = A;
      sAB[NT + tid] = B;
    } else {
      const T R[MX] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y};
      // TRiSK weights from prefix sums of the kite areas:
      // w(i,j) = S_j - S_i - 1/2 (j>i), S_6 - S_i + S_j - 1/2 (j<i), w(i,i) = 0
      T S[MX + 1];
      S[0] = (T)0;
#pragma unroll
      for (int j = 0; j < MX; ++j) S[j + 1] = S[j] + R[j];
      const T rest = S[MX] - (T)0.5;
      // P_i = sum_j G_j (q_i + q_j)/2 w(i,j) = (q_i sum_j G_j w + sum_j G_j q_j w)/2
      T H[MX];
#pragma unroll
      for (int j = 0; j < MX; ++j) H[j] = G[j] * qe[j];
#pragma unroll
      for (int i = 0; i < MX; ++i) {
        T x = (T)0, y = (T)0;
#pragma unroll
        for (int j = 0; j < MX; ++j)
          if (j != i) {
            const T w = (j > i) ? (S[j] - S[i]) - (T)0.5 : rest - (S[i] - S[j]);
            x = fma_(G[j], w, x);
            y = fma_(H[j], w, y);
          }
        const T P = flip((T)0.5 * fma_(qe[i], x, y), (f[i] << 1) & 0x80000000u);
        // for the block's own edges: by its owner or by its other cell
        T *to = (f[i] >> (16 + SB_OWN)) & 1 ? sP : sPo;
        if (ed[i] < 3 * nown && (i < MX - 1 || hex)) to[ed[i]] = P;
        if constexpr (DF) {
          // the tangential part: the jump of K zeta between the edge's triangles
          const T jump = sZ[ts[i]] - sZ[ts[i ? i - 1 : hex ? MX - 1 : MX - 2]];
          if (tid < nown && ((f[i] >> (16 + SB_OWN)) & 1) && (i < MX - 1 || hex))
            sE[ed[i]] = flip(jump, (tp.w << (31 - SW_FZ - i)) & 0x80000000u);
        }
      }
    }
  }
  __syncthreads();

  // P3: own edges
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    const int i = tid + r * NT;
    if (i >= 3 * nown) continue;
    const uint32_t w = ow[r];
    if (w == 0xFFFFu) continue;
    const int o = i / 3, c2 = w & LID;
    const bool own_v2 = (w >> SB_OWN) & 1;
    const T d = own_v2 ? sPhi[o] - sPhi[c2] : sPhi[c2] - sPhi[o];
    T du;
    if constexpr (PX) {
      const T ql = sE[i];
      const Tri<T> A1 = sAB[o], A2 = sAB[c2], B1 = sAB[NT + o], B2 = sAB[NT + c2];
      const T uhq = (T)0.25 * (en[r].x * (ql * (A1.x + A2.x) + (B1.x + B2.x)) +
                               en[r].y * (ql * (A1.y + A2.y) + (B1.y + B2.y)) +
                               en[r].z * (ql * (A1.z + A2.z) + (B1.z + B2.z)));
      du = -d * inverse_length(el[r].x) - uhq;
    } else {
      T P = sP[i] + sPo[i];
      if constexpr (DF) P += length_ratio(el[r].x, el[r].y) * a.inv_a * sE[i];
      du = -(d + P) * inverse_length(el[r].x);
    }
    if (a.zero_mom) du = (T)0;
    T ca = a.cat, cb = a.cbt;
    if (a.dte) {
      const T dt = at(a.dte + 3 * (size_t)own0, i);
      ca = a.whole ? dt : (T)0.5 * dt;
      cb = MODE == 1 ? dt / (T)3 : dt / (T)6;
    }
    if (MODE == 3) {
      put(a.du_out + 3 * (size_t)own0, i, du);
    } else if (MODE < 2) {
      put(a.uout + 3 * (size_t)own0, i, v0[r] + ca * du);
      put(a.accu + 3 * (size_t)own0, i, MODE == 0 ? cb * du : av[r] + cb * du);
    } else {
      put(a.uout + 3 * (size_t)own0, i, v0[r] + (av[r] + cb * du));
    }
  }
}

// ------------------------------------------------------------- host side ---
// an array whose elements are written before they are read
template <typename X>
struct Raw {
  std::unique_ptr<X[]> p;
  size_t n = 0;
  explicit Raw(size_t count = 0) : p(new X[count]), n(count) {}
  X &operator[](size_t i) { return p[i]; }
  const X &operator[](size_t i) const { return p[i]; }
};
template <typename X>
static bool down(Raw<X> &h, const void *d, size_t n) {
  h = Raw<X>(n);
  return n == 0 || hipMemcpy(h.p.get(), d, n * sizeof(X), hipMemcpyDeviceToHost) == hipSuccess;
}
template <typename X>
static X *up(Alloc &A, const Raw<X> &h) {
  return A.put(h.p.get(), h.n);
}

void stage_free(imx_swm *s) {
  if (!s->stg) return;
  s->stg->A.release();
  s->stg->O.release();
  delete s->stg;
  s->stg = nullptr;
}

int stage_threads(const imx_swm *s) { return s->stg ? s->stg->nt : 0; }
int stage_scheme(const imx_swm *s) { return s->stg ? s->stg->scheme : -1; }
void stage_set_remap(imx_swm *s, int remap) {
  if (s->stg) s->stg->remap = remap;
}
size_t stage_bytes(const imx_swm *s) { return s->stg ? s->stg->A.bytes + s->stg->O.bytes : 0; }

// A block's local cells and triangles: small open-addressing tables that are
// emptied by raising the stamp (a block holds far fewer entries than slots).
struct LocalSet {
  static constexpr int kSlots = 1 << 13;
  struct Entry {
    int32_t stamp = 0, key = 0, id = 0, level = 0;  // cells: 1 in L, 2 in C; triangles: 1 around C
  };
  std::vector<Entry> e{(size_t)kSlots};
  std::vector<int32_t> keys;
  int32_t stamp = 1;
  void clear() {
    ++stamp;
    keys.clear();
  }
  // the entry of key, added when absent
  Entry &at(int32_t key) {
    uint32_t p = (uint32_t)key * 2654435761u >> 19;
    while (e[p].stamp == stamp && e[p].key != key) p = (p + 1) & (kSlots - 1);
    if (e[p].stamp != stamp) {
      e[p] = Entry{stamp, key, 0, 0};
      keys.push_back(key);
    }
    return e[p];
  }
};
struct LocalSets {
  LocalSet L, tri;
  int nC = 0, nL = 0, nG = 0, own = 0;
  void clear() {
    L.clear();
    tri.clear();
    nC = nL = nG = own = 0;
  }
};

// The cut of the curve into blocks of nt threads, as the device takes it, with
// every value that stage_fill writes zero.
struct Cut {
  int nblk = 0;
  Raw<int4> head;
  Raw<int32_t> halo;
  Raw<uint4> topo;
  Raw<uint16_t> oth, tslot;
  Raw<uint32_t> tv;
  Raw<ushort4> tn;
};

static int cut_blocks(imx_swm *s, int nt, bool wide, Cut &C, bool *local) {
  const int nv = s->nv, NE = s->NE, NTri = s->NT;
  const int LC = cap_a(nt), CL = cap_l(nt, wide), TC = cap_t(nt, wide), GC = cap_g(nt);
  Raw<int32_t> nbr, bA, bB, oth, tab, teb, atn;
  if (!down(nbr, s->x_c_nb, (size_t)MX * nv) || !down(bA, s->x_c_bitsA, nv) || !down(bB, s->x_c_bitsB, nv) ||
      !down(oth, s->x_e_oth, NE) || !down(tab, s->x_t_ab, (size_t)2 * NTri) || !down(teb, s->x_t_eb, NTri) ||
      (wide && !down(atn, s->x_ap_tnb, (size_t)3 * NTri)))
    return set_error(IMX_EDEVICE, "stage tables: copy from the device failed");

  auto tri_of = [&](int c, int j) {
    const int ts = (bB[c] >> (BB_TSEL + 2 * j)) & 3;
    const int to = ts == 0 ? c : ts == 1 ? nbr[(size_t)j * nv + c] : nbr[(size_t)((j + 1) % MX) * nv + c];
    return 2 * to + ((bB[c] >> (BB_KT + j)) & 1);
  };
  // adds own cell c to the sets of the current block; false past a cap
  auto add = [&](LocalSets &w, int c) {
    auto in_l = [&](int k) {
      LocalSet::Entry &q = w.L.at(k);
      if (q.level) return;
      q.level = 1;
      ++w.nL;
      if (!wide) return;
      // APVM takes the velocity at k and the PV of the triangles around it
      const int n = bA[k] & 7;
      for (int j = 0; j < n; ++j) {
        (void)w.L.at(nbr[(size_t)j * nv + k]);
        (void)w.tri.at(tri_of(k, j));
      }
    };
    auto in_c = [&](int k) {
      in_l(k);
      LocalSet::Entry &q = w.L.at(k);
      if (q.level == 2) return;
      q.level = 2;
      ++w.nC;
      const int n = bA[k] & 7;
      for (int j = 0; j < n; ++j) {
        in_l(nbr[(size_t)j * nv + k]);
        LocalSet::Entry &t = w.tri.at(tri_of(k, j));
        w.nG += !t.level;
        t.level = 1;
      }
    };
    in_c(c);
    const int n = bA[c] & 7;
    for (int j = 0; j < n; ++j)
      if ((bA[c] >> (BA_OWN + j)) & 1) in_c(nbr[(size_t)j * nv + c]);
    ++w.own;
    const int nA = (int)w.L.keys.size();
    return w.nC <= nt && nA <= LC && nA - w.own <= nt && (int)w.tri.keys.size() <= TC &&
           (!wide || (w.nL <= CL && w.nG <= GC));
  };

  // Where the blocks start: the curve in at most 16 segments, one host thread
  // each, and every segment greedily into blocks. Kept with the handle (a few
  // thousand numbers), so that a scheme that is back need not look for them.
  std::vector<int32_t> &start = s->stg_start[{nt, wide}];
  std::atomic<bool> memory{true};
  auto parallel = [&](int n, auto fn) {
    parallel_ranges(n, [&](int i0, int i1) {
      try {
        fn(i0, i1);
      } catch (const std::bad_alloc &) {
        memory = false;
      }
    }, 1);
  };
  const char *out_of = "stage tables: host out of memory";
  if (start.empty()) {
    const int seg = std::max(64 * nt, (nv + 15) / 16), nseg = (nv + seg - 1) / seg;
    std::vector<std::vector<int32_t>> cuts(nseg);
    std::vector<char> fine(nseg, 1);
    parallel(nseg, [&](int g0, int g1) {
      LocalSets w;
      for (int g = g0; g < g1; ++g) {
        const int c0 = g * seg, c1 = std::min(nv, c0 + seg);
        w.clear();
        cuts[g].push_back(c0);
        for (int c = c0; c < c1 && fine[g]; ++c) {
          if (add(w, c)) continue;
          cuts[g].push_back(c);
          w.clear();
          fine[g] = add(w, c);  // a single cell within the caps
        }
      }
    });
    if (!memory) return set_error(IMX_ENOMEM, out_of);
    std::vector<int32_t> all;
    for (const auto &c : cuts) all.insert(all.end(), c.begin(), c.end());
    // Numberings that are not local (a mesh in its caller's order) cut into
    // blocks that are mostly rim: the three passes run instead.
    *local = all.size() <= 1 || (int64_t)all.size() * nt <= (int64_t)3 * nv;
    for (char ok : fine) *local = *local && ok;
    if (!*local) return IMX_OK;
    all.push_back(nv);
    start.swap(all);
  }
  const int nblk = (int)start.size() - 1;

  C.nblk = nblk;
  C.head = Raw<int4>(nblk);
  C.halo = Raw<int32_t>((size_t)nblk * nt);
  C.topo = Raw<uint4>((size_t)nblk * CL);
  C.oth = Raw<uint16_t>(NE);
  C.tslot = Raw<uint16_t>((size_t)nblk * TC);
  C.tv = Raw<uint32_t>((size_t)nblk * TC);
  C.tn = Raw<ushort4>(wide ? (size_t)nblk * GC : 0);
  parallel(nblk, [&](int b0, int b1) {
    LocalSets w;
    std::vector<uint64_t> cells, tris;  // rank above the id
    for (int b = b0; b < b1; ++b) {
      const int o0 = start[b], nown = start[b + 1] - o0;
      w.clear();
      for (int c = o0; c < o0 + nown; ++c) (void)add(w, c);
      // own cells, the rest of C, the rest of L, the others, each ascending;
      // own triangles, the others around C, the others
      auto own = [&](int k) { return k >= o0 && k < o0 + nown; };
      auto ranked = [](uint64_t rank, int k) { return rank << 32 | (uint32_t)k; };
      cells.clear();
      for (int k : w.L.keys) cells.push_back(ranked(own(k) ? 0 : 3 - w.L.at(k).level, k));
      tris.clear();
      for (int k : w.tri.keys) tris.push_back(ranked(own(k / 2) ? 0 : 2 - w.tri.at(k).level, k));
      std::sort(cells.begin(), cells.end());
      std::sort(tris.begin(), tris.end());
      const int nA = (int)cells.size(), nTri = (int)tris.size(), nL = w.nL, nC = w.nC;
      for (int k = 0; k < nA; ++k) w.L.at((int32_t)cells[k]).id = k;
      auto id = [&](int k) { return (uint32_t)w.L.at(k).id; };
      int32_t *halo = &C.halo[(size_t)b * nt];
      for (int k = 0; k < nt; ++k) halo[k] = nown + k < nA ? (int32_t)cells[nown + k] : 0;
      C.head[b] = int4{o0, nown | nL << 16, nC | w.nG << 16, nA | nTri << 16};
      uint4 *topo = &C.topo[(size_t)b * CL];
      for (int k = 0; k < CL; ++k) {
        topo[k] = uint4{0, 0, 0, 0};
        if (k >= (wide ? nL : nC)) continue;
        const int c = (int32_t)cells[k];
        uint32_t f[MX], t3 = (uint32_t)((bA[c] & 7) == MX) << SW_HEX;
        for (int j = 0; j < MX; ++j) {
          f[j] = id(nbr[(size_t)j * nv + c]);
          f[j] |= ((bA[c] >> (BA_OWN + j)) & 1u) << SB_OWN;
          f[j] |= ((bB[c] >> (2 * j)) & 3u) << SB_K;
          t3 |= ((bB[c] >> (BB_TSEL + 2 * j)) & 3u) << (2 * j);
          t3 |= ((bB[c] >> (BB_KT + j)) & 1u) << (SW_KT + j);
        }
        topo[k] = uint4{f[0] | f[1] << 16, f[2] | f[3] << 16, f[4] | f[5] << 16, t3};
      }
      for (int k = 0; k < TC; ++k) {
        const size_t p = (size_t)b * TC + k;
        C.tv[p] = 0;
        C.tslot[p] = 0;
        if (k >= nTri) continue;
        const int t = (int32_t)tris[k];
        C.tv[p] = id(tab[t]) | id(tab[(size_t)NTri + t]) << 10 | (uint32_t)(teb[t] & 511) << 20;
        C.tslot[p] = (uint16_t)(2 * id(t / 2) + t % 2);
      }
      for (int k = 0; wide && k < GC; ++k) {
        ushort4 &q = C.tn[(size_t)b * GC + k];
        q = ushort4{0, 0, 0, 0};
        if (k >= w.nG) continue;
        const int t = (int32_t)tris[k];
        auto slot = [&](int i) { return (unsigned short)(2 * id(i / 2) + i % 2); };
        q = ushort4{slot(atn[t]), slot(atn[(size_t)NTri + t]), slot(atn[(size_t)2 * NTri + t]), slot(t)};
      }
      for (int e = 3 * o0; e < 3 * (o0 + nown); ++e)
        C.oth[e] = oth[e] < 0 ? (uint16_t)0xFFFF : (uint16_t)id(oth[e] & OTH_MASK);
    }
  });
  return memory ? IMX_OK : set_error(IMX_ENOMEM, out_of);
}

// The handle's tables, and where their values go in the blocks' order.
template <typename T>
struct FillArgs {
  const int4 *head;
  const int32_t *halo;
  const uint16_t *tslot;
  const int32_t *bitsA, *e_oth;
  const T *R, *ika, *kh, *kt, *ceta, *kap, *f;
  const double *iaa, *leng, *dleng, *tarea;
  const Quad<T> *awc, *awt, *pn;
  uint4 *topo;
  Quad<T> *cw, *tk;
  Pair<T> *eld;
  uint16_t *oth;
  uint32_t *tv;
  T *tf, *tkt;
  Tri<T> *wc, *wt, *en;
  int nv, NE, NT, nt, CL, TC, GC;
  double ea;
};

// One block per block of the stage. The values are those of the host's
// arithmetic (IEEE divisions in FP64, rounded once to T). 0.3 ms at glevel 8,
// where making the tables on the host and copying them took 67.
template <typename T, int SCHEME>
__global__ __launch_bounds__(256) void stage_fill(const FillArgs<T> a) {
  constexpr bool AP = SCHEME == kApvm, PX = SCHEME == kPerot, DF = SCHEME == kDiff;
  const int b = blockIdx.x, nv = a.nv, NT = a.NT;
  const int4 hd = a.head[b];
  const int own0 = hd.x, nown = hd.y & 0xFFFF, nL = hd.y >> 16, nC = hd.z & 0xFFFF, nG = hd.z >> 16;
  const int nTri = hd.w >> 16;
  const int32_t *halo = a.halo + (size_t)b * a.nt;
  auto cell = [&](int k) { return k < nown ? own0 + k : halo[k - nown]; };
  for (int k = threadIdx.x; k < (AP ? nL : nC); k += blockDim.x) {
    const int c = cell(k), A = a.bitsA[c];
    uint4 &tp = a.topo[(size_t)b * a.CL + k];
    uint32_t w[3] = {tp.x & 0x3FFF3FFFu, tp.y & 0x3FFF3FFFu, tp.z & 0x3FFF3FFFu};
    for (int j = 0; j < MX; ++j) {
      const uint32_t f = ((A >> (BA_TTG + j)) & 1u) << SB_TTG | ((A >> (BA_TNR + j)) & 1u) << SB_TNR;
      w[j / 2] |= f << (16 * (j % 2));
    }
    const uint32_t fz = DF ? ((uint32_t)A >> BA_FZ & 63u) << SW_FZ : 0u;
    tp = uint4{w[0], w[1], w[2], (tp.w & ~(63u << SW_FZ)) | fz};
    if constexpr (AP || PX)
      for (int j = 0; j < MX; ++j) {
        const Quad<T> q = a.awc[(size_t)j * nv + c];
        a.wc[((size_t)b * MX + j) * a.CL + k] = Tri<T>{q.x, q.y, q.z};
      }
    if (k >= nC) continue;
    T r[MX];
    for (int j = 0; j < MX; ++j) r[j] = a.R[(size_t)j * nv + c];
    a.cw[((size_t)b * 2) * a.nt + k] = Quad<T>{r[0], r[1], r[2], r[3]};
    // ika = 1 / sum (l l~ / 4)
    a.cw[((size_t)b * 2 + 1) * a.nt + k] =
        Quad<T>{r[4], r[5], (T)0.25 * a.ika[c], DF ? (T)((double)a.kh[c] * a.iaa[c]) : (T)0};
  }
  for (int k = threadIdx.x; k < nTri; k += blockDim.x) {
    const size_t p = (size_t)b * a.TC + k;
    const int sl = a.tslot[p], t = 2 * cell(sl >> 1) + (sl & 1);
    uint32_t v = a.tv[p] & 0x1FFFFFFFu;
    for (int m = 0; m < 3; ++m) v |= (a.ceta[(size_t)m * NT + t] < (T)0 ? 1u : 0u) << (29 + m);
    a.tv[p] = v;
    a.tk[p] = Quad<T>{a.kap[t], a.kap[(size_t)NT + t], a.kap[(size_t)2 * NT + t], (T)(1.0 / (a.tarea[t] * a.ea))};
    a.tf[p] = a.f[t];
    if constexpr (DF) a.tkt[p] = a.kt[t];
    if constexpr (AP) {
      if (k >= nG) continue;
      for (int m = 0; m < 3; ++m) {
        const Quad<T> q = a.awt[(size_t)m * NT + t];
        a.wt[((size_t)b * 3 + m) * a.GC + k] = Tri<T>{q.x, q.y, q.z};
      }
    }
  }
  for (int e = 3 * own0 + threadIdx.x; e < 3 * (own0 + nown); e += blockDim.x) {
    a.eld[e] = Pair<T>{stored_length<T>(a.leng[e]), (T)a.dleng[e]};
    const int o = a.e_oth[e];
    if (o < 0) continue;
    a.oth[e] = (uint16_t)((a.oth[e] & LID) | ((uint32_t)(o >> OTH_V2) & 1u) << SB_OWN);
    if constexpr (PX) {
      const Quad<T> q = a.pn[e];
      a.en[e] = Tri<T>{q.x, q.y, q.z};
    }
  }
}

static int no_memory(hipError_t e) {
  return set_error(e == hipErrorOutOfMemory ? IMX_ENOMEM : IMX_EDEVICE,
                   std::string("stage tables: ") + hipGetErrorString(e));
}

// The cut for nt threads, or that the handle has where it fits the scheme too.
template <typename T>
static int ensure_cut(imx_swm *s, int nt, bool wide, bool *local) {
  if (s->stg && s->stg->nt == nt && s->stg->wide == wide &&
      (!s->stg_limit || s->stg->A.bytes <= s->stg_limit))
    return IMX_OK;
  stage_free(s);
  // the kernel addresses its tables by 32-bit byte offsets
  if ((uint64_t)s->NE * sizeof(Tri<T>) >> 32) return IMX_OK;
  Cut C;
  const int rc = cut_blocks(s, nt, wide, C, local);
  if (rc || !*local) return rc;
  // the handle has the tables once they are whole
  struct Drop {
    void operator()(Stage *p) const {
      p->A.release();
      delete p;
    }
  };
  std::unique_ptr<Stage, Drop> g(new Stage());
  Alloc &A = g->A;
  A.limit = s->stg_limit;
  const size_t nc = (size_t)C.nblk * nt, ntr = C.tv.n;
  g->nt = nt;
  g->nblk = C.nblk;
  g->wide = wide;
  g->head = up(A, C.head);
  g->halo = up(A, C.halo);
  g->topo = up(A, C.topo);
  g->cw = A.get<Quad<T>>(2 * nc);
  g->eld = A.get<Pair<T>>(s->NE);
  g->oth = up(A, C.oth);
  g->tv = up(A, C.tv);
  g->tslot = up(A, C.tslot);
  g->tk = A.get<Quad<T>>(ntr);
  g->tf = A.get<T>(ntr);
  if (wide) g->tn = up(A, C.tn);
  if (A.err != hipSuccess) return no_memory(A.err);
  s->stg = g.release();
  return IMX_OK;
}

template <typename T, int SCHEME>
static void fill(const FillArgs<T> &a, int nblk, hipStream_t st) {
  stage_fill<T, SCHEME><<<nblk, 256, 0, st>>>(a);
}

template <typename T>
static int build(imx_swm *s, int nt, int scheme, bool *local) {
  const bool ap = scheme == kApvm, px = scheme == kPerot, df = scheme == kDiff;
  int rc = ensure_cut<T>(s, nt, ap, local);
  if (rc || !s->stg) return rc;
  Stage &g = *s->stg;
  const int CL = cap_l(nt, ap), TC = cap_t(nt, ap), GC = cap_g(nt);
  Alloc &O = g.O;
  O.release();
  O = Alloc();
  g.wc = g.wt = g.en = g.tkt = nullptr;
  if (s->stg_limit) O.limit = std::max<size_t>(s->stg_limit - g.A.bytes, 1);
  if (ap || px) g.wc = O.get<Tri<T>>((size_t)g.nblk * MX * CL);
  if (ap) g.wt = O.get<Tri<T>>((size_t)g.nblk * 3 * GC);
  if (px) g.en = O.get<Tri<T>>(s->NE);
  if (df) g.tkt = O.get<T>((size_t)g.nblk * TC);
  if (O.err != hipSuccess) {
    rc = no_memory(O.err);
    stage_free(s);
    return rc;
  }
  g.scheme = scheme;
  FillArgs<T> a;
  a.head = g.head;
  a.halo = g.halo;
  a.tslot = g.tslot;
  a.bitsA = s->x_c_bitsA;
  a.e_oth = s->x_e_oth;
  a.R = (const T *)(px ? s->x_px_wq : s->x_c_R);
  a.ika = (const T *)s->x_c_ika;
  a.kh = (const T *)s->x_kh;
  a.kt = (const T *)s->x_kt;
  a.ceta = (const T *)s->x_t_ceta;
  a.kap = (const T *)s->x_t_kap;
  a.f = (const T *)s->x_t_f;
  a.iaa = s->x_c_iaa;
  a.leng = s->e_leng;
  a.dleng = s->e_dleng;
  a.tarea = s->t_area;
  a.awc = (const Quad<T> *)s->x_ap_wc;
  a.awt = (const Quad<T> *)s->x_ap_wt;
  a.pn = (const Quad<T> *)s->x_px_n;
  a.topo = g.topo;
  a.cw = (Quad<T> *)g.cw;
  a.tk = (Quad<T> *)g.tk;
  a.eld = (Pair<T> *)g.eld;
  a.oth = g.oth;
  a.tv = g.tv;
  a.tf = (T *)g.tf;
  a.tkt = (T *)g.tkt;
  a.wc = (Tri<T> *)g.wc;
  a.wt = (Tri<T> *)g.wt;
  a.en = (Tri<T> *)g.en;
  a.nv = s->nv;
  a.NE = s->NE;
  a.NT = s->NT;
  a.nt = nt;
  a.CL = CL;
  a.TC = TC;
  a.GC = GC;
  a.ea = s->o.erad;
  forget_error();
  switch (scheme) {
    case kApvm: fill<T, kApvm>(a, g.nblk, s->stream); break;
    case kPerot: fill<T, kPerot>(a, g.nblk, s->stream); break;
    case kDiff: fill<T, kDiff>(a, g.nblk, s->stream); break;
    default: fill<T, kPlain>(a, g.nblk, s->stream); break;
  }
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(s->stream);
  if (e == hipSuccess) return IMX_OK;
  stage_free(s);
  return set_error(IMX_EDEVICE, std::string("stage tables: ") + hipGetErrorString(e));
}

int stage_build(imx_swm *s, int nt, int scheme, bool *local) {
  *local = true;
  try {
    return s->single ? build<float>(s, nt, scheme, local) : build<double>(s, nt, scheme, local);
  } catch (const std::bad_alloc &) {
    stage_free(s);
    return set_error(IMX_ENOMEM, "stage tables: host out of memory");
  }
}

template <typename T, int NT, int S>
static void launch_nt(const StageOpts<T> &a, int stage, int grid, hipStream_t st) {
  using Args = std::conditional_t<S == kPlain, StageArgs<T>, StageOpts<T>>;
  switch (stage) {
    case 0: fast_stage<T, NT, 0, S, Args><<<grid, NT, 0, st>>>(a); break;
    case 1:
    case 2: fast_stage<T, NT, 1, S, Args><<<grid, NT, 0, st>>>(a); break;
    case 3: fast_stage<T, NT, 2, S, Args><<<grid, NT, 0, st>>>(a); break;
    default: fast_stage<T, NT, 3, S, Args><<<grid, NT, 0, st>>>(a); break;
  }
}

template <typename T, int S>
static void launch_threads(const StageOpts<T> &a, int nt, int stage, int grid, hipStream_t st) {
  switch (nt) {
    case 128: launch_nt<T, 128, S>(a, stage, grid, st); break;
    case 512:
      if constexpr (sizeof(T) == 4) launch_nt<T, 512, S>(a, stage, grid, st);
      break;
    default: launch_nt<T, 256, S>(a, stage, grid, st); break;
  }
}

template <typename T>
void stage_launch(imx_swm *s, int stage, const T *hs, const T *us, T *hout, T *uout) {
  const Stage &g = *s->stg;
  StageOpts<T> a;
  a.head = g.head;
  a.halo = g.halo;
  a.topo = g.topo;
  a.cw = (const Quad<T> *)g.cw;
  a.eld = (const Pair<T> *)g.eld;
  a.oth = g.oth;
  a.tv = g.tv;
  a.tslot = g.tslot;
  a.tk = (const Quad<T> *)g.tk;
  a.tf = (const T *)g.tf;
  a.wc = (const Tri<T> *)g.wc;
  a.wt = (const Tri<T> *)g.wt;
  a.tn = g.tn;
  a.en = (const Tri<T> *)g.en;
  a.tkt = (const T *)g.tkt;
  a.pvsdt = (T)(s->sc.pvspar * s->o.dt);
  a.iaa = s->x_c_iaa;
  a.hs = hs;
  a.us = us;
  a.h0 = (const T *)s->h0;
  a.u0 = (const T *)s->u0;
  a.gb = (const T *)s->x_gb;
  a.dte = (const T *)s->dt_e;
  a.dtc = s->dt_c;
  a.hout = hout;
  a.uout = uout;
  a.acch = (T *)s->acch;
  a.accu = (T *)s->accu;
  a.q = (T *)s->q;
  a.du_out = (T *)s->du_out;
  a.dh_out = s->dh_out;
  a.flag = s->flag;
  a.href = s->href;
  const double dt = s->o.dt;
  const T dtt = (T)dt;
  a.ca = stage == 2 ? dt : 0.5 * dt;
  a.cb = stage == 1 || stage == 2 ? dt / 3.0 : dt / 6.0;
  a.cat = stage == 2 ? dtt : (T)0.5 * dtt;
  a.cbt = stage == 1 || stage == 2 ? dtt / (T)3 : dtt / (T)6;
  a.grav = (T)s->o.grav;
  a.inv_a = (T)(1.0 / s->o.erad);
  a.nblk = g.nblk;
  a.remap = g.remap;
  a.whole = stage == 2;
  a.use_pv = s->o.testcase >= 2;
  a.flin = s->f_lin ? 1 : 0;
  a.zero_mom = s->o.testcase <= 1;
  const int grid = (g.nblk + NXCD - 1) / NXCD * NXCD;
  switch (g.scheme) {
    case kApvm: launch_threads<T, kApvm>(a, g.nt, stage, grid, s->stream); break;
    case kPerot: launch_threads<T, kPerot>(a, g.nt, stage, grid, s->stream); break;
    case kDiff: launch_threads<T, kDiff>(a, g.nt, stage, grid, s->stream); break;
    default: launch_threads<T, kPlain>(a, g.nt, stage, grid, s->stream); break;
  }
}
template void stage_launch<float>(imx_swm *, int, const float *, const float *, float *, float *);
template void stage_launch<double>(imx_swm *, int, const double *, const double *, double *, double *);

}  // namespace imx
