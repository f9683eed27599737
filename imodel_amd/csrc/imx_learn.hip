// libimx learned correction coupled to the shallow-water step.
//
// A coarse FAST handle advances with the plain RK4 step; the per-edge MLP
// (imx_mlp.hip) then predicts, from the 2-ring of every edge, the correction
// (du_e, dh) that maps the plain coarse step toward the restricted state of
// a finer run. Features of edge e (48, normalised by the caller's mean/std):
//   0-10   s_k u_k at e and the other ring edges of its two cells (TRiSK
//          orientation signs s_k), state before the step
//   11-21  the plain step's increment of the same
//   22-31  h - h_ref at the edge's 2 cells, the 2 triangle apexes (left,
//          right of v1->v2) and the other ring cells of both cells
//   32-41  the plain step's increment of the same
//   42-47  z and sqrt(1-z^2) of the edge midpoint, l_e, l~_e, A_c1, A_c2
//          relative to their means
// Outputs per edge: du_e, added to the edge velocity, and a mass flux F_e
// whose discrete divergence D F is added to the cell depths,
//   (D F)_c = -kappa/A_c sum_{e in c} ttgout_ce l~_e F_e,
// so the h correction moves mass between neighbours and the total mass
// sum_c A_c h_c is unchanged. Training fits du to its target directly and
// fits D F to the dh target through D (the gradient D^T r is handed to the
// MLP backward pass). The correction is skipped (plain step kept) when its
// RMS exceeds a bound. The corrected step (RK4 step, network with the features
// formed in its kernel, correction) is captured; one graph launch runs up to 16 of them.
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>

#include <cmath>
#include <cstring>
#include <new>
#include <string>
#include <vector>

#include "imx_device.h"
#include "imx_mlp_dev.h"

#define NF 48
#define NSE 11  // stencil edges
#define NSC 10  // stencil cells
#define LTPB 256
#define LPART 1024  // blocks of the correction-norm pass
#define SREC 32    // words per edge stencil record (128 bytes)
static constexpr int kLossSteps = 16;  // a fit returns the mean loss of its last steps

struct imx_learn {
  imx_swm *s = nullptr;
  imx_mlp *m = nullptr;
  int nv = 0, NE = 0;
  imx::Alloc A;
  int32_t *stn = nullptr;   // [NE][SREC] stencil record per edge slot (see learn_featx)
  float *dc = nullptr;      // [6][nv] coefficient of F_{c_ed[j][c]} in (D F)_c
  float *de = nullptr;      // [2][NE] coefficient of F_e in (D F) at e_v[0/1][e]
  void *hn = nullptr, *un = nullptr;  // state before the last step or sample (T)
  float *raw = nullptr;     // [NE][NF]
  float *mu = nullptr, *sig = nullptr, *norm = nullptr;  // norm: FeatLoader's order
  void *hq = nullptr, *uq = nullptr;  // state after the plain step of a corrected one (T)
  float tsu = 1.f, tsh = 1.f;
  float *Y = nullptr;       // [NE][2]
  float *wv = nullptr;      // [NE] 1/ne on real edges
  float *dhc = nullptr;     // [nv] (D F)_c, or its residual in training
  float *th = nullptr;      // [nv] scaled dh target
  double *part = nullptr;   // [LPART] partial sums of the correction norm
  double *rms = nullptr;    // [1] correction RMS of the last step
  double *bound = nullptr;  // [2] RMS bound, limiter mode (IMX_LIMIT_*)
  double *lh = nullptr;     // [kLossSteps] h losses of a fit's last steps
  float *lossu = nullptr;   // [kLossSteps][(NE + 63) / 64] their u loss partials
  int *nfb = nullptr;       // [1] limited steps since the counter was cleared
  imx::StepGraphs graphs;
  uint64_t gen = 0;           // the step handle's generation at capture
  // device sample store: normalised features, scaled targets
  int cap = 0, count = 0;
  int64_t xstride = 0;      // shorts per stored feature matrix
  short *Xb = nullptr;      // [cap][xstride]
  float *tub = nullptr;     // [cap][NE] scaled du target, internal order
  float *thb = nullptr;     // [cap][nv] scaled dh target
};


template <typename T>
__global__ __launch_bounds__(LTPB) void learn_save(int nv, int NE, const T *__restrict__ h,
                                                   const T *__restrict__ u, T *__restrict__ hn,
                                                   T *__restrict__ un) {
  const int i = blockIdx.x * LTPB + threadIdx.x;
  if (i < NE) un[i] = u[i];
  if (i < nv) hn[i] = h[i];
}

// Stencil record of an edge, 32 words in four quarters of 8, one per lane
// group of the network kernel (mlp_feature_slot): words 0-4 the quarter's ids
// j = 0..4 (id << 1 | sign, -1 pad), word 5 id 5 (quarter 3), words 6, 7 two
// geometry features (FP32 bits; quarters 0-2). Dummy slots: no ids, zeros.
__host__ __device__ inline int rec_edge(int k) { return k / 5 * 8 + k % 5; }
__host__ __device__ inline int rec_cell(int k) { return k < 4 ? 17 + k : 20 + k; }
__host__ __device__ inline int rec_geo(int k) { return k / 2 * 8 + 6 + k % 2; }

// Features of (saved state un/hn, plain step up/hp) for sampling and
// training, one thread per edge slot: the stencil record is read with vector
// loads and all 42 state gathers are issued before any is used, so a thread
// keeps its loads in flight together (one feature per thread would chain a
// record read and a gather for every feature). Dummy slots get all-zero raw
// features.
template <typename T>
__global__ __launch_bounds__(LTPB) void learn_featx(int NE, const int32_t *__restrict__ stn,
                                                    const T *__restrict__ un, const T *__restrict__ hn,
                                                    const T *__restrict__ up, const T *__restrict__ hp,
                                                    const float *__restrict__ mu,
                                                    const float *__restrict__ sig,
                                                    float *__restrict__ raw, short *__restrict__ X) {
  const int e = blockIdx.x * LTPB + threadIdx.x;
  if (e >= NE) return;
  int32_t r[SREC];
  const int4 *rv = reinterpret_cast<const int4 *>(stn + (int64_t)e * SREC);
#pragma unroll
  for (int q = 0; q < SREC / 4; ++q) {
    const int4 v = rv[q];
    r[4 * q] = v.x;
    r[4 * q + 1] = v.y;
    r[4 * q + 2] = v.z;
    r[4 * q + 3] = v.w;
  }
  float f[NF];
  T a[NSE], b[NSE], c0[NSC], c1[NSC];
#pragma unroll
  for (int k = 0; k < NSE; ++k) {
    const int w = r[rec_edge(k)];
    const int ek = w >= 0 ? w >> 1 : 0;
    a[k] = un[ek];
    b[k] = up[ek];
  }
#pragma unroll
  for (int k = 0; k < NSC; ++k) {
    const int w = r[rec_cell(k)];
    const int c = w >= 0 ? w >> 1 : 0;
    c0[k] = hn[c];
    c1[k] = hp[c];
  }
#pragma unroll
  for (int k = 0; k < NSE; ++k) {
    const int w = r[rec_edge(k)];
    const bool ok = w >= 0;
    const float sg = (w & 1) ? -1.f : 1.f;
    f[k] = ok ? sg * (float)a[k] : 0.f;
    f[NSE + k] = ok ? sg * (float)(b[k] - a[k]) : 0.f;
  }
#pragma unroll
  for (int k = 0; k < NSC; ++k) {
    const bool ok = r[rec_cell(k)] >= 0;
    f[2 * NSE + k] = ok ? (float)c0[k] : 0.f;
    f[2 * NSE + NSC + k] = ok ? (float)(c1[k] - c0[k]) : 0.f;
  }
#pragma unroll
  for (int k = 0; k < 6; ++k) f[2 * NSE + 2 * NSC + k] = __int_as_float(r[rec_geo(k)]);
  const int64_t o = (int64_t)e * NF;
  if (raw) {
    float4 *rw = reinterpret_cast<float4 *>(raw + o);
#pragma unroll
    for (int q = 0; q < NF / 4; ++q) rw[q] = make_float4(f[4 * q], f[4 * q + 1], f[4 * q + 2], f[4 * q + 3]);
  }
  if (X) {
    v4s *xw = reinterpret_cast<v4s *>(X + o);
#pragma unroll
    for (int q = 0; q < NF / 4; ++q) {
      v4s x;
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = f2bf((f[4 * q + i] - mu[4 * q + i]) / sig[4 * q + i]);
      xw[q] = x;
    }
  }
}

// Input fragments of the network formed in its own kernel: the features of
// learn_featx in the slots of mlp_feature_slot. The four lanes of an edge read
// its record as consecutive 32-byte quarters and gather six ids each; the
// normalised row (96 bytes written and read per edge) never exists: 355 to 382 us
// at glevel 8 instead of 147 for the rows and 259 to 279 for the network on them.
// Both kernels keep the vector units busy 92 % of the time (counters: 46 % of
// each wave's cycles issue vector work, two waves a SIMD). Of the cycles that the
// gathers add, 45 % are vector work (27 % more instructions: ids, signs, the
// normalisation's divisions) and 41 % waits, mostly for memory; gathering a tile
// ahead takes 1 % off there and adds as much at glevel 6. norm: per lane group 12 means, 12 deviations.
template <typename T>
struct FeatLoader {
  static constexpr int kNorm = 24;
  const int32_t *stn;
  const T *un, *hn, *up, *hp;
  const float *norm;
  __device__ __forceinline__ void prepare(float *sh) const {
    for (int i = threadIdx.x; i < 4 * kNorm; i += blockDim.x) sh[64 * (i / kNorm) + i % kNorm] = norm[i];
  }
  template <int ET>
  __device__ __forceinline__ void operator()(int64_t e0, int64_t n, int lane, v4s (&x)[3][ET], const float *sh) const {
    const int g = lane / 16;
    // id 0 is an edge's in groups 0-2, the others in groups 0 and 1
    const T *a0 = g < 3 ? un : hn, *b0 = g < 3 ? up : hp, *a1 = g < 2 ? un : hn, *b1 = g < 2 ? up : hp;
    int w[ET][8];
    T a[ET][6], b[ET][6];
#pragma unroll
    for (int t = 0; t < ET; ++t) {
      int64_t e = e0 + 16 * t + lane % 16;
      if (e >= n) e = n - 1;
      const int4 *r = reinterpret_cast<const int4 *>(stn + e * SREC + 8 * g);
      const int4 p = r[0], q = r[1];
      w[t][0] = p.x, w[t][1] = p.y, w[t][2] = p.z, w[t][3] = p.w;
      w[t][4] = q.x, w[t][5] = q.y, w[t][6] = q.z, w[t][7] = q.w;
    }
#pragma unroll
    for (int t = 0; t < ET; ++t)
#pragma unroll
      for (int j = 0; j < 6; ++j) {
        const int id = w[t][j] < 0 ? 0 : w[t][j] >> 1;
        a[t][j] = (j ? a1 : a0)[id];
        b[t][j] = (j ? b1 : b0)[id];
      }
    const float *m = sh + 64 * g;
#pragma unroll
    for (int t = 0; t < ET; ++t) {
      float f[12];
#pragma unroll
      for (int j = 0; j < 6; ++j) {
        const bool ok = w[t][j] >= 0;
        const float sg = (w[t][j] & 1) ? -1.f : 1.f;
        f[2 * j] = ok ? sg * (float)a[t][j] : 0.f;
        f[2 * j + 1] = ok ? sg * (float)(b[t][j] - a[t][j]) : 0.f;
      }
      if (g < 3) {
        f[10] = __int_as_float(w[t][6]);
        f[11] = __int_as_float(w[t][7]);
      }
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        float q[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int s = 4 * k + i;
          q[i] = (f[s] - m[s]) / m[12 + s];
        }
        const uint32_t v[2] = {f2bf2(q[0], q[1]), f2bf2(q[2], q[3])};
        x[k][t] = __builtin_bit_cast(v4s, v);
      }
    }
  }
};

// (D F)_c of the flux output F = Y[.][1]: all gathers in flight, then the sum
// in ring order
__device__ __forceinline__ float div_flux(int c, int nv, const int32_t *__restrict__ c_nnb,
                                          const int32_t *__restrict__ c_ed, const float *__restrict__ dc,
                                          const float *__restrict__ Y) {
  const int n = c_nnb[c];
  float f[IMX_MAXNB], d[IMX_MAXNB];
#pragma unroll
  for (int j = 0; j < IMX_MAXNB; ++j) {  // padded slots name edge slot 0
    f[j] = Y[2 * c_ed[j * nv + c] + 1];
    d[j] = dc[j * nv + c];
  }
  float v = 0.f;
#pragma unroll
  for (int j = 0; j < IMX_MAXNB; ++j)
    if (j < n) v += d[j] * f[j];
  return v;
}

// out_c = (D F)_c - t_c (t may be NULL)
__global__ __launch_bounds__(LTPB) void learn_div(int nv, const int32_t *__restrict__ c_nnb,
                                                  const int32_t *__restrict__ c_ed,
                                                  const float *__restrict__ dc, const float *__restrict__ Y,
                                                  const float *__restrict__ t, float *__restrict__ out) {
  const int c = blockIdx.x * LTPB + threadIdx.x;
  if (c >= nv) return;
  const float v = div_flux(c, nv, c_nnb, c_ed, dc, Y);
  out[c] = t ? v - t[c] : v;
}

// dL/dF_e = scale * (D^T r)_e into T[e][1] (the MLP's gradient input)
__global__ __launch_bounds__(LTPB) void learn_divT(int NE, const int32_t *__restrict__ e_v,
                                                   const float *__restrict__ de, const float *__restrict__ r,
                                                   float scale, float *__restrict__ T) {
  const int e = blockIdx.x * LTPB + threadIdx.x;
  if (e >= NE) return;
  const int c1 = e_v[e], c2 = e_v[NE + e];
  T[2 * e + 1] = (c1 < 0) ? 0.f : scale * (de[e] * r[c1] + de[NE + e] * r[c2]);
}

// T[e] = (scaled du target, scale * (D^T r)_e) for a stored sample's step
__global__ __launch_bounds__(LTPB) void learn_targets(int NE, const int32_t *__restrict__ e_v,
                                                      const float *__restrict__ de,
                                                      const float *__restrict__ r, float scale,
                                                      const float *__restrict__ tu, float *__restrict__ T) {
  const int e = blockIdx.x * LTPB + threadIdx.x;
  if (e >= NE) return;
  const int c1 = e_v[e], c2 = e_v[NE + e];
  T[2 * e] = tu[e];
  T[2 * e + 1] = (c1 < 0) ? 0.f : scale * (de[e] * r[c1] + de[NE + e] * r[c2]);
}

// out = sqrt(sum_e w_e a_e^2 + sb sum_c b_c^2) (one block; a strided by sa)
__global__ __launch_bounds__(1024) void learn_norm2(int na, const float *__restrict__ a, int sa,
                                                    const float *__restrict__ w, int nb,
                                                    const float *__restrict__ b, double sb, int take_sqrt,
                                                    double *__restrict__ out) {
  double s = 0.0;
  if (a)
    for (int e = threadIdx.x; e < na; e += 1024) s += (double)w[e] * (double)a[sa * e] * (double)a[sa * e];
  double t = 0.0;
  if (b)
#pragma unroll 8
    for (int c = threadIdx.x; c < nb; c += 1024) t += (double)b[c] * (double)b[c];
  s += sb * t;
  __shared__ double red[1024];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int o = 512; o > 0; o >>= 1) {
    if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = take_sqrt ? sqrt(red[0]) : red[0];
}

// Sum of one value per thread of a block, the same in every thread: lanes by
// butterfly, then the waves in order.
__device__ __forceinline__ double block_sum(double v) {
  __shared__ double red[LTPB / 64];
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = v;
  __syncthreads();
  double r = red[0];
#pragma unroll
  for (int w = 1; w < LTPB / 64; ++w) r += red[w];
  return r;
}

// (D F)_c of the flux output into dhc, and per-block partial sums of the
// correction's squared norm sum_e w_e Y0^2 + (1/nv) sum_c (D F)_c^2
// (grid-stride over max(nv, NE), LPART blocks). 17.4 us at glevel 8 and 4.8 at
// 6, with each gather waiting for the one before 24.5 and 6.5; 57 MB at glevel
// 8, mostly latency still.
__global__ __launch_bounds__(LTPB) void learn_div_part(int nv, int NE, const int32_t *__restrict__ c_nnb,
                                                       const int32_t *__restrict__ c_ed,
                                                       const float *__restrict__ dc,
                                                       const float *__restrict__ Y,
                                                       const float *__restrict__ w,
                                                       float *__restrict__ dhc, double *__restrict__ part) {
  double s = 0.0, t = 0.0;
  const int nmax = nv > NE ? nv : NE;
  for (int i = blockIdx.x * LTPB + threadIdx.x; i < nmax; i += gridDim.x * LTPB) {
    if (i < NE) s += (double)w[i] * (double)Y[2 * i] * (double)Y[2 * i];
    if (i >= nv) continue;
    const float v = div_flux(i, nv, c_nnb, c_ed, dc, Y);
    dhc[i] = v;
    t += (double)v * (double)v;
  }
  const double r = block_sum(s + t / nv);
  if (threadIdx.x == 0) part[blockIdx.x] = r;
}

// every block sums the LPART partials (fixed order: the same RMS in every
// block), then the state u, h becomes the plain step's up, hp plus Y0/tsu and
// (D F)/tsh, or the plain step's where RMS > bound. K elements a thread, their
// operands loaded before the sum's barrier: with one a thread every element's
// block sums the partials first, 15.4 us at glevel 8 against 9.0 with four (47
// MB at a copy's rate); from half a million elements on there are blocks enough.
template <typename T, int K>
__global__ __launch_bounds__(LTPB) void learn_apply(int nv, int NE, const float *__restrict__ wv,
                                                    const float *__restrict__ Y,
                                                    const float *__restrict__ dhc, float inv_tsu,
                                                    float inv_tsh, const double *__restrict__ part,
                                                    const double *__restrict__ bound, const T *__restrict__ up,
                                                    const T *__restrict__ hp, T *__restrict__ u, T *__restrict__ h,
                                                    double *__restrict__ rms, int *__restrict__ nfb) {
  const int i0 = blockIdx.x * (LTPB * K) + threadIdx.x;
  float y[K], d[K], wt[K];
  T us[K], hq[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int i = i0 + k * LTPB, e = min(i, NE - 1), c = min(i, nv - 1);
    wt[k] = wv[e];
    y[k] = Y[2 * e];
    us[k] = up[e];
    d[k] = dhc[c];
    hq[k] = hp[c];
  }
  double p = 0.0;
#pragma unroll
  for (int k = 0; k < LPART; k += LTPB) p += part[k + threadIdx.x];
  // limiter (bound[0] the RMS bound, bound[1] the mode): a correction whose
  // RMS exceeds the bound is dropped and the plain step kept (mode 0), or
  // scaled down to the bound (mode 1); a non-finite one (or bound 0) always
  // leaves the plain step untouched
  const double r = sqrt(block_sum(p));
  const bool ok = r <= bound[0];
  const bool scale = bound[1] > 0.5;
  const float sc = ok ? 1.f : ((scale && r < 1e300) ? (float)(bound[0] / r) : 0.f);
  if (i0 == 0) {
    rms[0] = r;
    if (!ok) nfb[0] = nfb[0] + 1;  // one thread of the grid counts
  }
  const bool on = sc > 0.f;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int i = i0 + k * LTPB;
    if (i < NE && wt[k] > 0.f) u[i] = on ? (T)((float)us[k] + sc * (y[k] * inv_tsu)) : us[k];
    if (i < nv) h[i] = on ? (T)((float)hq[k] + sc * (d[k] * inv_tsh)) : hq[k];
  }
}

namespace imx {

static int lfail(hipError_t e, const char *what) {
  return set_error(IMX_EDEVICE, std::string(what) + ": " + hipGetErrorString(e));
}
#define LTRY(expr, what)                        \
  do {                                          \
    hipError_t _e = (expr);                     \
    if (_e != hipSuccess) return imx::lfail(_e, what); \
  } while (0)

static void learn_drop_graph(imx_learn *L) { L->graphs.drop(); }

// enqueue: save x_n
template <typename T>
static void learn_enqueue_save(imx_learn *L) {
  imx_swm *s = L->s;
  const int g = (L->NE + LTPB - 1) / LTPB;
  learn_save<T><<<g, LTPB, 0, s->stream>>>(s->nv, L->NE, (const T *)s->h0, (const T *)s->u0, (T *)L->hn,
                                           (T *)L->un);
}

// enqueue: save x_n, one plain step
template <typename T>
static void learn_enqueue_sample(imx_learn *L) {
  learn_enqueue_save<T>(L);
  swm_launch_step(L->s);
}

// enqueue: features of (saved state, current state) into raw and/or X
template <typename T>
static void learn_enqueue_featx_t(imx_learn *L, hipStream_t st, float *raw, short *X) {
  imx_swm *s = L->s;
  learn_featx<T><<<(unsigned)((L->NE + LTPB - 1) / LTPB), LTPB, 0, st>>>(
      L->NE, L->stn, (const T *)L->un, (const T *)L->hn, (const T *)s->u0, (const T *)s->h0, L->mu, L->sig,
      raw, X);
}

static void learn_enqueue_featx(imx_learn *L, hipStream_t st, float *raw, short *X) {
  if (L->s->single) learn_enqueue_featx_t<float>(L, st, raw, X);
  else learn_enqueue_featx_t<double>(L, st, raw, X);
}

static void learn_free_store(imx_learn *L) {
  (void)hipFree(L->Xb);
  (void)hipFree(L->tub);
  (void)hipFree(L->thb);
  L->Xb = nullptr;
  L->tub = L->thb = nullptr;
  L->cap = L->count = 0;
}

// enqueue: one corrected step: the plain step into hq, uq, the network on
// features gathered from both states, the correction (with the RMS bound)
// back into the handle's state. save: x_n is kept as a sample's is; the last
// step of a run has it (with every graph's last step, 1 of up to 16: a copy of
// the state, 15 us at glevel 8), so that imx_learn_train and imx_learn_store
// after it take that step's features
template <typename T>
static int learn_enqueue_step(imx_learn *L, bool save) {
  imx_swm *s = L->s;
  hipStream_t st = s->stream;
  if (save) learn_enqueue_save<T>(L);
  swm_launch_step(s, L->hq, L->uq);
  const FeatLoader<T> ld{L->stn, (const T *)s->u0, (const T *)s->h0, (const T *)L->uq, (const T *)L->hq, L->norm};
  LTRY(mlp_fwd_launch(L->m->F1g, L->m->Ff32, L->m->P, L->NE, ld, L->Y, st), "mlp_fwd_lds");
  const int nmax = s->nv > L->NE ? s->nv : L->NE;
  learn_div_part<<<LPART, LTPB, 0, st>>>(s->nv, L->NE, s->c_nnb, s->c_ed, L->dc, L->Y, L->wv, L->dhc,
                                         L->part);
  auto apply = [&](auto kern, int k) {
    kern<<<(nmax + k * LTPB - 1) / (k * LTPB), LTPB, 0, st>>>(
        s->nv, L->NE, L->wv, L->Y, L->dhc, 1.f / L->tsu, 1.f / L->tsh, L->part, L->bound, (const T *)L->uq,
        (const T *)L->hq, (T *)s->u0, (T *)s->h0, L->rms, L->nfb);
  };
  if (nmax < 1 << 19) apply(learn_apply<T, 1>, 1);
  else apply(learn_apply<T, 4>, 4);
  LTRY(hipGetLastError(), "learn_apply");
  return IMX_OK;
}

static int learn_sample(imx_learn *L) {
  if (L->s->single) learn_enqueue_sample<float>(L);
  else learn_enqueue_sample<double>(L);
  LTRY(hipGetLastError(), "learn sample");
  return IMX_OK;
}

static int learn_ensure_graphs(imx_learn *L, int nsteps, int32_t *made = nullptr) {
  // recapture when the handle's step changed (scheme, tuning, topography, h_ref)
  if (L->gen != L->s->generation) learn_drop_graph(L);
  L->gen = L->s->generation;
  hipError_t e;
  const int rc = L->graphs.ensure(nsteps, L->s->stream, [&](bool last) {
    return L->s->single ? learn_enqueue_step<float>(L, last) : learn_enqueue_step<double>(L, last);
  }, e, made);
  if (rc) return rc;
  LTRY(e, "learn graph capture");
  return IMX_OK;
}

// FeatLoader's normalisation from the features' means and deviations
static std::vector<float> learn_norm(const float *mu, const float *sig) {
  constexpr int K = FeatLoader<float>::kNorm;
  std::vector<float> v(4 * K, 0.f);
  for (int q = 0; q < 4; ++q)
    for (int s = 0; s < 12; ++s) v[K * q + 12 + s] = 1.f;
  for (int f = 0; f < NF; ++f) {
    int g, s;
    mlp_feature_slot(f, &g, &s);
    v[K * g + s] = mu[f];
    v[K * g + 12 + s] = sig[f];
  }
  return v;
}

}  // namespace imx

extern "C" {

int imx_learn_create(imx_swm *s, imx_mlp *m, const imx_mesh_desc *d, imx_learn **out) {
  if (!s || !m || !d || !out) return imx::set_error(IMX_EINVAL, "imx_learn_create: NULL argument");
  *out = nullptr;
  if (!s->fast) return imx::set_error(IMX_ENOTSUP, "imx_learn_create: needs an FP32/FP64 fused handle");
  if (d->nv != s->nv || d->ne != s->ne || d->nt != s->nt)
    return imx::set_error(IMX_EINVAL, "imx_learn_create: mesh does not match the handle");
  imx_learn *L = new (std::nothrow) imx_learn();
  if (!L) return imx::set_error(IMX_ENOMEM, "imx_learn_create: out of memory");
  L->s = s;
  L->m = m;
  L->nv = s->nv;
  L->NE = s->NE;
  const int NE = s->NE, nv = s->nv, MX = IMX_MAXNB;
  const std::vector<int32_t> &cn = s->lay.cell_new, &en = s->lay.edge_new;
  std::vector<int32_t> stn((size_t)SREC * NE, 0);
  for (int e = 0; e < NE; ++e)
    for (int k = 0; k < SREC; ++k)
      if (k % 8 < 6) stn[(size_t)e * SREC + k] = -1;
  std::vector<float> wv(NE, 0.f);
  std::vector<float> dc((size_t)6 * nv, 0.f), de((size_t)2 * NE, 0.f);
  double ml = 0, md = 0, ma = 0;
  for (int eo = 0; eo < d->ne; ++eo) {
    ml += d->ed_leng[eo];
    md += d->edhx_leng[eo];
  }
  for (int c = 0; c < d->nv; ++c) ma += d->hx_areag[c];
  ml /= d->ne;
  md /= d->ne;
  ma /= d->nv;
  // (D F)_c coefficients, scaled by kappa = mean area / mean dual length
  const double kappa = ma / md;
  for (int co = 0; co < d->nv; ++co) {
    const int c = cn[co];
    for (int j = 0; j < d->v_nnb[co]; ++j) {
      const int eo = d->v_ed[MX * co + j] - 1, e = en[eo];
      const double sg = d->hx_ttgout[MX * co + j] < 0 ? -1.0 : 1.0;
      const float coef = (float)(-kappa * sg * d->edhx_leng[eo] / d->hx_areag[co]);
      dc[(size_t)j * nv + c] = coef;
      de[(size_t)((d->ed_v[2 * eo] - 1 == co) ? 0 : 1) * NE + e] = coef;
    }
  }
  for (int eo = 0; eo < d->ne; ++eo) {
    const int e = en[eo];
    int cell[2] = {d->ed_v[2 * eo] - 1, d->ed_v[2 * eo + 1] - 1};
    int slot[2] = {-1, -1};
    for (int q = 0; q < 2; ++q)
      for (int j = 0; j < d->v_nnb[cell[q]]; ++j)
        if (d->v_ed[MX * cell[q] + j] == eo + 1) slot[q] = j;
    int32_t *rec = stn.data() + (size_t)e * SREC;
    rec[rec_edge(0)] = e << 1;
    int k = 1;
    for (int q = 0; q < 2; ++q) {
      const int c = cell[q], n = d->v_nnb[c], i = slot[q];
      for (int t = 1; t < 6; ++t, ++k) {
        if (t >= n) continue;  // pentagon: one slot stays padded
        const int j = (i + t) % n;
        const int neg = d->hx_ttgout[MX * c + j] * d->hx_tnrccw[MX * c + i] < 0 ? 1 : 0;
        rec[rec_edge(k)] = (en[d->v_ed[MX * c + j] - 1] << 1) | neg;
      }
    }
    // cells: c1, c2, left apex, right apex, other ring cells of c1 and c2
    const double *p1 = d->v_p + 3 * cell[0], *p2 = d->v_p + 3 * cell[1];
    double nrm[3];
    imx::cross3(p1, p2, nrm);
    int apex[2] = {-1, -1};
    for (int q = 0; q < 2; ++q) {
      const int t = d->ed_sh[2 * eo + q] - 1;
      for (int l = 0; l < 3; ++l) {
        const int v = d->tr_v[3 * t + l] - 1;
        if (v != cell[0] && v != cell[1]) {
          if (imx::dot3(nrm, d->v_p + 3 * v) > 0) apex[0] = v;
          else apex[1] = v;
        }
      }
    }
    int cl[NSC];
    for (int q = 0; q < NSC; ++q) cl[q] = -1;
    cl[0] = cell[0];
    cl[1] = cell[1];
    cl[2] = apex[0];
    cl[3] = apex[1];
    int kc = 4;
    for (int q = 0; q < 2; ++q) {
      const int c = cell[q], n = d->v_nnb[c], i = slot[q];
      for (int t = 2; t <= 4; ++t, ++kc) {
        if (t > n - 2) continue;
        cl[kc] = d->v_nb[MX * c + (i + t) % n] - 1;
      }
    }
    for (int q = 0; q < NSC; ++q) rec[rec_cell(q)] = cl[q] >= 0 ? cn[cl[q]] << 1 : -1;
    const double z = d->ed_c[3 * eo + 2];
    const float geo[6] = {(float)z, (float)std::sqrt(std::max(0.0, 1 - z * z)),
                          (float)(d->ed_leng[eo] / ml), (float)(d->edhx_leng[eo] / md),
                          (float)(d->hx_areag[cell[0]] / ma), (float)(d->hx_areag[cell[1]] / ma)};
    for (int q = 0; q < 6; ++q) std::memcpy(rec + rec_geo(q), geo + q, 4);
    wv[e] = 1.f / (float)d->ne;
  }
  imx::Alloc &A = L->A;
  L->stn = A.put(stn);
  L->wv = A.put(wv);
  L->dc = A.put(dc);
  L->de = A.put(de);
  const size_t es = s->single ? 4 : 8;
  L->hn = A.get<char>(es * nv);
  L->un = A.get<char>(es * NE);
  L->raw = A.get<float>((size_t)NE * NF);
  L->mu = A.put(std::vector<float>(NF, 0.f));
  L->sig = A.put(std::vector<float>(NF, 1.f));
  {
    const std::vector<float> zero(NF, 0.f), one(NF, 1.f);
    L->norm = A.put(imx::learn_norm(zero.data(), one.data()));
  }
  L->hq = A.get<char>(es * nv);
  L->uq = A.get<char>(es * NE);
  L->Y = A.get<float>((size_t)2 * NE);
  L->dhc = A.get<float>(nv);
  L->th = A.get<float>(nv);
  L->part = A.get<double>(LPART);
  L->rms = A.get<double>(1);
  L->bound = A.put(std::vector<double>{1e300, (double)IMX_LIMIT_FALLBACK});
  L->lh = A.get<double>(kLossSteps);
  L->lossu = A.get<float>((size_t)kLossSteps * ((NE + 63) / 64));
  L->nfb = A.get<int>(1);
  if (A.err != hipSuccess) {
    int rc = imx::lfail(A.err, "imx_learn_create");
    imx_learn_destroy(L);
    return rc;
  }
  *out = L;
  return IMX_OK;
}

int imx_learn_sample(imx_learn *L, float *raw) {
  if (!L) return imx::set_error(IMX_EINVAL, "imx_learn_sample: NULL handle");
  int rc = imx::learn_sample(L);
  if (rc) return rc;
  if (raw) imx::learn_enqueue_featx(L, L->s->stream, L->raw, nullptr);
  LTRY(hipGetLastError(), "learn_featx");
  LTRY(hipStreamSynchronize(L->s->stream), "learn sample");
  if (raw) {  // caller edge order
    std::vector<float> b((size_t)L->NE * NF);
    LTRY(hipMemcpy(b.data(), L->raw, b.size() * 4, hipMemcpyDeviceToHost), "learn raw");
    for (int eo = 0; eo < L->s->ne; ++eo)
      std::memcpy(raw + (size_t)eo * NF, b.data() + (size_t)L->s->lay.edge_new[eo] * NF, NF * 4);
  }
  return IMX_OK;
}

int imx_learn_set_scaling(imx_learn *L, const float *mu, const float *sig, float tscale_u, float tscale_h) {
  if (!L || !mu || !sig || !(tscale_u > 0) || !(tscale_h > 0))
    return imx::set_error(IMX_EINVAL, "imx_learn_set_scaling: bad argument");
  for (int j = 0; j < NF; ++j)
    if (!(sig[j] > 0)) return imx::set_error(IMX_EINVAL, "imx_learn_set_scaling: sig must be positive");
  LTRY(hipMemcpy(L->mu, mu, NF * 4, hipMemcpyHostToDevice), "learn scaling");
  LTRY(hipMemcpy(L->sig, sig, NF * 4, hipMemcpyHostToDevice), "learn scaling");
  const std::vector<float> norm = imx::learn_norm(mu, sig);
  LTRY(hipMemcpy(L->norm, norm.data(), norm.size() * 4, hipMemcpyHostToDevice), "learn scaling");
  L->tsu = tscale_u;
  L->tsh = tscale_h;
  imx::learn_drop_graph(L);  // the scales are launch arguments of the graph
  return IMX_OK;
}

// Train on the features of the last imx_learn_sample against the targets
// du[ne], dh[nv] (caller numbering): `epochs` AdamW steps on all edges.
// loss[0] = mean_e (du_e - t_e)^2, loss[1] = mean_c ((D F)_c - t_c)^2 in
// the scaled units, before the last step.
int imx_learn_train(imx_learn *L, const double *du, const double *dh, int32_t epochs, float lr, float wd,
                    double *loss) {
  if (!L || !du || !dh || epochs < 1) return imx::set_error(IMX_EINVAL, "imx_learn_train: bad argument");
  imx_swm *s = L->s;
  imx_mlp *m = L->m;
  int rc = imx::mlp_reserve(m, L->NE);
  if (rc) return rc;
  const int NE = L->NE, nv = s->nv;
  imx::learn_enqueue_featx(L, s->stream, nullptr, m->X);
  LTRY(hipGetLastError(), "learn_featx");
  LTRY(hipStreamSynchronize(s->stream), "learn train");
  std::vector<float> T((size_t)2 * NE, 0.f), w(NE, 0.f), th(nv);
  for (int c = 0; c < nv; ++c) th[s->lay.cell_new[c]] = (float)(dh[c] * L->tsh);
  for (int eo = 0; eo < s->ne; ++eo) {
    const int e = s->lay.edge_new[eo];
    T[2 * e] = (float)(du[eo] * L->tsu);
    w[e] = 1.f / (float)s->ne;
  }
  hipStream_t st = m->stream;
  LTRY(hipMemcpyAsync(m->T, T.data(), T.size() * 4, hipMemcpyHostToDevice, st), "learn train");
  LTRY(hipMemcpyAsync(m->w, w.data(), w.size() * 4, hipMemcpyHostToDevice, st), "learn train");
  LTRY(hipMemcpyAsync(L->th, th.data(), th.size() * 4, hipMemcpyHostToDevice, st), "learn train");
  const int g = (NE + LTPB - 1) / LTPB, gc = (nv + LTPB - 1) / LTPB;
  double lu = 0.0;
  for (int k = 0; k < epochs; ++k) {
    const bool last = (k == epochs - 1);
    rc = imx::mlp_forward_dev(m, NE, m->X, L->Y, st);
    if (rc) return rc;
    learn_div<<<gc, LTPB, 0, st>>>(nv, s->c_nnb, s->c_ed, L->dc, L->Y, L->th, L->dhc);
    if (last) learn_norm2<<<1, 1024, 0, st>>>(0, nullptr, 1, nullptr, nv, L->dhc, 1.0 / nv, 0, L->lh);
    learn_divT<<<g, LTPB, 0, st>>>(NE, s->e_v, L->de, L->dhc, 2.f / (float)nv, m->T);
    LTRY(hipGetLastError(), "learn train");
    rc = imx::mlp_train_dev(m, NE, nullptr, lr, wd, 1, nullptr, 2);
    if (rc) return rc;
  }
  if ((rc = imx::mlp_loss(m, NE, nullptr, 1, &lu))) return rc;
  double lh = 0.0;
  LTRY(hipMemcpyAsync(&lh, L->lh, 8, hipMemcpyDeviceToHost, st), "learn train");
  LTRY(hipStreamSynchronize(st), "learn train");
  if (loss) {
    loss[0] = lu;
    loss[1] = lh;
  }
  return IMX_OK;
}

// nsteps corrected steps: plain RK4, then the MLP correction, scaled down
// to RMS `bound` (scaled units) where it exceeds it; *nlimited counts the
// scaled steps.
int imx_learn_set_limiter(imx_learn *L, int32_t mode) {
  if (!L || (mode != IMX_LIMIT_FALLBACK && mode != IMX_LIMIT_SCALE))
    return imx::set_error(IMX_EINVAL, "imx_learn_set_limiter: bad argument");
  const double m = (double)mode;
  LTRY(hipMemcpyAsync(L->bound + 1, &m, 8, hipMemcpyHostToDevice, L->s->stream), "imx_learn_set_limiter");
  LTRY(hipStreamSynchronize(L->s->stream), "imx_learn_set_limiter");
  return IMX_OK;
}

int imx_learn_prepare(imx_learn *L, int32_t nsteps, int32_t *made) {
  if (!L || nsteps < 0) return imx::set_error(IMX_EINVAL, "imx_learn_prepare: bad argument");
  return imx::learn_ensure_graphs(L, nsteps, made);
}

int imx_learn_step(imx_learn *L, int32_t nsteps, double bound, int32_t *nlimited) {
  if (!L || nsteps < 0) return imx::set_error(IMX_EINVAL, "imx_learn_step: bad argument");
  imx_swm *s = L->s;
  int rc = imx::learn_ensure_graphs(L, nsteps);
  if (rc) return rc;
  LTRY(hipMemcpyAsync(L->bound, &bound, 8, hipMemcpyHostToDevice, s->stream), "learn step");
  LTRY(hipMemsetAsync(L->nfb, 0, 4, s->stream), "learn step");
  LTRY(L->graphs.launch(nsteps, s->stream), "learn step");
  int nfb = 0;
  LTRY(hipMemcpyAsync(&nfb, L->nfb, 4, hipMemcpyDeviceToHost, s->stream), "learn step");
  rc = imx::swm_check_flag(s, "imx_learn_step");
  if (nlimited) *nlimited = nfb;
  return rc;
}

// Device sample store (capacity `cap` samples; existing samples dropped).
int imx_learn_reserve(imx_learn *L, int32_t cap) {
  if (!L || cap < 1) return imx::set_error(IMX_EINVAL, "imx_learn_reserve: bad argument");
  imx::learn_free_store(L);
  const int64_t npad = ((int64_t)L->NE + 63) / 64 * 64;
  L->xstride = npad * NF;
  LTRY(hipMalloc(&L->Xb, (size_t)cap * L->xstride * 2), "imx_learn_reserve");
  LTRY(hipMalloc(&L->tub, (size_t)cap * L->NE * 4), "imx_learn_reserve");
  LTRY(hipMalloc(&L->thb, (size_t)cap * L->nv * 4), "imx_learn_reserve");
  L->cap = cap;
  return IMX_OK;
}

// Store the last sample's normalised features with its targets du[ne],
// dh[nv] (caller numbering); the oldest sample is replaced when full.
int imx_learn_store(imx_learn *L, const double *du, const double *dh, int32_t *slot) {
  if (!L || !du || !dh) return imx::set_error(IMX_EINVAL, "imx_learn_store: bad argument");
  if (L->cap < 1) return imx::set_error(IMX_ESTATE, "imx_learn_store: no store (imx_learn_reserve)");
  imx_swm *s = L->s;
  const int k = L->count % L->cap;
  imx::learn_enqueue_featx(L, s->stream, nullptr, L->Xb + (size_t)k * L->xstride);
  LTRY(hipGetLastError(), "learn_featx");
  std::vector<float> tu(L->NE, 0.f), th(s->nv);
  for (int c = 0; c < s->nv; ++c) th[s->lay.cell_new[c]] = (float)(dh[c] * L->tsh);
  for (int eo = 0; eo < s->ne; ++eo) tu[s->lay.edge_new[eo]] = (float)(du[eo] * L->tsu);
  LTRY(hipMemcpyAsync(L->tub + (size_t)k * L->NE, tu.data(), tu.size() * 4, hipMemcpyHostToDevice,
                      s->stream), "imx_learn_store");
  LTRY(hipMemcpyAsync(L->thb + (size_t)k * s->nv, th.data(), th.size() * 4, hipMemcpyHostToDevice,
                      s->stream), "imx_learn_store");
  LTRY(hipStreamSynchronize(s->stream), "imx_learn_store");
  ++L->count;
  if (slot) *slot = k;
  return IMX_OK;
}

// nsteps AdamW steps, each on one stored sample drawn uniformly (SplitMix64
// from `seed`); the learning rate goes linearly from lr0 to lr1. loss[2]:
// mean scaled (u, h) losses over the last min(nsteps, 16) steps.
int imx_learn_fit(imx_learn *L, int32_t nsteps, float lr0, float lr1, float wd, uint64_t seed,
                  double loss[2]) {
  if (!L || nsteps < 1) return imx::set_error(IMX_EINVAL, "imx_learn_fit: bad argument");
  const int n = L->count < L->cap ? L->count : L->cap;
  if (n < 1) return imx::set_error(IMX_ESTATE, "imx_learn_fit: the store is empty");
  imx_swm *s = L->s;
  imx_mlp *m = L->m;
  int rc = imx::mlp_reserve(m, L->NE);
  if (rc) return rc;
  const int NE = L->NE, nv = s->nv;
  hipStream_t st = m->stream;
  LTRY(hipStreamSynchronize(s->stream), "imx_learn_fit");
  LTRY(hipMemcpyAsync(m->w, L->wv, (size_t)NE * 4, hipMemcpyDeviceToDevice, st), "imx_learn_fit");
  const int g = (NE + LTPB - 1) / LTPB, gc = (nv + LTPB - 1) / LTPB;
  const int tail = nsteps < kLossSteps ? nsteps : kLossSteps, nb = (NE + 63) / 64;
  uint64_t x = seed;
  for (int k = 0; k < nsteps; ++k) {
    x += 0x9E3779B97F4A7C15ull;  // SplitMix64
    uint64_t z = x;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    const int j = (int)(z % (uint64_t)n);
    const short *X = L->Xb + (size_t)j * L->xstride;
    const float lr = nsteps > 1 ? lr0 + (lr1 - lr0) * (float)k / (float)(nsteps - 1) : lr0;
    const bool last = k >= nsteps - tail;
    const int slot = k - (nsteps - tail);
    rc = imx::mlp_forward_dev(m, NE, X, L->Y, st);
    if (rc) return rc;
    learn_div<<<gc, LTPB, 0, st>>>(nv, s->c_nnb, s->c_ed, L->dc, L->Y, L->thb + (size_t)j * nv, L->dhc);
    if (last) learn_norm2<<<1, 1024, 0, st>>>(0, nullptr, 1, nullptr, nv, L->dhc, 1.0 / nv, 0, L->lh + slot);
    learn_targets<<<g, LTPB, 0, st>>>(NE, s->e_v, L->de, L->dhc, 2.f / (float)nv,
                                      L->tub + (size_t)j * NE, m->T);
    LTRY(hipGetLastError(), "imx_learn_fit");
    // the last steps' losses stay on the device until the end
    rc = imx::mlp_train_dev(m, NE, X, lr, wd, 1, last ? L->lossu + (size_t)slot * nb : nullptr, 2);
    if (rc) return rc;
  }
  double lu[kLossSteps], lh[kLossSteps];
  if ((rc = imx::mlp_loss(m, NE, L->lossu, tail, lu))) return rc;
  LTRY(hipMemcpy(lh, L->lh, tail * sizeof(double), hipMemcpyDeviceToHost), "imx_learn_fit");
  double su = 0.0, sh = 0.0;
  for (int k = 0; k < tail; ++k) {
    su += lu[k];
    sh += lh[k];
  }
  if (loss) {
    loss[0] = su / tail;
    loss[1] = sh / tail;
  }
  return IMX_OK;
}

int imx_learn_last_rms(imx_learn *L, double *rms) {
  if (!L || !rms) return imx::set_error(IMX_EINVAL, "imx_learn_last_rms: bad argument");
  LTRY(hipMemcpy(rms, L->rms, 8, hipMemcpyDeviceToHost), "learn rms");
  return IMX_OK;
}

void imx_learn_destroy(imx_learn *L) {
  if (!L) return;
  imx::learn_drop_graph(L);
  imx::learn_free_store(L);
  L->A.release();
  delete L;
}

}  // extern "C"
