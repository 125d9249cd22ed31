// bfa_assembly.hip -- CDNA4 kernels of the VIE assembly path and its C ABI.
//
// Cold (once per mesh): Taylor-Duffy moments of every tetrahedron pair with
// >= 2 shared vertices, then one 6-double static (FIBBI) record per touching
// BF pair.  Warm (per frequency): dense far-field Helmholtz cubature over
// the upper triangle, a sparse pass over touching pairs (desingularised
// kernel + static record + Gram/chi^-1 block) that overwrites those entries,
// RHS vectors and EMT power.
//
// Reference behaviour followed (HomerReid/buff-em):
//   AssembleVIEMatrix / AssembleGBlock / AssembleOverlapBlocks
//                                  src/libs/libbuff/VIEMatrix.cc:321-460
//   GetGMatrixElement, GMEIntegrand, GetExpRelTable
//                                  src/libs/libbuff/GMatrixElements.cc:59-424
//   BFBFInt/TetTetInt/TetInt fixed rules  src/libs/libbuff/Cubature.cc:161-527
//   GetOverlaps, Invert3x3Matrix   src/libs/libbuff/VIEMatrix.cc:51-72,122-316
//   TTaylorDuffy (static kernels)  src/libs/libTTaylorDuffy/TTaylorDuffy.cc:151-498
//   AssembleRHSVector              src/libs/libbuff/RHSVector.cc:62-124
//   GetEMTPFT                      src/libs/libbuff/EMTPFT.cc:85-546
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "bfa_internal.h"
#include "bfa_group.h"
#include "bfa_rules.h"
#include "bfa_expr.h"
#include "bfa_math.h"
#include "bfa_power.h"
#define TD_QUAL __constant__
#include "td_regions.h"

using namespace bfa;

#define ZVAC 376.73031346177
#define FOURPI 12.566370614359172954

#define HIPCHECK(call)                                                              \
  do {                                                                              \
    hipError_t e_ = (call);                                                         \
    if (e_ != hipSuccess)                                                           \
      return fail(e_ == hipErrorOutOfMemory ? BFA_ERR_OOM : BFA_ERR_HIP, "%s: %s (%s:%d)", \
                  #call, hipGetErrorString(e_), __FILE__, __LINE__);                \
  } while (0)

// ---------------------------------------------------------------------------
// small complex helpers
struct cd { double re, im; };
__device__ __forceinline__ cd cmul(cd a, cd b) { return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re}; }
__device__ __forceinline__ cd cadd(cd a, cd b) { return {a.re + b.re, a.im + b.im}; }
__device__ __forceinline__ cd cdiv(cd a, cd b)
{
  double d = b.re * b.re + b.im * b.im;
  return {(a.re * b.re + a.im * b.im) / d, (a.im * b.re - a.re * b.im) / d};
}
__device__ __forceinline__ cd cscale(cd a, double s) { return {a.re * s, a.im * s}; }

// ---------------------------------------------------------------------------
// device-memory helpers
static int dev_upload(void **dst, const void *src, size_t bytes)
{
  if (*dst) { hipFree(*dst); *dst = nullptr; }
  if (bytes == 0) return BFA_OK;
  HIPCHECK(hipMalloc(dst, bytes));
  HIPCHECK(hipMemcpy(*dst, src, bytes, hipMemcpyHostToDevice));
  return BFA_OK;
}

static void dev_free_all(bfa::DevBuffers &d)
{
  void **ptrs[] = {&d.V, &d.tetVI, &d.tetFI, &d.tetVol, &d.q4, &d.q16, &d.q33, &d.bfV, &d.bfT,
                   &d.bfPF, &d.bfQ, &d.bfRad, &d.rowptr, &d.cols, &d.pairRow, &d.ftTab, &d.tdPairs,
                   &d.tdVerts, &d.tdMom, &d.pairTD, &d.table, &d.tpTab, &d.gram};
  for (void **p : ptrs)
    if (*p) { hipFree(*p); *p = nullptr; }
  if (d.turnEv) { (void)hipEventDestroy((hipEvent_t)d.turnEv); d.turnEv = nullptr; }
  d.tpTabBytes = 0;
}

extern "C" void bfa_geometry_destroy(bfa_geometry *g)
{
  if (!g) return;
  if (g->uploaded) dev_free_all(g->d);
  delete g;
}

// tetrahedron centroids live after tetVol in one buffer: [nt] vol, [3nt] cen
extern "C" int bfa_geometry_upload(bfa_geometry *g, void *stream)
{
  (void)stream;
  if (!g) return fail(BFA_ERR_ARG, "null geometry");
  int dev = 0;
  HIPCHECK(hipGetDevice(&dev));
  g->device = dev;
  const int nt = g->nt, N = g->nbf;
  // cubature tables per tetrahedron (iQ = 0 vertex order)
  std::vector<double> q[3];
  const int rules[3] = {4, 16, 33};
  for (int r = 0; r < 3; r++) {
    double tab[33 * 4];
    int np = tet_rule(rules[r], tab);
    q[r].resize((size_t)nt * np * 4);
    for (int t = 0; t < nt; t++) {
      const int *vi = &g->tetVI[4 * t];
      const double *P0 = &g->V[3 * vi[0]];
      double L[3][3];
      for (int k = 0; k < 3; k++)
        for (int d = 0; d < 3; d++) L[k][d] = g->V[3 * vi[k + 1] + d] - P0[d];
      for (int i = 0; i < np; i++) {
        double *o = &q[r][((size_t)t * np + i) * 4];
        for (int d = 0; d < 3; d++)
          o[d] = P0[d] + tab[4 * i] * L[0][d] + tab[4 * i + 1] * L[1][d] + tab[4 * i + 2] * L[2][d];
        o[3] = 6.0 * g->tetVol[t] * tab[4 * i + 3];
      }
    }
  }
  std::vector<int> bfV(5 * (size_t)N), bfT(2 * (size_t)N), pairRow(g->cols.size());
  std::vector<double> bfPF(2 * (size_t)N), bfQ(6 * (size_t)N), volcen(4 * (size_t)nt);
  for (int a = 0; a < N; a++) {
    bfV[5 * a] = g->fQP[a]; bfV[5 * a + 1] = g->fV[3 * a]; bfV[5 * a + 2] = g->fV[3 * a + 1];
    bfV[5 * a + 3] = g->fV[3 * a + 2]; bfV[5 * a + 4] = g->fQM[a];
    bfT[2 * a] = g->fPT[a]; bfT[2 * a + 1] = g->fMT[a];
    bfPF[2 * a] = g->fArea[a] / (3.0 * g->tetVol[g->fPT[a]]);
    bfPF[2 * a + 1] = -g->fArea[a] / (3.0 * g->tetVol[g->fMT[a]]);
    for (int d = 0; d < 3; d++) {
      bfQ[6 * a + d] = g->V[3 * g->fQP[a] + d];
      bfQ[6 * a + 3 + d] = g->V[3 * g->fQM[a] + d];
    }
    for (int j = g->rowptr[a]; j < g->rowptr[a + 1]; j++) pairRow[j] = a;
  }
  // far-field tiles: distinct tetrahedra of each FT2-BF tile, in order of
  // first appearance, and the slot of every (BF, side) in that list
  const int nft = (N + FT2 - 1) / FT2;
  g->ft_max = 0;
  std::vector<int> ftTab((size_t)nft * FTAB, -1);
  for (int tile = 0; tile < nft; tile++) {
    int *row = &ftTab[(size_t)tile * FTAB];
    int n = 0;
    for (int k = 0; k < 2 * FT2; k++) {
      const int a = tile * FT2 + k / 2;
      if (a >= N) { row[2 * FT2 + k] = 0; continue; }
      const int t = bfT[2 * a + (k & 1)];
      int u = 0;
      while (u < n && row[u] != t) u++;
      if (u == n) row[n++] = t;
      row[2 * FT2 + k] = u;
    }
    row[4 * FT2] = n;
    g->ft_max = std::max(g->ft_max, n);
  }
  for (int t = 0; t < nt; t++) {
    volcen[t] = g->tetVol[t];
    for (int d = 0; d < 3; d++) volcen[nt + 3 * t + d] = g->tetCen[3 * t + d];
  }
  int rc;
  auto &d = g->d;
  if ((rc = dev_upload(&d.V, g->V.data(), g->V.size() * 8)) ||
      (rc = dev_upload(&d.tetVI, g->tetVI.data(), g->tetVI.size() * 4)) ||
      (rc = dev_upload(&d.tetFI, g->tetFI.data(), g->tetFI.size() * 4)) ||
      (rc = dev_upload(&d.tetVol, volcen.data(), volcen.size() * 8)) ||
      (rc = dev_upload(&d.q4, q[0].data(), q[0].size() * 8)) ||
      (rc = dev_upload(&d.q16, q[1].data(), q[1].size() * 8)) ||
      (rc = dev_upload(&d.q33, q[2].data(), q[2].size() * 8)) ||
      (rc = dev_upload(&d.bfV, bfV.data(), bfV.size() * 4)) ||
      (rc = dev_upload(&d.bfT, bfT.data(), bfT.size() * 4)) ||
      (rc = dev_upload(&d.bfPF, bfPF.data(), bfPF.size() * 8)) ||
      (rc = dev_upload(&d.bfQ, bfQ.data(), bfQ.size() * 8)) ||
      (rc = dev_upload(&d.bfRad, g->fRad.data(), (size_t)N * 8)) ||
      (rc = dev_upload(&d.rowptr, g->rowptr.data(), g->rowptr.size() * 4)) ||
      (rc = dev_upload(&d.cols, g->cols.data(), g->cols.size() * 4)) ||
      (rc = dev_upload(&d.pairRow, pairRow.data(), pairRow.size() * 4)) ||
      (rc = dev_upload(&d.ftTab, ftTab.data(), ftTab.size() * 4))) {
    dev_free_all(d);
    return rc;
  }
  if (d.gram) { hipFree(d.gram); d.gram = nullptr; }
  if (d.turnEv) { (void)hipEventDestroy((hipEvent_t)d.turnEv); d.turnEv = nullptr; }
  if (hipMalloc(&d.gram, (size_t)std::max(nt, 1) * 16 * sizeof(cd)) != hipSuccess ||
      hipEventCreateWithFlags((hipEvent_t *)&d.turnEv, hipEventDisableTiming) != hipSuccess) {
    dev_free_all(d);
    return fail(BFA_ERR_OOM, "bfa_geometry_upload: allocation");
  }
  DevGeom &dg = g->dg;
  dg.nv = g->nv; dg.nt = nt; dg.nbf = N; dg.nnz = (int64_t)g->cols.size();
  dg.V = (const double *)d.V; dg.tetVI = (const int *)d.tetVI; dg.tetFI = (const int *)d.tetFI;
  dg.tetVol = (const double *)d.tetVol;
  dg.q4 = (const double *)d.q4; dg.q16 = (const double *)d.q16; dg.q33 = (const double *)d.q33;
  dg.bfV = (const int *)d.bfV; dg.bfT = (const int *)d.bfT; dg.bfPF = (const double *)d.bfPF;
  dg.bfQ = (const double *)d.bfQ; dg.bfRad = (const double *)d.bfRad;
  dg.rowptr = (const int *)d.rowptr; dg.cols = (const int *)d.cols; dg.pairRow = (const int *)d.pairRow;
  dg.ftTab = (const int *)d.ftTab;
  g->uploaded = true;
  g->static_built = false;
  return BFA_OK;
}

// ===========================================================================
// Cold step 1: Taylor-Duffy moments.  One workgroup per tetrahedron pair.
// Per base simplex the displacement L and the radial coefficients X1 and
// Y1 = X1 + L (the columns of Mx and My that multiply the remaining variables
// belong to the common vertices) are affine in sigma; the radial and
// remaining-variable integrals are closed-form (Beta integrals, simplex
// covariance).  Bound by FP64 instructions.  The collapsed coordinates are
// t_d = g_0 g_1 ... g_d, so along the last one L = LA + g LB and
// X1 = XA + g XB: a thread takes one line of n nodes and sums f, f g and
// f g^2 for f = w/r and w r (w alone gives constants), about 25 instructions a
// node, and turns them into the 24 moments once a line (~150).  Point by
// point, with the barycentric coordinates read from a table, a node took ~115
// and the pairs of a 3,072-tetrahedron ball (order 12) 20.5 ms; now 7.6 ms,
// what the FP64 instructions of 7.7e9 nodes take to issue.
// ===========================================================================
#define TD_MAXORDER 32
struct TDNodes {          // Gauss nodes and weights on [0, 1] for 4, 3, 2 common vertices
  double x[3][TD_MAXORDER], w[3][TD_MAXORDER];
  int n[3];
};
struct TDShared {
  double E[20][5][6];     // per simplex: L, X1 at vertex 0, then the edges between successive vertices
  double det[20];
  double red[4 * 24];
  double x[TD_MAXORDER], w[TD_MAXORDER], wx[TD_MAXORDER], wxx[TD_MAXORDER], ww[3];
  double Mx[3][3], My[3][3], cov[3][3], tbar[3], tot[24];
};

template <int NCV> struct TDCase;
template <> struct TDCase<4> {
  static constexpr int D = 3, M = 3, NSIMP = TD4_NSIMP;
  __device__ static const double *simp(int s) { return &TD4_SIMP_V[s][0][0]; }
  __device__ static const double *off(int s) { return &TD4_OFFSET[TD4_SIMP_PAT[s]][0][0]; }
  __device__ static double det(int s) { return TD4_SIMP_DET[s]; }
};
template <> struct TDCase<3> {
  static constexpr int D = 4, M = 2, NSIMP = TD3_NSIMP;
  __device__ static const double *simp(int s) { return &TD3_SIMP_V[s][0][0]; }
  __device__ static const double *off(int s) { return &TD3_OFFSET[TD3_SIMP_PAT[s]][0][0]; }
  __device__ static double det(int s) { return TD3_SIMP_DET[s]; }
};
template <> struct TDCase<2> {
  static constexpr int D = 5, M = 1, NSIMP = TD2_NSIMP;
  __device__ static const double *simp(int s) { return &TD2_SIMP_V[s][0][0]; }
  __device__ static const double *off(int s) { return &TD2_OFFSET[TD2_SIMP_PAT[s]][0][0]; }
  __device__ static double det(int s) { return TD2_SIMP_DET[s]; }
};

// xs = Sx s, es = Se s for each case (x' - x = My es - Mx xs)
template <int NCV> __device__ __forceinline__ void td_split(const double *s, double *xs, double *es)
{
  if (NCV == 4) { xs[0] = xs[1] = xs[2] = 0.0; es[0] = s[0]; es[1] = s[1]; es[2] = s[2]; }
  else if (NCV == 3) { xs[0] = 0.0; xs[1] = 0.0; xs[2] = s[2]; es[0] = s[0]; es[1] = s[1]; es[2] = s[3]; }
  else { xs[0] = 0.0; xs[1] = s[1]; xs[2] = s[2]; es[0] = s[0]; es[1] = s[3]; es[2] = s[4]; }
}

__device__ __forceinline__ double beta_int(int a, int b)
{
  double r = 1.0;
  for (int i = 1; i <= b; i++) r *= (double)i / (double)(a + i);
  return r / (a + b + 1);
}

__device__ __forceinline__ double wave_sum(double v)
{
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  return v;
}

template <int NCV>
__device__ void td_pair(const double *VA, const double *VB, const double *cA, const double *cB, const TDNodes &td,
                        int ic, double *out, TDShared &sh)
{
  using C = TDCase<NCV>;
  constexpr int D = C::D, M = C::M, K = D - 1;
  static_assert(C::NSIMP <= 20 && D <= 5, "TDShared");
  const int n = td.n[ic];
  const int tid = threadIdx.x;
  double Mx[3][3], My[3][3];
  for (int d = 0; d < 3; d++) {
    Mx[d][0] = VA[3 + d] - VA[d]; Mx[d][1] = VA[6 + d] - VA[3 + d]; Mx[d][2] = VA[9 + d] - VA[6 + d];
    My[d][0] = VB[3 + d] - VB[d]; My[d][1] = VB[6 + d] - VB[3 + d]; My[d][2] = VB[9 + d] - VB[6 + d];
  }
  // remaining-variable simplex statistics (degree-2 exact rule)
  double tbar[3] = {0, 0, 0}, cov[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}}, vol = 0.0;
  {
    double tau[4][3], tw[4];
    int nt;
    if (M == 3) {
      const double a = 0.58541019662496845446, b = 0.13819660112501051518;
      const double Nv[4][3] = {{0, 0, 0}, {1, 0, 0}, {1, 1, 0}, {1, 1, 1}};
      for (int i = 0; i < 4; i++) {
        for (int d = 0; d < 3; d++) {
          double s = 0.0;
          for (int j = 0; j < 4; j++) s += (i == j ? a : b) * Nv[j][d];
          tau[i][d] = s;
        }
        tw[i] = 1.0 / 24.0;
      }
      nt = 4;
    } else if (M == 2) {
      const double Nv[3][2] = {{0, 0}, {1, 0}, {1, 1}};
      for (int i = 0; i < 3; i++) {
        for (int d = 0; d < 2; d++) {
          double s = 0.0;
          for (int j = 0; j < 3; j++) s += (i == j ? 2.0 / 3.0 : 1.0 / 6.0) * Nv[j][d];
          tau[i][d] = s;
        }
        tau[i][2] = 0.0;
        tw[i] = 1.0 / 6.0;
      }
      nt = 3;
    } else {
      tau[0][0] = 0.5 - 0.5 / sqrt(3.0); tw[0] = 0.5;
      tau[1][0] = 0.5 + 0.5 / sqrt(3.0); tw[1] = 0.5;
      nt = 2;
    }
    for (int i = 0; i < nt; i++) {
      vol += tw[i];
      for (int a = 0; a < M; a++) tbar[a] += tw[i] * tau[i][a];
    }
    for (int a = 0; a < M; a++) tbar[a] /= vol;
    for (int i = 0; i < nt; i++)
      for (int a = 0; a < M; a++)
        for (int b = 0; b < M; b++) cov[a][b] += tw[i] * (tau[i][a] - tbar[a]) * (tau[i][b] - tbar[b]) / vol;
  }
  if (tid < n) {
    const double x = td.x[ic][tid], w = td.w[ic][tid];
    sh.x[tid] = x;
    sh.w[tid] = w;
    sh.wx[tid] = w * x;
    sh.wxx[tid] = w * x * x;
  }
  if (tid < C::NSIMP) sh.det[tid] = C::det(tid);
  if (tid == 0) {   // for the last step: not held in registers over the loop
    for (int d = 0; d < 3; d++) {
      sh.tbar[d] = tbar[d];
      for (int c = 0; c < 3; c++) { sh.Mx[d][c] = Mx[d][c]; sh.My[d][c] = My[d][c]; sh.cov[d][c] = cov[d][c]; }
    }
  }
  // rem -> physical maps: the first M columns of Mx / My
  if (tid < C::NSIMP * D) {
    const int is = tid / D, q = tid % D;
    const double *sv = C::simp(is), *O = C::off(is);
    double v[2][6];
    for (int e = 0; e < 2; e++) {
      const double *s = sv + (q > 0 ? q - 1 + e : 0) * D;
      double rem[3], xs[3], es[3];
      for (int a = 0; a < M; a++) {
        double o = 0.0;
        for (int d = 0; d < D; d++) o += O[a * D + d] * s[d];
        rem[a] = o - tbar[a];
      }
      td_split<NCV>(s, xs, es);
      for (int d = 0; d < 3; d++) {
        double l = 0, x1 = 0;
        for (int c = 0; c < 3; c++) {
          l += My[d][c] * es[c] - Mx[d][c] * xs[c];
          x1 += Mx[d][c] * xs[c];
        }
        for (int a = 0; a < M; a++) x1 += Mx[d][a] * rem[a];
        v[e][d] = l; v[e][3 + d] = x1;
      }
    }
    for (int d = 0; d < 6; d++) sh.E[is][q][d] = q > 0 ? v[1][d] - v[0][d] : v[0][d];
  }
  __syncthreads();
  if (tid < 3) {
    double c = 0.0;
    for (int i = 0; i < n; i++) c += tid == 0 ? sh.w[i] : tid == 1 ? sh.wx[i] : sh.wxx[i];
    sh.ww[tid] = c;
  }
  __syncthreads();
  double acc[3][8];
#pragma unroll
  for (int p = 0; p < 3; p++)
#pragma unroll
    for (int q = 0; q < 8; q++) acc[p][q] = 0.0;
  unsigned nl = 1;
  for (int d = 0; d < K - 1; d++) nl *= n;
  for (unsigned task = tid; task < C::NSIMP * nl; task += 256) {
    const unsigned is = task / nl;
    unsigned ri = task - is * nl;
    const double *E = &sh.E[is][0][0];
    double LX[6], LXg[6];
#pragma unroll
    for (int d = 0; d < 6; d++) LX[d] = E[d];
    double W = sh.det[is], t = 1.0;
#pragma unroll
    for (int d = 0; d < K - 1; d++) {
      const unsigned rn = ri / n, id = ri - rn * n;
      ri = rn;
      const double v = sh.x[id];
      t *= v;
      W *= sh.w[id];
#pragma unroll
      for (int e = 0; e < K - 1 - d; e++) W *= v;
#pragma unroll
      for (int c = 0; c < 6; c++) LX[c] += t * E[6 * (d + 1) + c];
    }
#pragma unroll
    for (int c = 0; c < 6; c++) LXg[c] = t * E[6 * K + c];
    double s[3][3] = {};
#pragma unroll 2
    for (int i = 0; i < n; i++) {
      const double gx = sh.x[i], w0 = sh.w[i], w1 = sh.wx[i], w2 = sh.wxx[i];
      const double L0 = LX[0] + gx * LXg[0], L1 = LX[1] + gx * LXg[1], L2 = LX[2] + gx * LXg[2];
      const double r2 = L0 * L0 + L1 * L1 + L2 * L2;
      const double f0 = rsqrt_nr(r2), f2 = f0 * r2;
      s[0][0] += w0 * f0; s[0][1] += w1 * f0; s[0][2] += w2 * f0;
      s[2][0] += w0 * f2; s[2][1] += w1 * f2; s[2][2] += w2 * f2;
    }
#pragma unroll
    for (int q = 0; q < 3; q++) s[1][q] = sh.ww[q];
    const double *XA = LX + 3, *XB = LXg + 3;
    double YA[3], YB[3], aa = 0, ab = 0, bb = 0;
#pragma unroll
    for (int d = 0; d < 3; d++) {
      YA[d] = XA[d] + LX[d]; YB[d] = XB[d] + LXg[d];
      aa += XA[d] * YA[d];
      ab += XA[d] * YB[d] + XB[d] * YA[d];
      bb += XB[d] * YB[d];
    }
#pragma unroll
    for (int p = 0; p < 3; p++) {
      const double m0 = W * s[p][0], m1 = W * s[p][1], m2 = W * s[p][2];
      acc[p][0] += m0;
#pragma unroll
      for (int d = 0; d < 3; d++) {
        acc[p][1 + d] += m0 * XA[d] + m1 * XB[d];
        acc[p][4 + d] += m0 * YA[d] + m1 * YB[d];
      }
      acc[p][7] += m0 * aa + m1 * ab + m2 * bb;
    }
  }
  // block reduction of the 24 accumulators
  double *red = sh.red;
  const int lane = tid & 63, wid = tid >> 6, nw = blockDim.x >> 6;
#pragma unroll
  for (int p = 0; p < 3; p++)
#pragma unroll
    for (int q = 0; q < 8; q++) {
      double v = wave_sum(acc[p][q]);
      if (lane == 0) red[wid * 24 + p * 8 + q] = v;
    }
  __syncthreads();
  if (tid < 24) {
    double v = 0.0;
    for (int w = 0; w < nw; w++) v += red[w * 24 + tid];
    sh.tot[tid] = v;
  }
  __syncthreads();
  if (tid < 3) {   // one kernel power each
    const int p = tid;
    const double *tot = sh.tot + 8 * p;
    const auto &Mx = sh.Mx, &My = sh.My, &cov = sh.cov;
    const auto &tbar = sh.tbar;
    double detA = Mx[0][0] * (Mx[1][1] * Mx[2][2] - Mx[2][1] * Mx[1][2])
                - Mx[0][1] * (Mx[1][0] * Mx[2][2] - Mx[2][0] * Mx[1][2])
                + Mx[0][2] * (Mx[1][0] * Mx[2][1] - Mx[2][0] * Mx[1][1]);
    double detB = My[0][0] * (My[1][1] * My[2][2] - My[2][1] * My[1][2])
                - My[0][1] * (My[1][0] * My[2][2] - My[2][0] * My[1][2])
                + My[0][2] * (My[1][0] * My[2][1] - My[2][0] * My[1][1]);
    double jac = fabs(detA) * fabs(detB);
    double X0[3], Y0[3], kappa = 0.0;
    for (int d = 0; d < 3; d++) {
      X0[d] = VA[d] - cA[d]; Y0[d] = VB[d] - cB[d];
      for (int a = 0; a < M; a++) { X0[d] += Mx[d][a] * tbar[a]; Y0[d] += My[d][a] * tbar[a]; }
    }
    for (int a = 0; a < M; a++)
      for (int b = 0; b < M; b++)
        kappa += cov[a][b] * (Mx[0][a] * My[0][b] + Mx[1][a] * My[1][b] + Mx[2][a] * My[2][b]);
    double s0 = jac * vol;
    {
      double b0 = beta_int(D - 2 + p, M), b1 = beta_int(D - 1 + p, M), b2 = beta_int(D + p, M);
      double bk = beta_int(D - 2 + p, M + 2);
      double a0 = tot[0];
      out[p * 8] = s0 * b0 * a0;
      for (int d = 0; d < 3; d++) {
        out[p * 8 + 1 + d] = s0 * (b0 * X0[d] * a0 + b1 * tot[1 + d]);
        out[p * 8 + 4 + d] = s0 * (b0 * Y0[d] * a0 + b1 * tot[4 + d]);
      }
      double x0y0 = X0[0] * Y0[0] + X0[1] * Y0[1] + X0[2] * Y0[2];
      double cross = X0[0] * tot[4] + X0[1] * tot[5] + X0[2] * tot[6]
                   + Y0[0] * tot[1] + Y0[1] * tot[2] + Y0[2] * tot[3];
      out[p * 8 + 7] = s0 * (b0 * x0y0 * a0 + b1 * cross + b2 * tot[7] + bk * kappa * a0);
    }
  }
}

__global__ __launch_bounds__(256) void k_td_moments(const int *pairs, const double *verts,
                                                    const double *tetCen, TDNodes td, double *mom)
{
  __shared__ TDShared sh;
  const int p = blockIdx.x;
  const int tA = pairs[4 * p], tB = pairs[4 * p + 1], ncv = pairs[4 * p + 2];
  const double *VA = verts + 24 * (size_t)p, *VB = VA + 12;
  const double *cA = tetCen + 3 * tA, *cB = tetCen + 3 * tB;
  double *out = mom + 24 * (size_t)p;
  if (ncv == 4) td_pair<4>(VA, VB, cA, cB, td, 0, out, sh);
  else if (ncv == 3) td_pair<3>(VA, VB, cA, cB, td, 1, out, sh);
  else td_pair<2>(VA, VB, cA, cB, td, 2, out, sh);
}

// ---------------------------------------------------------------------------
// Cold step 2: FIBBI record per touching pair (GetGME_TetTetInt with the
// static kernel, GMatrixElements.cc:295-375).
__global__ __launch_bounds__(256) void k_fibbi(DevGeom g, const int *tdPairs, const double *tdMom,
                                               const int *pairTD, double *table)
{
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= g.nnz) return;
  const int a = g.pairRow[j], b = g.cols[j];
  const double *tetCen = g.tetVol + g.nt;
  double G[6] = {0, 0, 0, 0, 0, 0};
  const double inv4pi = 1.0 / FOURPI, inv8pi = 0.5 / FOURPI;
  for (int sa = 0; sa < 2; sa++)
    for (int sb = 0; sb < 2; sb++) {
      const int ta = g.bfT[2 * a + sa], tb = g.bfT[2 * b + sb];
      const double pfa = g.bfPF[2 * a + sa], pfb = g.bfPF[2 * b + sb];
      const double *Qa = g.bfQ + 6 * a + 3 * sa, *Qb = g.bfQ + 6 * b + 3 * sb;
      const int code = pairTD[4 * j + 2 * sa + sb];
      if (code < 0) {
        // 16 x 16 point product rule, static kernels r^-1, r^0, r^1
        const double dd = 9.0 * pfa * pfb;
        const double *qa = g.q16 + (size_t)ta * 64, *qb = g.q16 + (size_t)tb * 64;
        for (int i = 0; i < 16; i++) {
          const double xa0 = qa[4 * i], xa1 = qa[4 * i + 1], xa2 = qa[4 * i + 2], wa = qa[4 * i + 3];
          const double ba0 = pfa * (xa0 - Qa[0]), ba1 = pfa * (xa1 - Qa[1]), ba2 = pfa * (xa2 - Qa[2]);
          for (int k = 0; k < 16; k++) {
            const double xb0 = qb[4 * k], xb1 = qb[4 * k + 1], xb2 = qb[4 * k + 2], wb = qb[4 * k + 3];
            const double R0 = xa0 - xb0, R1 = xa1 - xb1, R2 = xa2 - xb2;
            const double r = sqrt(R0 * R0 + R1 * R1 + R2 * R2);
            if (r < 1.0e-12) continue;
            const double dot = ba0 * pfb * (xb0 - Qb[0]) + ba1 * pfb * (xb1 - Qb[1]) + ba2 * pfb * (xb2 - Qb[2]);
            const double ww = wa * wb;
            const double r0 = inv4pi / r, r2 = r * inv8pi;
            G[0] += ww * r0 * dot; G[1] += ww * r0 * dd;
            G[2] += ww * inv4pi * dot; G[3] += ww * inv4pi * dd;
            G[4] += ww * r2 * dot; G[5] += ww * r2 * dd;
          }
        }
      } else {
        const int idx = code >> 1, sw = code & 1;
        const double *Mm = tdMom + 24 * (size_t)idx;
        const int tA = tdPairs[4 * idx], tB = tdPairs[4 * idx + 1];
        const int ox = sw ? 4 : 1, oy = sw ? 1 : 4;       // moment slots of ta / tb
        const double *cx = tetCen + 3 * (sw ? tB : tA), *cy = tetCen + 3 * (sw ? tA : tB);
        double dA[3], dB[3];
        for (int d = 0; d < 3; d++) { dA[d] = cx[d] - Qa[d]; dB[d] = cy[d] - Qb[d]; }
        const double ua = g.tetVol[ta] < 0.0 ? -pfa : pfa, ub = g.tetVol[tb] < 0.0 ? -pfb : pfb;
        const double gpre[3] = {inv4pi, inv4pi, inv8pi};
        for (int p = 0; p < 3; p++) {
          const double *Mp = Mm + 8 * p;
          double bb = Mp[7] + dA[0] * Mp[oy] + dA[1] * Mp[oy + 1] + dA[2] * Mp[oy + 2]
                    + dB[0] * Mp[ox] + dB[1] * Mp[ox + 1] + dB[2] * Mp[ox + 2]
                    + (dA[0] * dB[0] + dA[1] * dB[1] + dA[2] * dB[2]) * Mp[0];
          G[2 * p] += gpre[p] * ua * ub * bb;
          G[2 * p + 1] += gpre[p] * 9.0 * ua * ub * Mp[0];
        }
      }
    }
  for (int i = 0; i < 6; i++) table[6 * j + i] = G[i];
}

extern "C" int bfa_static_build(bfa_geometry *g, int td_order, void *stream)
{
  if (!g || !g->uploaded) return fail(BFA_ERR_STATE, "bfa_static_build: geometry not uploaded");
  hipStream_t st = (hipStream_t)stream;
  if (td_order <= 0) td_order = 12;
  if (td_order > 28) return fail(BFA_ERR_ARG, "td_order %d too large (max 28)", td_order);
  auto &d = g->d;
  const size_t ntd = g->tdA.size();
  int rc;
  // Taylor-Duffy inputs
  std::vector<int> pairs(4 * ntd);
  std::vector<double> verts(24 * ntd);
  for (size_t p = 0; p < ntd; p++) {
    pairs[4 * p] = g->tdA[p]; pairs[4 * p + 1] = g->tdB[p]; pairs[4 * p + 2] = g->tdNcv[p]; pairs[4 * p + 3] = 0;
    for (int q = 0; q < 8; q++)
      for (int c = 0; c < 3; c++) verts[24 * p + 3 * q + c] = g->V[3 * g->tdOV[8 * p + q] + c];
  }
  if ((rc = dev_upload(&d.tdPairs, pairs.data(), pairs.size() * 4)) ||
      (rc = dev_upload(&d.tdVerts, verts.data(), verts.size() * 8)) ||
      (rc = dev_upload(&d.pairTD, g->pairTD.data(), g->pairTD.size() * 4)))
    return rc;
  const int orders[3] = {std::min(td_order + 4, TD_MAXORDER), std::min(td_order + 2, TD_MAXORDER), td_order};
  TDNodes td;
  for (int c = 0; c < 3; c++) {
    td.n[c] = orders[c];
    gauss01(orders[c], td.x[c], td.w[c]);
  }
  if (d.tdMom) hipFree(d.tdMom);
  d.tdMom = nullptr;
  if (d.table) hipFree(d.table);
  d.table = nullptr;
  hipError_t e1 = hipMalloc(&d.tdMom, std::max<size_t>(ntd, 1) * 24 * 8);
  hipError_t e2 = hipMalloc(&d.table, std::max<int64_t>(g->dg.nnz, 1) * 6 * 8);
  if (e1 != hipSuccess || e2 != hipSuccess) return fail(BFA_ERR_OOM, "bfa_static_build: allocation failed");
  if (ntd > 0)
    hipLaunchKernelGGL(k_td_moments, dim3((unsigned)ntd), dim3(256), 0, st, (const int *)d.tdPairs,
                       (const double *)d.tdVerts, g->dg.tetVol + g->nt, td, (double *)d.tdMom);
  const int64_t nnz = g->dg.nnz;
  if (nnz > 0)
    hipLaunchKernelGGL(k_fibbi, dim3((unsigned)((nnz + 255) / 256)), dim3(256), 0, st, g->dg,
                       (const int *)d.tdPairs, (const double *)d.tdMom, (const int *)d.pairTD,
                       (double *)d.table);
  hipError_t e3 = hipGetLastError();
  hipError_t e4 = hipStreamSynchronize(st);
  if (e3 != hipSuccess || e4 != hipSuccess)
    return fail(BFA_ERR_HIP, "static build kernels failed: %s", hipGetErrorString(e3 != hipSuccess ? e3 : e4));
  g->static_built = true;
  g->td_order = td_order;
  return BFA_OK;
}

// static records supplied by the caller (nnz x 6, CSR order), e.g. from a
// FIBBI cache file; replaces any table built before
extern "C" int bfa_static_upload(bfa_geometry *g, const double *table)
{
  if (!g || !g->uploaded) return fail(BFA_ERR_STATE, "bfa_static_upload: geometry not uploaded");
  if (!table) return fail(BFA_ERR_ARG, "bfa_static_upload: null table");
  int rc = dev_upload(&g->d.table, table, (size_t)std::max<int64_t>(g->dg.nnz, 1) * 6 * 8);
  if (rc) return rc;
  g->static_built = true;
  return BFA_OK;
}

extern "C" int bfa_static_download(const bfa_geometry *g, double *table)
{
  if (!g || !g->static_built) return fail(BFA_ERR_STATE, "static table not built");
  if (!table) return fail(BFA_ERR_ARG, "null table");
  HIPCHECK(hipMemcpy(table, g->d.table, (size_t)g->dg.nnz * 6 * 8, hipMemcpyDeviceToHost));
  return BFA_OK;
}

// ===========================================================================
// Warm step: dense far field over the upper triangle (touching pairs are
// skipped: the sparse near-field pass writes them), from tetrahedron-pair
// moments; the precision form evaluates the kernel of those moments with
// its rounding-sensitive part in FP32 (tp_moments_split).
// ===========================================================================

__device__ __forceinline__ int bf_ncv(const int *va, const int *vb)
{
  int n = 0;
#pragma unroll
  for (int i = 0; i < 5; i++)
#pragma unroll
    for (int j = 0; j < 5; j++) n += (va[i] == vb[j]);
  return n;
}

// point data of BF a: 8 points (P-tet 4, M-tet 4) x {x,y,z, wbx,wby,wbz, wdiv}
__device__ __forceinline__ void bf_points4(const DevGeom &g, int a, int pt, double *o)
{
  const int side = pt >> 2, i = pt & 3;
  const int t = g.bfT[2 * a + side];
  const double *q = g.q4 + ((size_t)t * 4 + i) * 4;
  const double pf = g.bfPF[2 * a + side];
  const double *Q = g.bfQ + 6 * a + 3 * side;
  const double w = q[3];
  o[0] = q[0]; o[1] = q[1]; o[2] = q[2];
  o[3] = w * pf * (q[0] - Q[0]); o[4] = w * pf * (q[1] - Q[1]); o[5] = w * pf * (q[2] - Q[2]);
  o[6] = 3.0 * w * pf;
}

__device__ __forceinline__ void tile_coords(int64_t bid, int ntiles, int &ti, int &tj)
{
  // upper-triangular tile enumeration: row ti has (ntiles - ti) tiles
  double n = ntiles;
  int r = (int)floor(((2.0 * n + 1.0) - sqrt((2.0 * n + 1.0) * (2.0 * n + 1.0) - 8.0 * (double)bid)) / 2.0);
  if (r < 0) r = 0;
  auto start = [ntiles](int64_t row) { return row * ntiles - row * (row - 1) / 2; };
  while (r > 0 && start(r) > bid) r--;
  while (start(r + 1) <= bid) r++;
  ti = r;
  tj = r + (int)(bid - start(r));
}

// Tetrahedron-pair form of the far field.  Consecutive BFs share
// tetrahedra, so a 32 x 32 BF tile touches ~31 x 31 distinct tetrahedron
// pairs instead of 4 x 1024.  Per tetrahedron pair (S, T) the 4-point rule's
// moments about the centroids cS, cT (signed weights w = 6 V w_rule):
//   I0 = sum w w' g, Ix = sum w w' g (x - cS), Iy = sum w w' g (y - cT),
//   Ixy = sum w w' g (x - cS).(y - cT),   g = exp(ikr) / r,
// then per BF pair and side combination, with a = Q_a - cS, b = Q_b - cT:
//   sum w w' g b_a.b_b - div div/k^2 = pf_a pf_b [Ixy - b.Ix - a.Iy + (a.b) I0 - 9 I0/k^2]
// -- the same 64-point sum as GetGME_BFBFInt's fixed rule, regrouped.
#define FTT_MAX 1024   // tetrahedron pairs whose moments fit in LDS (larger tiles: direct path)
#define FT_THREADS 512

// Structure-of-arrays so that lanes on consecutive tetrahedra hit
// consecutive LDS banks.
struct FarTpShared {
  double mom[16][FTT_MAX];       // per tetrahedron pair: I0, Ix, Iy, Ixy (re, im)
  double pts[2][16][2 * FT2];    // [row/col][point*4 + {x,y,z,w}][distinct tet]
  double cen[2][3][2 * FT2];
  int slot[2][2 * FT2];          // (BF local * 2 + side) -> distinct tet
};

// 4-point product-rule moments of one tetrahedron pair (signed weights):
// row tetrahedron us of the tile (points in sh), column tetrahedron's points
// ys and centroid cT in registers; out[i * stride] for i < 16
// one point pair (x, y) of tp_moments: g(|x - y|) times the quadrature
// weights, accumulated into the 16 moments
template <bool REALK>
__device__ __forceinline__ void tp_point_pair(const double *x, const double *y, double xi0, double xi1, double xi2,
                                              const double *cT, double kre, double kim, double *m)
{
  const double R0 = x[0] - y[0], R1 = x[1] - y[1], R2 = x[2] - y[2];
  const double r2 = R0 * R0 + R1 * R1 + R2 * R2, ir = rsqrt_nr(r2), r = r2 * ir;
  double sn, co;
  sincos_mod(kre * r, &sn, &co);
  double amp = x[3] * y[3] * ir;
  if (!REALK) amp *= exp(-kim * r);
  const double gr = amp * co, gi = amp * sn;
  const double e0 = y[0] - cT[0], e1 = y[1] - cT[1], e2 = y[2] - cT[2];
  const double xy = xi0 * e0 + xi1 * e1 + xi2 * e2;
  m[0] += gr; m[1] += gi;
  m[2] += gr * xi0; m[3] += gi * xi0; m[4] += gr * xi1; m[5] += gi * xi1; m[6] += gr * xi2; m[7] += gi * xi2;
  m[8] += gr * e0; m[9] += gi * e0; m[10] += gr * e1; m[11] += gi * e1; m[12] += gr * e2; m[13] += gi * e2;
  m[14] += gr * xy; m[15] += gi * xy;
}

// LDSY: the column tetrahedron's points are read from LDS (pts[1][.][ut])
// two points at a time instead of from ys, which keeps the table kernel at
// four waves per SIMD instead of three; the single-pass kernel keeps ys (with
// LDSY it would spill).  The arithmetic
// and its order are the same either way; the time did not change
// measurably (the kernel is bound by its FP64 arithmetic).
template <bool REALK, bool LDSY = false, typename SH>
__device__ __forceinline__ void tp_moments(const SH &sh, int us, int ut, const double *cS, const double *ys,
                                           const double *cT, double kre, double kim, double *out, int stride)
{
  double m[16];
#pragma unroll
  for (int i = 0; i < 16; i++) m[i] = 0.0;
#pragma unroll 1
  for (int p = 0; p < 4; p++) {
    // row tetrahedron's point p read from LDS: a register array indexed by
    // this rolled loop's counter would be placed in scratch memory
    double x[4];
#pragma unroll
    for (int e = 0; e < 4; e++) x[e] = sh.pts[0][4 * p + e][us];
    const double xi0 = x[0] - cS[0], xi1 = x[1] - cS[1], xi2 = x[2] - cS[2];
    if constexpr (LDSY) {
#pragma unroll 2
      for (int q = 0; q < 4; q++) {
        double y[4];
#pragma unroll
        for (int e = 0; e < 4; e++) y[e] = sh.pts[1][4 * q + e][ut];
        tp_point_pair<REALK>(x, y, xi0, xi1, xi2, cT, kre, kim, m);
      }
    } else {
#pragma unroll
      for (int q = 0; q < 4; q++) tp_point_pair<REALK>(x, ys + 4 * q, xi0, xi1, xi2, cT, kre, kim, m);
    }
  }
#pragma unroll
  for (int i = 0; i < 16; i++) out[i * stride] = m[i];
}

// The far-field kernel with its point evaluations in FP32 (the precision
// form).  Plain FP32 evaluation of g at each point pair misses 1e-8 in the
// powers by ~40x: the scalar-potential term of a BF pair is a second
// difference of g over its four tetrahedron pairs, (h/D)^2 of the terms it
// sums, so the terms' 6e-8 relative rounding reaches the result amplified.
// Split instead, about the centroid separation d = cS - cT (length D,
// direction e), with w = (x - cS) - (y - cT), p = e.w, s = |w|^2 - p^2:
//   g(|d + w|) = g(D) [T2 + E3],
//   T2 = 1 + c1 (p + s / 2D) + c2 p^2 / 2,  c1 = ik - 1/D,  c2 = c1^2 + 1/D^2,
// the second-order Taylor part (FP64: one complex exponential per
// tetrahedron pair, a polynomial per point pair), and E3, the remainder of
// third order in |w| / D, evaluated in FP32 from formulas in which no two
// large terms cancel, so that its rounding error stays relative to itself:
//   r = sqrt((D + p)^2 + |w - p e|^2),  e1 = |w - p e|^2 / (D + p + r),
//   Delta = r - D = p + e1,  u = Delta / D,  x = ik Delta,
//   X3 = e^x - 1 - x - x^2/2 (its series for |x| <= 1),  U3 = u^3 / (1 + u),
//   R3 = X3 / (1 + u) - (1 + x + x^2/2) U3 + x u^2 + x^2 u (u - 1) / 2
//        [= e^x / (1 + u) - 1 - c1 Delta - c2 Delta^2 / 2],
//   E3 = R3 + c1 (Delta - p - s/2D) + c2 (Delta^2 - p^2) / 2,
//   Delta - p - s/2D = -s (p + Delta) / (2 D (D + p + r)),
//   (Delta^2 - p^2) / 2 = e1 (p + Delta) / 2.
// The sum is the same 4-point rule as tp_moments; with E3 rounded to FP32
// the far-field elements move by ~1e-9 relative (emulated on the 1,350-BF
// sphere: powers within 1.3e-9 of the FP64 rule).  The series holds for
// k |Delta| <= 1; beyond it X3 comes from e^x directly.
struct SplitK {
  double g0r, g0i;                   // g(D) = e^{ikD} / D
  double c1r, c1i, c2r, c2i;         // c1, c2 (FP64, for T2)
  double e0, e1, e2, D, hiD;         // e, D, 1 / 2D
  float f_e0, f_e1, f_e2, f_D, f_iD, f_kr, f_ki, f_c1r, f_c1i, f_c2r, f_c2i;
};

template <bool REALK>
__device__ __forceinline__ SplitK split_setup(const double *cS, const double *cT, double kre, double kim)
{
  SplitK z;
  const double d0 = cS[0] - cT[0], d1 = cS[1] - cT[1], d2 = cS[2] - cT[2];
  const double D2 = d0 * d0 + d1 * d1 + d2 * d2, iD = rsqrt_nr(D2), D = D2 * iD;
  z.e0 = d0 * iD; z.e1 = d1 * iD; z.e2 = d2 * iD; z.D = D; z.hiD = 0.5 * iD;
  double sn, co;
  sincos_mod(kre * D, &sn, &co);
  double amp = iD;
  if (!REALK) amp *= exp(-kim * D);
  z.g0r = amp * co; z.g0i = amp * sn;
  // c1 = ik - 1/D = (-kim - 1/D) + i kre;  c2 = c1^2 + 1/D^2
  z.c1r = -kim - iD; z.c1i = kre;
  z.c2r = z.c1r * z.c1r - z.c1i * z.c1i + iD * iD;
  z.c2i = 2.0 * z.c1r * z.c1i;
  z.f_e0 = (float)z.e0; z.f_e1 = (float)z.e1; z.f_e2 = (float)z.e2;
  z.f_D = (float)D; z.f_iD = (float)iD; z.f_kr = (float)kre; z.f_ki = (float)kim;
  z.f_c1r = (float)z.c1r; z.f_c1i = (float)z.c1i; z.f_c2r = (float)z.c2r; z.f_c2i = (float)z.c2i;
  return z;
}

// E3 (above) for one point pair, w in FP32
template <bool REALK>
__device__ __forceinline__ void split_e3(const SplitK &z, float w0, float w1, float w2, float &er, float &ei)
{
  const float p = z.f_e0 * w0 + z.f_e1 * w1 + z.f_e2 * w2;
  const float q0 = w0 - p * z.f_e0, q1 = w1 - p * z.f_e1, q2 = w2 - p * z.f_e2;
  const float s = q0 * q0 + q1 * q1 + q2 * q2;
  const float dp = z.f_D + p;
  const float r = sqrtf(dp * dp + s);
  const float den = dp + r, iden = 1.0f / den;
  const float e1 = s * iden, Dl = p + e1, u = Dl * z.f_iD;
  const float i1u = 1.0f / (1.0f + u);
  const float U3 = u * u * u * i1u;
  const float pD = p + Dl;
  const float m = -s * pD * iden * 0.5f * z.f_iD;   // Delta - p - s/2D
  const float h = 0.5f * e1 * pD;                  // (Delta^2 - p^2) / 2
  float r3r, r3i;
  if (REALK) {
    // x = i t
    const float t = z.f_kr * Dl, t2 = t * t;
    float xr, xi;
    if (fabsf(t) <= 1.0f) {
      xr = t2 * t2 * (1.0f / 24 + t2 * (-1.0f / 720 + t2 * (1.0f / 40320 + t2 * (-1.0f / 3628800 + t2 * (1.0f / 479001600)))));
      xi = t * t2 * (-1.0f / 6 + t2 * (1.0f / 120 + t2 * (-1.0f / 5040 + t2 * (1.0f / 362880 + t2 * (-1.0f / 39916800)))));
    } else {
      float sn, co;
      sincosf(t, &sn, &co);
      xr = (co - 1.0f) + 0.5f * t2;
      xi = sn - t;
    }
    // (1 + x + x^2/2) = (1 - t^2/2) + i t;  x u^2 + x^2 u (u - 1)/2 = i t u^2 - t^2 u (u - 1)/2
    r3r = xr * i1u - (1.0f - 0.5f * t2) * U3 - 0.5f * t2 * u * (u - 1.0f);
    r3i = xi * i1u - t * U3 + t * u * u;
  } else {
    const float xr = -z.f_ki * Dl, xi = z.f_kr * Dl;
    const float x2r = xr * xr - xi * xi, x2i = 2.0f * xr * xi;
    float Xr, Xi;
    if (xr * xr + xi * xi <= 1.0f) {
      // x^3 (1/3! + x (1/4! + x (...))), Horner from 1/12!
      const float c[10] = {1.0f / 6, 1.0f / 24, 1.0f / 120, 1.0f / 720, 1.0f / 5040, 1.0f / 40320,
                           1.0f / 362880, 1.0f / 3628800, 1.0f / 39916800, 1.0f / 479001600};
      float ar = c[9], ai = 0.0f;
#pragma unroll
      for (int n = 8; n >= 0; n--) {
        const float tr = ar * xr - ai * xi + c[n];
        ai = ar * xi + ai * xr;
        ar = tr;
      }
      const float x3r = x2r * xr - x2i * xi, x3i = x2r * xi + x2i * xr;
      Xr = ar * x3r - ai * x3i;
      Xi = ar * x3i + ai * x3r;
    } else {
      float sn, co;
      sincosf(xi, &sn, &co);
      const float ex = expf(xr);
      Xr = ex * co - 1.0f - xr - 0.5f * x2r;
      Xi = ex * sn - xi - 0.5f * x2i;
    }
    const float ar = 1.0f + xr + 0.5f * x2r, ai = xi + 0.5f * x2i;
    const float uu = u * u, hu = 0.5f * u * (u - 1.0f);
    r3r = Xr * i1u - ar * U3 + xr * uu + x2r * hu;
    r3i = Xi * i1u - ai * U3 + xi * uu + x2i * hu;
  }
  er = r3r + z.f_c1r * m + z.f_c2r * h;
  ei = r3i + z.f_c1i * m + z.f_c2i * h;
}

// tp_moments with g from the split above.  The column tetrahedron's points
// are read from LDS (pts[1][.][ut]) one point at a time rather than from
// ys: the real-k table kernel then holds 155 VGPRs (three waves per SIMD)
// instead of 217 (two), with the same arithmetic in the same order (the
// kernel's time did not change measurably: it is bound by its arithmetic).
template <bool REALK, typename SH>
__device__ __forceinline__ void tp_moments_split(const SH &sh, int us, int ut, const double *cS, const double *ys,
                                                 const double *cT, double kre, double kim, double *out, int stride)
{
  const SplitK z = split_setup<REALK>(cS, cT, kre, kim);
  double m[16];
#pragma unroll
  for (int i = 0; i < 16; i++) m[i] = 0.0;
#pragma unroll 1
  for (int p = 0; p < 4; p++) {
    double x[4];
#pragma unroll
    for (int e = 0; e < 4; e++) x[e] = sh.pts[0][4 * p + e][us];
    const double xi0 = x[0] - cS[0], xi1 = x[1] - cS[1], xi2 = x[2] - cS[2];
#pragma unroll 1
    for (int q = 0; q < 4; q++) {
      double y[4];
#pragma unroll
      for (int e = 0; e < 4; e++) y[e] = sh.pts[1][4 * q + e][ut];
      const double e0 = y[0] - cT[0], e1 = y[1] - cT[1], e2 = y[2] - cT[2];
      const double w0 = xi0 - e0, w1 = xi1 - e1, w2 = xi2 - e2;
      const double pp = z.e0 * w0 + z.e1 * w1 + z.e2 * w2;
      const double ww = w0 * w0 + w1 * w1 + w2 * w2;
      // T2 - 1 = c1 (p + s/2D) + c2 p^2/2
      const double l = pp + (ww - pp * pp) * z.hiD, hp = 0.5 * pp * pp;
      float fr, fi;
      split_e3<REALK>(z, (float)w0, (float)w1, (float)w2, fr, fi);
      const double vr = 1.0 + (z.c1r * l + z.c2r * hp) + (double)fr;
      const double vi = (z.c1i * l + z.c2i * hp) + (double)fi;
      const double amp = x[3] * y[3];
      const double gr = amp * (z.g0r * vr - z.g0i * vi), gi = amp * (z.g0r * vi + z.g0i * vr);
      const double xy = xi0 * e0 + xi1 * e1 + xi2 * e2;
      m[0] += gr; m[1] += gi;
      m[2] += gr * xi0; m[3] += gi * xi0; m[4] += gr * xi1; m[5] += gi * xi1; m[6] += gr * xi2; m[7] += gi * xi2;
      m[8] += gr * e0; m[9] += gi * e0; m[10] += gr * e1; m[11] += gi * e1; m[12] += gr * e2; m[13] += gi * e2;
      m[14] += gr * xy; m[15] += gi * xy;
    }
  }
#pragma unroll
  for (int i = 0; i < 16; i++) out[i * stride] = m[i];
}

// one of the two moment routines
template <bool REALK, bool SPLIT, bool LDSY = false, typename SH>
__device__ __forceinline__ void tp_moments_any(const SH &sh, int us, int ut, const double *cS, const double *ys,
                                               const double *cT, double kre, double kim, double *out, int stride)
{
  if (SPLIT)
    tp_moments_split<REALK>(sh, us, ut, cS, ys, cT, kre, kim, out, stride);
  else
    tp_moments<REALK, LDSY>(sh, us, ut, cS, ys, cT, kre, kim, out, stride);
}

// points and centroid of distinct tetrahedron u of side `which` into registers
template <typename SH>
__device__ __forceinline__ void tp_load(const SH &sh, int which, int u, double *x, double *c)
{
#pragma unroll
  for (int e = 0; e < 16; e++) x[e] = sh.pts[which][e][u];
#pragma unroll
  for (int d = 0; d < 3; d++) c[d] = sh.cen[which][d][u];
}

template <bool REALK, bool SPLIT = false>
__device__ void far_tp_tile(const DevGeom &g, double kre, double kim, cd *M, int64_t ld, int ti, int tj,
                            FarTpShared &sh)
{
  const int tid = threadIdx.x, nth = blockDim.x, N = g.nbf;
  const int *tab[2] = {g.ftTab + (size_t)ti * FTAB, g.ftTab + (size_t)tj * FTAB};
  const int nr = tab[0][4 * FT2], nc = tab[1][4 * FT2];
  for (int idx = tid; idx < 2 * 2 * FT2; idx += nth) {
    const int which = idx / (2 * FT2), k = idx % (2 * FT2);
    sh.slot[which][k] = tab[which][2 * FT2 + k];
  }
  // quadrature points of the distinct tetrahedra
  for (int idx = tid; idx < 2 * 2 * FT2 * 16; idx += nth) {
    const int which = idx / (2 * FT2 * 16), rem = idx % (2 * FT2 * 16);
    const int u = rem / 16, e = rem % 16;
    if (u < (which ? nc : nr)) sh.pts[which][e][u] = g.q4[(size_t)tab[which][u] * 16 + e];
  }
  __syncthreads();
  for (int idx = tid; idx < 2 * 2 * FT2; idx += nth) {
    const int which = idx / (2 * FT2), u = idx % (2 * FT2);
    if (u < (which ? nc : nr))
      for (int d = 0; d < 3; d++)
        sh.cen[which][d][u] = 0.25 * (sh.pts[which][d][u] + sh.pts[which][4 + d][u] + sh.pts[which][8 + d][u] +
                                      sh.pts[which][12 + d][u]);
  }
  __syncthreads();
  // moments of every (row tet, col tet) pair; a tile with more pairs than
  // fit in LDS computes each needed pair on the fly in the combination below
  const bool direct = nr * nc > FTT_MAX;
  if (!direct) {
    for (int pidx = tid; pidx < nr * nc; pidx += nth) {
      const int us = pidx / nc, ut = pidx % nc;
      double xs[16], cS[3], ys[16], cT[3];
      tp_load(sh, 0, us, xs, cS);
      tp_load(sh, 1, ut, ys, cT);
      tp_moments_any<REALK, SPLIT>(sh, us, ut, cS, ys, cT, kre, kim, &sh.mom[0][pidx], FTT_MAX);
    }
  }
  __syncthreads();
  // 1/k^2
  const double k2re = kre * kre - kim * kim, k2im = 2.0 * kre * kim;
  const double ik2d = k2re * k2re + k2im * k2im;
  const double ik2re = k2re / ik2d, ik2im = -k2im / ik2d;
  // lanes run along the column BF so that moment reads are consecutive
  for (int pidx = tid; pidx < FT2 * FT2; pidx += nth) {
    const int lb = pidx % FT2, la = pidx / FT2;
    const int a = ti * FT2 + la, b = tj * FT2 + lb;
    if (a >= N || b >= N || b < a) continue;
    if (bf_ncv(g.bfV + 5 * a, g.bfV + 5 * b) > 0) continue;
    double accr = 0.0, acci = 0.0;
    for (int sa = 0; sa < 2; sa++) {
      const int us = sh.slot[0][2 * la + sa];
      const double pfa = g.bfPF[2 * a + sa];
      const double *Qa = g.bfQ + 6 * a + 3 * sa;
      const double al0 = Qa[0] - sh.cen[0][0][us], al1 = Qa[1] - sh.cen[0][1][us], al2 = Qa[2] - sh.cen[0][2][us];
      for (int sb = 0; sb < 2; sb++) {
        const int ut = sh.slot[1][2 * lb + sb];
        const double pfb = g.bfPF[2 * b + sb];
        const double *Qb = g.bfQ + 6 * b + 3 * sb;
        const double be0 = Qb[0] - sh.cen[1][0][ut], be1 = Qb[1] - sh.cen[1][1][ut], be2 = Qb[2] - sh.cen[1][2][ut];
        double m[16];
        if (direct) {
          double xs[16], cS[3], ys[16], cT[3];
          tp_load(sh, 0, us, xs, cS);
          tp_load(sh, 1, ut, ys, cT);
          tp_moments_any<REALK, SPLIT>(sh, us, ut, cS, ys, cT, kre, kim, m, 1);
        } else {
#pragma unroll
          for (int i = 0; i < 16; i++) m[i] = sh.mom[i][us * nc + ut];
        }
        const double ab = al0 * be0 + al1 * be1 + al2 * be2;
        // Ixy - b.Ix - a.Iy + (a.b) I0
        double dr = m[14] - (be0 * m[2] + be1 * m[4] + be2 * m[6]) - (al0 * m[8] + al1 * m[10] + al2 * m[12]) + ab * m[0];
        double di = m[15] - (be0 * m[3] + be1 * m[5] + be2 * m[7]) - (al0 * m[9] + al1 * m[11] + al2 * m[13]) + ab * m[1];
        // - 9 I0 / k^2
        dr -= 9.0 * (m[0] * ik2re - m[1] * ik2im);
        di -= 9.0 * (m[0] * ik2im + m[1] * ik2re);
        const double f = pfa * pfb;
        accr += f * dr;
        acci += f * di;
      }
    }
    const cd v = {accr / FOURPI, acci / FOURPI};
    M[(size_t)b * ld + a] = v;
    M[(size_t)a * ld + b] = v;
  }
}

template <bool REALK, bool SPLIT>
__global__ __launch_bounds__(FT_THREADS) void k_far_tp(DevGeom g, double kre, double kim, cd *M, int64_t ld,
                                                       int ntiles)
{
  __shared__ FarTpShared sh;
  int ti, tj;
  tile_coords(blockIdx.x, ntiles, ti, tj);
  far_tp_tile<REALK, SPLIT>(g, kre, kim, M, ld, ti, tj, sh);
}

// Two-pass far field.  A 32 x 32 BF tile evaluates ~31 x 31 tetrahedron
// pairs, and a tetrahedron lies in the support of BFs that fall in ~1.9
// different tiles per side, so the single pass evaluates each pair 3.45
// times on average.  Pass 1 evaluates every tetrahedron pair S <= T once
// (32 x 32 tetrahedron tiles) and stores its 16 moments, 128 B, at
// S nt - S (S - 1) / 2 + (T - S); pass 2 is the single pass's combination
// with the moments gathered from that table (for S > T the record of (T, S)
// with Ix and Iy exchanged: the kernel g is symmetric).  Pairs of one
// tetrahedron with itself are never needed (their BF pairs touch) and are
// stored as zeros.
__device__ __forceinline__ size_t tp_index(int S, int T, int nt)
{
  return (size_t)S * nt - (size_t)S * (S - 1) / 2 + (size_t)(T - S);
}

// points and centroids of a 32 x 32 tetrahedron tile (pass 1 keeps no
// moments in LDS: 19 KB, so that several workgroups share a CU)
struct TpTileShared {
  double pts[2][16][2 * FT2];
  double cen[2][3][2 * FT2];
};
#define TPT_THREADS 256

// one 32 x 32 tile (bs, bt) of tetrahedron pairs of pass 1
template <bool REALK, bool SPLIT>
__device__ __forceinline__ void tp_table_tile(const DevGeom &g, double kre, double kim, double *tab, int bs, int bt,
                                              TpTileShared &sh)
{
  const int tid = threadIdx.x, nt = g.nt;
  // points of the tile's 32 row and 32 column tetrahedra
  for (int idx = tid; idx < 2 * 32 * 16; idx += TPT_THREADS) {
    const int which = idx / (32 * 16), u = (idx / 16) % 32, e = idx % 16;
    const int t = (which ? bt : bs) * 32 + u;
    sh.pts[which][e][u] = t < nt ? g.q4[(size_t)t * 16 + e] : 0.0;
  }
  __syncthreads();
  for (int idx = tid; idx < 2 * 32; idx += TPT_THREADS) {
    const int which = idx / 32, u = idx % 32;
    for (int d = 0; d < 3; d++)
      sh.cen[which][d][u] = 0.25 * (sh.pts[which][d][u] + sh.pts[which][4 + d][u] + sh.pts[which][8 + d][u] +
                                    sh.pts[which][12 + d][u]);
  }
  __syncthreads();
  // lanes along the column tetrahedron: consecutive records
  for (int pidx = tid; pidx < 32 * 32; pidx += TPT_THREADS) {
    const int us = pidx / 32, ut = pidx % 32;
    const int S = bs * 32 + us, T = bt * 32 + ut;
    if (S >= nt || T >= nt || S > T) continue;
    double m[16];
    if (S == T) {
#pragma unroll
      for (int i = 0; i < 16; i++) m[i] = 0.0;
    } else {
      double xs[16], cS[3], ys[16], cT[3];
      tp_load(sh, 0, us, xs, cS);
      tp_load(sh, 1, ut, ys, cT);
      tp_moments_any<REALK, SPLIT, true>(sh, us, ut, cS, ys, cT, kre, kim, m, 1);
    }
    double2 *o = (double2 *)(tab + tp_index(S, T, nt) * 16);
#pragma unroll
    for (int i = 0; i < 8; i++) o[i] = make_double2(m[2 * i], m[2 * i + 1]);
  }
}

template <bool REALK, bool SPLIT>
__global__ __launch_bounds__(TPT_THREADS) void k_tp_table(DevGeom g, double kre, double kim, double *tab, int ntb)
{
  __shared__ TpTileShared sh;
  int bs, bt;
  tile_coords(blockIdx.x, ntb, bs, bt);
  tp_table_tile<REALK, SPLIT>(g, kre, kim, tab, bs, bt, sh);
}

// Pass 2: a 32 x 32 BF tile combines the table's records in two steps.  A BF
// pair's element is a sum over its four tetrahedron pairs (S, T) of
//   pf_a pf_b [Ixy - b.Ix - a.Iy + (a.b) I0 - 9 I0/k^2],
// so for a row tetrahedron S and a column BF the sum over the BF's two T is
//   s - a.v,  s = sum pf_b [Ixy - b.Ix - 9 I0/k^2],  v = sum pf_b [Iy - b I0],
// four complex numbers that every row BF on S shares: 992 + 2,048 short
// combinations a tile instead of 4,096 long ones, and a quarter of the LDS
// reads.  Row tetrahedra go through LDS four at a time (records, then s and
// v; the next four's records are on their way meanwhile), so a workgroup holds
// 35 KB of LDS, not the tile's 151 KB of records, and four share a CU.
// N = 19,872: 11.8 -> 5.4 ms (before: one workgroup a CU, all of a tile's
// records in LDS, bound by the latency of its dependent phases).  Tried on
// top of it: tiles dealt to the XCDs in bands that share records, 6.1 -> 6.3
// ms at the time -- the records' traffic is not the bound, issue is.
#define GS_CH 4            // row tetrahedra at a time
#define GS_NT 256
typedef double dv2 __attribute__((ext_vector_type(2)));
template <int NC> struct GatherShared {
  dv2 rec[GS_CH][NC][9];       // a record's 8 entries, padded: lanes on consecutive tetrahedra read distinct banks
  double H[GS_CH][8][FT2];         // s, v (re, im) of each column BF
  int rt[2 * FT2], ct[2 * FT2];    // distinct tetrahedra
  double rpf[2][FT2], ral[2][3][FT2];
  int rslot[2][FT2], rv[5][FT2], cv[5][FT2];
};

// x plus the other half-wave's x
__device__ __forceinline__ double half_sum(double x)
{
  const unsigned long long b = (unsigned long long)__double_as_longlong(x);
  const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)b, (unsigned)b, false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(b >> 32), (unsigned)(b >> 32), false, false);
  return __longlong_as_double((long long)(((unsigned long long)hi[0] << 32) | lo[0])) +
         __longlong_as_double((long long)(((unsigned long long)hi[1] << 32) | lo[1]));
}

template <int NC>
__device__ __forceinline__ void far_gather_tile(const DevGeom &g, double kre, double kim,
                                                const double *__restrict__ tpt, cd *M, int64_t ld, int ti, int tj,
                                                GatherShared<NC> &sh)
{
  const int tid = threadIdx.x, lane = tid & 63, N = g.nbf, nt = g.nt;
  const int *rtab = g.ftTab + (size_t)ti * FTAB, *ctab = g.ftTab + (size_t)tj * FTAB;
  const int nr = rtab[4 * FT2], nc = ctab[4 * FT2];
  const double *tetCen = g.tetVol + nt;
  // this thread's column BF and side (one wave: 32 BFs x 2 sides)
  const int lb = tid & 31, sb = (tid >> 5) & 1, b = tj * FT2 + lb;
  const int cslot = ctab[2 * FT2 + 2 * lb + sb];
  double pfb = 0.0, be[3] = {0.0, 0.0, 0.0};
  if (b < N) {
    const int T = g.bfT[2 * b + sb];
    pfb = g.bfPF[2 * b + sb];
#pragma unroll
    for (int d = 0; d < 3; d++) be[d] = g.bfQ[6 * b + 3 * sb + d] - tetCen[3 * T + d];
  }
  if (tid < 4 * FT2) {
    const int side = tid / (2 * FT2), u = tid % (2 * FT2);
    const int t = u < (side ? nc : nr) ? (side ? ctab : rtab)[u] : 0;
    (side ? sh.ct : sh.rt)[u] = t;
  } else if (tid < 6 * FT2) {
    const int k = tid - 4 * FT2, la = k >> 1, sa = k & 1, a = ti * FT2 + la;
    sh.rslot[sa][la] = rtab[2 * FT2 + k];
    double pf = 0.0, al[3] = {0.0, 0.0, 0.0};
    if (a < N) {
      const int S = g.bfT[2 * a + sa];
      pf = g.bfPF[2 * a + sa];
#pragma unroll
      for (int d = 0; d < 3; d++) al[d] = g.bfQ[6 * a + 3 * sa + d] - tetCen[3 * S + d];
    }
    sh.rpf[sa][la] = pf;
#pragma unroll
    for (int d = 0; d < 3; d++) sh.ral[sa][d][la] = al[d];
  } else if (tid < 7 * FT2) {
    const int la = tid - 6 * FT2, a = ti * FT2 + la;
#pragma unroll
    for (int v = 0; v < 5; v++) sh.rv[v][la] = a < N ? g.bfV[5 * a + v] : -2;
  } else {
#pragma unroll
    for (int v = 0; v < 5; v++) sh.cv[v][lb] = b < N ? g.bfV[5 * b + v] : -1;
  }
  __syncthreads();
  const double k2re = kre * kre - kim * kim, k2im = 2.0 * kre * kim, ik2d = k2re * k2re + k2im * k2im;
  const double q9re = 9.0 * k2re / ik2d, q9im = -9.0 * k2im / ik2d;        // 9 / k^2
  const int a0 = (tid >> 5) * 4;                   // this thread's four row BFs
  int slot[2][4];
#pragma unroll
  for (int sa = 0; sa < 2; sa++)
#pragma unroll
    for (int i = 0; i < 4; i++) slot[sa][i] = sh.rslot[sa][a0 + i];
  cd acc[4];
#pragma unroll
  for (int i = 0; i < 4; i++) acc[i] = {0.0, 0.0};
  // records of row tetrahedra s0 .. s0 + 3, one a wave, eight threads a
  // record; for S > T the record of (T, S), with Ix and Iy exchanged.  Record
  // numbers fit 32 bits (2^32 of them would fill 550 GB).
  constexpr int NL = NC / 8;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), e = tid & 7, u0 = (tid >> 3) & 7;
  const int ex = e >= 1 && e <= 3 ? e + 3 : e >= 4 && e <= 6 ? e - 3 : e;
  int T[NL];
  unsigned tbase[NL];                              // row T's first record, less T
#pragma unroll
  for (int k = 0; k < NL; k++) {
    T[k] = sh.ct[u0 + 8 * k];
    tbase[k] = (unsigned)((int64_t)T[k] * nt - (int64_t)T[k] * (T[k] + 1) / 2);
  }
  dv2 pre[NL];
  auto fetch = [&](int s0) __attribute__((always_inline)) {
    const int S = __builtin_amdgcn_readfirstlane(sh.rt[min(s0 + wv, 2 * FT2 - 1)]);
    const unsigned sbase = (unsigned)((int64_t)S * nt - (int64_t)S * (S + 1) / 2);
#pragma unroll
    for (int k = 0; k < NL; k++) {
      const bool sw = S > T[k];
      const unsigned row = sw ? tbase[k] + S : sbase + T[k];
      pre[k] = ((const dv2 *)tpt)[(size_t)row * 8 + (sw ? ex : e)];
    }
  };
  fetch(0);
#pragma unroll 1
  for (int s0 = 0; s0 < nr; s0 += GS_CH) {
#pragma unroll
    for (int k = 0; k < NL; k++) sh.rec[wv][u0 + 8 * k][e] = pre[k];
    __syncthreads();
    if (s0 + GS_CH < nr) fetch(s0 + GS_CH);
    // s and v of wave `si`'s row tetrahedron: one side a thread, the two added across the wave's halves
    {
      const int si = tid >> 6;
      double h[8];
      const dv2 *m = sh.rec[si][cslot];
      const dv2 i0 = m[0], xy = m[7];
      double sr = xy.x - (i0.x * q9re - i0.y * q9im), sm = xy.y - (i0.x * q9im + i0.y * q9re);
#pragma unroll
      for (int d = 0; d < 3; d++) {
        const dv2 ix = m[1 + d], iy = m[4 + d];
        sr -= be[d] * ix.x;
        sm -= be[d] * ix.y;
        h[2 + 2 * d] = pfb * (iy.x - be[d] * i0.x);
        h[3 + 2 * d] = pfb * (iy.y - be[d] * i0.y);
      }
      h[0] = pfb * sr;
      h[1] = pfb * sm;
#pragma unroll
      for (int i = 0; i < 8; i++) h[i] = half_sum(h[i]);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const double lo = h[i], hi = h[4 + i];
        sh.H[si][4 * sb + i][lb] = sb ? hi : lo;
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int sa = 0; sa < 2; sa++) {
        const int u = slot[sa][i] - s0;
        if (u < 0 || u >= GS_CH) continue;
        const double pf = sh.rpf[sa][a0 + i];
        double re = sh.H[u][0][lb], im = sh.H[u][1][lb];
#pragma unroll
        for (int d = 0; d < 3; d++) {
          const double al = sh.ral[sa][d][a0 + i];
          re -= al * sh.H[u][2 + 2 * d][lb];
          im -= al * sh.H[u][3 + 2 * d][lb];
        }
        acc[i].re += pf * re;
        acc[i].im += pf * im;
      }
  }
  int vb[5];
#pragma unroll
  for (int v = 0; v < 5; v++) vb[v] = sh.cv[v][lb];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int a = ti * FT2 + a0 + i;
    if (a >= N || b >= N || b < a) continue;
    int va[5];
#pragma unroll
    for (int v = 0; v < 5; v++) va[v] = sh.rv[v][a0 + i];
    if (bf_ncv(va, vb) > 0) continue;
    const cd v = {acc[i].re * (1.0 / FOURPI), acc[i].im * (1.0 / FOURPI)};
    M[(size_t)b * ld + a] = v;
    M[(size_t)a * ld + b] = v;
  }
}

// NC: most distinct tetrahedra of a tile (31 on average on the Kuhn spheres,
// 34 at most; 64 is any mesh's bound).  64 slots hold 49 KB of LDS, three
// workgroups a CU, 40 hold 35 KB, four: N = 19,872 assembled in 8.5 ms with the
// tetrahedra in the mesh's order and 12.5 in random order, which needs the 64
// and gathers records further apart (all moments in LDS: 17.0 and 27.2)
template <int NC>
__global__ __launch_bounds__(GS_NT, 4) void k_far_gather(DevGeom g, double kre, double kim,
                                                      const double *__restrict__ tpt, cd *M, int64_t ld, int ntiles)
{
  __shared__ GatherShared<NC> sh;
  int ti, tj;
  tile_coords(blockIdx.x, ntiles, ti, tj);
  far_gather_tile<NC>(g, kre, kim, tpt, M, ld, ti, tj, sh);
}

// ---------------------------------------------------------------------------
// near field + static record + Gram, one thread per touching pair
// 1/n for the series below, correctly rounded at compile time (the same
// values a division gives, without a division per term)
struct InvIntTable {
  double v[100];
  constexpr InvIntTable() : v()
  {
    for (int i = 1; i < 100; i++) v[i] = 1.0 / i;
  }
};
__constant__ InvIntTable c_inv_int = InvIntTable();

__device__ __forceinline__ cd exprel3(cd x)
{
  // GetExpRelTable(x, 3, 3): x^3/3! + sum_{n>=4} x^n/n!, relative 1e-8 break
  cd term = {1.0, 0.0};
  term = cscale(cmul(term, x), 1.0);
  term = cscale(cmul(term, x), 0.5);
  term = cscale(cmul(term, x), 1.0 / 3.0);
  cd first = term, sum = {0.0, 0.0};
  for (int n = 4; n < 100; n++) {
    term = cscale(cmul(term, x), c_inv_int.v[n]);
    sum = cadd(sum, term);
    const double mt = term.re * term.re + term.im * term.im;
    const double ms = sum.re * sum.re + sum.im * sum.im;
    if (mt < 1.0e-16 * ms) break;
  }
  return cadd(first, sum);
}

// ---- compiled SVTensor expressions (bfa_expr.h): complex functions and a
// postfix interpreter over a small complex stack
__device__ __forceinline__ cd csub(cd a, cd b) { return {a.re - b.re, a.im - b.im}; }
__device__ cd cexp_d(cd a)
{
  double s, c;
  sincos(a.im, &s, &c);
  const double e = exp(a.re);
  return {e * c, e * s};
}
__device__ cd clog_d(cd a) { return {log(hypot(a.re, a.im)), atan2(a.im, a.re)}; }
__device__ cd csqrt_d(cd a)
{
  const double m = hypot(a.re, a.im);
  if (m == 0.0) return {0.0, 0.0};
  const double t = sqrt(0.5 * (m + fabs(a.re)));
  return a.re >= 0.0 ? cd{t, a.im / (2.0 * t)} : cd{fabs(a.im) / (2.0 * t), a.im >= 0.0 ? t : -t};
}
__device__ cd csin_d(cd a) { double s, c; sincos(a.re, &s, &c); return {s * cosh(a.im), c * sinh(a.im)}; }
__device__ cd ccos_d(cd a) { double s, c; sincos(a.re, &s, &c); return {c * cosh(a.im), -s * sinh(a.im)}; }
__device__ cd csinh_d(cd a) { double s, c; sincos(a.im, &s, &c); return {sinh(a.re) * c, cosh(a.re) * s}; }
__device__ cd ccosh_d(cd a) { double s, c; sincos(a.im, &s, &c); return {cosh(a.re) * c, sinh(a.re) * s}; }
// principal branches: asin z = -i log(iz + sqrt(1 - z^2)), acos z = pi/2 - asin z,
// atan z = (i/2) log((i + z)/(i - z))
__device__ cd casin_d(cd z)
{
  const cd w = cadd(cd{-z.im, z.re}, csqrt_d(csub(cd{1.0, 0.0}, cmul(z, z))));
  const cd l = clog_d(w);
  return {l.im, -l.re};
}
__device__ cd catan_d(cd z)
{
  const cd l = clog_d(cdiv(cd{z.re, 1.0 + z.im}, cd{-z.re, 1.0 - z.im}));
  return {-0.5 * l.im, 0.5 * l.re};
}
__device__ cd expr_fn(int f, cd a)
{
  switch (f) {
    case EFN_EXP: return cexp_d(a);
    case EFN_LOG: return clog_d(a);
    case EFN_SQRT: return csqrt_d(a);
    case EFN_SIN: return csin_d(a);
    case EFN_COS: return ccos_d(a);
    case EFN_TAN: return cdiv(csin_d(a), ccos_d(a));
    case EFN_COT: return cdiv(ccos_d(a), csin_d(a));
    case EFN_SEC: return cdiv(cd{1.0, 0.0}, ccos_d(a));
    case EFN_CSC: return cdiv(cd{1.0, 0.0}, csin_d(a));
    case EFN_ASIN: return casin_d(a);
    case EFN_ACOS: { const cd s = casin_d(a); return {0.5 * M_PI - s.re, -s.im}; }
    case EFN_ATAN: return catan_d(a);
    case EFN_SINH: return csinh_d(a);
    case EFN_COSH: return ccosh_d(a);
    case EFN_TANH: return cdiv(csinh_d(a), ccosh_d(a));
    case EFN_ABS: return {hypot(a.re, a.im), 0.0};
    case EFN_STEP: return {a.re >= 0.0 ? 1.0 : 0.0, 0.0};
    default: return {0.0, 0.0};
  }
}
// a^b = exp(b log a); integer powers by repeated products (exact w^2 etc.)
__device__ cd expr_pow(cd a, cd b)
{
  if (b.im == 0.0 && b.re == floor(b.re) && fabs(b.re) <= 16.0) {
    int n = (int)fabs(b.re);
    cd r = {1.0, 0.0}, x = a;
    while (n) {
      if (n & 1) r = cmul(r, x);
      x = cmul(x, x);
      n >>= 1;
    }
    return b.re < 0.0 ? cdiv(cd{1.0, 0.0}, r) : r;
  }
  if (a.re == 0.0 && a.im == 0.0) return {0.0, 0.0};
  return cexp_d(cmul(b, clog_d(a)));
}
__device__ cd expr_run(const ExprHeader *h, int slot, const cd *vars)
{
  const ExprOp *ops = (const ExprOp *)(h + 1);
  const double *k = (const double *)(ops + h->nops);
  cd st[EXPR_STACK];
  int sp = 0;
  for (int i = h->start[slot], e = h->start[slot] + h->len[slot]; i < e; i++) {
    const ExprOp o = ops[i];
    if (o.op == EOP_CONST) { st[sp++] = {k[2 * o.arg], k[2 * o.arg + 1]}; continue; }
    if (o.op == EOP_VAR) { st[sp++] = vars[o.arg]; continue; }
    if (o.op == EOP_NEG) { st[sp - 1] = {-st[sp - 1].re, -st[sp - 1].im}; continue; }
    if (o.op == EOP_FN) { st[sp - 1] = expr_fn(o.arg, st[sp - 1]); continue; }
    const cd b = st[--sp], a = st[sp - 1];
    st[sp - 1] = o.op == EOP_ADD ? cadd(a, b) : o.op == EOP_SUB ? csub(a, b) : o.op == EOP_MUL ? cmul(a, b)
               : o.op == EOP_DIV ? cdiv(a, b) : expr_pow(a, b);
  }
  return st[0];
}

// Permittivity tensor at x (SVTensor::Evaluate, SVTensor.cc:306-373); kinds
// 0-3 are the closed forms documented with bfa_material, kind 4 a compiled
// SVTensor evaluated at w = omega * FreqUnit.  EXPR = false leaves kind 4
// out of the code (its interpreter's registers and stack would otherwise
// set the calling kernel's occupancy for every material).
template <bool EXPR = true>
__device__ void eps_tensor(const bfa_material &m, const double *x, double omega, cd Q[3][3])
{
  for (int r = 0; r < 3; r++)
    for (int c = 0; c < 3; c++) Q[r][c] = {0.0, 0.0};
  switch (m.kind) {
    case 1:
      Q[0][0] = {m.p[0], m.p[1]}; Q[1][1] = {m.p[2], m.p[3]}; Q[2][2] = {m.p[4], m.p[5]};
      return;
    case 2: {
      const double re = m.p[0] + m.p[2] * sin(M_PI * x[0]) * cos(M_PI * x[1]);
      Q[0][0] = Q[1][1] = Q[2][2] = {re, m.p[1]};
    } return;
    case 3: {
      const bool up = x[2] > 0.0;
      Q[0][0] = Q[1][1] = Q[2][2] = up ? cd{m.p[0], m.p[1]} : cd{m.p[2], m.p[3]};
    } return;
    case 4: if constexpr (EXPR) {
      const ExprHeader *h = (const ExprHeader *)m.expr;
      cd v[EV_COUNT];
      const double rho = sqrt(x[0] * x[0] + x[1] * x[1]);
      v[EV_W] = {omega * h->freq_unit, 0.0};
      v[EV_X] = {x[0], 0.0}; v[EV_Y] = {x[1], 0.0}; v[EV_Z] = {x[2], 0.0};
      v[EV_R] = {sqrt(rho * rho + x[2] * x[2]), 0.0};
      v[EV_THETA] = {atan2(rho, x[2]), 0.0};
      v[EV_PHI] = {atan2(x[1], x[0]), 0.0};
      v[EV_EPS1] = v[EV_EPS2] = v[EV_EPS3] = {0.0, 0.0};
      for (int k = 0; k < h->num_mp && k < 3; k++) v[EV_EPS1 + k] = expr_run(h, 9 + k, v);
      if (h->matprop) {
        Q[0][0] = Q[1][1] = Q[2][2] = v[EV_EPS1];
        return;
      }
      for (int s = 0; s < 9; s++) {
        if (h->len[s]) Q[s / 3][s % 3] = expr_run(h, s, v);
        else if (s % 4 == 0) Q[s / 3][s % 3] = {1.0, 0.0};
      }
      for (int mu = 0; mu < 3; mu++) {
        const int nu = (mu + 1) % 3;
        const cd avg = cscale(cadd(Q[mu][nu], Q[nu][mu]), 0.5);
        Q[mu][nu] = Q[nu][mu] = avg;
      }
      if (h->len[0]) {
        if (!h->len[4]) Q[1][1] = Q[0][0];
        if (!h->len[8]) Q[2][2] = Q[0][0];
      }
    } return;
    default:
      Q[0][0] = Q[1][1] = Q[2][2] = {m.p[0], m.p[1]};
  }
}

// (eps - 1)^-1 by the cofactor formula of Invert3x3Matrix (VIEMatrix.cc:51-72)
__device__ void inv_chi(const cd Q[3][3], cd W[3][3])
{
  cd Mm[3][3];
  for (int r = 0; r < 3; r++)
    for (int c = 0; c < 3; c++) Mm[r][c] = r == c ? cd{Q[r][c].re - 1.0, Q[r][c].im} : Q[r][c];
  auto sub = [](cd a, cd b) { return cd{a.re - b.re, a.im - b.im}; };
  cd M11 = Mm[0][0], M12 = Mm[0][1], M13 = Mm[0][2], M21 = Mm[1][0], M22 = Mm[1][1], M23 = Mm[1][2];
  cd M31 = Mm[2][0], M32 = Mm[2][1], M33 = Mm[2][2];
  cd Det = cadd(cadd(cmul(cmul(M12, M23), M31), cmul(cmul(M13, M21), M32)), cmul(cmul(M11, M22), M33));
  Det = sub(sub(sub(Det, cmul(cmul(M13, M22), M31)), cmul(cmul(M11, M23), M32)), cmul(cmul(M12, M21), M33));
  W[0][0] = cdiv(sub(cmul(M22, M33), cmul(M23, M32)), Det);
  W[0][1] = cdiv(sub(cmul(M13, M32), cmul(M12, M33)), Det);
  W[0][2] = cdiv(sub(cmul(M12, M23), cmul(M13, M22)), Det);
  W[1][0] = cdiv(sub(cmul(M23, M31), cmul(M21, M33)), Det);
  W[1][1] = cdiv(sub(cmul(M11, M33), cmul(M13, M31)), Det);
  W[1][2] = cdiv(sub(cmul(M13, M21), cmul(M11, M23)), Det);
  W[2][0] = cdiv(sub(cmul(M21, M32), cmul(M22, M31)), Det);
  W[2][1] = cdiv(sub(cmul(M12, M31), cmul(M11, M32)), Det);
  W[2][2] = cdiv(sub(cmul(M11, M22), cmul(M12, M21)), Det);
}

// permittivity tensors at points (row-major 3x3 complex per point)
__global__ void k_eps_points(bfa_material m, double omega, int n, const double *pts, double *Q)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  cd T[3][3];
  eps_tensor(m, pts + 3 * (size_t)i, omega, T);
  for (int r = 0; r < 3; r++)
    for (int c = 0; c < 3; c++) {
      Q[18 * (size_t)i + 2 * (3 * r + c)] = T[r][c].re;
      Q[18 * (size_t)i + 2 * (3 * r + c) + 1] = T[r][c].im;
    }
}

extern "C" int bfa_material_eval(const bfa_material *mat, double omega, int npts, const double *pts, double *Q)
{
  if (!mat || npts < 0 || (npts > 0 && (!pts || !Q))) return fail(BFA_ERR_ARG, "bfa_material_eval: bad argument");
  if (mat->kind == 4 && !mat->expr) return fail(BFA_ERR_ARG, "bfa_material_eval: compiled material without program");
  if (npts == 0) return BFA_OK;
  double *dp = nullptr, *dq = nullptr;
  HIPCHECK(hipMalloc(&dp, (size_t)npts * 3 * 8));
  hipError_t e = hipMalloc(&dq, (size_t)npts * 18 * 8);
  if (e != hipSuccess) { (void)hipFree(dp); return fail(BFA_ERR_OOM, "bfa_material_eval: allocation"); }
  int rc = BFA_OK;
  if (hipMemcpy(dp, pts, (size_t)npts * 24, hipMemcpyHostToDevice) != hipSuccess) rc = fail(BFA_ERR_HIP, "upload");
  if (!rc) {
    hipLaunchKernelGGL(k_eps_points, dim3((npts + 127) / 128), dim3(128), 0, 0, *mat, omega, npts, dp, dq);
    if (hipMemcpy(Q, dq, (size_t)npts * 18 * 8, hipMemcpyDeviceToHost) != hipSuccess) rc = fail(BFA_ERR_HIP, "download");
  }
  (void)hipFree(dp);
  (void)hipFree(dq);
  return rc;
}

// -(1/omega^2) int_t F_i . chi^-1 . F_j over TetCR33 (GetOverlapIntegrand) for
// the 4 x 4 faces (i, j) of tetrahedron t, by one wave: chi^-1 once per point
// (a lane each), then sixteen (i, j) by four shares of the points.  The pairs
// of BFs that share t read their entry; evaluated pair by pair, each point's
// permittivity and inverse would be formed ten times over, by the few lanes of
// k_near's waves that need them (a compiled expression, N = 3,822: assembly
// 3.97 -> 0.59 ms; closed forms, N = 19,872: near field 2.4 -> 1.0 ms).
struct GramShared { cd W[33][9]; };
template <bool EXPR>
__device__ void gram_tet(const DevGeom &g, int t, double omega, const bfa_material &mat, cd *out, GramShared &sh)
{
  const int lane = threadIdx.x;
  const double *q = g.q33 + (size_t)t * 33 * 4;
  if (lane < 33) {
    const double x[3] = {q[4 * lane], q[4 * lane + 1], q[4 * lane + 2]}, w = q[4 * lane + 3];
    cd Q[3][3], W[3][3];
    eps_tensor<EXPR>(mat, x, omega, Q);
    inv_chi(Q, W);
#pragma unroll
    for (int r = 0; r < 3; r++)
#pragma unroll
      for (int c = 0; c < 3; c++) sh.W[lane][3 * r + c] = cscale(W[r][c], w);
  }
  __syncthreads();
  const int i = (lane >> 2) & 3, j = lane & 3, part = lane >> 4;
  const int a = g.tetFI[4 * t + i], b = g.tetFI[4 * t + j];
  cd acc = {0.0, 0.0};
  if (a < g.nbf && b < g.nbf) {
    const int sa = g.bfT[2 * a] == t ? 0 : 1, sb = g.bfT[2 * b] == t ? 0 : 1;
    const double *QA = g.bfQ + 6 * a + 3 * sa, *QB = g.bfQ + 6 * b + 3 * sb;
    const double pp = g.bfPF[2 * a + sa] * g.bfPF[2 * b + sb];
    for (int p = part; p < 33; p += 4) {
      double FA[3], FB[3];
#pragma unroll
      for (int d = 0; d < 3; d++) { FA[d] = q[4 * p + d] - QA[d]; FB[d] = pp * (q[4 * p + d] - QB[d]); }
#pragma unroll
      for (int r = 0; r < 3; r++)
#pragma unroll
        for (int c = 0; c < 3; c++) acc = cadd(acc, cscale(sh.W[p][3 * r + c], FA[r] * FB[c]));
    }
  }
#pragma unroll
  for (int off = 16; off < 64; off <<= 1) {
    acc.re += __shfl_xor(acc.re, off, 64);
    acc.im += __shfl_xor(acc.im, off, 64);
  }
  if (part == 0) out[4 * i + j] = cscale(acc, -1.0 / (omega * omega));
}

template <bool EXPR>
__global__ __launch_bounds__(64) void k_gram(DevGeom g, double omega, bfa_material mat, cd *gram)
{
  __shared__ GramShared sh;
  gram_tet<EXPR>(g, blockIdx.x, omega, mat, gram + (size_t)blockIdx.x * 16, sh);
}

// ---------------------------------------------------------------------------
// AssembleOverlapBlocks / GetOverlaps (VIEMatrix.cc:122-360): per row a the
// self entry (both tetrahedra) then the other interior faces of a's positive
// and negative tetrahedra in FI order (<= 7 entries), each the TetCR33
// integral of F_a . M . F_b with
//   V:     -Omega^2 (eps - 1)        VInv: -(eps - 1)^-1 / Omega^2
//   Rytov: 4 Omega RelDeltaTheta / (pi Z0) Im(eps - 1)
// RelDeltaTheta = Theta(Omega, T(x)) - Theta_env, divided by
// DeltaThetaHat = Theta(T_avg) - Theta_env when that is nonzero;
// Theta(Omega, T) = Omega / (exp(Omega / (k T)) - 1), k = 4.36763e-4,
// Theta = 0 at T = 0 (GetThetaFactor, VIEMatrix.cc:78-84).
#define BOLTZMANN_K 4.36763e-4
#define MAXOVERLAP 7
__device__ double theta_factor(double omega, double T)
{
  if (T == 0.0) return 0.0;
  return omega / (exp(omega / (BOLTZMANN_K * T)) - 1.0);
}

__device__ void overlap_entry(const DevGeom &g, int t, const double *QA, double pfA, const double *QB, double pfB,
                              double omega, const bfa_material &mat, const bfa_material &temp, bool has_temp,
                              double theta_env, double dtheta_hat, cd &V, cd &VI, double &R)
{
  const double *q = g.q33 + (size_t)t * 33 * 4;
  cd v = {0.0, 0.0}, vi = {0.0, 0.0};
  double ry = 0.0;
  for (int i = 0; i < 33; i++) {
    const double x[3] = {q[4 * i], q[4 * i + 1], q[4 * i + 2]};
    cd Q[3][3], W[3][3];
    eps_tensor(mat, x, omega, Q);
    inv_chi(Q, W);
    double rel = 1.0;
    if (has_temp) {
      cd Tq[3][3];
      eps_tensor(temp, x, 0.0, Tq);
      rel = theta_factor(omega, Tq[0][0].re) - theta_env;
      if (dtheta_hat != 0.0) rel /= dtheta_hat;
    }
    double FA[3], FB[3];
    for (int d = 0; d < 3; d++) { FA[d] = pfA * (x[d] - QA[d]); FB[d] = pfB * (x[d] - QB[d]); }
    cd sv = {0.0, 0.0}, sw = {0.0, 0.0};
    double sr = 0.0;
    for (int r = 0; r < 3; r++)
      for (int c = 0; c < 3; c++) {
        const double f = FA[r] * FB[c];
        const cd em1 = r == c ? cd{Q[r][c].re - 1.0, Q[r][c].im} : Q[r][c];
        sv = cadd(sv, cscale(em1, f));
        sw = cadd(sw, cscale(W[r][c], f));
        sr += f * em1.im;
      }
    const double w = q[4 * i + 3];
    v = cadd(v, cscale(sv, w));
    vi = cadd(vi, cscale(sw, w));
    ry += w * sr * rel;
  }
  V = cscale(v, -omega * omega);
  VI = cscale(vi, -1.0 / (omega * omega));
  R = ry * 4.0 * omega / (M_PI * ZVAC);
}

// Eight lanes a basis function, one for each face of its two tetrahedra: with
// one thread for all of them, 2,376 unknowns had 38 wavefronts and took
// 1.44 ms, now 0.11.  The row's first entry is the diagonal, the sum of both
// sides; the others follow in the order of the faces.
__global__ __launch_bounds__(128) void k_overlap_rows(DevGeom g, double omega, bfa_material mat, bfa_material temp,
                                                      int has_temp, double theta_env, double dtheta_hat, int *cnt,
                                                      int *cols, cd *V, cd *VI, double *R)
{
  const int id = blockIdx.x * blockDim.x + threadIdx.x, a = id >> 3, e = id & 7, side = e >> 2;
  const int base = threadIdx.x & 56;   // the basis function's first lane
  cd v = {0.0, 0.0}, vi = {0.0, 0.0};
  double r = 0.0;
  int b = -1;
  if (a < g.nbf) {
    const int t = g.bfT[2 * a + side];
    b = g.tetFI[4 * t + (e & 3)];
    if (b >= g.nbf) b = -1;
    if (b >= 0) {
      const int sb = g.bfT[2 * b] == t ? 0 : 1;
      overlap_entry(g, t, g.bfQ + 6 * a + 3 * side, g.bfPF[2 * a + side], g.bfQ + 6 * b + 3 * sb, g.bfPF[2 * b + sb],
                    omega, mat, temp, has_temp != 0, theta_env, dtheta_hat, v, vi, r);
    }
  }
  const unsigned diag = (unsigned)(__ballot(b >= 0 && b == a) >> base) & 0xFF;
  const unsigned off = (unsigned)(__ballot(b >= 0 && b != a) >> base) & 0xFF;
  // the diagonal's two parts, one of each side
  const int l0 = base + __ffs(diag & 0xF) - 1, l1 = base + 3 + __ffs(diag >> 4);
  const cd s0 = {__shfl(v.re, l0, 64), __shfl(v.im, l0, 64)}, s1 = {__shfl(v.re, l1, 64), __shfl(v.im, l1, 64)};
  const cd i0 = {__shfl(vi.re, l0, 64), __shfl(vi.im, l0, 64)}, i1 = {__shfl(vi.re, l1, 64), __shfl(vi.im, l1, 64)};
  const double r0 = __shfl(r, l0, 64), r1 = __shfl(r, l1, 64);
  if (a >= g.nbf) return;
  const size_t o = (size_t)a * MAXOVERLAP;
  if (e == 0) {
    cols[o] = a; V[o] = cadd(s0, s1); VI[o] = cadd(i0, i1); R[o] = r0 + r1;
    cnt[a] = 1 + __popc(off);
  }
  if (b >= 0 && b != a) {
    const size_t n = o + 1 + __popc(off & ((1u << e) - 1));
    cols[n] = b; V[n] = v; VI[n] = vi; R[n] = r;
  }
}

// Theta factors of AssembleOverlapBlocks' Rytov entries: the environment's
// and Theta(T_avg) - Theta_env, with T_avg the volume-weighted temperature at
// the tetrahedron centroids (GetThetaFactor, GetAverageTemperature,
// VIEMatrix.cc:78-101), both evaluated at omega = 0 as the reference does
static int rytov_thetas(const bfa_geometry *g, double omega, const bfa_material *temperature, double t_env,
                        double &theta_env, double &dhat)
{
  theta_env = dhat = 0.0;
  if (!temperature) return BFA_OK;
  const int nt = g->nt;
  std::vector<double> cen(3 * (size_t)nt), Tq(18 * (size_t)nt);
  for (int t = 0; t < nt; t++)
    for (int d = 0; d < 3; d++) cen[3 * t + d] = g->tetCen[3 * t + d];
  int rc = bfa_material_eval(temperature, 0.0, nt, cen.data(), Tq.data());
  if (rc) return rc;
  double tv = 0.0, vol = 0.0;
  for (int t = 0; t < nt; t++) { vol += g->tetVol[t]; tv += g->tetVol[t] * Tq[18 * (size_t)t]; }
  const double TAvg = tv / vol;
  auto theta = [](double w, double T) { return T == 0.0 ? 0.0 : w / (std::exp(w / (BOLTZMANN_K * T)) - 1.0); };
  theta_env = theta(omega, t_env);
  dhat = theta(omega, TAvg) - theta_env;
  return BFA_OK;
}

namespace bfa {
// overlap rows into device arrays (N x MAXOVERLAP each), on stream st
int overlap_rows_device(bfa_geometry *g, double omega, const bfa_material *eps, const bfa_material *temperature,
                        double t_env, int *dcnt, int *dcols, void *dV, void *dVI, double *dR, hipStream_t st)
{
  double theta_env = 0.0, dhat = 0.0;
  int rc = rytov_thetas(g, omega, temperature, t_env, theta_env, dhat);
  if (rc) return rc;
  bfa_material temp;
  memset(&temp, 0, sizeof temp);
  if (temperature) temp = *temperature;
  hipLaunchKernelGGL(k_overlap_rows, dim3((g->nbf + 15) / 16), dim3(128), 0, st, g->dg, omega, *eps, temp,
                     temperature ? 1 : 0, theta_env, dhat, dcnt, dcols, (cd *)dV, (cd *)dVI, dR);
  HIPCHECK(hipGetLastError());
  return BFA_OK;
}
}  // namespace bfa

// AssembleOverlapBlocks for one object: row a holds cnt[a] <= 7 entries at
// [a*7, a*7 + cnt[a]) of cols / V / VInv / Rytov (host arrays)
extern "C" int bfa_overlap_blocks(bfa_geometry *g, double omega, const bfa_material *eps,
                                  const bfa_material *temperature, double t_env, int *cnt, int *cols, double *V,
                                  double *VInv, double *Rytov)
{
  if (!g || !g->uploaded || !eps || !cnt || !cols || !V || !VInv || !Rytov)
    return fail(BFA_ERR_ARG, "bfa_overlap_blocks: bad argument");
  if (omega == 0.0) return fail(BFA_ERR_ARG, "bfa_overlap_blocks: omega = 0");
  const int N = g->nbf;
  int *dc = nullptr, *dcols = nullptr;
  cd *dV = nullptr, *dVI = nullptr;
  double *dR = nullptr;
  const size_t m = (size_t)N * MAXOVERLAP;
  int rc = BFA_OK;
  if (hipMalloc(&dc, (size_t)N * 4) != hipSuccess || hipMalloc(&dcols, m * 4) != hipSuccess ||
      hipMalloc(&dV, m * 16) != hipSuccess || hipMalloc(&dVI, m * 16) != hipSuccess || hipMalloc(&dR, m * 8) != hipSuccess)
    rc = fail(BFA_ERR_OOM, "bfa_overlap_blocks: allocation");
  if (!rc) rc = bfa::overlap_rows_device(g, omega, eps, temperature, t_env, dc, dcols, dV, dVI, dR, 0);
  if (!rc) {
    if (hipMemcpy(cnt, dc, (size_t)N * 4, hipMemcpyDeviceToHost) != hipSuccess ||
        hipMemcpy(cols, dcols, m * 4, hipMemcpyDeviceToHost) != hipSuccess ||
        hipMemcpy(V, dV, m * 16, hipMemcpyDeviceToHost) != hipSuccess ||
        hipMemcpy(VInv, dVI, m * 16, hipMemcpyDeviceToHost) != hipSuccess ||
        hipMemcpy(Rytov, dR, m * 8, hipMemcpyDeviceToHost) != hipSuccess)
      rc = fail(BFA_ERR_HIP, "bfa_overlap_blocks: %s", hipGetErrorString(hipGetLastError()));
  }
  (void)hipFree(dc); (void)hipFree(dcols); (void)hipFree(dV); (void)hipFree(dVI); (void)hipFree(dR);
  return rc;
}

// gram: gram_tet's blocks; null asks for the G block alone (AssembleGBlock)
__device__ __forceinline__ void near_entry(const DevGeom &g, double kre, double kim, const double *table,
                                           const cd *gram, cd *M, int64_t ld, int64_t j)
{
  const int a = g.pairRow[j], b = g.cols[j];
  const cd k = {kre, kim}, ik = {-kim, kre};
  const cd k2 = cmul(k, k);
  const cd ik2 = cmul(ik, ik);
  // column BF's 8 points in registers (the inner loop is unrolled); the row
  // BF's point is built per outer iteration, so no array is indexed by a
  // loop counter the compiler keeps rolled (that would spill to scratch)
  double bp[8][7];
#pragma unroll
  for (int pt = 0; pt < 8; pt++) bf_points4(g, b, pt, bp[pt]);
  cd acc = {0.0, 0.0};
  const cd ik2inv = cdiv({1.0, 0.0}, k2);          // 1/k^2, once per pair
  for (int ip = 0; ip < 8; ip++) {
    double ap[7];
    bf_points4(g, a, ip, ap);
#pragma unroll
    for (int jp = 0; jp < 8; jp++) {
      const double R0 = ap[0] - bp[jp][0], R1 = ap[1] - bp[jp][1], R2 = ap[2] - bp[jp][2];
      const double r2 = R0 * R0 + R1 * R1 + R2 * R2;
      if (r2 < 1.0e-24) continue;                  // r < 1e-12
      const double ir = rsqrt_nr(r2), r = r2 * ir;
      const double dot = ap[3] * bp[jp][3] + ap[4] * bp[jp][4] + ap[5] * bp[jp][5];
      const double dd = ap[6] * bp[jp][6];
      const cd pe = {dot - dd * ik2inv.re, -dd * ik2inv.im};
      const cd ef = exprel3(cscale(ik, r));
      acc = cadd(acc, cmul(pe, cscale(ef, ir * (1.0 / FOURPI))));
    }
  }
  // static part (GMatrixElements.cc:415-419)
  const double *G = table + 6 * j;
  const cd t0 = {G[0] - cdiv({G[1], 0.0}, k2).re, -cdiv({G[1], 0.0}, k2).im};
  const cd t1 = {G[2] - cdiv({G[3], 0.0}, k2).re, -cdiv({G[3], 0.0}, k2).im};
  const cd t2 = {G[4] - cdiv({G[5], 0.0}, k2).re, -cdiv({G[5], 0.0}, k2).im};
  acc = cadd(acc, cadd(t0, cadd(cmul(ik, t1), cmul(ik2, t2))));
  // Gram / chi^-1 block on shared tetrahedra (GetOverlaps)
  for (int sa = 0; sa < 2 && gram; sa++)
    for (int sb = 0; sb < 2; sb++) {
      const int t = g.bfT[2 * a + sa];
      if (t != g.bfT[2 * b + sb] || (a == b && sa != sb)) continue;
      int fa = 0, fb = 0;
      for (int f = 1; f < 4; f++) {
        const int i = g.tetFI[4 * t + f];
        if (i == a) fa = f;
        if (i == b) fb = f;
      }
      acc = cadd(acc, gram[(size_t)t * 16 + 4 * fa + fb]);
    }
  M[(size_t)b * ld + a] = acc;
  M[(size_t)a * ld + b] = acc;
}

__global__ __launch_bounds__(256) void k_near(DevGeom g, double kre, double kim, const double *table, const cd *gram,
                                              cd *M, int64_t ld)
{
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j < g.nnz) near_entry(g, kre, kim, table, gram, M, ld, j);
}

// The geometry has one moment table and one set of Gram blocks, for one
// frequency and one material, so assemblies of it on several streams or
// threads take turns: one call at a time is put on its stream, which waits for
// the last call's kernels.  (A captured call records no wait: its replays are
// ordered by whoever launches them.)
struct AssemblyTurn {
  bfa_geometry *g;
  hipStream_t st;
  std::lock_guard<std::mutex> lock;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  AssemblyTurn(bfa_geometry *g, hipStream_t st) : g(g), st(st), lock(g->turn)
  {
    (void)hipStreamIsCapturing(st, &cap);
    if (cap == hipStreamCaptureStatusNone) (void)hipStreamWaitEvent(st, (hipEvent_t)g->d.turnEv, 0);
  }
  ~AssemblyTurn()
  {
    if (cap == hipStreamCaptureStatusNone) (void)hipEventRecord((hipEvent_t)g->d.turnEv, st);
  }
};

// The closed-form materials' Gram kernel is compiled without the expression
// interpreter, whose stack is scratch memory.  kind < 0: no Gram block.
// Called within the geometry's AssemblyTurn.
static void launch_near(bfa_geometry *g, double omega_re, double omega_im, const bfa_material *mat, cd *M,
                        int64_t ld, hipStream_t st)
{
  const int64_t nnz = g->dg.nnz;
  cd *gram = mat->kind < 0 ? nullptr : (cd *)g->d.gram;
  if (nnz <= 0) return;
  if (gram && mat->kind == 4)
    hipLaunchKernelGGL(k_gram<true>, dim3(g->nt), dim3(64), 0, st, g->dg, omega_re, *mat, gram);
  else if (gram)
    hipLaunchKernelGGL(k_gram<false>, dim3(g->nt), dim3(64), 0, st, g->dg, omega_re, *mat, gram);
  hipLaunchKernelGGL(k_near, dim3((unsigned)((nnz + 255) / 256)), dim3(256), 0, st, g->dg, omega_re, omega_im,
                     (const double *)g->d.table, (const cd *)gram, M, ld);
}

// The two-pass far field's moment table (nt (nt + 1) / 2 records of 128 B,
// 6.9 GB at 10,368 tetrahedra), allocated on first use and kept with the
// geometry; null -- the single-pass kernel -- when it would take more than a
// quarter of the free device memory, when the allocation fails, or with
// BFA_FAR_TABLE=0.
static double *far_table(bfa_geometry *g)
{
  static int use = -1;
  if (use < 0) {
    const char *e = getenv("BFA_FAR_TABLE");
    use = !(e && strcmp(e, "0") == 0);
  }
  if (!use) return nullptr;
  const size_t need = (size_t)g->nt * (g->nt + 1) / 2 * 16 * sizeof(double);
  if (g->d.tpTab && g->d.tpTabBytes >= need) return (double *)g->d.tpTab;
  size_t fr = 0, tot = 0;
  if (hipMemGetInfo(&fr, &tot) != hipSuccess || need > fr / 4) return nullptr;
  void *p = nullptr;
  if (hipMalloc(&p, need) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  if (g->d.tpTab) (void)hipFree(g->d.tpTab);
  g->d.tpTab = p;
  g->d.tpTabBytes = need;
  return (double *)p;
}

static int assemble_vie(bfa_geometry *g, double omega_re, double omega_im, const bfa_material *mat, void *d_M,
                        int64_t ld, bool far32, void *stream)
{
  if (!g || !mat || !d_M) return fail(BFA_ERR_ARG, "bfa_assemble_vie: null argument");
  if (!g->uploaded || !g->static_built)
    return fail(BFA_ERR_STATE, "bfa_assemble_vie: call bfa_geometry_upload and bfa_static_build first");
  if (ld < g->nbf) return fail(BFA_ERR_ARG, "bfa_assemble_vie: ld %lld < N %d", (long long)ld, g->nbf);
  if (omega_re == 0.0 && omega_im == 0.0) return fail(BFA_ERR_ARG, "bfa_assemble_vie: omega = 0");
  hipStream_t st = (hipStream_t)stream;
  const int N = g->nbf;
  cd *M = (cd *)d_M;
  const int nt2 = (N + FT2 - 1) / FT2;
  const int64_t nblk2 = (int64_t)nt2 * (nt2 + 1) / 2;
  const bool rk = omega_im == 0.0;
  AssemblyTurn turn(g, st);
  double *tpt = far_table(g);
  if (tpt) {
    const int ntb = (g->nt + 31) / 32;
    const dim3 gr1((unsigned)((int64_t)ntb * (ntb + 1) / 2)), bl1(TPT_THREADS);
    if (far32) {
      if (rk) hipLaunchKernelGGL((k_tp_table<true, true>), gr1, bl1, 0, st, g->dg, omega_re, 0.0, tpt, ntb);
      else hipLaunchKernelGGL((k_tp_table<false, true>), gr1, bl1, 0, st, g->dg, omega_re, omega_im, tpt, ntb);
    } else {
      if (rk) hipLaunchKernelGGL((k_tp_table<true, false>), gr1, bl1, 0, st, g->dg, omega_re, 0.0, tpt, ntb);
      else hipLaunchKernelGGL((k_tp_table<false, false>), gr1, bl1, 0, st, g->dg, omega_re, omega_im, tpt, ntb);
    }
    if (g->ft_max <= 40)
      hipLaunchKernelGGL(k_far_gather<40>, dim3((unsigned)nblk2), dim3(GS_NT), 0, st, g->dg, omega_re, omega_im,
                         (const double *)tpt, M, ld, nt2);
    else
      hipLaunchKernelGGL(k_far_gather<64>, dim3((unsigned)nblk2), dim3(GS_NT), 0, st, g->dg, omega_re, omega_im,
                         (const double *)tpt, M, ld, nt2);
  } else {
    const dim3 gr2((unsigned)nblk2), bl2(FT_THREADS);
    if (far32) {
      if (rk) hipLaunchKernelGGL((k_far_tp<true, true>), gr2, bl2, 0, st, g->dg, omega_re, 0.0, M, ld, nt2);
      else hipLaunchKernelGGL((k_far_tp<false, true>), gr2, bl2, 0, st, g->dg, omega_re, omega_im, M, ld, nt2);
    } else {
      if (rk) hipLaunchKernelGGL((k_far_tp<true, false>), gr2, bl2, 0, st, g->dg, omega_re, 0.0, M, ld, nt2);
      else hipLaunchKernelGGL((k_far_tp<false, false>), gr2, bl2, 0, st, g->dg, omega_re, omega_im, M, ld, nt2);
    }
  }
  launch_near(g, omega_re, omega_im, mat, M, ld, st);
  HIPCHECK(hipGetLastError());
  return BFA_OK;
}

extern "C" int bfa_assemble_vie(bfa_geometry *g, double omega_re, double omega_im, const bfa_material *mat,
                                void *d_M, int64_t ld, void *stream)
{
  return assemble_vie(g, omega_re, omega_im, mat, d_M, ld, false, stream);
}

// SWGGeometry::AssembleGBlock(no, no, ...) (VIEMatrix.cc:365-426): the G
// block without the chi^-1 overlap terms
extern "C" int bfa_assemble_g(bfa_geometry *g, double omega_re, double omega_im, void *d_M, int64_t ld, void *stream)
{
  bfa_material none;
  memset(&none, 0, sizeof none);
  none.kind = -1;
  return assemble_vie(g, omega_re, omega_im, &none, d_M, ld, false, stream);
}

extern "C" int bfa_assemble_vie_far32(bfa_geometry *g, double omega_re, double omega_im, const bfa_material *mat,
                                      void *d_M, int64_t ld, void *stream)
{
  return assemble_vie(g, omega_re, omega_im, mat, d_M, ld, true, stream);
}

int bfa::assemble_near_only(bfa_geometry *g, double omega_re, double omega_im, const bfa_material *mat, void *d_M,
                            int64_t ld, void *stream)
{
  if (!g || !mat || !d_M) return fail(BFA_ERR_ARG, "assemble_near_only: null argument");
  if (!g->uploaded || !g->static_built) return fail(BFA_ERR_STATE, "assemble_near_only: static table not built");
  AssemblyTurn turn(g, (hipStream_t)stream);
  launch_near(g, omega_re, omega_im, mat, (cd *)d_M, ld, (hipStream_t)stream);
  HIPCHECK(hipGetLastError());
  return BFA_OK;
}

// ===========================================================================
// RHS: v_a = -1/(i omega Z0) int b_a . E_inc (TetCR33 on both tetrahedra)
// ===========================================================================
__device__ cd bf_dot_pw(const DevGeom &g, int a, const bfa_planewave &pw, double k)
{
  cd acc = {0.0, 0.0};
  for (int side = 0; side < 2; side++) {
    const int t = g.bfT[2 * a + side];
    const double pf = g.bfPF[2 * a + side];
    const double *Q = g.bfQ + 6 * a + 3 * side;
    const double *q = g.q33 + (size_t)t * 33 * 4;
    for (int i = 0; i < 33; i++) {
      const double x0 = q[4 * i], x1 = q[4 * i + 1], x2 = q[4 * i + 2], w = q[4 * i + 3];
      double s, c;
      sincos(k * (pw.dir[0] * x0 + pw.dir[1] * x1 + pw.dir[2] * x2), &s, &c);
      const double b0 = pf * (x0 - Q[0]), b1 = pf * (x1 - Q[1]), b2 = pf * (x2 - Q[2]);
      const double er = b0 * pw.E0[0] + b1 * pw.E0[2] + b2 * pw.E0[4];
      const double ei = b0 * pw.E0[1] + b1 * pw.E0[3] + b2 * pw.E0[5];
      acc.re += w * (er * c - ei * s);
      acc.im += w * (er * s + ei * c);
    }
  }
  return acc;
}

#define MAXPW 32
struct PWList { bfa_planewave pw[MAXPW]; };

__global__ void k_rhs(DevGeom g, double omega, PWList pws, int npw, cd *B, int64_t ldb)
{
  const int a = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y;
  if (a >= g.nbf || j >= npw) return;
  const cd v = bf_dot_pw(g, a, pws.pw[j], omega);
  // -1/(i omega Z0) * v = (i / (omega Z0)) * v
  const double s = 1.0 / (omega * ZVAC);
  B[(size_t)j * ldb + a] = {-v.im * s, v.re * s};
}

extern "C" int bfa_assemble_rhs(bfa_geometry *g, double omega, const bfa_planewave *pw, int npw, void *d_B,
                                int64_t ldb, void *stream)
{
  if (!g || !pw || !d_B || npw <= 0) return fail(BFA_ERR_ARG, "bfa_assemble_rhs: bad argument");
  if (!g->uploaded) return fail(BFA_ERR_STATE, "bfa_assemble_rhs: geometry not uploaded");
  if (npw > MAXPW) return fail(BFA_ERR_ARG, "bfa_assemble_rhs: at most %d plane waves per call", MAXPW);
  if (ldb < g->nbf) return fail(BFA_ERR_ARG, "bfa_assemble_rhs: ldb < N");
  if (omega == 0.0) return fail(BFA_ERR_ARG, "bfa_assemble_rhs: omega = 0");
  PWList l;
  memset(&l, 0, sizeof l);
  for (int j = 0; j < npw; j++) l.pw[j] = pw[j];
  hipLaunchKernelGGL(k_rhs, dim3((g->nbf + 127) / 128, npw), dim3(128), 0, (hipStream_t)stream, g->dg, omega, l,
                     npw, (cd *)d_B, ldb);
  HIPCHECK(hipGetLastError());
  return BFA_OK;
}

// ===========================================================================
// EMT power.  Q_ab = omega * int int PEFIE sin(kr)/(4 pi r) (same object,
// EMTPFT.cc:216-319), rule size by ncv and kR; dense symmetric Q in a
// scratch buffer, then P_scat = Z0 * sum_{a<=b} Re(J_a^* J_b) Q_ab
// = Z0/2 * [Re(J^H Q J) + sum_a |J_a|^2 Q_aa];  P_ext = 1/2 sum Re(J^* <b,E>).
// ===========================================================================
__device__ double emt_tetpair(const DevGeom &g, int ta, double pfa, const double *Qa, int tb, double pfb,
                              const double *Qb, int np, double k)
{
  const double *qa = np == 4 ? g.q4 : np == 16 ? g.q16 : g.q33;
  const double *qb = qa + (size_t)tb * np * 4;
  qa += (size_t)ta * np * 4;
  const double divdiv = 9.0 * pfa * pfb;
  double acc = 0.0;
  for (int i = 0; i < np; i++) {
    const double xa0 = qa[4 * i], xa1 = qa[4 * i + 1], xa2 = qa[4 * i + 2], wa = qa[4 * i + 3];
    const double ba0 = pfa * (xa0 - Qa[0]), ba1 = pfa * (xa1 - Qa[1]), ba2 = pfa * (xa2 - Qa[2]);
    for (int j = 0; j < np; j++) {
      const double xb0 = qb[4 * j], xb1 = qb[4 * j + 1], xb2 = qb[4 * j + 2], wb = qb[4 * j + 3];
      const double R0 = xa0 - xb0, R1 = xa1 - xb1, R2 = xa2 - xb2;
      const double r = sqrt(R0 * R0 + R1 * R1 + R2 * R2), kr = k * r;
      const double dot = ba0 * pfb * (xb0 - Qb[0]) + ba1 * pfb * (xb1 - Qb[1]) + ba2 * pfb * (xb2 - Qb[2]);
      const double pe = dot - divdiv / (k * k);
      double im;
      if (fabs(kr) < 2.0e-2) im = (1.0 - kr * kr / 6.0) * k / FOURPI;
      else im = sin(kr) / (FOURPI * r);
      acc += wa * wb * k * pe * im;
    }
  }
  return acc;
}

// Tetrahedron-pair form of Q for the pairs on the 4-point rule (no shared
// vertex, |omega| max(r_a, r_b) <= 5): the same regrouping as the far field
// with the real kernel k Im g / 4pi = k sin(kr) / (4 pi r) (series below
// |kr| = 0.02); other pairs run emt_tetpair's rule directly.
// Row tetrahedron us's points are read from sh (as in tp_moments).
__device__ __forceinline__ void emt_moments(const FarTpShared &sh, int us, const double *cS, const double *ys,
                                            const double *cT, double k, double *out, int stride)
{
  double m[8];
#pragma unroll
  for (int i = 0; i < 8; i++) m[i] = 0.0;
#pragma unroll 1
  for (int p = 0; p < 4; p++) {
    double x[4];
#pragma unroll
    for (int e = 0; e < 4; e++) x[e] = sh.pts[0][4 * p + e][us];
    const double xi0 = x[0] - cS[0], xi1 = x[1] - cS[1], xi2 = x[2] - cS[2];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const double *y = ys + 4 * q;
      const double R0 = x[0] - y[0], R1 = x[1] - y[1], R2 = x[2] - y[2];
      const double r = sqrt(R0 * R0 + R1 * R1 + R2 * R2), kr = k * r;
      double im;
      if (fabs(kr) < 2.0e-2) im = (1.0 - kr * kr / 6.0) * k / FOURPI;
      else im = sin(kr) / (FOURPI * r);
      const double gv = x[3] * y[3] * k * im;
      const double e0 = y[0] - cT[0], e1 = y[1] - cT[1], e2 = y[2] - cT[2];
      m[0] += gv;
      m[1] += gv * xi0; m[2] += gv * xi1; m[3] += gv * xi2;
      m[4] += gv * e0; m[5] += gv * e1; m[6] += gv * e2;
      m[7] += gv * (xi0 * e0 + xi1 * e1 + xi2 * e2);
    }
  }
#pragma unroll
  for (int i = 0; i < 8; i++) out[i * stride] = m[i];
}

__device__ void emt_tp_tile(const DevGeom &g, double omega, double *Q, int64_t ldq, int ti, int tj, FarTpShared &sh)
{
  const int tid = threadIdx.x, nth = blockDim.x, N = g.nbf;
  const int *tab[2] = {g.ftTab + (size_t)ti * FTAB, g.ftTab + (size_t)tj * FTAB};
  const int nr = tab[0][4 * FT2], nc = tab[1][4 * FT2];
  for (int idx = tid; idx < 2 * 2 * FT2; idx += nth) {
    const int which = idx / (2 * FT2), k = idx % (2 * FT2);
    sh.slot[which][k] = tab[which][2 * FT2 + k];
  }
  for (int idx = tid; idx < 2 * 2 * FT2 * 16; idx += nth) {
    const int which = idx / (2 * FT2 * 16), rem = idx % (2 * FT2 * 16);
    const int u = rem / 16, e = rem % 16;
    if (u < (which ? nc : nr)) sh.pts[which][e][u] = g.q4[(size_t)tab[which][u] * 16 + e];
  }
  __syncthreads();
  for (int idx = tid; idx < 2 * 2 * FT2; idx += nth) {
    const int which = idx / (2 * FT2), u = idx % (2 * FT2);
    if (u < (which ? nc : nr))
      for (int d = 0; d < 3; d++)
        sh.cen[which][d][u] = 0.25 * (sh.pts[which][d][u] + sh.pts[which][4 + d][u] + sh.pts[which][8 + d][u] +
                                      sh.pts[which][12 + d][u]);
  }
  __syncthreads();
  const bool direct = nr * nc > FTT_MAX;
  if (!direct) {
    for (int pidx = tid; pidx < nr * nc; pidx += nth) {
      const int us = pidx / nc, ut = pidx % nc;
      double xs[16], cS[3], ys[16], cT[3];
      tp_load(sh, 0, us, xs, cS);
      tp_load(sh, 1, ut, ys, cT);
      emt_moments(sh, us, cS, ys, cT, omega, &sh.mom[0][pidx], FTT_MAX);
    }
  }
  __syncthreads();
  const double ik2 = 9.0 / (omega * omega);
  for (int pidx = tid; pidx < FT2 * FT2; pidx += nth) {
    const int lb = pidx % FT2, la = pidx / FT2;
    const int a = ti * FT2 + la, b = tj * FT2 + lb;
    if (a >= N || b >= N || b < a) continue;
    // pairs sharing a vertex: emt_near_pair
    if (bf_ncv(g.bfV + 5 * a, g.bfV + 5 * b) > 0) continue;
    double q = 0.0;
    if (fabs(omega) * fmax(g.bfRad[a], g.bfRad[b]) > 5.0) {
      for (int sa = 0; sa < 2; sa++)
        for (int sb = 0; sb < 2; sb++)
          q += emt_tetpair(g, g.bfT[2 * a + sa], g.bfPF[2 * a + sa], g.bfQ + 6 * a + 3 * sa, g.bfT[2 * b + sb],
                           g.bfPF[2 * b + sb], g.bfQ + 6 * b + 3 * sb, 16, omega);
    } else {
      for (int sa = 0; sa < 2; sa++) {
        const int us = sh.slot[0][2 * la + sa];
        const double pfa = g.bfPF[2 * a + sa];
        const double *Qa = g.bfQ + 6 * a + 3 * sa;
        const double al0 = Qa[0] - sh.cen[0][0][us], al1 = Qa[1] - sh.cen[0][1][us], al2 = Qa[2] - sh.cen[0][2][us];
        for (int sb = 0; sb < 2; sb++) {
          const int ut = sh.slot[1][2 * lb + sb];
          const double pfb = g.bfPF[2 * b + sb];
          const double *Qb = g.bfQ + 6 * b + 3 * sb;
          const double be0 = Qb[0] - sh.cen[1][0][ut], be1 = Qb[1] - sh.cen[1][1][ut],
                       be2 = Qb[2] - sh.cen[1][2][ut];
          double m[8];
          if (direct) {
            double xs[16], cS[3], ys[16], cT[3];
            tp_load(sh, 0, us, xs, cS);
            tp_load(sh, 1, ut, ys, cT);
            emt_moments(sh, us, cS, ys, cT, omega, m, 1);
          } else {
#pragma unroll
            for (int i = 0; i < 8; i++) m[i] = sh.mom[i][us * nc + ut];
          }
          const double ab = al0 * be0 + al1 * be1 + al2 * be2;
          q += pfa * pfb *
               (m[7] - (be0 * m[1] + be1 * m[2] + be2 * m[3]) - (al0 * m[4] + al1 * m[5] + al2 * m[6]) + ab * m[0] -
                ik2 * m[0]);
        }
      }
    }
    Q[(size_t)b * ldq + a] = q;
    Q[(size_t)a * ldq + b] = q;
  }
}

// Q for touching pair j of the CSR list (16-point rule, 33 at high kR)
__device__ __forceinline__ void emt_near_pair(const DevGeom &g, double omega, double *Q, int64_t ldq, int64_t j)
{
  const int a = g.pairRow[j], b = g.cols[j];
  const bool hf = fabs(omega) * fmax(g.bfRad[a], g.bfRad[b]) > 5.0;
  const int np = hf ? 33 : 16;
  double q = 0.0;
  for (int sa = 0; sa < 2; sa++)
    for (int sb = 0; sb < 2; sb++)
      q += emt_tetpair(g, g.bfT[2 * a + sa], g.bfPF[2 * a + sa], g.bfQ + 6 * a + 3 * sa, g.bfT[2 * b + sb],
                       g.bfPF[2 * b + sb], g.bfQ + 6 * b + 3 * sb, np, omega);
  Q[(size_t)b * ldq + a] = q;
  Q[(size_t)a * ldq + b] = q;
}

__global__ __launch_bounds__(256) void k_emt_near(DevGeom g, double omega, double *Q, int64_t ldq)
{
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j < g.nnz) emt_near_pair(g, omega, Q, ldq, j);
}

__global__ __launch_bounds__(FT_THREADS) void k_emt_q(DevGeom g, double omega, double *Q, int64_t ldq, int ntiles)
{
  __shared__ FarTpShared sh;
  int ti, tj;
  tile_coords(blockIdx.x, ntiles, ti, tj);
  emt_tp_tile(g, omega, Q, ldq, ti, tj, sh);
}

// extinction: per (a, j) Re(conj(J_aj) <b_a, E_j>), summed over the block's rows
__device__ __forceinline__ void emt_ext_block(const DevGeom &g, double omega, const cd *Jj, const bfa_planewave &pw,
                                              int blk, double *out)
{
  __shared__ double re[256];
  const int a = blk * 256 + threadIdx.x;
  double e = 0.0;
  if (a < g.nbf) {
    const cd qe = bf_dot_pw(g, a, pw, omega), ja = Jj[a];
    e = ja.re * qe.re + ja.im * qe.im;
  }
  re[threadIdx.x] = e;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) re[threadIdx.x] += re[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = re[0];
}

__global__ __launch_bounds__(256) void k_emt_ext(DevGeom g, double omega, const cd *J, int64_t ldj, PWList pws,
                                                 double *part)
{
  const int j = blockIdx.y;
  emt_ext_block(g, omega, J + (size_t)j * ldj, pws.pw[j], blockIdx.x, part + (size_t)j * gridDim.x + blockIdx.x);
}

// ===========================================================================
// Fields at evaluation points (SWGGeometry::GetFields, GetFields.cc:288-382):
// per point X and BF a, Get1BFFields' volume integral (GetFields.cc:181-224,
// 285-299) with the 4-point rule when |X - centroid| > 10 radius, else 16:
//   E = i Omega Z0 sum_x w G(X - x).b(x),   H = -i Omega sum_x w C(X - x).b(x),
// G = (I + grad grad / k^2) e^{ikr}/(4 pi r), C.b = -(1 + i/kr) e^{ikr}/(4 pi r) Rhat x b
// (the dyadic Green's function pair of CalcGC in vacuum, k = Omega; H = curl
// of the vector potential, so curl E = i Omega Z0 H), times J_a, summed; plus
// the incident plane waves, H_inc = nhat x E_inc / Z0.
// ===========================================================================
#define FLD_TETS 1024      // tetrahedra of a workgroup ...
#define FLD_FEW 256        // ... where that would leave CUs idle
#define FLD_BLOCKS 1024

// sum_i w_i G.j, C.j over a rule's points of tetrahedron t, j = A (x - c) - B
// complex; o: E (re, im) x 3, H (re, im) x 3
__device__ __forceinline__ void tet_field(const double *q, int np, const double *c, const double *x, double k,
                                          double invk, const double *A, const double *B, double *o)
{
  for (int i = 0; i < np; i++) {
    const double xs[3] = {q[4 * i], q[4 * i + 1], q[4 * i + 2]}, w = q[4 * i + 3] * (1.0 / FOURPI);
    const double R0 = x[0] - xs[0], R1 = x[1] - xs[1], R2 = x[2] - xs[2];
    const double r2 = R0 * R0 + R1 * R1 + R2 * R2, ir = rsqrt_nr(r2);
    const double u[3] = {R0 * ir, R1 * ir, R2 * ir};
    double sn, cs;
    sincos_mod(k * (r2 * ir), &sn, &cs);
    const double gw = w * ir, h = invk * ir, h2 = h * h;
    const cd gf = {cs * gw, sn * gw};
    // f1 = 1 + i/(kr) - 1/(kr)^2, f2 = -1 - 3i/(kr) + 3/(kr)^2, f3 = -(1 + i/(kr))
    const cd f1 = cmul(gf, cd{1.0 - h2, h}), f2 = cmul(gf, cd{3.0 * h2 - 1.0, -3.0 * h}), f3 = cmul(gf, cd{-1.0, -h});
    cd j[3];
#pragma unroll
    for (int m = 0; m < 3; m++) {
      const double d = xs[m] - c[m];
      j[m] = {A[0] * d - B[2 * m], A[1] * d - B[2 * m + 1]};
    }
    const cd uj = {u[0] * j[0].re + u[1] * j[1].re + u[2] * j[2].re, u[0] * j[0].im + u[1] * j[1].im + u[2] * j[2].im};
    const cd g = cmul(f2, uj);
#pragma unroll
    for (int m = 0; m < 3; m++) {
      const int m1 = (m + 1) % 3, m2 = (m + 2) % 3;
      const cd cr = {u[m1] * j[m2].re - u[m2] * j[m1].re, u[m1] * j[m2].im - u[m2] * j[m1].im};
      o[2 * m] += f1.re * j[m].re - f1.im * j[m].im + u[m] * g.re;
      o[2 * m + 1] += f1.re * j[m].im + f1.im * j[m].re + u[m] * g.im;
      o[6 + 2 * m] += f3.re * cr.re - f3.im * cr.im;
      o[7 + 2 * m] += f3.re * cr.im + f3.im * cr.re;
    }
  }
}

// Thread: tetrahedra of a chunk, workgroup: (chunk, point).  Bound by FP64
// arithmetic.  The currents of a tetrahedron's BFs on the same rule add up to
// one polynomial A (x - c) - B, so each cubature point is evaluated once for
// up to four BFs, with a complex current; a BF's own choice of the rule stays.
// BF by BF (two tetrahedra each, library sqrt, division and sincos), 5,760
// BFs at 1,000 points took 1.35 ms, now 0.47.
__global__ __launch_bounds__(256) void k_fields(DevGeom g, double omega, const cd *__restrict__ J, const double *X,
                                                int nchunk, int chunk, cd *part)
{
  const int p = blockIdx.y, tid = threadIdx.x;
  const int t0 = blockIdx.x * chunk, t1 = min(g.nt, t0 + chunk);
  const double x[3] = {X[3 * p], X[3 * p + 1], X[3 * p + 2]};
  const double k = omega, invk = 1.0 / omega;
  double acc[12];
#pragma unroll
  for (int c = 0; c < 12; c++) acc[c] = 0.0;
  for (int t = t0 + tid; t < t1; t += 256) {
    const double *cen = g.tetVol + g.nt + 3 * t;
    const double c[3] = {cen[0], cen[1], cen[2]};
    double A[2][2] = {}, B[2][6] = {};   // 16-point, 4-point rule
    bool any[2] = {false, false};
#pragma unroll
    for (int f = 0; f < 4; f++) {
      const int a = g.tetFI[4 * t + f];
      if (a >= g.nbf) continue;
      const double *v1 = g.V + 3 * g.bfV[5 * a + 1], *v2 = g.V + 3 * g.bfV[5 * a + 2], *v3 = g.V + 3 * g.bfV[5 * a + 3];
      const double d0 = x[0] - (v1[0] + v2[0] + v3[0]) / 3.0, d1 = x[1] - (v1[1] + v2[1] + v3[1]) / 3.0,
                   d2 = x[2] - (v1[2] + v2[2] + v3[2]) / 3.0;
      const bool farp = sqrt(d0 * d0 + d1 * d1 + d2 * d2) > 10.0 * g.bfRad[a];
      const int side = g.bfT[2 * a] == t ? 0 : 1;
      const double pf = g.bfPF[2 * a + side];
      const double *Q = g.bfQ + 6 * a + 3 * side;
      const cd j = {pf * J[a].re, pf * J[a].im};
      const double q[3] = {Q[0] - c[0], Q[1] - c[1], Q[2] - c[2]};
#pragma unroll
      for (int e = 0; e < 2; e++) {
        if (farp != (e == 1)) continue;
        any[e] = true;
        A[e][0] += j.re; A[e][1] += j.im;
#pragma unroll
        for (int m = 0; m < 3; m++) { B[e][2 * m] += j.re * q[m]; B[e][2 * m + 1] += j.im * q[m]; }
      }
    }
    if (any[0]) tet_field(g.q16 + (size_t)t * 64, 16, c, x, k, invk, A[0], B[0], acc);
    if (any[1]) tet_field(g.q4 + (size_t)t * 16, 4, c, x, k, invk, A[1], B[1], acc);
  }
  __shared__ double red[4][12];
#pragma unroll
  for (int c = 0; c < 12; c++) {
    const double v = wave_sum(acc[c]);
    if ((tid & 63) == 0) red[tid >> 6][c] = v;
  }
  __syncthreads();
  // E *= i Omega Z0, H *= -i Omega
  if (tid < 6) {
    const cd v = {red[0][2 * tid] + red[1][2 * tid] + red[2][2 * tid] + red[3][2 * tid],
                  red[0][2 * tid + 1] + red[1][2 * tid + 1] + red[2][2 * tid + 1] + red[3][2 * tid + 1]};
    part[((size_t)p * nchunk + blockIdx.x) * 6 + tid] = cmul(v, cd{0.0, tid < 3 ? omega * ZVAC : -omega});
  }
}

__global__ void k_fields_final(int npts, int nchunk, const cd *part, double omega, PWList pws, int npw, const double *X,
                               cd *F)
{
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= npts) return;
  cd f[6];
  for (int c = 0; c < 6; c++) {
    f[c] = {0.0, 0.0};
    for (int q = 0; q < nchunk; q++) f[c] = cadd(f[c], part[((size_t)p * nchunk + q) * 6 + c]);
  }
  const double *x = X + 3 * p;
  for (int j = 0; j < npw; j++) {
    const bfa_planewave &w = pws.pw[j];
    double sn, cs;
    sincos(omega * (w.dir[0] * x[0] + w.dir[1] * x[1] + w.dir[2] * x[2]), &sn, &cs);
    cd e[3];
    for (int m = 0; m < 3; m++) e[m] = cmul(cd{w.E0[2 * m], w.E0[2 * m + 1]}, cd{cs, sn});
    const double *n = w.dir;
    const cd h[3] = {csub(cscale(e[2], n[1]), cscale(e[1], n[2])), csub(cscale(e[0], n[2]), cscale(e[2], n[0])),
                     csub(cscale(e[1], n[0]), cscale(e[0], n[1]))};
    for (int m = 0; m < 3; m++) {
      f[m] = cadd(f[m], e[m]);
      f[3 + m] = cadd(f[3 + m], cscale(h[m], 1.0 / ZVAC));
    }
  }
  for (int c = 0; c < 6; c++) F[(size_t)p * 6 + c] = f[c];
}

extern "C" int bfa_get_fields(bfa_geometry *g, double omega, const bfa_planewave *pw, int npw, const void *d_J,
                              int npts, const double *X, double *F, void *stream)
{
  if (!g || !g->uploaded) return fail(BFA_ERR_STATE, "bfa_get_fields: geometry not uploaded");
  if (npts < 0 || npw < 0 || npw > MAXPW || (npts > 0 && (!X || !F)) || (npw > 0 && !pw))
    return fail(BFA_ERR_ARG, "bfa_get_fields: bad argument");
  if (npts == 0) return BFA_OK;
  hipStream_t st = (hipStream_t)stream;
  const int chunk = (int64_t)npts * ((g->nt + FLD_TETS - 1) / FLD_TETS) < FLD_BLOCKS ? FLD_FEW : FLD_TETS;
  const int nchunk = d_J ? (g->nt + chunk - 1) / chunk : 0;
  double *dX = nullptr;
  cd *dF = nullptr, *part = nullptr;
  HIPCHECK(hipMalloc(&dX, (size_t)npts * 24));
  int rc = BFA_OK;
  if (hipMalloc(&dF, (size_t)npts * 6 * 16) != hipSuccess ||
      hipMalloc(&part, std::max<size_t>((size_t)npts * nchunk * 6 * 16, 16)) != hipSuccess)
    rc = fail(BFA_ERR_OOM, "bfa_get_fields: allocation");
  if (!rc && hipMemcpyAsync(dX, X, (size_t)npts * 24, hipMemcpyHostToDevice, st) != hipSuccess)
    rc = fail(BFA_ERR_HIP, "bfa_get_fields: upload");
  if (!rc) {
    PWList l;
    memset(&l, 0, sizeof l);
    for (int j = 0; j < npw; j++) l.pw[j] = pw[j];
    if (nchunk)
      hipLaunchKernelGGL(k_fields, dim3(nchunk, npts), dim3(256), 0, st, g->dg, omega, (const cd *)d_J,
                         (const double *)dX, nchunk, chunk, part);
    hipLaunchKernelGGL(k_fields_final, dim3((npts + 63) / 64), dim3(64), 0, st, npts, nchunk, (const cd *)part, omega,
                       l, npw, (const double *)dX, dF);
    if (hipMemcpyAsync(F, dF, (size_t)npts * 6 * 16, hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
      rc = fail(BFA_ERR_HIP, "bfa_get_fields: %s", hipGetErrorString(hipGetLastError()));
  }
  (void)hipFree(dX);
  (void)hipFree(dF);
  (void)hipFree(part);
  return rc;
}

namespace bfa {
// Q_ab = Im Q_PSCAT of GetScatteredPFTIntegrals for every BF pair, both
// triangles (N x N real, ld >= N): far pairs by tetrahedron-pair tiles,
// touching pairs by the 16/33-point rule
void emt_q_matrix(const bfa_geometry *g, double omega, double *Q, int64_t ldq, hipStream_t st)
{
  const int N = g->nbf;
  const int nt2 = (N + FT2 - 1) / FT2;
  hipLaunchKernelGGL(k_emt_q, dim3((unsigned)((int64_t)nt2 * (nt2 + 1) / 2)), dim3(FT_THREADS), 0, st, g->dg, omega,
                     Q, ldq, nt2);
  if (g->dg.nnz > 0)
    hipLaunchKernelGGL(k_emt_near, dim3((unsigned)((g->dg.nnz + 255) / 256)), dim3(256), 0, st, g->dg, omega, Q,
                       ldq);
}
}  // namespace bfa

extern "C" int bfa_emt_power(bfa_geometry *g, double omega, const bfa_planewave *pw, int npw, const void *d_J,
                             int64_t ldj, double *out, void *stream)
{
  if (!g || !pw || !d_J || !out || npw <= 0) return fail(BFA_ERR_ARG, "bfa_emt_power: bad argument");
  if (!g->uploaded) return fail(BFA_ERR_STATE, "bfa_emt_power: geometry not uploaded");
  if (npw > MAXPW) return fail(BFA_ERR_ARG, "bfa_emt_power: at most %d plane waves", MAXPW);
  if (omega == 0.0) return fail(BFA_ERR_ARG, "bfa_emt_power: omega = 0");
  hipStream_t st = (hipStream_t)stream;
  const int N = g->nbf;
  // scattered sums [npw], extinction partials [npw][nb], then work space
  const int nb = (N + 255) / 256;
  const size_t nout = (size_t)npw * (nb + 1);
  double *d = nullptr;
  HIPCHECK(hipMalloc(&d, (nout + bfa::emt_work_doubles(g->nt, npw)) * 8));
  PWList l;
  memset(&l, 0, sizeof l);
  for (int j = 0; j < npw; j++) l.pw[j] = pw[j];
  bfa::launch_emt_scattered(g->dg, omega, d_J, ldj, npw, d + nout, d, st);
  hipLaunchKernelGGL(k_emt_ext, dim3(nb, npw), dim3(256), 0, st, g->dg, omega, (const cd *)d_J, ldj, l, d + npw);
  std::vector<double> h(nout);
  hipError_t e1 = hipGetLastError();
  hipError_t e2 = hipMemcpyAsync(h.data(), d, nout * 8, hipMemcpyDeviceToHost, st);
  hipError_t e3 = hipStreamSynchronize(st);
  hipFree(d);
  if (e1 != hipSuccess || e2 != hipSuccess || e3 != hipSuccess)
    return fail(BFA_ERR_HIP, "bfa_emt_power kernels failed");
  for (int j = 0; j < npw; j++) {
    const double s = h[j];
    double x = 0.0;
    for (int i = 0; i < nb; i++) x += h[(size_t)npw + (size_t)j * nb + i];
    const double pscat = ZVAC * 0.5 * s;
    const double pext = 0.5 * x;
    out[2 * j] = pext - pscat;
    out[2 * j + 1] = pscat;
  }
  return BFA_OK;
}

// ===========================================================================
// Grouped (batch) kernels: every instance's work in one launch; the
// frequency comes from device memory so that one captured graph serves a
// whole sweep.
// ===========================================================================
enum { GF_FAR = 0, GF_NEAR, GF_ROW, GF_TAB };
__device__ __forceinline__ int inst_first(const AsmInst &q, int which)
{
  return which == GF_FAR ? q.far0 : which == GF_NEAR ? q.near0 : which == GF_ROW ? q.row0 : q.tab0;
}
__device__ __forceinline__ int find_inst(const AsmInst *__restrict__ d, int n, int bid, int which)
{
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (inst_first(d[mid], which) <= bid) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// REALK: the host guarantees omega_im == 0 for every frequency replayed
// through this launch (one kernel holding both variants spills 592 B/lane,
// the real-k one alone 144 B/lane, as the single-matrix k_far_tp<true>)
template <bool REALK>
__global__ __launch_bounds__(FT_THREADS) void kg_far(const AsmInst *__restrict__ d, int ni, const FreqState *fs)
{
  __shared__ FarTpShared sh;
  const AsmInst &q = d[find_inst(d, ni, blockIdx.x, GF_FAR)];
  int ti, tj;
  tile_coords(blockIdx.x - q.far0, q.ntiles, ti, tj);
  far_tp_tile<REALK>(q.g, fs->omega_re, REALK ? 0.0 : fs->omega_im, (cd *)q.M, q.ldm, ti, tj, sh);
}

// the two-pass far field over the instances (as k_tp_table, k_far_gather)
template <bool REALK>
__global__ __launch_bounds__(TPT_THREADS) void kg_tp_table(const AsmInst *__restrict__ d, int ni, const FreqState *fs)
{
  __shared__ TpTileShared sh;
  const AsmInst &q = d[find_inst(d, ni, blockIdx.x, GF_TAB)];
  int bs, bt;
  tile_coords(blockIdx.x - q.tab0, q.ntb, bs, bt);
  tp_table_tile<REALK, false>(q.g, fs->omega_re, REALK ? 0.0 : fs->omega_im, q.tpt, bs, bt, sh);
}

template <int NC>
__global__ __launch_bounds__(GS_NT, 4) void kg_far_gather(const AsmInst *__restrict__ d, int ni, const FreqState *fs)
{
  __shared__ GatherShared<NC> sh;
  const AsmInst &q = d[find_inst(d, ni, blockIdx.x, GF_FAR)];
  int ti, tj;
  tile_coords(blockIdx.x - q.far0, q.ntiles, ti, tj);
  far_gather_tile<NC>(q.g, fs->omega_re, fs->omega_im, q.tpt, (cd *)q.M, q.ldm, ti, tj, sh);
}

// EXPR: some instance's material is a compiled SVTensor (as k_gram)
template <bool EXPR>
__global__ __launch_bounds__(64) void kg_gram(const AsmInst *__restrict__ d, const FreqState *fs)
{
  __shared__ GramShared sh;
  const AsmInst &q = d[blockIdx.y];
  for (int t = blockIdx.x; t < q.g.nt; t += gridDim.x) {
    __syncthreads();
    gram_tet<EXPR>(q.g, t, fs->omega_re, q.mat, (cd *)q.gram + (size_t)t * 16, sh);
  }
}

__global__ __launch_bounds__(256) void kg_near(const AsmInst *__restrict__ d, int ni, const FreqState *fs)
{
  const AsmInst &q = d[find_inst(d, ni, blockIdx.x, GF_NEAR)];
  const int64_t j = (int64_t)(blockIdx.x - q.near0) * blockDim.x + threadIdx.x;
  if (j < q.g.nnz)
    near_entry(q.g, fs->omega_re, fs->omega_im, q.table, (const cd *)q.gram, (cd *)q.M, q.ldm, j);
}

__global__ __launch_bounds__(256) void kg_rhs(const AsmInst *__restrict__ d, int ni, const FreqState *fs,
                                              PWBatch pws, int npw)
{
  const AsmInst &q = d[find_inst(d, ni, blockIdx.x, GF_ROW)];
  const int a = (blockIdx.x - q.row0) * blockDim.x + threadIdx.x;
  const int j = blockIdx.y;
  if (a >= q.g.nbf || j >= npw) return;
  const double omega = fs->omega_re;
  const cd v = bf_dot_pw(q.g, a, pws.pw[j], omega);
  const double s = 1.0 / (omega * ZVAC);
  ((cd *)q.B)[(size_t)j * q.ldb + a] = {-v.im * s, v.re * s};
}

__global__ __launch_bounds__(256) void kg_emt_ext(const AsmInst *__restrict__ d, int ni, const FreqState *fs,
                                                  PWBatch pws, int npw)
{
  const AsmInst &q = d[find_inst(d, ni, blockIdx.x, GF_ROW)];
  const int rb = blockIdx.x - q.row0, j = blockIdx.y;
  emt_ext_block(q.g, fs->omega_re, (const cd *)q.B + (size_t)j * q.ldb, pws.pw[j], rb,
                q.part + (size_t)(npw + j) * q.nrowblk + rb);
}

// one workgroup per instance: the scattered sum (part[j][0]) and the fixed-order
// sum of the extinction's row-block partials
__global__ __launch_bounds__(64) void kg_emt_final(const AsmInst *__restrict__ d, int ni, const FreqState *fs, int npw,
                                                   double *out)
{
  const AsmInst &q = d[blockIdx.x];
  const int j = threadIdx.x;
  if (j >= npw) return;
  const double s = q.part[(size_t)j * q.nrowblk];
  double x = 0.0;
  for (int b = 0; b < q.nrowblk; b++) x += q.part[(size_t)(npw + j) * q.nrowblk + b];
  const double pscat = ZVAC * 0.5 * s, pext = 0.5 * x;
  double *o = out + 2 * (((size_t)fs->fidx * ni + blockIdx.x) * npw + j);
  o[0] = pext - pscat;
  o[1] = pscat;
}

namespace bfa {
void launch_tp_table_g(const AsmInst *d, int ni, int ntab, const FreqState *fs, bool realk, hipStream_t st)
{
  if (ntab <= 0) return;
  if (realk) hipLaunchKernelGGL(kg_tp_table<true>, dim3(ntab), dim3(TPT_THREADS), 0, st, d, ni, fs);
  else hipLaunchKernelGGL(kg_tp_table<false>, dim3(ntab), dim3(TPT_THREADS), 0, st, d, ni, fs);
}

void launch_far_gather_g(const AsmInst *d, int ni, int nfar, int ft_max, const FreqState *fs, hipStream_t st)
{
  if (nfar <= 0) return;
  if (ft_max <= 40) hipLaunchKernelGGL(kg_far_gather<40>, dim3(nfar), dim3(GS_NT), 0, st, d, ni, fs);
  else hipLaunchKernelGGL(kg_far_gather<64>, dim3(nfar), dim3(GS_NT), 0, st, d, ni, fs);
}

size_t tp_table_bytes(int nt) { return (size_t)nt * (nt + 1) / 2 * 16 * sizeof(double); }

void launch_far_g(const AsmInst *d, int ni, int nblk, const FreqState *fs, bool realk, hipStream_t st)
{
  if (nblk <= 0) return;
  if (realk) hipLaunchKernelGGL(kg_far<true>, dim3(nblk), dim3(FT_THREADS), 0, st, d, ni, fs);
  else hipLaunchKernelGGL(kg_far<false>, dim3(nblk), dim3(FT_THREADS), 0, st, d, ni, fs);
}
void launch_near_g(const AsmInst *d, int ni, int nblk, const FreqState *fs, bool expr, hipStream_t st)
{
  if (nblk <= 0) return;
  // a few workgroups an instance and CU; each walks the instance's tetrahedra
  const dim3 gr(std::max(64, 4096 / std::max(ni, 1)), ni);
  if (expr) hipLaunchKernelGGL(kg_gram<true>, gr, dim3(64), 0, st, d, fs);
  else hipLaunchKernelGGL(kg_gram<false>, gr, dim3(64), 0, st, d, fs);
  hipLaunchKernelGGL(kg_near, dim3(nblk), dim3(256), 0, st, d, ni, fs);
}
void launch_rhs_g(const AsmInst *d, int ni, int nblk, const FreqState *fs, const PWBatch &pw, int npw, hipStream_t st)
{
  if (nblk > 0) hipLaunchKernelGGL(kg_rhs, dim3(nblk, npw), dim3(256), 0, st, d, ni, fs, pw, npw);
}
void launch_emt_ext_g(const AsmInst *d, int ni, int nblk, const FreqState *fs, const PWBatch &pw, int npw,
                      hipStream_t st)
{
  if (nblk > 0) hipLaunchKernelGGL(kg_emt_ext, dim3(nblk, npw), dim3(256), 0, st, d, ni, fs, pw, npw);
}
void launch_emt_final_g(const AsmInst *d, int ni, const FreqState *fs, int npw, double *out, hipStream_t st)
{
  if (ni > 0) hipLaunchKernelGGL(kg_emt_final, dim3(ni), dim3(64), 0, st, d, ni, fs, npw, out);
}
}  // namespace bfa

// ---------------------------------------------------------------------------
extern "C" int bfa_device_malloc(void **ptr, size_t bytes)
{
  if (!ptr) return fail(BFA_ERR_ARG, "null pointer");
  HIPCHECK(hipMalloc(ptr, bytes));
  return BFA_OK;
}
extern "C" int bfa_device_free(void *ptr)
{
  HIPCHECK(hipFree(ptr));
  return BFA_OK;
}
extern "C" int bfa_memcpy_htod(void *dst, const void *src, size_t bytes, void *stream)
{
  HIPCHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, (hipStream_t)stream));
  HIPCHECK(hipStreamSynchronize((hipStream_t)stream));
  return BFA_OK;
}
extern "C" int bfa_memcpy_dtoh(void *dst, const void *src, size_t bytes, void *stream)
{
  HIPCHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, (hipStream_t)stream));
  HIPCHECK(hipStreamSynchronize((hipStream_t)stream));
  return BFA_OK;
}
extern "C" int bfa_stream_synchronize(void *stream)
{
  HIPCHECK(hipStreamSynchronize((hipStream_t)stream));
  return BFA_OK;
}
