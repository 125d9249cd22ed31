// bfa_power.hip -- scattered power of the EMT method (GetEMTPFT,
// src/libs/libbuff/EMTPFT.cc:216-319, 389-427) from tetrahedron currents.
//
// P_scat = Z0 sum_{a <= b} Re(J_a^* J_b) Q_ab, Q_ab the cubature of
// (b_a.b_b - div div/k^2) k sin(kr)/(4 pi r) over the four tetrahedron pairs
// of a BF pair, with 4 points a tetrahedron, 16 where the BFs share a vertex,
// 16 and 33 where k times a BF's radius exceeds 5.  Q is not formed: on
// tetrahedron T the BFs' currents add up to A_T (x - c_T) - B_T,
// A_T = sum J_a pf_a, B_T = sum J_a pf_a (Q_a - c_T), so the 4-point rule's
// sum over all BF pairs is a form in (A, B) with the 8 moments of each
// tetrahedron pair (I0, Ix, Iy, Ixy of the kernel); the pairs of BFs on a
// finer rule add the difference of the two rules, tetrahedron pair by
// tetrahedron pair.
#include <hip/hip_runtime.h>
#include <algorithm>

#include "bfa_internal.h"
#include "bfa_group.h"
#include "bfa_math.h"
#include "bfa_power.h"

using namespace bfa;

namespace {

#define ET_NT 256
#define ET_TILE 32
#define EMT_SPLIT 8
#define FOURPI 12.566370614359172954

struct cd { double re, im; };

// A_T and B_T of tetrahedron t for the currents J: A (re, im), Bx, By, Bz
__device__ __forceinline__ void tet_current(const DevGeom &g, int t, const cd *J, double *o)
{
  const double *cen = g.tetVol + g.nt + 3 * t;
  double v[8];
#pragma unroll
  for (int i = 0; i < 8; i++) v[i] = 0.0;
#pragma unroll
  for (int f = 0; f < 4; f++) {
    const int b = g.tetFI[4 * t + f];
    if (b >= g.nbf) continue;
    const int side = g.bfT[2 * b] == t ? 0 : 1;
    const double pf = g.bfPF[2 * b + side];
    const double *Q = g.bfQ + 6 * b + 3 * side;
    const double re = pf * J[b].re, im = pf * J[b].im;
    v[0] += re; v[1] += im;
#pragma unroll
    for (int d = 0; d < 3; d++) {
      const double al = Q[d] - cen[d];
      v[2 + 2 * d] += re * al;
      v[3 + 2 * d] += im * al;
    }
  }
#pragma unroll
  for (int i = 0; i < 8; i++) o[i] = v[i];
}

// k w w' sin(kr) / (4 pi r) and its moments about the centroids
__device__ __forceinline__ void sine_moments(const double *x, const double *xi, const double *y, const double *cT,
                                             double k, double *m)
{
  const double R0 = x[0] - y[0], R1 = x[1] - y[1], R2 = x[2] - y[2];
  const double r2 = R0 * R0 + R1 * R1 + R2 * R2, ir = rsqrt_nr(r2), kr = k * (r2 * ir);
  double im;
  if (r2 * k * k < 4.0e-4) im = (1.0 - k * k * r2 / 6.0) * k / FOURPI;   // |kr| < 0.02, r = 0 included
  else {
    double sn, cs;
    sincos_mod(kr, &sn, &cs);
    im = sn * ir * (1.0 / FOURPI);
  }
  const double gv = x[3] * y[3] * k * im;
  const double e0 = y[0] - cT[0], e1 = y[1] - cT[1], e2 = y[2] - cT[2];
  m[0] += gv;
  m[1] += gv * xi[0]; m[2] += gv * xi[1]; m[3] += gv * xi[2];
  m[4] += gv * e0; m[5] += gv * e1; m[6] += gv * e2;
  m[7] += gv * (xi[0] * e0 + xi[1] * e1 + xi[2] * e2);
}

template <int NJ> struct EmtShared {
  double pts[2][16][ET_TILE];
  double cen[2][3][ET_TILE];
  double cur[2][NJ][8][ET_TILE];
  double pf[2][4][ET_TILE], al[2][4][3][ET_TILE];
  int bf[2][4][ET_TILE], opp[2][4][ET_TILE], vi[2][4][ET_TILE];
  unsigned mask[ET_TILE * ET_TILE];            // low half: 16-point BF pairs (bit 4 i + j), high half: 33-point
  unsigned short list[ET_TILE * ET_TILE];
  int wcnt[4];
  double red[4][NJ];
};

// the three rules' moments of BF pair (i, j): pf pf' [Ixy - b.Ix - a.Iy + (a.b - 9/k^2) I0]
__device__ __forceinline__ double bf_form(const double *m, const double *a, const double *b, double pp, double ik2)
{
  const double ab = a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
  return pp * (m[7] - (b[0] * m[1] + b[1] * m[2] + b[2] * m[3]) - (a[0] * m[4] + a[1] * m[5] + a[2] * m[6]) +
               (ab - ik2) * m[0]);
}

// One 32 x 32 tile (bs <= bt) of tetrahedron pairs S <= T for right-hand sides
// j0 .. j0 + NJ - 1: their part of Re(J^H Q J) + sum_a |J_a|^2 Q_aa into
// part[j * stride].  Bound by its FP64 arithmetic: 16 point pairs of about 55
// operations for each tetrahedron pair, 272 for those with BF pairs on the
// 16-point rule (about 2 % of all pairs at 10,368 tetrahedra), which sixteen
// threads share.  Of the nz workgroups of a tile, one evaluates the 4-point
// rule, and they deal the finer rules' pairs among them: a mesh of a few
// tiles, where nearly every pair is such, would leave the chip idle
// (N = 270: 0.33 -> 0.19 ms with 8).
template <int NJ>
__device__ __forceinline__ void emt_tet_tile(const DevGeom &g, double omega, const cd *J, int64_t ldj,
                                             const double *cur, int npw, int j0, int bs, int bt, int z, int nz,
                                             double *part, int64_t stride, EmtShared<NJ> &sh)
{
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nt = g.nt;
  const double k = omega, ik2 = 9.0 / (omega * omega);
  for (int idx = tid; idx < 2 * ET_TILE * 16; idx += ET_NT) {
    const int side = idx / (ET_TILE * 16), u = (idx / 16) % ET_TILE, e = idx % 16;
    const int t = (side ? bt : bs) * ET_TILE + u;
    sh.pts[side][e][u] = t < nt ? g.q4[(size_t)t * 16 + e] : 0.0;
  }
  for (int idx = tid; idx < 2 * ET_TILE * 3; idx += ET_NT) {
    const int side = idx / (ET_TILE * 3), u = (idx / 3) % ET_TILE, d = idx % 3;
    const int t = (side ? bt : bs) * ET_TILE + u;
    sh.cen[side][d][u] = t < nt ? g.tetVol[nt + 3 * t + d] : 0.0;
  }
  // faces: prefactor, Q - centroid, opposite vertex of the BF's other tetrahedron (-1: no BF), high-kR flag
  for (int idx = tid; idx < 2 * ET_TILE * 4; idx += ET_NT) {
    const int side = idx / (ET_TILE * 4), u = (idx / 4) % ET_TILE, f = idx % 4;
    const int t = (side ? bt : bs) * ET_TILE + u;
    int b = -1, opp = -1, v = -2 - side;
    double pf = 0.0, al[3] = {0.0, 0.0, 0.0};
    if (t < nt) {
      v = g.tetVI[4 * t + f];
      b = g.tetFI[4 * t + f];
      if (b >= g.nbf) b = -1;
      if (b >= 0) {
        const int s = g.bfT[2 * b] == t ? 0 : 1;
        pf = g.bfPF[2 * b + s];
        opp = g.bfV[5 * b + (s ? 0 : 4)];
        for (int d = 0; d < 3; d++) al[d] = g.bfQ[6 * b + 3 * s + d] - g.tetVol[nt + 3 * t + d];
        if (fabs(omega) * g.bfRad[b] > 5.0) opp |= 1 << 30;
      }
    }
    sh.bf[side][f][u] = b; sh.opp[side][f][u] = opp; sh.vi[side][f][u] = v; sh.pf[side][f][u] = pf;
    for (int d = 0; d < 3; d++) sh.al[side][f][d][u] = al[d];
  }
  for (int idx = tid; idx < 2 * NJ * ET_TILE * 8; idx += ET_NT) {
    const int side = idx / (NJ * ET_TILE * 8), j = idx / (ET_TILE * 8) % NJ, u = idx / 8 % ET_TILE, e = idx % 8;
    const int t = (side ? bt : bs) * ET_TILE + u;
    sh.cur[side][j][e][u] = t < nt && j0 + j < npw ? cur[((size_t)(j0 + j) * nt + t) * 8 + e] : 0.0;
  }
  __syncthreads();
  double acc[NJ];
#pragma unroll
  for (int j = 0; j < NJ; j++) acc[j] = 0.0;
  // the 4-point rule on every pair
#pragma unroll 1
  for (int pidx = tid; pidx < ET_TILE * ET_TILE; pidx += ET_NT) {
    const int us = pidx / ET_TILE, ut = pidx % ET_TILE, S = bs * ET_TILE + us, T = bt * ET_TILE + ut;
    unsigned mask = 0;
    if (S < nt && T < nt && S <= T) {
      if (z == 0) {
        double m[8], cS[3], cT[3];
#pragma unroll
        for (int i = 0; i < 8; i++) m[i] = 0.0;
#pragma unroll
        for (int d = 0; d < 3; d++) { cS[d] = sh.cen[0][d][us]; cT[d] = sh.cen[1][d][ut]; }
#pragma unroll 1
        for (int p = 0; p < 4; p++) {
          double x[4], xi[3];
#pragma unroll
          for (int e = 0; e < 4; e++) x[e] = sh.pts[0][4 * p + e][us];
#pragma unroll
          for (int d = 0; d < 3; d++) xi[d] = x[d] - cS[d];
#pragma unroll 2
          for (int q = 0; q < 4; q++) {
            double y[4];
#pragma unroll
            for (int e = 0; e < 4; e++) y[e] = sh.pts[1][4 * q + e][ut];
            sine_moments(x, xi, y, cT, k, m);
          }
        }
        const double wgt = S == T ? 1.0 : 2.0;
#pragma unroll
        for (int j = 0; j < NJ; j++) {
          double a[8], b[8];
#pragma unroll
          for (int e = 0; e < 8; e++) { a[e] = sh.cur[0][j][e][us]; b[e] = sh.cur[1][j][e][ut]; }
          const double aa = a[0] * b[0] + a[1] * b[1];
          const double bb = a[2] * b[2] + a[3] * b[3] + a[4] * b[4] + a[5] * b[5] + a[6] * b[6] + a[7] * b[7];
          const double xr = m[1] * b[2] + m[2] * b[4] + m[3] * b[6], xm = m[1] * b[3] + m[2] * b[5] + m[3] * b[7];
          const double yr = m[4] * a[2] + m[5] * a[4] + m[6] * a[6], ym = m[4] * a[3] + m[5] * a[5] + m[6] * a[7];
          acc[j] += wgt * (aa * (m[7] - ik2 * m[0]) - (a[0] * xr + a[1] * xm) - (b[0] * yr + b[1] * ym) + m[0] * bb);
        }
      }
      // BF pairs on a finer rule: a shared vertex (of the tetrahedra: every
      // pair; of a BF's outer vertex: that BF's pairs), or k times a radius
      bool share = false;
      int vS[4], vT[4], oS[4], oT[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        vS[i] = sh.vi[0][i][us]; vT[i] = sh.vi[1][i][ut];
        oS[i] = sh.opp[0][i][us]; oT[i] = sh.opp[1][i][ut];
      }
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) share |= vS[i] == vT[j];
      const int vmask = (1 << 30) - 1;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int o = oS[i] & vmask;
        const bool ti = share || o == vT[0] || o == vT[1] || o == vT[2] || o == vT[3];
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const int q = oT[j] & vmask;
          const bool touch = ti || q == vS[0] || q == vS[1] || q == vS[2] || q == vS[3] || q == o;
          const bool hf = ((oS[i] | oT[j]) >> 30) & 1;
          if (oS[i] >= 0 && oT[j] >= 0 && (touch || hf)) mask |= (touch && hf ? 0x10000u : 1u) << (4 * i + j);
        }
      }
    }
    sh.mask[pidx] = mask;
  }
  __syncthreads();
  // those pairs in order: each thread counts four consecutive ones
  int total;
  {
    int c = 0, pre = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) c += sh.mask[4 * tid + i] != 0;
    pre = c;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int o = __shfl_up(pre, off, 64);
      if (lane >= off) pre += o;
    }
    if (lane == 63) sh.wcnt[wave] = pre;
    __syncthreads();
    int base = pre - c;
    for (int w = 0; w < wave; w++) base += sh.wcnt[w];
    total = sh.wcnt[0] + sh.wcnt[1] + sh.wcnt[2] + sh.wcnt[3];
#pragma unroll
    for (int i = 0; i < 4; i++)
      if (sh.mask[4 * tid + i]) sh.list[base++] = (unsigned short)(4 * tid + i);
    __syncthreads();
  }
  // sixteen threads a pair: thread `sub` takes a row point of each rule, and
  // afterwards BF pair (sub / 4, sub % 4)
  const int sub = tid & 15;
#pragma unroll 1
  for (int e0 = z * (ET_NT / 16); e0 < total; e0 += nz * (ET_NT / 16)) {
    const int e = e0 + (tid >> 4);
    const bool on = e < total;
    const int pidx = on ? sh.list[e] : 0, us = pidx / ET_TILE, ut = pidx % ET_TILE;
    const unsigned mask = on ? sh.mask[pidx] : 0;
    const int S = bs * ET_TILE + us, T = bt * ET_TILE + ut;
    double cS[3], cT[3], m4[8], mf[8];
#pragma unroll
    for (int d = 0; d < 3; d++) { cS[d] = sh.cen[0][d][us]; cT[d] = sh.cen[1][d][ut]; }
#pragma unroll
    for (int i = 0; i < 8; i++) m4[i] = mf[i] = 0.0;
    double v = 0.0;
    const int fi = sub >> 2, fj = sub & 3;
    double al[3], be[3];
#pragma unroll
    for (int d = 0; d < 3; d++) { al[d] = sh.al[0][fi][d][us]; be[d] = sh.al[1][fj][d][ut]; }
    const double pp = sh.pf[0][fi][us] * sh.pf[1][fj][ut];
    const int ba = sh.bf[0][fi][us], bb = sh.bf[1][fj][ut];
    if (on) {
      double x[4], xi[3], y[4];
#pragma unroll
      for (int c = 0; c < 4; c++) { x[c] = sh.pts[0][4 * fi + c][us]; y[c] = sh.pts[1][4 * fj + c][ut]; }
#pragma unroll
      for (int d = 0; d < 3; d++) xi[d] = x[d] - cS[d];
      sine_moments(x, xi, y, cT, k, m4);
    }
#pragma unroll
    for (int i = 0; i < 8; i++)
#pragma unroll
      for (int off = 1; off < 16; off <<= 1) m4[i] += __shfl_xor(m4[i], off, 64);
#pragma unroll 1
    for (int rule = 0; rule < 2; rule++) {
      // a rule that no pair of this wave needs is skipped by the whole wave
      const bool need = rule ? mask >> 16 : mask & 0xffffu;
      if (!__any(need)) continue;
      const int np = rule ? 33 : 16;
      const double *qs = (rule ? g.q33 : g.q16) + (size_t)S * np * 4, *qt = (rule ? g.q33 : g.q16) + (size_t)T * np * 4;
#pragma unroll
      for (int i = 0; i < 8; i++) mf[i] = 0.0;
      if (need)
#pragma unroll 1
        for (int p = sub; p < np; p += 16) {
          double x[4], xi[3];
#pragma unroll
          for (int c = 0; c < 4; c++) x[c] = qs[4 * p + c];
#pragma unroll
          for (int d = 0; d < 3; d++) xi[d] = x[d] - cS[d];
#pragma unroll 2
          for (int q = 0; q < np; q++) {
            double y[4];
#pragma unroll
            for (int c = 0; c < 4; c++) y[c] = qt[4 * q + c];
            sine_moments(x, xi, y, cT, k, mf);
          }
        }
#pragma unroll
      for (int i = 0; i < 8; i++)
#pragma unroll
        for (int off = 1; off < 16; off <<= 1) mf[i] += __shfl_xor(mf[i], off, 64);
      if ((mask >> (16 * rule + sub)) & 1) {
        const double full = bf_form(mf, al, be, pp, ik2), wgt = S == T ? 1.0 : 2.0;
        // the diagonal pairs a = b count once more
        v += wgt * (full - bf_form(m4, al, be, pp, ik2)) + (ba == bb ? wgt * full : 0.0);
      }
    }
    if (v != 0.0) {
#pragma unroll
      for (int j = 0; j < NJ; j++)
        if (j0 + j < npw) {
          const cd ja = J[(size_t)(j0 + j) * ldj + ba], jb = J[(size_t)(j0 + j) * ldj + bb];
          acc[j] += v * (ja.re * jb.re + ja.im * jb.im);
        }
    }
  }
#pragma unroll
  for (int j = 0; j < NJ; j++) {
    double v = acc[j];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    if (lane == 0) sh.red[wave][j] = v;
  }
  __syncthreads();
  if (tid < NJ && j0 + tid < npw) part[(int64_t)(j0 + tid) * stride] = sh.red[0][tid] + sh.red[1][tid] + sh.red[2][tid] + sh.red[3][tid];
}

__device__ __forceinline__ void tile_of(int64_t bid, int n, int &bi, int &bj)
{
  // row bi of the upper triangle starts at bi n - bi (bi - 1) / 2
  const double d = 2.0 * n + 1.0;
  int r = (int)((d - sqrt(d * d - 8.0 * (double)bid)) / 2.0);
  auto start = [n](int64_t i) { return i * n - i * (i - 1) / 2; };
  r = max(0, min(r, n - 1));
  while (r > 0 && start(r) > bid) r--;
  while (r + 1 < n && start(r + 1) <= bid) r++;
  bi = r;
  bj = r + (int)(bid - start(r));
}

__global__ void k_tet_current(DevGeom g, const cd *J, int64_t ldj, double *cur)
{
  const int t = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
  if (t < g.nt) tet_current(g, t, J + (size_t)j * ldj, cur + ((size_t)j * g.nt + t) * 8);
}

template <int NJ>
__global__ __launch_bounds__(ET_NT) void k_emt_tet(DevGeom g, double omega, const cd *J, int64_t ldj,
                                                   const double *cur, int npw, int ntb, double *part)
{
  __shared__ EmtShared<NJ> sh;
  int bs, bt;
  tile_of(blockIdx.x, ntb, bs, bt);
  emt_tet_tile<NJ>(g, omega, J, ldj, cur, npw, blockIdx.y * NJ, bs, bt, blockIdx.z, gridDim.z,
                   part + blockIdx.x * gridDim.z + blockIdx.z, (int64_t)gridDim.x * gridDim.z, sh);
}

// out[j] = sum of part[j][0 .. n), in a fixed order
__global__ __launch_bounds__(1024) void k_sum_rows(const double *part, int64_t n, double *out)
{
  __shared__ double red[1024];
  const double *p = part + (size_t)blockIdx.x * n;
  double s = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += 1024) s += p[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int off = 512; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[blockIdx.x] = red[0];
}

// ---- grouped over the instances of a batch
__device__ __forceinline__ int emt_inst(const AsmInst *__restrict__ d, int n, int bid)
{
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (d[mid].emt0 <= bid) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

__global__ void kg_tet_current(const AsmInst *__restrict__ d)
{
  const AsmInst &q = d[blockIdx.z];
  const int j = blockIdx.y;
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < q.g.nt; t += gridDim.x * blockDim.x)
    tet_current(q.g, t, (const cd *)q.B + (size_t)j * q.ldb, q.Q + ((size_t)j * q.g.nt + t) * 8);
}

template <int NJ>
__global__ __launch_bounds__(ET_NT) void kg_emt_tet(const AsmInst *__restrict__ d, int ni, const FreqState *fs, int npw)
{
  __shared__ EmtShared<NJ> sh;
  const AsmInst &q = d[emt_inst(d, ni, blockIdx.x)];
  const int ntb = (q.g.nt + ET_TILE - 1) / ET_TILE, blk = blockIdx.x - q.emt0;
  int bs, bt;
  tile_of(blk, ntb, bs, bt);
  double *part = q.Q + (size_t)npw * q.g.nt * 8;
  const int nz = gridDim.z;
  emt_tet_tile<NJ>(q.g, fs->omega_re, (const cd *)q.B, q.ldb, q.Q, npw, blockIdx.y * NJ, bs, bt, blockIdx.z, nz,
                   part + blk * nz + blockIdx.z, (int64_t)(ntb * (ntb + 1) / 2) * nz, sh);
}

// scattered sums of instance blockIdx.y, right-hand side blockIdx.x, into its part[j * nrowblk]
__global__ __launch_bounds__(256) void kg_emt_sum(const AsmInst *__restrict__ d, int npw, int nz)
{
  __shared__ double red[256];
  const AsmInst &q = d[blockIdx.y];
  const int ntb = (q.g.nt + ET_TILE - 1) / ET_TILE, n = ntb * (ntb + 1) / 2 * nz, j = blockIdx.x;
  const double *p = q.Q + (size_t)npw * q.g.nt * 8 + (size_t)j * n;
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) s += p[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) q.part[(size_t)j * q.nrowblk] = red[0];
}

}  // namespace

namespace bfa {
int emt_tiles(int nt)
{
  const int ntb = (nt + ET_TILE - 1) / ET_TILE;
  return ntb * (ntb + 1) / 2;
}

size_t emt_work_doubles(int nt, int npw) { return (size_t)npw * ((size_t)nt * 8 + (size_t)emt_tiles(nt) * EMT_SPLIT); }

// workgroups of a tile: enough for two on every CU
static int emt_split(int64_t wgs) { return (int)std::max<int64_t>(1, std::min<int64_t>(EMT_SPLIT, 512 / std::max<int64_t>(wgs, 1))); }

// right-hand sides evaluated together: the moments of a tetrahedron pair serve
// all of them, and the currents of more than 8 would leave one workgroup a CU
void launch_emt_scattered(const DevGeom &g, double omega, const void *J, int64_t ldj, int npw, double *work,
                          double *out, hipStream_t st)
{
  const int ntb = (g.nt + ET_TILE - 1) / ET_TILE, n = emt_tiles(g.nt);
  double *cur = work, *part = work + (size_t)npw * g.nt * 8;
  hipLaunchKernelGGL(k_tet_current, dim3((g.nt + 127) / 128, npw), dim3(128), 0, st, g, (const cd *)J, ldj, cur);
  const int nz = emt_split((int64_t)n * ((npw + 7) / 8));
#define EMT_LAUNCH(NJ) \
  hipLaunchKernelGGL(k_emt_tet<NJ>, dim3(n, (npw + NJ - 1) / NJ, nz), dim3(ET_NT), 0, st, g, omega, (const cd *)J, ldj, \
                     (const double *)cur, npw, ntb, part)
  if (npw == 1) EMT_LAUNCH(1);
  else if (npw == 2) EMT_LAUNCH(2);
  else if (npw <= 4) EMT_LAUNCH(4);
  else EMT_LAUNCH(8);
#undef EMT_LAUNCH
  hipLaunchKernelGGL(k_sum_rows, dim3(npw), dim3(1024), 0, st, (const double *)part, (int64_t)n * nz, out);
}

void launch_emt_scattered_g(const AsmInst *d, int ni, int nblk, const FreqState *fs, int npw, hipStream_t st)
{
  if (nblk <= 0) return;
  const int nz = emt_split(nblk);
  hipLaunchKernelGGL(kg_tet_current, dim3(8, npw, ni), dim3(256), 0, st, d);
  if (npw == 1) hipLaunchKernelGGL(kg_emt_tet<1>, dim3(nblk, 1, nz), dim3(ET_NT), 0, st, d, ni, fs, npw);
  else if (npw == 2) hipLaunchKernelGGL(kg_emt_tet<2>, dim3(nblk, 1, nz), dim3(ET_NT), 0, st, d, ni, fs, npw);
  else if (npw <= 4) hipLaunchKernelGGL(kg_emt_tet<4>, dim3(nblk, 1, nz), dim3(ET_NT), 0, st, d, ni, fs, npw);
  else hipLaunchKernelGGL(kg_emt_tet<8>, dim3(nblk, (npw + 7) / 8, nz), dim3(ET_NT), 0, st, d, ni, fs, npw);
  hipLaunchKernelGGL(kg_emt_sum, dim3(npw, ni), dim3(256), 0, st, d, npw, nz);
}
}  // namespace bfa
