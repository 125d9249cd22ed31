// bfa_panel.hip -- register-resident LU panel: an m x w block column (w up to
// 256) factored with partial pivoting by one launch of co-resident
// workgroups, one exchange through memory per column.
//
// Replaces the column loop of HMatrix::LUFactorize's zgetrf
// (src/applications/buff-scatter/buff-scatter.cc:285).
#include <hip/hip_runtime.h>
#include <algorithm>
#include <mutex>

#include "bfa_internal.h"
#include "bfa_panel.h"

using namespace bfa;

namespace {

template <typename T> struct zc { T re, im; };
template <typename T> __device__ __forceinline__ zc<T> z_mul(zc<T> a, zc<T> b)
{ return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re}; }
template <typename T> __device__ __forceinline__ T t_fma(T a, T b, T c) { return sizeof(T) == 8 ? (T)fma(a, b, c) : (T)fmaf(a, b, c); }
// l u, apart from the sum it goes into, so that one rounding and not two is at
// the sum's magnitude (random matrices: factor error 10 % less, 1 % of the time)
template <typename T> __device__ __forceinline__ zc<T> z_prod(zc<T> l, zc<T> u)
{ return {t_fma(-l.im, u.im, l.re * u.re), t_fma(l.im, u.re, l.re * u.im)}; }
// a - l u, a + l u
template <typename T> __device__ __forceinline__ zc<T> z_fms(zc<T> a, zc<T> l, zc<T> u)
{ const zc<T> p = z_prod(l, u); return {a.re - p.re, a.im - p.im}; }
template <typename T> __device__ __forceinline__ zc<T> z_fma(zc<T> a, zc<T> l, zc<T> u)
{ const zc<T> p = z_prod(l, u); return {a.re + p.re, a.im + p.im}; }
template <typename T> __device__ __forceinline__ zc<T> z_sub(zc<T> a, zc<T> b) { return {a.re - b.re, a.im - b.im}; }
template <typename T> __device__ __forceinline__ zc<T> z_pick(bool c, zc<T> a, zc<T> b)
{ return {c ? a.re : b.re, c ? a.im : b.im}; }
template <typename T> __device__ __forceinline__ T z_abs1(zc<T> a) { return fabs(a.re) + fabs(a.im); }

// agent-scope relaxed accesses: coherent between workgroups of one launch
// wherever they run, no cache maintenance
__device__ __forceinline__ void ag_store(unsigned long long *p, unsigned long long v)
{ __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ unsigned long long ag_load(const unsigned long long *p)
{ return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
// a row entry travels as 8-byte words of 32 data bits below the column's
// 32-bit sequence number, so that every word proves itself current; word k of
// all entries together (XP_PLANE apart), so that a wave's accesses are whole
// lines
__device__ __forceinline__ void put_word(unsigned long long *p, unsigned d, unsigned seq)
{ ag_store(p, ((unsigned long long)seq << 32) | d); }
__device__ __forceinline__ void put_entry(unsigned long long *p, zc<double> v, unsigned seq)
{
  const unsigned long long a = (unsigned long long)__double_as_longlong(v.re),
                           b = (unsigned long long)__double_as_longlong(v.im);
  put_word(p, (unsigned)a, seq);
  put_word(p + XP_PLANE, (unsigned)(a >> 32), seq);
  put_word(p + 2 * XP_PLANE, (unsigned)b, seq);
  put_word(p + 3 * XP_PLANE, (unsigned)(b >> 32), seq);
}
__device__ __forceinline__ void put_entry(unsigned long long *p, zc<float> v, unsigned seq)
{
  put_word(p, __float_as_uint(v.re), seq);
  put_word(p + XP_PLANE, __float_as_uint(v.im), seq);
}
// false while a word is not yet the column's
__device__ __forceinline__ bool get_entry(const unsigned long long *p, zc<double> &v, unsigned seq)
{
  const unsigned long long a = ag_load(p), b = ag_load(p + XP_PLANE), c = ag_load(p + 2 * XP_PLANE),
                           d = ag_load(p + 3 * XP_PLANE);
  v = {__longlong_as_double((long long)((a & 0xffffffffull) | (b << 32))),
       __longlong_as_double((long long)((c & 0xffffffffull) | (d << 32)))};
  return (unsigned)(a >> 32) == seq && (unsigned)(b >> 32) == seq && (unsigned)(c >> 32) == seq &&
         (unsigned)(d >> 32) == seq;
}
__device__ __forceinline__ bool get_entry(const unsigned long long *p, zc<float> &v, unsigned seq)
{
  const unsigned long long a = ag_load(p), b = ag_load(p + XP_PLANE);
  v = {__uint_as_float((unsigned)a), __uint_as_float((unsigned)b)};
  return (unsigned)(a >> 32) == seq && (unsigned)(b >> 32) == seq;
}
// 1 / a: on the path from one exchange to the next, so the reciprocal of
// |a|^2 comes from the hardware estimate and Newton steps where that cannot
// overflow, and each quotient is corrected by its own remainder: as exact as
// the two divisions it stands for
__device__ __forceinline__ double recip(double d)
{
  double y = __builtin_amdgcn_rcp(d);
  y = fma(y, fma(-d, y, 1.0), y);
  return fma(y, fma(-d, y, 1.0), y);
}
__device__ __forceinline__ float recip(float d)
{
  const float y = __builtin_amdgcn_rcpf(d);
  return fmaf(y, fmaf(-d, y, 1.0f), y);
}
template <typename T> __device__ __forceinline__ zc<T> z_inv(zc<T> a)
{
  constexpr T big = sizeof(T) == 8 ? (T)1e290 : (T)1e30;
  const T d = a.re * a.re + a.im * a.im;
  if (d > 1 / big && d < big) {
    const T y = recip(d), p = a.re * y, q = -a.im * y;
    return {t_fma(y, t_fma(-d, p, a.re), p), t_fma(y, t_fma(-d, q, -a.im), q)};
  }
  return {a.re / d, -a.im / d};
}

// value of lane `src` (wave-uniform)
__device__ __forceinline__ float lane_get(float v, int src)
{ return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), src)); }
__device__ __forceinline__ double lane_get(double v, int src)
{
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_readlane((unsigned)b, src), hi = __builtin_amdgcn_readlane((unsigned)(b >> 32), src);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
template <typename T> __device__ __forceinline__ zc<T> lane_get(zc<T> v, int src)
{ return {lane_get(v.re, src), lane_get(v.im, src)}; }

template <int CTRL> __device__ __forceinline__ unsigned dpp_max(unsigned v)
{
  const unsigned o = (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, false);
  return o > v ? o : v;
}
// maximum over the wave: row shifts, then the two row broadcasts
__device__ __forceinline__ unsigned wave_max(unsigned v)
{
  v = dpp_max<0x111>(v);
  v = dpp_max<0x112>(v);
  v = dpp_max<0x114>(v);
  v = dpp_max<0x118>(v);
  v = dpp_max<0x142>(v);
  v = dpp_max<0x143>(v);
  return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}

// a[i] for a wave-uniform i: a branch tree down to four rows, then selects (an
// array indexed by a variable would be moved to scratch memory; the leaves'
// distinct comments keep them from being merged into such an access)
template <int LO, int HI, typename T, int R> __device__ __forceinline__ void reg_get(const zc<T> (&a)[R], int i, zc<T> &x)
{
  if constexpr (HI - LO <= 4) {
    x = a[LO];
#pragma unroll
    for (int k = LO + 1; k < HI; k++) x = z_pick(i == k, a[k], x);
    asm volatile("; leaf %2" : "+v"(x.re), "+v"(x.im) : "i"(LO));
  } else {
    constexpr int MID = LO + ((HI - LO) / 4 + 1) / 2 * 4;
    if (i < MID) reg_get<LO, MID>(a, i, x);
    else reg_get<MID, HI>(a, i, x);
  }
}
template <int LO, int HI, typename T, int R> __device__ __forceinline__ void reg_put(zc<T> (&a)[R], int i, zc<T> x)
{
  if constexpr (HI - LO <= 4) {
#pragma unroll
    for (int k = LO; k < HI; k++) a[k] = z_pick(i == k, x, a[k]);
    asm volatile("; leaf %0" : : "i"(LO));
  } else {
    constexpr int MID = LO + ((HI - LO) / 4 + 1) / 2 * 4;
    if (i < MID) reg_put<LO, MID>(a, i, x);
    else reg_put<MID, HI>(a, i, x);
  }
}

#define XP_NT 256
#define XP_FOLD 32       // columns whose products are summed before they go into the values
#define XP_SPIN_LIMIT (1u << 24)

// org: each entry's value when its sum was last zero, rows 0 .. AL - 1 (the
// odd row length spreads a column over the banks)
template <typename T, int R, int AL> struct XpShared {
  zc<T> org[AL][XP_NT + 1];
  zc<T> col[4][R];
};

// One workgroup (rank of nwg) of the panel.  Thread t holds column t of rows
// r0 .. r0 + R - 1 for the whole panel: in registers the sum of the products
// l u to be subtracted from each entry, in LDS the value to subtract it from
// (rows AL .. R - 1: in registers too).  The difference is formed where an
// entry leaves the workgroup and every XP_FOLD columns, so an entry is rounded
// at its own magnitude about 10 times a panel and not once a column, as with
// the panels of 32 columns and the GEMM that accumulates from zero.
// |PA - LU| / |A| over u, complex64, VIE matrices of 270, 1,350 and 3,822
// unknowns: 0.82, 1.20, 1.57; subtracted from the entries product by product
// 4.8, 7.5, 9.3, by 32-column panels 1.55, 1.87, 2.20.  Random matrices of 200
// and 512, complex128: 15.5 and 36.9, 32-column panels 16.4 and 39.9.  Sums
// over the whole panel are better on the VIE matrices (0.66, 1.00, 1.44) and
// 4 % worse on random ones.  About as fast (n = 1,350 3.49 -> 3.57 ms): the
// values, read by row index, need no branch tree, and a column's time is the
// exchange's.
// Lanes also hold, redundantly in every wave, the next two columns row by row
// (lane = row), so that the multipliers of column j, the values of column
// j + 1 and its pivot candidate need no workgroup reduction.
//
// Exchange of column j: the owner of row j publishes that row (all columns) as
// soon as it is up to date; every workgroup publishes one word {sequence
// number, magnitude, row} of its candidate and, behind it, the candidate's
// row.  Every wave reads all workgroups' words until they carry this column's
// sequence number, so all see the same pivot (largest |re| + |im| rounded to
// float, first row among equals, as izamax does), and row j with them; only a
// pivot elsewhere costs a further read.  A row's words carry the sequence
// number as well: no store is waited for and nothing is cleared, the numbers
// never repeat between launches.  The register update of column j - 1
// overlaps the exchange.
// Words and rows rotate through XP_NBUF buffers: wave 0 publishes column
// j + 2 after the workgroup barrier of column j, which every wave passes only
// when it has read column j's, so a workgroup that has seen all words of
// j + 2 may overwrite column j's.
//
// Rows that are finished (global row <= j) are left out of the update.  The
// multipliers of column j go to A straight from the lanes, in the row order of
// step j: the interchanges of later columns are applied to them afterwards,
// with those of the columns left of the panel (k_laswp_left); U is written at
// the end.
template <typename T, int R, int AL>
__device__ __forceinline__ void xpanel_body(const XPanel &p, int rank, XpShared<T, R, AL> &sh)
{
  constexpr int EW = sizeof(T) / 2;   // words of an entry
  constexpr int NX = R > AL ? R - AL : 1;
  static_assert(R <= 64 && AL <= R, "a lane a row");
  typedef zc<T> Z;
  typedef unsigned long long u64;
  __builtin_amdgcn_s_setprio(3);
  const int t = threadIdx.x, lane = t & 63, t0 = __builtin_amdgcn_readfirstlane(t & ~63);
  const int m = p.m, w = p.w, nwg = p.nwg, r0 = rank * R;
  Z *A = (Z *)p.A;
  Z s[R], ox[NX];
#pragma unroll
  for (int i = 0; i < R; i++) {
    const int r = r0 + i;
    const Z v = (t < w && r < m) ? A[(size_t)t * p.lda + r] : Z{0, 0};
    if (i < AL) sh.org[i][t] = v;
    else ox[i < AL ? 0 : i - AL] = v;
    if (t < 2) sh.col[t][i] = v;   // columns 0, 1 to the lanes
    if (t == 2) sh.col[2][i] = i < AL ? Z{0, 0} : z_sub(Z{0, 0}, v);
    s[i] = {0, 0};
  }
  __syncthreads();
  const int il = lane < R ? lane : 0;
  const bool row_lane = lane < R;
  Z c0 = sh.col[0][il], c1 = sh.col[1][il], l = {0, 0};
  Z pt = {0, 0};
  bool dead = false;               // a wait gave up somewhere: finish without waiting
  auto wait_ok = [&](unsigned &spins) __attribute__((always_inline)) {
    if (dead) return true;
    if ((++spins & 255) == 0 && __hip_atomic_load(&p.err[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) dead = true;
    if (spins > XP_SPIN_LIMIT) {
      if (lane == 0) atomicOr(&p.err[0], 1);   // reported as an error by the host
      dead = true;
    }
    return dead;
  };
  auto row_slot = [&](int buf, int who) __attribute__((always_inline)) {
    return (u64 *)p.data + ((size_t)buf * (XP_MAXWG + 1) + who) * XP_PLANE * EW;
  };
  // this thread's entry of row i (wave-uniform): value, and the sum to subtract
  auto row_get = [&](int i, Z &o, Z &q) __attribute__((always_inline)) {
    if (AL == R || i < AL) o = sh.org[i][t];
    else reg_get<0, NX>(ox, i - AL, o);
    reg_get<0, R>(s, i, q);
  };
  auto row_set = [&](int i, Z v) __attribute__((always_inline)) {
    if (AL == R || i < AL) sh.org[i][t] = v;
    else reg_put<0, NX>(ox, i - AL, v);
    reg_put<0, R>(s, i, Z{0, 0});
  };
  // row jn's entry and its sum before step jn - 1, fetched while waiting
  Z xo = {0, 0}, xs = {0, 0};
  auto fetch = [&](int jn) __attribute__((always_inline)) {
    if (jn >= r0 && jn < r0 + R) row_get(jn - r0, xo, xs);
  };
  // row `row` of this workgroup, whose sum (q) misses step jn - 1 if elim
  auto send = [&](int row, Z o, Z q, u64 *dst, unsigned seq, bool elim) __attribute__((always_inline)) {
    if (elim) q = z_fma(q, lane_get(l, row), pt);
    put_entry(dst + t, z_sub(o, q), seq);
  };
  // row jn, then the candidate of column jn (lanes hold the column in c0)
  auto publish = [&](int jn, bool elim) __attribute__((always_inline)) {
    const unsigned seq = p.seq0 + jn;
    const int buf = jn & (XP_NBUF - 1), lj = jn - r0;
    if (lj >= 0 && lj < R) send(lj, xo, xs, row_slot(buf, XP_MAXWG), seq, elim);
    const int r = r0 + lane;
    const float v = (float)z_abs1(c0);
    const unsigned mg = (row_lane && r < m && r >= jn) ? (v == v ? __float_as_uint(v) : 0u) + 1u : 0u;
    const unsigned M = wave_max(mg);
    const int rp = M ? (int)__builtin_ctzll(__ballot(mg == M)) : -1;
    if (t == 0)
      ag_store(p.flags + ((size_t)buf * XP_MAXWG + rank) * XP_FSTRIDE,
               ((u64)seq << 40) | ((u64)M << 9) | (unsigned)(rp < 0 ? 0 : rp));
    if (rp >= 0 && rp != lj) {
      Z o, q;
      row_get(rp, o, q);
      send(rp, o, q, row_slot(buf, rank), seq, elim);
    }
  };
  fetch(0);
  publish(0, false);
  fetch(1);
#pragma unroll 1
  for (int j = 0; j < w; j++) {
    const int buf = j & (XP_NBUF - 1);
    const unsigned seq = p.seq0 + j;
    // every workgroup's candidate; beside it row j, which most often is the
    // pivot's (and otherwise moves to the pivot's place): this thread's column,
    // and columns j, j + 1, j + 2 once more on lanes 0 .. 2
    const int ib = min(j + (lane & 3), XP_NT - 1);
    Z ov = sh.org[AL == R ? il : min(il, AL - 1)][min(j + 2, XP_NT - 1)];   // see below
    const u64 *fl = p.flags + (size_t)buf * XP_MAXWG * XP_FSTRIDE, *rj = row_slot(buf, XP_MAXWG);
    const bool two = nwg > 64;
    u64 f, f2 = 0;
    Z rt, rb;
    bool have = false;
    for (unsigned spins = 0;;) {
      f = lane < nwg ? ag_load(fl + (size_t)lane * XP_FSTRIDE) : (u64)seq << 40;
      if (two) f2 = lane + 64 < nwg ? ag_load(fl + (size_t)(lane + 64) * XP_FSTRIDE) : (u64)seq << 40;
      if (!have) {
        const bool a1 = get_entry(rj + t, rt, seq), a2 = get_entry(rj + ib, rb, seq);
        have = __ballot(a1 && a2) == ~0ull;
      }
      const bool all = __ballot((unsigned)(f >> 40) == seq && (!two || (unsigned)(f2 >> 40) == seq)) == ~0ull;
      if ((all && have) || wait_ok(spins)) break;
    }
    const unsigned mg = lane < nwg ? (unsigned)(f >> 9) & 0x7fffffffu : 0u;
    const unsigned mg2 = two && lane + 64 < nwg ? (unsigned)(f2 >> 9) & 0x7fffffffu : 0u;
    const unsigned M = wave_max(mg > mg2 ? mg : mg2);
    const u64 wb = __ballot(lane < nwg && mg == M), wb2 = __ballot(mg2 == M);
    int win, lrow;
    if (wb) {
      win = (int)__builtin_ctzll(wb);
      lrow = (int)(__builtin_amdgcn_readlane((unsigned)f, win) & 511u);
    } else {
      win = wb2 ? (int)__builtin_ctzll(wb2) : 0;
      lrow = (int)(__builtin_amdgcn_readlane((unsigned)f2, win) & 511u);
      win = min(win + 64, nwg - 1);
    }
    const int prow = max(j, min(m - 1, win * R + lrow));
    const bool ownp = prow != j && prow >= r0 && prow < r0 + R;
    Z pb = rb;
    pt = rt;
    if (prow != j) {
      const u64 *pr = row_slot(buf, win);
      for (unsigned spins = 0;;) {
        const bool a1 = get_entry(pr + t, pt, seq), a2 = get_entry(pr + ib, pb, seq);
        if (__ballot(a1 && a2) == ~0ull || wait_ok(spins)) break;
      }
    }
    const Z pj = lane_get(pb, 0), pj1 = lane_get(pb, 1), pj2 = lane_get(pb, 2), inv = z_inv(pj);
    // rows j and prow change places
    const int lp = prow - r0;
    if (prow != j) {
      const int lj = j - r0;
      if (lj >= 0 && lj < R) row_set(lj, pt);
      if (ownp) {
        row_set(lp, rt);
        if (lp == j + 1 - r0) { xo = rt; xs = {0, 0}; }
        const Z r0v = lane_get(rb, 0), r1v = lane_get(rb, 1);
        if (lane == lp) { c0 = r0v; c1 = r1v; }
      }
    }
    if (t <= j) pt = {0, 0};       // finished columns: the update below leaves them alone
    const bool scale = z_abs1(pj) != (T)0, act = row_lane && r0 + lane > j;
    l = scale && act ? z_mul(c0, inv) : Z{0, 0};
    const Z lo = z_pick(scale, l, c0);   // column j of L as stored
    c0 = scale && act ? z_fms(c1, l, pj1) : c1;
    if (j + 1 < w) publish(j + 1, scale);
    if ((t >> 6) == (j & (XP_NT / 64 - 1))) {
      const int r = r0 + lane;
      if (row_lane && r > j && r < m) A[(size_t)j * p.lda + r] = lo;
    }
    if (rank == 0 && t == 0) {
      p.ipiv[j] = prow + p.piv_off;
      if (!scale && p.err[1] == 0) p.err[1] = p.piv_off + j + 1;
    }
    __syncthreads();
    // column j + 2 through step j - 1, then step j.  Its thread left the sums
    // in a buffer; the values were read from org before this step's barrier,
    // beside which only this step's interchange may have written
    {
      if (AL < R && il >= AL) ov = {0, 0};
      Z v = z_sub(ov, sh.col[2 + (j & 1)][il]);
      if (ownp && il == lp) v = lane_get(rb, 2);
      c1 = scale && act ? z_fms(v, l, pj2) : v;
    }
    // the other rows
    const int ist = max(0, j + 1 - r0);
    if (scale && ist < R && t0 + 63 > j) {
      if (ist == 0) {
#pragma unroll
        for (int i = 0; i < R; i++) s[i] = z_fma(s[i], lane_get(l, i), pt);
      } else {
#pragma unroll
        for (int i = 1; i < R; i++) s[i] = z_pick(i >= ist, z_fma(s[i], lane_get(l, i), pt), s[i]);
      }
    }
    // every XP_FOLD columns the sums go into the values, so that neither grows long
    if ((j & (XP_FOLD - 1)) == XP_FOLD - 1) {
#pragma unroll
      for (int i = 0; i < R; i++) {
        if (i < AL) sh.org[i < AL ? i : 0][t] = z_sub(sh.org[i < AL ? i : 0][t], s[i]);
        else ox[i < AL ? 0 : i - AL] = z_sub(ox[i < AL ? 0 : i - AL], s[i]);
        s[i] = {0, 0};
      }
      __syncthreads();             // the next step's lanes read org
    }
    if (t == j + 3) {
#pragma unroll
      for (int i = 0; i < R; i++)
        sh.col[2 + ((j + 1) & 1)][i] = i < AL ? s[i] : z_sub(s[i], ox[i < AL ? 0 : i - AL]);
    }
    fetch(j + 2);
  }
#pragma unroll
  for (int i = 0; i < R; i++) {
    const int r = r0 + i;
    if (t < w && r <= t && r < m)
      A[(size_t)t * p.lda + r] = z_sub(i < AL ? sh.org[i < AL ? i : 0][t] : ox[i < AL ? 0 : i - AL], s[i]);
  }
}

template <typename T, int R> __global__ __launch_bounds__(XP_NT) void k_xpanel(XPanel p)
{
  __shared__ XpShared<T, R, R> sh;
  xpanel_body<T, R, R>(p, blockIdx.x, sh);
}

// grouped: workgroups blk0 .. blk0 + nwg - 1 of the launch factor panel d[i].
// Two workgroups share a CU's LDS, so of 48 rows 38 fit in it.
template <int R> __global__ __launch_bounds__(XP_NT) void kg_xpanel(const XPanelProb *__restrict__ d, int np)
{
  constexpr int AL = R < 38 ? R : 38;
  __shared__ XpShared<float, R, AL> sh;
  int lo = 0, hi = np - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (d[mid].blk0 <= (int)blockIdx.x) lo = mid;
    else hi = mid - 1;
  }
  xpanel_body<float, R, AL>(d[lo].p, blockIdx.x - d[lo].blk0, sh);
}

const int g_rows[2][4] = {{8, 16, 32, 48}, {8, 16, 24, 32}};   // [f64]
const int g_group_rows[3] = {16, 32, 48};

// workgroups of each variant on one CU, and the CUs, of the current device
struct Occupancy { int cus, per[2][4], group[3]; };
const Occupancy &occupancy()
{
  static Occupancy none{}, tab[16];
  static bool have[16];
  static std::mutex mx;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16) return none;
  std::lock_guard<std::mutex> lock(mx);
  Occupancy &o = tab[dev];
  if (have[dev]) return o;
  const void *k[2][4] = {
      {(const void *)k_xpanel<float, 8>, (const void *)k_xpanel<float, 16>, (const void *)k_xpanel<float, 32>,
       (const void *)k_xpanel<float, 48>},
      {(const void *)k_xpanel<double, 8>, (const void *)k_xpanel<double, 16>, (const void *)k_xpanel<double, 24>,
       (const void *)k_xpanel<double, 32>}};
  const void *kg[3] = {(const void *)kg_xpanel<16>, (const void *)kg_xpanel<32>, (const void *)kg_xpanel<48>};
  auto count = [](const void *f) {
    int per = 0;
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, f, XP_NT, 0) == hipSuccess ? per : 0;
  };
  if (hipDeviceGetAttribute(&o.cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return none;
  for (int v = 0; v < 4; v++) { o.per[0][v] = count(k[0][v]); o.per[1][v] = count(k[1][v]); }
  for (int v = 0; v < 3; v++) o.group[v] = count(kg[v]);
  have[dev] = true;
  return o;
}
// workgroups of a grouped launch: two a CU at most
int resident_g(int v)
{
  const Occupancy &o = occupancy();
  return std::min(o.group[v], 2) * o.cus;
}

template <typename T, int R> void launch(XPanel p, hipStream_t st)
{
  p.nwg = (p.m + R - 1) / R;
  hipLaunchKernelGGL((k_xpanel<T, R>), dim3(p.nwg), dim3(XP_NT), 0, st, p);
}

}  // namespace

namespace bfa {
static size_t row_bytes(bool f64) { return (size_t)XP_NBUF * (XP_MAXWG + 1) * XP_PLANE * (f64 ? 32 : 16); }
size_t xpanel_bytes(bool f64) { return row_bytes(f64) + (size_t)XP_NBUF * XP_MAXWG * XP_FSTRIDE * 8; }

void xpanel_carve(bool f64, char *mem, XPanel *p)
{
  p->data = mem;
  p->flags = (unsigned long long *)(mem + row_bytes(f64));
}

// Rows a workgroup holds, fewest first: a column's time grows with them (the
// register update outlasts the exchange from about 16 complex128 / 32
// complex64 rows), the exchange's hardly with the workgroups.  Measured, us a
// column of 256: complex128 1.76 (8 rows, m = 256), 2.18 (16, 1,350), 2.75
// (24, 3,000), 3.03 (32, 4,000); complex64 1.48 (8, 256), 1.78 (16, 1,350),
// 2.36 (32, 4,000), 2.85 (48, 6,000); with an interchange in every column 2.21
// to 3.97 and 1.75 to 3.48.
// A panel's workgroups wait for each other, so all must run at once: XP_MAXWG
// of them at most, and what the device holds (a partition of it has fewer CUs).
int xpanel_max_rows(bool f64)
{
  const Occupancy &o = occupancy();
  int rows = 0;
  for (int v = 0; v < 4; v++) rows = std::max(rows, g_rows[f64][v] * std::min(XP_MAXWG, o.per[f64][v] * o.cus));
  return rows;
}

int launch_xpanel(bool f64, XPanel p, hipStream_t st)
{
  const Occupancy &o = occupancy();
  const int rows = bfa_xpanel_rows(f64, p.m, o.cus, o.per[f64]);
  if (p.m < 1 || !rows || p.w < 1 || p.w > XP_MAXW || p.w > p.m)
    return fail(BFA_ERR_ARG, "register panel of %d x %d", p.m, p.w);
  if (f64) {
    if (rows == 8) launch<double, 8>(p, st);
    else if (rows == 16) launch<double, 16>(p, st);
    else if (rows == 24) launch<double, 24>(p, st);
    else launch<double, 32>(p, st);
  } else {
    if (rows == 8) launch<float, 8>(p, st);
    else if (rows == 16) launch<float, 16>(p, st);
    else if (rows == 32) launch<float, 32>(p, st);
    else launch<float, 48>(p, st);
  }
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? BFA_OK : fail(BFA_ERR_HIP, "register panel launch: %s", hipGetErrorString(e));
}

// Fewest rows that keep the launch to two workgroups a CU (a column's time
// grows with the rows, see above, and with a second round of launches more)
int xpanel_group_rows(int m, int64_t total, int *resident)
{
  int pick = -1;
  for (int i = 0; i < 3; i++) {
    if (m > g_group_rows[i] * std::min(XP_MAXWG, resident_g(i))) continue;
    pick = i;
    if (total <= (int64_t)g_group_rows[i] * resident_g(i)) break;
  }
  *resident = pick < 0 ? 0 : resident_g(pick);
  return pick < 0 ? 0 : g_group_rows[pick];
}

int xpanel_group_max_rows()
{
  int rows = 0;
  for (int i = 0; i < 3; i++) rows = std::max(rows, g_group_rows[i] * std::min(XP_MAXWG, resident_g(i)));
  return rows;
}

void launch_xpanel_g(const XPanelProb *d, int np, int nblk, int rows, hipStream_t st)
{
  if (nblk <= 0) return;
  if (rows == 16) hipLaunchKernelGGL(kg_xpanel<16>, dim3(nblk), dim3(XP_NT), 0, st, d, np);
  else if (rows == 32) hipLaunchKernelGGL(kg_xpanel<32>, dim3(nblk), dim3(XP_NT), 0, st, d, np);
  else hipLaunchKernelGGL(kg_xpanel<48>, dim3(nblk), dim3(XP_NT), 0, st, d, np);
}
}  // namespace bfa

extern "C" int bfa_xpanel_rows(int f64, int m, int cus, const int *per_cu)
{
  const int *rows = g_rows[f64 ? 1 : 0];
  for (int v = 0; v < 4; v++)
    if (m <= rows[v] * std::min(XP_MAXWG, per_cu[v] * cus)) return rows[v];
  return 0;
}
