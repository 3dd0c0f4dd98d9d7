// agx_mg.hip -- multigrid self-gravity on gfx950 (plain FP64).
//
// The reference keeps a multigrid hierarchy per MeshBlock (levels bnx, bnx/2, .., 1) plus
// a root grid with one cell per MeshBlock (multigrid/multigrid.cpp:32-144,
// multigrid_driver.cpp:343-349), and refreshes a one-cell ghost layer from the
// neighbours before every stencil (task_list/mg_task_list.cpp:287-510).  On a uniform
// periodic mesh that hierarchy is exactly one periodic grid per level: the block
// levels and the root grid tile it, every ghost equals the neighbour's interior cell,
// and the block-coarsest level coincides with the root grid's finest.  This file keeps
// one HBM array per level for the whole mesh and reads neighbours through periodic
// index wrap, so the ghost exchanges disappear while every stencil value is the one
// the reference computes.  The control flow (V-cycle, FMG, iteration, average removal)
// follows MultigridDriver step for step.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <cfloat>
#include <cmath>

#include "agx_internal.hpp"

using namespace agx;

namespace {

constexpr int BS = 256;

__device__ __forceinline__ int wrapm(int i, int n) { return (i == 0) ? n - 1 : i - 1; }
__device__ __forceinline__ int wrapp(int i, int n) { return (i == n - 1) ? 0 : i + 1; }
__device__ __forceinline__ int wrap(int i, int n) { return (i < 0) ? i + n : (i >= n ? i - n : i); }

__device__ __forceinline__ int64_t LIX(int n1, int n2, int k, int j, int i) {
  return ((int64_t)k * n2 + j) * n1 + i;
}

// One red-black Gauss-Seidel update (MGGravity::Smooth, gravity/mg_gravity.cpp:259-267),
// the operand order of the reference.
template <typename T>
__device__ __forceinline__ T gs_value(T uc, T ukp, T ujp, T uip, T ukm, T ujm, T uim, T s, T dx2,
                                      T isix) {
  return uc - ((T(6.0) * uc - ukp - ujp - uip - ukm - ujm - uim) + s * dx2) * isix;
}

// MGGravity::Smooth (gravity/mg_gravity.cpp:220-273), omega = 1.15 (mg_gravity.hpp:43).
// The reference sweeps i = il + ((color + k + j) & 1) in steps of 2 in block-local
// indices with a one-cell ghost; with an even number of cells per block that is the set
// of global cells with (I + J + K + color) even.  One thread per updated cell.
template <typename T>
__global__ void __launch_bounds__(BS)
k_mg_smooth(const int *__restrict__ gate, T *__restrict__ u, const T *__restrict__ src, int n1, int n2, int n3,
            T dx2, T isix, int color) {
  if (gate && *gate) return;   // a closed gate: the recorded V-cycle loop has ended
  int nh = (n1 + 1) / 2;
  const unsigned t = xcd_slot(blockIdx.x, gridDim.x) * BS + threadIdx.x;   // < 2^32 cells per level
  int64_t tot = (int64_t)nh * n2 * n3;
  if (t >= tot) return;
  int h = (int)(t % (unsigned)nh);
  unsigned r = t / (unsigned)nh;
  int j = (int)(r % (unsigned)n2);
  int k = (int)(r / (unsigned)n2);
  int i = 2 * h + ((color + k + j) & 1);
  if (i >= n1) return;
  int64_t id = LIX(n1, n2, k, j, i);
  T uc = u[id];
  T ukp = u[LIX(n1, n2, wrapp(k, n3), j, i)], ujp = u[LIX(n1, n2, k, wrapp(j, n2), i)];
  T uip = u[LIX(n1, n2, k, j, wrapp(i, n1))];
  T ukm = u[LIX(n1, n2, wrapm(k, n3), j, i)], ujm = u[LIX(n1, n2, k, wrapm(j, n2), i)];
  T uim = u[LIX(n1, n2, k, j, wrapm(i, n1))];
  u[id] = gs_value(uc, ukp, ujp, uip, ukm, ujm, uim, src[id], dx2, isix);
}

// The sweep of a level with an odd extent of three or more, where the periodic wrap joins cells of
// one colour: out of place, so that every update reads the values from before the sweep, as the
// reference's do from ghosts filled ahead of it.  In place the value read across the wrap would be
// whichever of old and new another workgroup has stored.  Only a root grid's lowest level is odd.
template <typename T>
__global__ void __launch_bounds__(BS)
k_mg_smooth_wrap(const int *__restrict__ gate, const T *__restrict__ u, T *__restrict__ out, const T *__restrict__ src,
                 int n1, int n2, int n3, T dx2, T isix, int color) {
  if (gate && *gate) return;   // a closed gate: the recorded V-cycle loop has ended
  const unsigned t = blockIdx.x * BS + threadIdx.x;
  if (t >= (unsigned)n1 * n2 * n3) return;
  const unsigned r = t / (unsigned)n1;
  const int i = (int)(t - r * n1), j = (int)(r % (unsigned)n2), k = (int)(r / (unsigned)n2);
  T v = u[t];
  if (((color + i + j + k) & 1) == 0)
    v = gs_value(v, u[LIX(n1, n2, wrapp(k, n3), j, i)], u[LIX(n1, n2, k, wrapp(j, n2), i)],
                 u[LIX(n1, n2, k, j, wrapp(i, n1))], u[LIX(n1, n2, wrapm(k, n3), j, i)],
                 u[LIX(n1, n2, k, wrapm(j, n2), i)], u[LIX(n1, n2, k, j, wrapm(i, n1))], src[t], dx2, isix);
  out[t] = v;
}

// The same red/black sweep with one thread per (i, i+1) pair of a row (n1 even): the
// pair is read and written as one 16-B (8-B in FP32) vector, so rows are read and
// written as whole cache lines; the cell of the pair that is not of this colour is
// written back unchanged (no other thread writes it, and its readers see the same
// value either way).  Arithmetic as k_mg_smooth.
template <typename T> struct Vec2;
template <> struct Vec2<double> { using type = double2; };
template <> struct Vec2<float> { using type = float2; };

template <typename T>
__global__ void __launch_bounds__(BS)
k_mg_smooth_pairs(const int *__restrict__ gate, T *__restrict__ u, const T *__restrict__ src, int n1, int n2, int n3,
                  T dx2, T isix, int color) {
  if (gate && *gate) return;   // a closed gate: the recorded V-cycle loop has ended
  using V = typename Vec2<T>::type;
  const unsigned nh = (unsigned)n1 >> 1;
  const unsigned t = xcd_slot(blockIdx.x, gridDim.x) * BS + threadIdx.x;   // < 2^32 pairs per level
  if (t >= nh * (unsigned)n2 * (unsigned)n3) return;
  const unsigned h = t % nh;
  const unsigned r = t / nh;
  const int j = (int)(r % (unsigned)n2);
  const int k = (int)(r / (unsigned)n2);
  const int odd = (color + k + j) & 1;   // 0: update i = 2h, 1: update i = 2h + 1
  const int i = 2 * (int)h + odd;
  V *u2 = reinterpret_cast<V *>(u);
  const int64_t row = ((int64_t)k * n2 + j) * nh;
  V c = u2[row + h];
  V kp = u2[((int64_t)wrapp(k, n3) * n2 + j) * nh + h];
  V jp = u2[((int64_t)k * n2 + wrapp(j, n2)) * nh + h];
  V km = u2[((int64_t)wrapm(k, n3) * n2 + j) * nh + h];
  V jm = u2[((int64_t)k * n2 + wrapm(j, n2)) * nh + h];
  T uc = odd ? c.y : c.x;
  T ukp = odd ? kp.y : kp.x, ujp = odd ? jp.y : jp.x;
  T ukm = odd ? km.y : km.x, ujm = odd ? jm.y : jm.x;
  T uip = odd ? u[LIX(n1, n2, k, j, wrapp(i, n1))] : c.y;
  T uim = odd ? c.x : u[LIX(n1, n2, k, j, wrapm(i, n1))];
  T v = gs_value(uc, ukp, ujp, uip, ukm, ujm, uim, src[LIX(n1, n2, k, j, i)], dx2, isix);
  if (odd) c.y = v;
  else c.x = v;
  u2[row + h] = c;
}

template <typename T>
__device__ __forceinline__ T defect_at(const T *u, const T *src, int n1, int n2,
                                       int n3, int k, int j, int i, T idx2) {
  // MGGravity::CalculateDefect, gravity/mg_gravity.cpp:283-314
  int64_t id = LIX(n1, n2, k, j, i);
  T uc = u[id];
  return (T(6.0) * uc - u[LIX(n1, n2, wrapp(k, n3), j, i)] - u[LIX(n1, n2, k, wrapp(j, n2), i)] -
          u[LIX(n1, n2, k, j, wrapp(i, n1))] - u[LIX(n1, n2, wrapm(k, n3), j, i)] -
          u[LIX(n1, n2, k, wrapm(j, n2), i)] - u[LIX(n1, n2, k, j, wrapm(i, n1))]) * idx2 + src[id];
}

// 8-cell average of the fine defect over the children of coarse cell (k, j, i)
// (Restrict, multigrid.cpp:684-724).
template <typename T>
__device__ __forceinline__ T restricted_defect(const T *u, const T *src, int n1, int n2, int n3,
                                               int k, int j, int i, T idx2) {
  int fi = 2 * i, fj = 2 * j, fk = 2 * k;
  T d000 = defect_at(u, src, n1, n2, n3, fk, fj, fi, idx2);
  T d001 = defect_at(u, src, n1, n2, n3, fk, fj, fi + 1, idx2);
  T d010 = defect_at(u, src, n1, n2, n3, fk, fj + 1, fi, idx2);
  T d011 = defect_at(u, src, n1, n2, n3, fk, fj + 1, fi + 1, idx2);
  T d100 = defect_at(u, src, n1, n2, n3, fk + 1, fj, fi, idx2);
  T d101 = defect_at(u, src, n1, n2, n3, fk + 1, fj, fi + 1, idx2);
  T d110 = defect_at(u, src, n1, n2, n3, fk + 1, fj + 1, fi, idx2);
  T d111 = defect_at(u, src, n1, n2, n3, fk + 1, fj + 1, fi + 1, idx2);
  return T(0.125) * (d000 + d001 + d010 + d011 + d100 + d101 + d110 + d111);
}

template <typename T>
__device__ __forceinline__ typename Vec2<T>::type load2(const T *a, int64_t id) {   // id even
  return *reinterpret_cast<const typename Vec2<T>::type *>(a + id);
}

// restricted_defect with the fine values read as (i, i+1) pairs: a cross of 12 row pairs
// (k-1..k+2 x j-1..j+2 without the corners), 8 i-neighbours and 4 source pairs, 24 loads
// instead of 64.  Every defect and the average use the operands and order of
// restricted_defect / defect_at, so the result is the same bit for bit.
template <typename T>
__device__ __forceinline__ T restricted_defect_pairs(const T *u, const T *src, int n1, int n2, int n3,
                                                     int k, int j, int i, T idx2) {
  using V = typename Vec2<T>::type;
  const int fi = 2 * i, fj = 2 * j, fk = 2 * k;
  const int kk[4] = {wrapm(fk, n3), fk, fk + 1, wrapp(fk + 1, n3)};
  const int jj[4] = {wrapm(fj, n2), fj, fj + 1, wrapp(fj + 1, n2)};
  const int im = wrapm(fi, n1), ip = wrapp(fi + 1, n1);
  V P[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b)
      if ((a == 1 || a == 2) || (b == 1 || b == 2)) P[a][b] = load2(u, LIX(n1, n2, kk[a], jj[b], fi));
  T d[2][2][2];
#pragma unroll
  for (int dk = 0; dk < 2; ++dk)
#pragma unroll
    for (int dj = 0; dj < 2; ++dj) {
      const int a = 1 + dk, b = 1 + dj;
      const V sv = load2(src, LIX(n1, n2, kk[a], jj[b], fi));
      const T um = u[LIX(n1, n2, kk[a], jj[b], im)], up = u[LIX(n1, n2, kk[a], jj[b], ip)];
      // di = 0: cell fi (i+1 neighbour is the pair's second value)
      d[dk][dj][0] = (T(6.0) * P[a][b].x - P[a + 1][b].x - P[a][b + 1].x - P[a][b].y - P[a - 1][b].x -
                      P[a][b - 1].x - um) * idx2 + sv.x;
      // di = 1: cell fi + 1 (i-1 neighbour is the pair's first value)
      d[dk][dj][1] = (T(6.0) * P[a][b].y - P[a + 1][b].y - P[a][b + 1].y - up - P[a - 1][b].y -
                      P[a][b - 1].y - P[a][b].x) * idx2 + sv.y;
    }
  return T(0.125) * (d[0][0][0] + d[0][0][1] + d[0][1][0] + d[0][1][1] + d[1][0][0] + d[1][0][1] +
                     d[1][1][0] + d[1][1][1]);
}

// RestrictBlock (multigrid/multigrid.cpp:331-355): defect on the fine level, 8-cell
// average into the coarse source (Restrict, multigrid.cpp:684-724), coarse u zeroed
// (ZeroClearData, non-FAS).  One thread per coarse cell.
template <typename T>
__global__ void __launch_bounds__(BS)
k_mg_defect_restrict(const int *__restrict__ gate, const T *__restrict__ u, const T *__restrict__ src,
                     T *__restrict__ csrc, T *__restrict__ cu, int n1, int n2, int n3,
                     T idx2) {
  if (gate && *gate) return;   // a closed gate: the recorded V-cycle loop has ended
  int c1 = n1 >> 1, c2 = n2 >> 1, c3 = n3 >> 1;
  const unsigned t = xcd_slot(blockIdx.x, gridDim.x) * BS + threadIdx.x;   // < 2^32 cells per level
  if (t >= (int64_t)c1 * c2 * c3) return;
  int i = (int)(t % (unsigned)c1);
  unsigned r = t / (unsigned)c1;
  int j = (int)(r % (unsigned)c2);
  int k = (int)(r / (unsigned)c2);
  csrc[t] = restricted_defect_pairs(u, src, n1, n2, n3, k, j, i, idx2);
  cu[t] = T(0.0);
}

// Restrict (multigrid.cpp:684-724) of the source only, for RestrictFMGSource
// (multigrid.cpp:253-262).
template <typename T>
__global__ void __launch_bounds__(BS)
k_mg_restrict_src(const T *__restrict__ src, T *__restrict__ csrc, int n1, int n2,
                  int n3) {
  int c1 = n1 >> 1, c2 = n2 >> 1, c3 = n3 >> 1;
  const unsigned t = xcd_slot(blockIdx.x, gridDim.x) * BS + threadIdx.x;   // < 2^32 cells per level
  if (t >= (int64_t)c1 * c2 * c3) return;
  int i = (int)(t % (unsigned)c1);
  unsigned r = t / (unsigned)c1;
  int j = (int)(r % (unsigned)c2);
  int k = (int)(r / (unsigned)c2);
  int fi = 2 * i, fj = 2 * j, fk = 2 * k;
#define S(kk, jj, ii) src[LIX(n1, n2, kk, jj, ii)]
  csrc[t] = T(0.125) * (S(fk, fj, fi) + S(fk, fj, fi + 1) + S(fk, fj + 1, fi) + S(fk, fj + 1, fi + 1) +
                     S(fk + 1, fj, fi) + S(fk + 1, fj, fi + 1) + S(fk + 1, fj + 1, fi) +
                     S(fk + 1, fj + 1, fi + 1));
#undef S
}

// Trilinear correction of fine cell (fk, fj, fi) from the coarse level (c1, c2, c3)
// (ProlongateAndCorrect, multigrid.cpp:733-829).
template <typename T>
__device__ __forceinline__ T prolong_corr(const T *cu, int c1, int c2, int c3, int fk, int fj, int fi) {
  int i = fi >> 1, j = fj >> 1, k = fk >> 1;
  int ip = wrap(i + ((fi & 1) ? 1 : -1), c1);
  int jp = wrap(j + ((fj & 1) ? 1 : -1), c2);
  int kp = wrap(k + ((fk & 1) ? 1 : -1), c3);
#define C(kk, jj, ii) cu[LIX(c1, c2, kk, jj, ii)]
  return T(0.015625) * (T(27.0) * C(k, j, i) + C(kp, jp, ip) + T(9.0) * (C(k, j, ip) + C(k, jp, i) + C(kp, j, i)) +
                        T(3.0) * (C(kp, jp, i) + C(kp, j, ip) + C(k, jp, ip)));
#undef C
}

// ProlongateAndCorrect (multigrid/multigrid.cpp:733-829): trilinear (27,9,3,1)/64
// correction.  One thread per fine cell; (dk,dj,di) = -1 for the low child, +1 for the
// high child along each axis.
template <typename T>
__global__ void __launch_bounds__(BS)
k_mg_prolong(const int *__restrict__ gate, const T *__restrict__ cu, T *__restrict__ u, int n1, int n2, int n3) {
  if (gate && *gate) return;   // a closed gate: the recorded V-cycle loop has ended
  const unsigned t = xcd_slot(blockIdx.x, gridDim.x) * BS + threadIdx.x;   // < 2^32 cells per level
  if (t >= (int64_t)n1 * n2 * n3) return;
  int fi = (int)(t % (unsigned)n1);
  unsigned r = t / (unsigned)n1;
  int fj = (int)(r % (unsigned)n2);
  int fk = (int)(r / (unsigned)n2);
  u[t] += prolong_corr(cu, n1 >> 1, n2 >> 1, n3 >> 1, fk, fj, fi);
}

// k_mg_prolong with one thread per (i, i+1) pair of fine cells, the two children of coarse
// cell i along x1: they share the coarse values at i-1, i, i+1 of four coarse rows, and
// the fine pair is read and written as one vector.  Per cell the arithmetic of
// prolong_corr.
template <typename T>
__global__ void __launch_bounds__(BS)
k_mg_prolong_pairs(const int *__restrict__ gate, const T *__restrict__ cu, T *__restrict__ u, int n1, int n2, int n3) {
  if (gate && *gate) return;   // a closed gate: the recorded V-cycle loop has ended
  using V = typename Vec2<T>::type;
  const unsigned nh = (unsigned)n1 >> 1;
  const unsigned t = xcd_slot(blockIdx.x, gridDim.x) * BS + threadIdx.x;   // < 2^32 pairs per level
  if (t >= nh * (unsigned)n2 * (unsigned)n3) return;
  const int i = (int)(t % nh);
  const unsigned r = t / nh;
  const int fj = (int)(r % (unsigned)n2), fk = (int)(r / (unsigned)n2);
  const int c1 = n1 >> 1, c2 = n2 >> 1, c3 = n3 >> 1;
  const int j = fj >> 1, k = fk >> 1;
  const int jp = wrap(j + ((fj & 1) ? 1 : -1), c2), kp = wrap(k + ((fk & 1) ? 1 : -1), c3);
  const int im = wrap(i - 1, c1), ipp = wrap(i + 1, c1);
#define C(kk, jj, ii) cu[LIX(c1, c2, kk, jj, ii)]
  const T a0 = C(k, j, i), am = C(k, j, im), ap = C(k, j, ipp);
  const T b0 = C(k, jp, i), bm = C(k, jp, im), bp = C(k, jp, ipp);
  const T c0 = C(kp, j, i), cm = C(kp, j, im), cp = C(kp, j, ipp);
  const T e0 = C(kp, jp, i), em = C(kp, jp, im), ep = C(kp, jp, ipp);
#undef C
  // prolong_corr with ip = i - 1 (low child) and i + 1 (high child)
  const T lo = T(0.015625) * (T(27.0) * a0 + em + T(9.0) * (am + b0 + c0) + T(3.0) * (e0 + cm + bm));
  const T hi = T(0.015625) * (T(27.0) * a0 + ep + T(9.0) * (ap + b0 + c0) + T(3.0) * (e0 + cp + bp));
  V *u2 = reinterpret_cast<V *>(u);
  const int64_t id = ((int64_t)fk * n2 + fj) * nh + i;
  V v = u2[id];
  v.x += lo;
  v.y += hi;
  u2[id] = v;
}

// FMGProlongate (multigrid/multigrid.cpp:838-1048): 27-point interpolation whose
// weights are products of the 1-D weights (5,30,-3) (low child) or (-3,30,5) (high
// child) over (c-1, c, c+1); summed in (k,j,i) row-major order, then / 32768.
template <typename T>
__global__ void __launch_bounds__(BS)
k_mg_fmg_prolong(const T *__restrict__ cu, T *__restrict__ u, int n1, int n2, int n3) {
  const unsigned t = xcd_slot(blockIdx.x, gridDim.x) * BS + threadIdx.x;   // < 2^32 cells per level
  if (t >= (int64_t)n1 * n2 * n3) return;
  int fi = (int)(t % (unsigned)n1);
  unsigned r = t / (unsigned)n1;
  int fj = (int)(r % (unsigned)n2);
  int fk = (int)(r / (unsigned)n2);
  int c1 = n1 >> 1, c2 = n2 >> 1, c3 = n3 >> 1;
  int i = fi >> 1, j = fj >> 1, k = fk >> 1;
  const T wlo[3] = {T(5.0), T(30.0), T(-3.0)}, whi[3] = {T(-3.0), T(30.0), T(5.0)};
  const T *wk = (fk & 1) ? whi : wlo;
  const T *wj = (fj & 1) ? whi : wlo;
  const T *wi = (fi & 1) ? whi : wlo;
  T acc = T(0.0);
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    int kk = wrap(k - 1 + a, c3);
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      int jj = wrap(j - 1 + b, c2);
#pragma unroll
      for (int e = 0; e < 3; ++e) {
        int ii = wrap(i - 1 + e, c1);
        T term = (wk[a] * wj[b] * wi[e]) * cu[LIX(c1, c2, kk, jj, ii)];
        acc = (a == 0 && b == 0 && e == 0) ? term : acc + term;
      }
    }
  }
  u[t] = acc / T(32768.0);
}

// Reductions: a launch of at most NPART workgroups, workgroup w summing the contiguous
// range [t0, t1) of the level (XCD-aware order); the partials are summed by one
// workgroup (k_mg_final).  The order is fixed, so results are deterministic.
constexpr int NPART = 2048;
__device__ __forceinline__ void wg_range(unsigned n, unsigned &t0, unsigned &t1) {
  const unsigned w = xcd_slot(blockIdx.x, gridDim.x);
  const unsigned per = ((n + gridDim.x - 1) / gridDim.x + BS - 1) / BS * BS;
  t0 = w * per;
  t1 = (t0 + per < n) ? t0 + per : n;
  if (t0 > n) t0 = n;
}

// block-partial sums of a level array in FP64
template <typename T>
__global__ void __launch_bounds__(BS)
k_mg_partial(const int *__restrict__ gate, const T *__restrict__ a, unsigned ncell, double *__restrict__ part) {
  if (gate && *gate) return;   // a closed gate: the recorded V-cycle loop has ended
  __shared__ double sh[BS];
  unsigned t0, t1;
  wg_range(ncell, t0, t1);   // < 2^32 cells per level
  double v = 0.0;
  for (unsigned t = t0 + threadIdx.x; t < t1; t += BS) v += a[t];
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int s = BS / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

// block-partial sums of the squared defect, a thread's cells as (i, i+1) pairs of a row read as one
// vector and stepped from pair to pair without divisions, which were most of the instructions of a
// cell at a time: 256^3 FP64 93 -> 66 us, 4.0 TB/s of u and source.  For the finest level, whose rows
// are even (a MeshBlock has at least two cells along i, a power of two).
template <typename T>
__global__ void __launch_bounds__(BS)
k_mg_norm_pairs(const int *__restrict__ gate, const T *__restrict__ u, const T *__restrict__ src, int n1, int n2,
                int n3, T idx2, double *__restrict__ part) {
  if (gate && *gate) return;   // a closed gate: the recorded V-cycle loop has ended
  using V = typename Vec2<T>::type;
  __shared__ double sh[BS];
  const unsigned nh = (unsigned)n1 >> 1;
  unsigned t0, t1;
  wg_range(nh * (unsigned)n2 * (unsigned)n3, t0, t1);
  const unsigned dh = BS % nh, dr = BS / nh;   // a step: pairs along the row, rows
  const unsigned dj = dr % (unsigned)n2, dk = dr / (unsigned)n2;
  unsigned t = t0 + threadIdx.x;
  unsigned h = t % nh, r = t / nh, j = r % (unsigned)n2, k = r / (unsigned)n2;
  double v = 0.0;
  for (; t < t1; t += BS) {
    const int64_t row = LIX(n1, n2, k, j, 0);
    const T *c = u + row + 2 * h;
    const V uc = load2(c, 0), f = load2(src, row + 2 * h);
    const V kp = load2(u, LIX(n1, n2, wrapp(k, n3), j, 2 * h)), km = load2(u, LIX(n1, n2, wrapm(k, n3), j, 2 * h));
    const V jp = load2(u, LIX(n1, n2, k, wrapp(j, n2), 2 * h)), jm = load2(u, LIX(n1, n2, k, wrapm(j, n2), 2 * h));
    const T im = u[row + (h == 0 ? n1 - 1 : 2 * (int)h - 1)], ip = u[row + (h == nh - 1 ? 0 : 2 * h + 2)];
    const double d0 = (T(6.0) * uc.x - kp.x - jp.x - uc.y - km.x - jm.x - im) * idx2 + f.x;
    const double d1 = (T(6.0) * uc.y - kp.y - jp.y - ip - km.y - jm.y - uc.x) * idx2 + f.y;
    v += d0 * d0;
    v += d1 * d1;
    h += dh; j += dj; k += dk;
    if (h >= nh) { h -= nh; ++j; }
    if (j >= (unsigned)n2) { j -= n2; ++k; }
  }
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int s = BS / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

// the sum of n partials, in thread 0 (fixed order)
__device__ __forceinline__ double part_sum(const double *__restrict__ part, int64_t n) {
  __shared__ double sh[BS];
  double v = 0.0;
#pragma unroll 8
  for (int64_t q = threadIdx.x; q < n; q += BS) v += part[q];
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int s = BS / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
    __syncthreads();
  }
  return sh[0];
}

__global__ void __launch_bounds__(BS) k_mg_final(const int *__restrict__ gate, const double *__restrict__ part,
                                                 int64_t n, double *__restrict__ out) {
  if (gate && *gate) return;   // a closed gate: the recorded V-cycle loop has ended
  const double sum = part_sum(part, n);
  if (threadIdx.x == 0) *out = sum;
}

// finish_norm on the device: sqrt(sum * dv / volume)
__global__ void k_mg_gate_open(MGGate *g, const double *__restrict__ scal, double dv, double vol, double eps) {
  if (threadIdx.x) return;
  const double def = sqrt(scal[0] * dv / vol);
  g->iters = 0;
  g->def = def;
  g->first = def;
  g->closed = (def > eps) ? 0 : 1;
}

// SolveIterative's tests after a V-cycle (multigrid_driver.cpp:733-753); n is the
// loop's count before its increment
__device__ __forceinline__ void gate_check(MGGate *g, double sum, double dv, double vol, double eps) {
  const double olddef = g->def;
  const double def = sqrt(sum * dv / vol);
  const int n = g->iters;
  g->iters = n + 1;
  g->def = def;
  if ((def / olddef > 0.8 && eps == 0.0) || n > 100 || !(def > eps)) g->closed = 1;
}

// k_mg_final for the norm that ends a pass of the recorded loop, and the gate's check of it:
// one launch of 4.6 us where the two took 9
__global__ void __launch_bounds__(BS) k_mg_final_check(const double *__restrict__ part, int64_t n,
                                                       double *__restrict__ out, MGGate *g, double dv, double vol,
                                                       double eps) {
  const int closed = g->closed;
  const double sum = part_sum(part, n);
  if (closed || threadIdx.x) return;
  *out = sum;
  gate_check(g, sum, dv, vol, eps);
}

template <typename T>
__global__ void __launch_bounds__(BS) k_mg_add(const int *__restrict__ gate, T *__restrict__ a, int64_t n,
                                               const double *__restrict__ val, double scale) {
  if (gate && *gate) return;   // a closed gate: the recorded V-cycle loop has ended
  const unsigned t = xcd_slot(blockIdx.x, gridDim.x) * BS + threadIdx.x;   // < 2^32 cells per level
  if (t < n) a[t] -= T((*val) * scale);
}

template <typename T>
__global__ void __launch_bounds__(BS) k_mg_zero(const int *__restrict__ gate, T *__restrict__ a, int64_t n) {
  if (gate && *gate) return;   // a closed gate: the recorded V-cycle loop has ended
  const unsigned t = xcd_slot(blockIdx.x, gridDim.x) * BS + threadIdx.x;   // < 2^32 cells per level
  if (t < n) a[t] = T(0.0);
}

// Mixed-precision defect correction, FP64 side.  The FP64 defect d = src - L(phi)
// (the form of MGGravity::CalculateDefect) becomes the FP32 source of the correction
// problem L(e) = d, and its squares are summed in FP64 for the defect norm.  With ein,
// phi is first corrected by the FP32 correction of the previous cycle (phi + e, into
// uout, read back by no other thread of this launch), so the correction and the next
// defect take one pass.  e0 (not ein) receives the start of the next correction V-cycle: its first
// sweep (colour cred) from e = 0 gives gs_value(0, ..., 0, d) at those cells and 0
// elsewhere, so that cycle starts with its second sweep.
__global__ void __launch_bounds__(BS)
k_mg_defect_to32(const int *__restrict__ gate,
                 const double *__restrict__ u, const float *__restrict__ ein, double *__restrict__ uout,
                 const double *__restrict__ src, float *__restrict__ d32, float *__restrict__ e0, int n1, int n2,
                 int n3, double idx2, float dx2f, float isixf, int cred, double *__restrict__ part) {
  if (gate && *gate) return;   // a closed gate: the recorded V-cycle loop has ended
  __shared__ double sh[BS];
  const unsigned ncell = (unsigned)n1 * n2 * n3;   // < 2^32 cells per level
  unsigned t0, t1;
  wg_range(ncell, t0, t1);
  double v = 0.0;
  auto phi = [&](int64_t q) { return ein ? u[q] + (double)ein[q] : u[q]; };
  for (unsigned t = t0 + threadIdx.x; t < t1; t += BS) {
    const int i = (int)(t % (unsigned)n1);
    const unsigned r = t / (unsigned)n1;
    const int j = (int)(r % (unsigned)n2);
    const int k = (int)(r / (unsigned)n2);
    const double uc = phi(t);
    const double d = (6.0 * uc - phi(LIX(n1, n2, wrapp(k, n3), j, i)) - phi(LIX(n1, n2, k, wrapp(j, n2), i)) -
                      phi(LIX(n1, n2, k, j, wrapp(i, n1))) - phi(LIX(n1, n2, wrapm(k, n3), j, i)) -
                      phi(LIX(n1, n2, k, wrapm(j, n2), i)) - phi(LIX(n1, n2, k, j, wrapm(i, n1)))) * idx2 + src[t];
    if (uout) uout[t] = uc;
    const float df = (float)d;
    d32[t] = df;
    e0[t] = (((i + j + k + cred) & 1) == 0)
                ? gs_value(0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, df, dx2f, isixf)
                : 0.0f;
    v += d * d;
  }
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int s = BS / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

// k_mg_defect_to32 for levels with n1 % DT_TI == 0 and n2 % DT_TJ == 0, tiled like
// k_mg_down: a workgroup owns a DT_TI x DT_TJ tile of (i,j) columns and a chunk of
// DT_KC planes, and keeps phi (= u + e) of three planes of (tile + 1-cell ring) in LDS,
// the next plane being fetched into registers while the current one is processed, so
// u and e are read about once instead of seven times.  Per cell the arithmetic is that
// of k_mg_defect_to32 (bit for bit); the partial sums of d^2 are per workgroup.
constexpr int DT_TI = 64, DT_TJ = 8, DT_KC = 16;
template <bool CORR>
__global__ void __launch_bounds__(DT_TI * DT_TJ)
k_mg_defect_to32_t(const int *__restrict__ gate,
                   const double *__restrict__ u, const float *__restrict__ ein, double *__restrict__ uout,
                   const double *__restrict__ src, float *__restrict__ d32, float *__restrict__ e0, int n1,
                   int n2, int n3, double idx2, float dx2f, float isixf, int cred, double *__restrict__ part) {
  if (gate && *gate) return;   // a closed gate: the recorded V-cycle loop has ended
  constexpr int TI = DT_TI, TJ = DT_TJ, NT = TI * TJ, RI = TI + 2, RJ = TJ + 2;
  constexpr int NPF = (RI * RJ + NT - 1) / NT;
  __shared__ double s_phi[3][RJ][RI];
  __shared__ double sh[NT];
  const int tid = threadIdx.x;
  const int nti = n1 / TI, ntj = n2 / TJ;
  const unsigned wg = xcd_slot(blockIdx.x, gridDim.x);
  const int tile = wg % (unsigned)(nti * ntj), chunk = wg / (unsigned)(nti * ntj);
  const int i0 = (tile % nti) * TI, j0 = (tile / nti) * TJ;
  const int k0 = chunk * DT_KC, k1 = min(k0 + DT_KC, n3);   // planes [k0, k1) of this workgroup
  auto slot = [](int q) { return ((q % 3) + 3) % 3; };
  auto wr = [](int a, int n) { return a < 0 ? a + n : (a >= n ? a - n : a); };
  double pf[NPF];
  auto fetch = [&](int q) {
    const int kq = wr(q, n3);
#pragma unroll
    for (int r = 0; r < NPF; ++r) {
      const int t = tid + r * NT;
      if (t < RI * RJ) {
        const int jj = t / RI, ii = t - jj * RI;
        const int64_t id = LIX(n1, n2, kq, wr(j0 - 1 + jj, n2), wr(i0 - 1 + ii, n1));
        pf[r] = CORR ? u[id] + (double)ein[id] : u[id];
      }
    }
  };
  auto stash = [&](int q) {
    const int sl = slot(q);
#pragma unroll
    for (int r = 0; r < NPF; ++r) {
      const int t = tid + r * NT;
      if (t < RI * RJ) {
        const int jj = t / RI, ii = t - jj * RI;
        s_phi[sl][jj][ii] = pf[r];
      }
    }
  };
  const int jj = tid / TI, ii = tid - (tid / TI) * TI;
  const int gj = j0 + jj, gi = i0 + ii;
  double v = 0.0;
  fetch(k0 - 1);
  stash(k0 - 1);
  fetch(k0);
  stash(k0);
  fetch(k0 + 1);
  for (int q = k0; q < k1; ++q) {
    stash(q + 1);   // the slot of plane q - 2, last read before the previous barrier
    if (q + 2 <= k1) fetch(q + 2);
    __syncthreads();
    const int so = slot(q), sm = slot(q - 1), sp = slot(q + 1);
    const double uc = s_phi[so][jj + 1][ii + 1];
    const double d = (6.0 * uc - s_phi[sp][jj + 1][ii + 1] - s_phi[so][jj + 2][ii + 1] - s_phi[so][jj + 1][ii + 2] -
                      s_phi[sm][jj + 1][ii + 1] - s_phi[so][jj][ii + 1] - s_phi[so][jj + 1][ii]) * idx2;
    const int64_t id = LIX(n1, n2, q, gj, gi);
    const double dd = d + src[id];
    if (CORR) uout[id] = uc;
    const float df = (float)dd;
    d32[id] = df;
    e0[id] = (((gi + gj + q + cred) & 1) == 0)
                 ? gs_value(0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, df, dx2f, isixf)
                 : 0.0f;
    v += dd * dd;
    __syncthreads();
  }
  sh[tid] = v;
  __syncthreads();
  for (int s = NT / 2; s > 0; s >>= 1) {
    if (tid < s) sh[tid] += sh[tid + s];
    __syncthreads();
  }
  if (tid == 0) part[blockIdx.x] = sh[0];
}

// phi += e (mode 0) or phi = e (mode 1), FP32 correction into the FP64 iterate; mode 2
// converts an FP64 array to FP32 (src32 = src).
__global__ void __launch_bounds__(BS)
k_mg_mix(double *__restrict__ u, float *__restrict__ e, int64_t n, int mode) {
  const unsigned t = xcd_slot(blockIdx.x, gridDim.x) * BS + threadIdx.x;   // < 2^32 cells per level
  if (t >= n) return;
  if (mode == 0) u[t] += (double)e[t];
  else if (mode == 1) u[t] = (double)e[t];
  else e[t] = (float)u[t];
}

// Source mask of MultigridDriver::SetupMultigrid (multigrid_driver.cpp:430-436), in the
// form of the reference's collapse problem (pgen/collapse.cpp:66-82): the source is zero
// at cell centres with |x - c|^2 > r^2.  Centres as MGCoordinates (whole-mesh faces,
// end faces exact).
struct SrcMask {
  int on;
  int n[3];
  double xmin[3], xmax[3], c[3], r2;
};
__device__ __forceinline__ double mask_centre(const SrcMask &k, int d, int i) {   // cell i = 0 .. n-1
  const double h = (k.xmax[d] - k.xmin[d]) / k.n[d];
  const double a = (i == 0) ? k.xmin[d] : k.xmin[d] + i * h;
  const double b = (i + 1 == k.n[d]) ? k.xmax[d] : k.xmin[d] + (i + 1) * h;
  return 0.5 * (a + b);
}
__device__ __forceinline__ bool masked_out(const SrcMask &k, int I, int J, int K) {
  if (!k.on) return false;
  const double x = mask_centre(k, 0, I) - k.c[0], y = mask_centre(k, 1, J) - k.c[1],
               z = mask_centre(k, 2, K) - k.c[2];
  return x * x + y * y + z * z > k.r2;
}

// LoadSource (multigrid.cpp:194-231): src = fac * u(IDN) over every block interior,
// and in MGI mode LoadFinestData (multigrid.cpp:160-180): u = phi.
__global__ void __launch_bounds__(BS)
k_mg_load(Geo g, const double *__restrict__ u, const double *__restrict__ phi,
          double *__restrict__ src, double *__restrict__ mu, double fac, int load_phi, SrcMask mk) {
  int N1 = g.nb1 * g.bx1, N2 = g.nb2 * g.bx2, N3 = g.nb3 * g.bx3;
  const unsigned t = xcd_slot(blockIdx.x, gridDim.x) * BS + threadIdx.x;   // < 2^32 cells per level
  if (t >= (int64_t)N1 * N2 * N3) return;
  int I = (int)(t % (unsigned)N1);
  unsigned r = t / (unsigned)N1;
  int J = (int)(r % (unsigned)N2);
  int K = (int)(r / (unsigned)N2);
  int b = ((K / g.bx3) * g.nb2 + (J / g.bx2)) * g.nb1 + (I / g.bx1);
  int64_t id = IDX(g, K % g.bx3 + g.ng, J % g.bx2 + g.ng, I % g.bx1 + g.ng);
  double v = u[(int64_t)b * NHYDRO * g.S + id];
  src[t] = masked_out(mk, I, J, K) ? 0.0 : ((fac == 1.0) ? v : v * fac);
  if (load_phi) mu[t] = phi[(int64_t)b * g.S + id];
}

// RetrieveResult with one ghost layer (multigrid.cpp:269-288).
__global__ void __launch_bounds__(BS)
k_mg_retrieve(Geo g, const double *__restrict__ mu, double *__restrict__ phi) {
  int m1 = g.bx1 + 2, m2 = g.bx2 + 2, m3 = g.bx3 + 2;
  const unsigned t = xcd_slot(blockIdx.x, gridDim.x) * BS + threadIdx.x;   // < 2^32 cells per level
  if (t >= (int64_t)m1 * m2 * m3 * g.nb) return;
  int li = (int)(t % (unsigned)m1);
  unsigned r = t / (unsigned)m1;
  int lj = (int)(r % (unsigned)m2);
  r /= (unsigned)m2;
  int lk = (int)(r % (unsigned)m3);
  int b = (int)(r / (unsigned)m3);
  int N1 = g.nb1 * g.bx1, N2 = g.nb2 * g.bx2, N3 = g.nb3 * g.bx3;
  int lx1 = b % g.nb1, lx2 = (b / g.nb1) % g.nb2, lx3 = b / (g.nb1 * g.nb2);
  int I = wrap(lx1 * g.bx1 + li - 1, N1), J = wrap(lx2 * g.bx2 + lj - 1, N2),
      K = wrap(lx3 * g.bx3 + lk - 1, N3);
  phi[(int64_t)b * g.S + IDX(g, lk - 1 + g.ng, lj - 1 + g.ng, li - 1 + g.ng)] = mu[LIX(N1, N2, K, J, I)];
}


// ================================================================ multipole boundaries
// Non-periodic multigrid with MGMultipole* boundaries (multigrid/mgbval_multipole.cpp)
// and the full approximation scheme the reference uses with them
// (multigrid_driver.cpp:292-295).  Each level is one grid over the whole mesh with a
// one-cell ghost frame (MGLevelB).  A ghost is 2 phi_s(p) - (the cell inside it), phi_s
// the multipole potential at the boundary point p; edge and corner ghosts take "the cell
// inside" along the last face that writes them (x3 after x2 after x1,
// MGBoundaryValues::ApplyPhysicalBoundaries, bvals_mg.cpp:321-368), resolved here as a
// chain so that one launch fills every ghost.  mp[0..2] is the expansion origin,
// mp[3..27] the scaled coefficients.
__device__ __forceinline__ unsigned BX(int n1, int n2, int k, int j, int i) {
  return ((unsigned)k * (unsigned)(n2 + 2) + (unsigned)j) * (unsigned)(n1 + 2) + (unsigned)i;
}

struct MPGeom {
  int n1, n2, n3;
  double xmin[3], xmax[3], h[3];
};

// MGCoordinates::CalculateMGCoordinates (multigrid.cpp:1321-1350) on the whole mesh:
// face i (1 .. n+1, end faces exact) and centre i (0 .. n+1) along direction d
__device__ __forceinline__ double mp_face(const MPGeom &G, int d, int i) {
  const int n = d == 0 ? G.n1 : (d == 1 ? G.n2 : G.n3);
  if (i == 1) return G.xmin[d];
  if (i == n + 1) return G.xmax[d];
  return G.xmin[d] + (i - 1) * G.h[d];
}
__device__ __forceinline__ double mp_centre(const MPGeom &G, int d, int i) {
  return 0.5 * (mp_face(G, d, i) + mp_face(G, d, i + 1));
}

// phi_s at (x, y, z) relative to the origin, mgbval_multipole.cpp:36-88 (mporder 2, 4)
__device__ double mp_phis(const double *__restrict__ mpc, int order, double x, double y, double z) {
  double x2 = x * x, y2 = y * y, z2 = z * z;
  double xy = x * y, yz = y * z, zx = z * x;
  double r2 = x2 + y2 + z2;
  double ir2 = 1.0 / r2, ir1 = sqrt(ir2);
  double ir3 = ir2 * ir1, ir5 = ir3 * ir2;
  if (order == 2)
    return ir1 * mpc[0] + ir3 * (mpc[1] * y + mpc[2] * z + mpc[3] * x) +
           ir5 * (mpc[4] * xy + mpc[5] * yz + (3.0 * z2 - r2) * mpc[6] + mpc[7] * zx + mpc[8] * 0.5 * (x2 - y2));
  double ir7 = ir5 * ir2, ir9 = ir7 * ir2;
  double hx2my2 = 0.5 * (x2 - y2);
  double x2mty2 = x2 - 3.0 * y2;
  double tx2my2 = 3.0 * x2 - y2;
  return ir1 * mpc[0] + ir3 * (mpc[1] * y + mpc[2] * z + mpc[3] * x) +
         ir5 * (mpc[4] * xy + mpc[5] * yz + (3.0 * z2 - r2) * mpc[6] + mpc[7] * zx + mpc[8] * 0.5 * (x2 - y2)) +
         ir7 * (y * tx2my2 * mpc[9] + x * x2mty2 * mpc[15] + xy * z * mpc[10] + z * hx2my2 * mpc[14] +
                (5.0 * z2 - r2) * (y * mpc[11] + x * mpc[13]) + z * (z2 - 3.0 * r2) * mpc[12]) +
         ir9 * (xy * hx2my2 * mpc[16] + 0.125 * (x2 * x2mty2 - y2 * tx2my2) * mpc[24] + yz * tx2my2 * mpc[17] +
                zx * x2mty2 * mpc[23] + (7.0 * z2 - r2) * (xy * mpc[18] + hx2my2 * mpc[22]) +
                (7.0 * z2 - 3.0 * r2) * (yz * mpc[19] + zx * mpc[21]) +
                (35.0 * z2 * z2 - 30.0 * z2 * r2 + 3.0 * r2 * r2) * mpc[20]);
}

// Ghost q of a level's frame and its chain of boundary points inwards.  q enumerates the
// shell: the two k planes, then the two j rows of each inner plane, then the two i ends
// of each inner row.  The reference fills x1 faces, then x2 faces over all i, then x3
// faces over all (i, j), so an edge or corner ghost is 2 phi_s(p) minus the value inside
// it along the last face that writes it (at most three points); the chain ends at the
// interior cell (kk, jj, ii).  False past the last ghost.
struct GhostChain {
  int k, j, i, kk, jj, ii, depth;
  double px[3], py[3], pz[3];
};
__device__ __forceinline__ bool ghost_chain(const MPGeom &G, unsigned q, GhostChain &c) {
  const int n1 = G.n1, n2 = G.n2, n3 = G.n3;
  const unsigned w1 = n1 + 2, w2 = n2 + 2;
  const unsigned np = 2 * w1 * w2, nr = 2 * (unsigned)n3 * w1, nc = 2 * (unsigned)n3 * n2;
  if (q < np) {
    const unsigned side = q / (w1 * w2), r = q - side * w1 * w2;
    c.k = side ? n3 + 1 : 0; c.j = r / w1; c.i = r - c.j * w1;
  } else if ((q -= np) < nr) {
    const unsigned row = q / w1;
    c.i = q - row * w1; c.k = 1 + row / 2; c.j = (row & 1) ? n2 + 1 : 0;
  } else if ((q -= nr) < nc) {
    const unsigned row = q / 2;
    c.i = (q & 1) ? n1 + 1 : 0; c.k = 1 + row / n2; c.j = 1 + row % n2;
  } else {
    return false;
  }
  c.depth = 0;
  c.kk = c.k; c.jj = c.j; c.ii = c.i;
  while (c.depth < 3) {
    const int d = c.depth;
    if (c.kk == 0 || c.kk == n3 + 1) {
      c.px[d] = mp_centre(G, 0, c.ii); c.py[d] = mp_centre(G, 1, c.jj);
      c.pz[d] = mp_face(G, 2, c.kk == 0 ? 1 : n3 + 1);
      c.kk = (c.kk == 0) ? 1 : n3;
    } else if (c.jj == 0 || c.jj == n2 + 1) {
      c.px[d] = mp_centre(G, 0, c.ii); c.pz[d] = mp_centre(G, 2, c.kk);
      c.py[d] = mp_face(G, 1, c.jj == 0 ? 1 : n2 + 1);
      c.jj = (c.jj == 0) ? 1 : n2;
    } else if (c.ii == 0 || c.ii == n1 + 1) {
      c.py[d] = mp_centre(G, 1, c.jj); c.pz[d] = mp_centre(G, 2, c.kk);
      c.px[d] = mp_face(G, 0, c.ii == 0 ? 1 : n1 + 1);
      c.ii = (c.ii == 0) ? 1 : n1;
    } else {
      break;
    }
    ++c.depth;
  }
  return true;
}

// The multipole expansion at every boundary point of every ghost's chain, once per solve
// and level (the coefficients and origin are fixed during a solve): bcv[3q + d].
__global__ void __launch_bounds__(BS)
k_mb_bc_fill(double *__restrict__ bcv, MPGeom G, const double *__restrict__ mp, int order) {
  const unsigned q = xcd_slot(blockIdx.x, gridDim.x) * BS + threadIdx.x;
  GhostChain c;
  if (!ghost_chain(G, q, c)) return;
  for (int d = 0; d < c.depth; ++d)
    bcv[3 * (int64_t)q + d] = mp_phis(mp + 3, order, c.px[d] - mp[0], c.py[d] - mp[1], c.pz[d] - mp[2]);
}

// MGMultipoleInnerX1..OuterX3 (mgbval_multipole.cpp:28-426) on every ghost of a level in
// one launch: ghost = 2 phi_s(p) - (the value inside it), along the chain, with phi_s from
// bcv (the same doubles k_mb_bc_fill computed).
__global__ void __launch_bounds__(BS)
k_mb_bc(const int *__restrict__ gate, double *__restrict__ u, MPGeom G, const double *__restrict__ bcv) {
  if (gate && *gate) return;   // a closed gate: the recorded V-cycle loop has ended
  const unsigned q = xcd_slot(blockIdx.x, gridDim.x) * BS + threadIdx.x;
  GhostChain c;
  if (!ghost_chain(G, q, c)) return;
  const int n1 = G.n1, n2 = G.n2;
  double v = u[BX(n1, n2, c.kk, c.jj, c.ii)];
  for (int d = c.depth - 1; d >= 0; --d) v = 2.0 * bcv[3 * (int64_t)q + d] - v;
  u[BX(n1, n2, c.k, c.j, c.i)] = v;
}

// The same chain for a correction of the potential: the boundary values are those of
// the potential itself, so the correction's ghosts take 2 * 0 - (the value inside).
__global__ void __launch_bounds__(BS)
k_mb_bc_hom(const int *__restrict__ gate, float *__restrict__ u, MPGeom G) {
  if (gate && *gate) return;   // a closed gate: the recorded V-cycle loop has ended
  const unsigned q = xcd_slot(blockIdx.x, gridDim.x) * BS + threadIdx.x;
  GhostChain c;
  if (!ghost_chain(G, q, c)) return;
  const int n1 = G.n1, n2 = G.n2;
  float v = u[BX(n1, n2, c.kk, c.jj, c.ii)];
  for (int d = c.depth - 1; d >= 0; --d) v = -v;
  u[BX(n1, n2, c.k, c.j, c.i)] = v;
}

// red-black update of the framed level (MGGravity::Smooth, mg_gravity.cpp:220-273)
template <typename T>
__global__ void __launch_bounds__(BS)
k_mb_smooth(const int *__restrict__ gate,
            T *__restrict__ u, const T *__restrict__ src, int n1, int n2, int n3, T dx2, T isix, int color) {
  if (gate && *gate) return;   // a closed gate: the recorded V-cycle loop has ended
  const int nh = (n1 + 1) / 2;
  const unsigned t = xcd_slot(blockIdx.x, gridDim.x) * BS + threadIdx.x;
  if (t >= (unsigned)nh * n2 * n3) return;
  const int h = t % nh, r = t / nh;
  const int j = 1 + r % n2, k = 1 + r / n2;
  const int i = 1 + 2 * h + ((color + k + j) & 1);   // (color + k + j) parity in framed indices
  if (i > n1) return;
  const unsigned id = BX(n1, n2, k, j, i), sj = n1 + 2, sk = (unsigned)(n1 + 2) * (n2 + 2);
  u[id] = gs_value(u[id], u[id + sk], u[id + sj], u[id + 1], u[id - sk], u[id - sj], u[id - 1], src[id], dx2,
                   isix);
}


template <typename T>
__device__ __forceinline__ T mb_defect(const T *u, const T *src, unsigned id, unsigned sj, unsigned sk, T idx2) {
  return (T(6.0) * u[id] - u[id + sk] - u[id + sj] - u[id + 1] - u[id - sk] - u[id - sj] - u[id - 1]) * idx2 +
         src[id];
}

// FAS: uold = u over the framed level (StoreOldData, multigrid.cpp:645-653), then
// src -= (6u - sum of neighbours) idx2 on the interior (CalculateFASRHS,
// mg_gravity.cpp:324-351)
template <typename T>
__global__ void __launch_bounds__(BS)
k_mb_fas(const int *__restrict__ gate,
         const T *__restrict__ u, T *__restrict__ src, T *__restrict__ uold, int n1, int n2, int n3, T idx2) {
  if (gate && *gate) return;   // a closed gate: the recorded V-cycle loop has ended
  const unsigned t = xcd_slot(blockIdx.x, gridDim.x) * BS + threadIdx.x;
  const unsigned w1 = n1 + 2, w2 = n2 + 2;
  if (t >= w1 * w2 * (unsigned)(n3 + 2)) return;
  uold[t] = u[t];
  const int i = t % w1, r = t / w1, j = r % w2, k = r / w2;
  if (i < 1 || i > n1 || j < 1 || j > n2 || k < 1 || k > n3) return;
  const unsigned sj = w1, sk = w1 * w2;
  src[t] -= (T(6.0) * u[t] - u[t + sk] - u[t + sj] - u[t + 1] - u[t - sk] - u[t - sj] - u[t - 1]) * idx2;
}

// RestrictBlock (multigrid.cpp:331-355): defect average into the coarse source and, in
// FAS, the average of u into the coarse u.  One thread per coarse interior cell.
template <typename T>
__global__ void __launch_bounds__(BS)
k_mb_restrict(const int *__restrict__ gate,
              const T *__restrict__ u, const T *__restrict__ src, T *__restrict__ csrc, T *__restrict__ cu,
              int n1, int n2, int n3, T idx2) {
  if (gate && *gate) return;   // a closed gate: the recorded V-cycle loop has ended
  const int c1 = n1 >> 1, c2 = n2 >> 1, c3 = n3 >> 1;
  const unsigned t = xcd_slot(blockIdx.x, gridDim.x) * BS + threadIdx.x;
  if (t >= (unsigned)c1 * c2 * c3) return;
  const int i = 1 + t % c1, r = t / c1, j = 1 + r % c2, k = 1 + r / c2;
  const int fi = 2 * i - 1, fj = 2 * j - 1, fk = 2 * k - 1;
  const unsigned sj = n1 + 2, sk = (unsigned)(n1 + 2) * (n2 + 2);
#define F(kk, jj, ii) BX(n1, n2, kk, jj, ii)
  const unsigned f[8] = {F(fk, fj, fi), F(fk, fj, fi + 1), F(fk, fj + 1, fi), F(fk, fj + 1, fi + 1),
                         F(fk + 1, fj, fi), F(fk + 1, fj, fi + 1), F(fk + 1, fj + 1, fi), F(fk + 1, fj + 1, fi + 1)};
#undef F
  T d[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) d[q] = mb_defect(u, src, f[q], sj, sk, idx2);
  const unsigned c = BX(c1, c2, k, j, i);
  csrc[c] = T(0.125) * (d[0] + d[1] + d[2] + d[3] + d[4] + d[5] + d[6] + d[7]);
  cu[c] = T(0.125) * (u[f[0]] + u[f[1]] + u[f[2]] + u[f[3]] + u[f[4]] + u[f[5]] + u[f[6]] + u[f[7]]);
}

// ProlongateAndCorrect with FAS (multigrid.cpp:361-379, 733-829): the fine interior
// gains the trilinear interpolation of (u - uold) of the framed coarse level.
template <typename T>
__global__ void __launch_bounds__(BS)
k_mb_prolong(const int *__restrict__ gate,
             const T *__restrict__ cu, const T *__restrict__ cuold, T *__restrict__ fu, int n1, int n2, int n3) {
  if (gate && *gate) return;   // a closed gate: the recorded V-cycle loop has ended
  const unsigned t = xcd_slot(blockIdx.x, gridDim.x) * BS + threadIdx.x;
  if (t >= (unsigned)n1 * n2 * n3) return;
  const int fi = 1 + t % n1, r = t / n1, fj = 1 + r % n2, fk = 1 + r / n2;
  const int c1 = n1 >> 1, c2 = n2 >> 1;
  const int i = (fi - 1) / 2 + 1, j = (fj - 1) / 2 + 1, k = (fk - 1) / 2 + 1;
  const int di = ((fi - 1) & 1) ? 1 : -1, dj = ((fj - 1) & 1) ? 1 : -1, dk = ((fk - 1) & 1) ? 1 : -1;
#define C(kk, jj, ii) (cu[BX(c1, c2, kk, jj, ii)] - cuold[BX(c1, c2, kk, jj, ii)])
  fu[BX(n1, n2, fk, fj, fi)] +=
      T(0.015625) * (T(27.0) * C(k, j, i) + C(k + dk, j + dj, i + di) +
                     T(9.0) * (C(k, j, i + di) + C(k, j + dj, i) + C(k + dk, j, i)) +
                     T(3.0) * (C(k + dk, j + dj, i) + C(k + dk, j, i + di) + C(k, j + dj, i + di)));
#undef C
}

// k_mb_prolong for the two x1 children (2i-1, 2i) of each coarse cell i, which share the
// coarse (u - uold) values at i-1, i, i+1; every fine cell's sum is k_mb_prolong's, term
// for term.  n1 even (every level above the root grid).
template <typename T>
__global__ void __launch_bounds__(BS)
k_mb_prolong_pairs(const int *__restrict__ gate, const T *__restrict__ cu, const T *__restrict__ cuold,
                   T *__restrict__ fu, int n1, int n2, int n3) {
  if (gate && *gate) return;   // a closed gate: the recorded V-cycle loop has ended
  const int c1 = n1 >> 1, c2 = n2 >> 1;
  const unsigned t = xcd_slot(blockIdx.x, gridDim.x) * BS + threadIdx.x;
  if (t >= (unsigned)c1 * n2 * n3) return;
  const int i = 1 + t % c1, r = t / c1, fj = 1 + r % n2, fk = 1 + r / n2;
  const int j = (fj - 1) / 2 + 1, k = (fk - 1) / 2 + 1;
  const int dj = ((fj - 1) & 1) ? 1 : -1, dk = ((fk - 1) & 1) ? 1 : -1;
#define C(kk, jj, ii) (cu[BX(c1, c2, kk, jj, ii)] - cuold[BX(c1, c2, kk, jj, ii)])
  const T c0 = C(k, j, i), cj = C(k, j + dj, i), ck = C(k + dk, j, i), cjk = C(k + dk, j + dj, i);
  const unsigned f = BX(n1, n2, fk, fj, 2 * i - 1);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int di = h ? 1 : -1;
    const T ci = C(k, j, i + di), cij = C(k, j + dj, i + di), cik = C(k + dk, j, i + di),
            cijk = C(k + dk, j + dj, i + di);
    fu[f + h] += T(0.015625) * (T(27.0) * c0 + cijk + T(9.0) * (ci + cj + ck) + T(3.0) * (cjk + cik + cij));
  }
#undef C
}

// Mixed precision with multipole boundaries: the FP64 defect of the framed finest level
// (ghosts filled) becomes the FP32 source of the correction cycle, whose correction
// starts at zero over the framed level.
__global__ void __launch_bounds__(BS)
k_mb_defect32(const int *__restrict__ gate,
              const double *__restrict__ u, const double *__restrict__ src, float *__restrict__ src32,
              float *__restrict__ e32, int n1, int n2, int n3, double idx2) {
  if (gate && *gate) return;   // a closed gate: the recorded V-cycle loop has ended
  const unsigned t = xcd_slot(blockIdx.x, gridDim.x) * BS + threadIdx.x;
  const unsigned w1 = n1 + 2, w2 = n2 + 2;
  if (t >= w1 * w2 * (unsigned)(n3 + 2)) return;
  e32[t] = 0.f;
  const int i = t % w1, r = t / w1, j = r % w2, k = r / w2;
  if (i < 1 || i > n1 || j < 1 || j > n2 || k < 1 || k > n3) return;
  src32[t] = (float)mb_defect(u, src, t, w1, w1 * w2, idx2);
}

// phi += e on the interior of the framed finest level
__global__ void __launch_bounds__(BS)
k_mb_add32(const int *__restrict__ gate, double *__restrict__ u, const float *__restrict__ e, int n1, int n2, int n3) {
  if (gate && *gate) return;   // a closed gate: the recorded V-cycle loop has ended
  const unsigned t = xcd_slot(blockIdx.x, gridDim.x) * BS + threadIdx.x;
  const unsigned w1 = n1 + 2, w2 = n2 + 2;
  if (t >= w1 * w2 * (unsigned)(n3 + 2)) return;
  const int i = t % w1, r = t / w1, j = r % w2, k = r / w2;
  if (i < 1 || i > n1 || j < 1 || j > n2 || k < 1 || k > n3) return;
  u[t] += (double)e[t];
}

// The coarse end of a V(1,1) cycle (vcycle, vcycle_b, vcycle_b32) in one workgroup: levels
// `top` down to 0 and back, held in LDS from the first load to the last store.  Each step is
// the per-cell arithmetic of the per-level kernels (k_mg_smooth, k_mg_defect_restrict,
// k_mg_prolong; k_mb_fas, k_mb_smooth, k_mb_restrict, k_mb_prolong with the chain of k_mb_bc,
// or k_mb_bc_hom for the FP32 correction), separated by workgroup barriers, so the result
// equals the per-level launches bit for bit.  What bounds it is the latency of a step: about
// 35 (multipole) or 24 (periodic) steps run one after the other on one CU.  Through global
// memory the periodic levels of 16^3 and below took 28 us, from LDS 18; the multipole levels
// of 8^3 and below took 44 us, with ghost fills between the steps, and those of 16^3 and
// below (14 launches more) now 35.
//
// Framed levels keep u with its frame, where each face ghost holds the constant 2 phi_s and
// a stencil next to it takes 2 phi_s - (its own cell), the value a ghost fill would have
// stored; so no fills run between the steps.  The frame of (u - uold) that the prolongation
// reads, edges and corners included, comes from the chains when the coarse level is done.
// Every barrier is reached by every thread: loops have workgroup-uniform bounds.
enum : int { BC_PER, BC_MP, BC_HOM };   // periodic wrap; multipole values; homogeneous chain
constexpr int COARSE_CELLS = 4096, COARSE_BS = 1024, MAXC = 8;
constexpr int COARSE_LDS = 15872;   // elements: 124 KB of the CU's 160 KB in FP64

template <typename T>
struct CoarseLevel {
  T *u, *src, *old;
  const double *bcv;
  int n1, n2, n3;
  T dx2, idx2;
  int lu, ls, lo, lb;   // offsets in LDS of u, src, old (below top) and bcv (below top)
};
template <typename T>
struct CoarseSet {
  CoarseLevel<T> lv[MAXC];
};

// t / n for t < 2^14: the quotient in FP32 is within 2^-8 / n of (t + 1/2) / n, which is at
// least 1 / (2n) away from a whole number
struct FastDiv {
  float inv;
  __device__ __forceinline__ explicit FastDiv(int n) : inv(1.0f / (float)n) {}
  __device__ __forceinline__ int operator()(int t) const { return (int)(((float)t + 0.5f) * inv); }
};

// Ghost q of a framed level in the order of ghost_chain: its cell, the interior cell at the
// end of its chain and the chain's length
struct GhostCell {
  int k, j, i, kk, jj, ii, depth;
};
__host__ __device__ __forceinline__ int ghost_count(int n1, int n2, int n3) {
  return 2 * (n1 + 2) * (n2 + 2) + 2 * n3 * (n1 + 2) + 2 * n3 * n2;
}
__device__ __forceinline__ GhostCell ghost_cell(int n1, int n2, int n3, int q) {
  const int w1 = n1 + 2, w2 = n2 + 2, np = 2 * w1 * w2, nr = 2 * n3 * w1;
  GhostCell c;
  if (q < np) {
    const int side = q >= w1 * w2, r = q - side * w1 * w2;
    c.k = side ? n3 + 1 : 0; c.j = FastDiv(w1)(r); c.i = r - c.j * w1;
  } else if ((q -= np) < nr) {
    const int row = FastDiv(w1)(q);
    c.i = q - row * w1; c.k = 1 + row / 2; c.j = (row & 1) ? n2 + 1 : 0;
  } else {
    q -= nr;
    const int row = q / 2, kr = FastDiv(n2)(row);
    c.i = (q & 1) ? n1 + 1 : 0; c.k = 1 + kr; c.j = 1 + row - kr * n2;
  }
  c.kk = min(max(c.k, 1), n3); c.jj = min(max(c.j, 1), n2); c.ii = min(max(c.i, 1), n1);
  c.depth = (c.k != c.kk) + (c.j != c.jj) + (c.i != c.ii);
  return c;
}
// the chain's value from the interior value v and its boundary values b[0 .. depth)
template <int KIND, typename T>
__device__ __forceinline__ T chain_value(T v, int depth, const double *b) {
  for (int d = depth - 1; d >= 0; --d) {
    if constexpr (KIND == BC_MP) v = 2.0 * b[d] - v;
    else v = -v;
  }
  return v;
}

// u and its six neighbours at interior cell (k, j, i) of a level in LDS (0-based)
template <typename T>
struct Cross {
  T c, kp, jp, ip, km, jm, im;
};
template <int KIND, typename T>
__device__ __forceinline__ int coarse_id(const CoarseLevel<T> &L, int k, int j, int i) {
  return KIND == BC_PER ? (k * L.n2 + j) * L.n1 + i : ((k + 1) * (L.n2 + 2) + j + 1) * (L.n1 + 2) + i + 1;
}
template <int KIND, typename T>
__device__ __forceinline__ Cross<T> cross_at(const CoarseLevel<T> &L, const T *u, int k, int j, int i) {
  const int n1 = L.n1, n2 = L.n2, n3 = L.n3;
  const int id = coarse_id<KIND>(L, k, j, i);
  Cross<T> x;
  x.c = u[id];
  if constexpr (KIND == BC_PER) {
    const int sk = n1 * n2;
    x.kp = u[k == n3 - 1 ? id - (n3 - 1) * sk : id + sk];
    x.km = u[k == 0 ? id + (n3 - 1) * sk : id - sk];
    x.jp = u[j == n2 - 1 ? id - (n2 - 1) * n1 : id + n1];
    x.jm = u[j == 0 ? id + (n2 - 1) * n1 : id - n1];
    x.ip = u[i == n1 - 1 ? id - (n1 - 1) : id + 1];
    x.im = u[i == 0 ? id + n1 - 1 : id - 1];
  } else {
    const int sj = n1 + 2, sk = sj * (n2 + 2);
    x.kp = u[id + sk]; x.km = u[id - sk];
    x.jp = u[id + sj]; x.jm = u[id - sj];
    x.ip = u[id + 1]; x.im = u[id - 1];
    if (k == n3 - 1) x.kp -= x.c;
    if (k == 0) x.km -= x.c;
    if (j == n2 - 1) x.jp -= x.c;
    if (j == 0) x.jm -= x.c;
    if (i == n1 - 1) x.ip -= x.c;
    if (i == 0) x.im -= x.c;
  }
  return x;
}
template <typename T>
__device__ __forceinline__ T cross_lap(const Cross<T> &x) {   // operand order of mb_defect / defect_at
  return T(6.0) * x.c - x.kp - x.jp - x.ip - x.km - x.jm - x.im;
}

template <int KIND, typename T>
__device__ __forceinline__ void coarse_smooth(const CoarseLevel<T> &L, T *s, int color, T isix) {
  const int nh = (L.n1 + 1) / 2;
  const FastDiv dh(nh), d2(L.n2);
  T *u = s + L.lu;
  const T *src = s + L.ls;
  for (int t = threadIdx.x; t < nh * L.n2 * L.n3; t += COARSE_BS) {
    const int r = dh(t), k = d2(r), j = r - k * L.n2;
    const int i = 2 * (t - r * nh) + ((color + k + j) & 1);
    if (i >= L.n1) continue;
    const Cross<T> x = cross_at<KIND>(L, u, k, j, i);
    u[coarse_id<KIND>(L, k, j, i)] = gs_value(x.c, x.kp, x.jp, x.ip, x.km, x.jm, x.im,
                                              src[(k * L.n2 + j) * L.n1 + i], L.dx2, isix);
  }
  __syncthreads();
}

template <int KIND, typename T>
__device__ __forceinline__ void coarse_fas(const CoarseLevel<T> &L, T *s, T *old, const double *bcv) {
  const FastDiv d1(L.n1), d2(L.n2);
  const T *u = s + L.lu;
  T *src = s + L.ls;
  for (int t = threadIdx.x; t < L.n1 * L.n2 * L.n3; t += COARSE_BS) {
    const int r = d1(t), i = t - r * L.n1, k = d2(r), j = r - k * L.n2;
    const Cross<T> x = cross_at<KIND>(L, u, k, j, i);
    old[coarse_id<KIND>(L, k, j, i)] = x.c;
    src[t] -= cross_lap(x) * L.idx2;
  }
  for (int q = threadIdx.x; q < ghost_count(L.n1, L.n2, L.n3); q += COARSE_BS) {
    const GhostCell c = ghost_cell(L.n1, L.n2, L.n3, q);
    old[BX(L.n1, L.n2, c.k, c.j, c.i)] = chain_value<KIND>(u[BX(L.n1, L.n2, c.kk, c.jj, c.ii)], c.depth, bcv + 3 * q);
  }
  __syncthreads();
}

template <int KIND, typename T>
__device__ __forceinline__ void coarse_restrict(const CoarseLevel<T> &F, const CoarseLevel<T> &C, T *s) {
  const FastDiv d1(C.n1), d2(C.n2);
  const T *u = s + F.lu, *src = s + F.ls;
  for (int t = threadIdx.x; t < C.n1 * C.n2 * C.n3; t += COARSE_BS) {
    const int r = d1(t), i = t - r * C.n1, k = d2(r), j = r - k * C.n2;
    T sd = T(0.0), su = T(0.0);
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int fk = 2 * k + (q >> 2), fj = 2 * j + ((q >> 1) & 1), fi = 2 * i + (q & 1);
      const Cross<T> x = cross_at<KIND>(F, u, fk, fj, fi);
      const T d = cross_lap(x) * F.idx2 + src[(fk * F.n2 + fj) * F.n1 + fi];
      sd = q ? sd + d : d;
      su = q ? su + x.c : x.c;
    }
    s[C.ls + t] = T(0.125) * sd;
    s[C.lu + coarse_id<KIND>(C, k, j, i)] = KIND == BC_PER ? T(0.0) : T(0.125) * su;
  }
  __syncthreads();
}

// old = u - old over the framed level (the values k_mb_prolong interpolates)
template <int KIND, typename T>
__device__ __forceinline__ void coarse_change(const CoarseLevel<T> &L, T *s, const double *bcv) {
  const FastDiv d1(L.n1), d2(L.n2);
  const T *u = s + L.lu;
  T *old = s + L.lo;
  for (int t = threadIdx.x; t < L.n1 * L.n2 * L.n3; t += COARSE_BS) {
    const int r = d1(t), k = d2(r), id = coarse_id<KIND>(L, k, r - k * L.n2, t - r * L.n1);
    old[id] = u[id] - old[id];
  }
  for (int q = threadIdx.x; q < ghost_count(L.n1, L.n2, L.n3); q += COARSE_BS) {
    const GhostCell c = ghost_cell(L.n1, L.n2, L.n3, q);
    const unsigned id = BX(L.n1, L.n2, c.k, c.j, c.i);
    old[id] = chain_value<KIND>(u[BX(L.n1, L.n2, c.kk, c.jj, c.ii)], c.depth, bcv + 3 * q) - old[id];
  }
  __syncthreads();
}

template <int KIND, typename T>
__device__ __forceinline__ void coarse_prolong(const CoarseLevel<T> &F, const CoarseLevel<T> &C, T *s) {
  const FastDiv d1(F.n1), d2(F.n2);
  T *u = s + F.lu;
  const T *c = s + (KIND == BC_PER ? C.lu : C.lo);
  for (int t = threadIdx.x; t < F.n1 * F.n2 * F.n3; t += COARSE_BS) {
    const int r = d1(t), fi = t - r * F.n1, fk = d2(r), fj = r - fk * F.n2;
    const int i = fi >> 1, j = fj >> 1, k = fk >> 1;
    int ip = i + ((fi & 1) ? 1 : -1), jp = j + ((fj & 1) ? 1 : -1), kp = k + ((fk & 1) ? 1 : -1);
    if constexpr (KIND == BC_PER) { ip = wrap(ip, C.n1); jp = wrap(jp, C.n2); kp = wrap(kp, C.n3); }
#define V(kk, jj, ii) c[coarse_id<KIND>(C, kk, jj, ii)]
    u[coarse_id<KIND>(F, fk, fj, fi)] +=
        T(0.015625) * (T(27.0) * V(k, j, i) + V(kp, jp, ip) + T(9.0) * (V(k, j, ip) + V(k, jp, i) + V(kp, j, i)) +
                       T(3.0) * (V(kp, jp, i) + V(kp, j, ip) + V(k, jp, ip)));
#undef V
  }
  __syncthreads();
}

template <typename T, int KIND>
__global__ void __launch_bounds__(COARSE_BS)
k_mg_coarse(const int *__restrict__ gate, CoarseSet<T> S, int top, int fmglevel, int coffset, int ni, T isix,
            int first_sweep_done) {
  const int closed = gate ? *gate : 0;   // a closed gate: the recorded V-cycle loop has ended
  __shared__ T s[COARSE_LDS];
  // every global value into registers before the first is used: the interior of top, and with
  // multipole values its face constants and the boundary values of the levels below (the
  // chunks that a cubic hierarchy has; loops take the rest)
  constexpr int NI = COARSE_CELLS / COARSE_BS, NG = 2, NL = KIND == BC_MP ? 4 : 1;
  const CoarseLevel<T> &LT = S.lv[top];
  const int nt = LT.n1 * LT.n2 * LT.n3, gt = KIND == BC_PER ? 0 : ghost_count(LT.n1, LT.n2, LT.n3);
  T uv[NI], sv[NI], gv[NG];
  double bl[NL][NG];
  int ut[NI];
  {
    const FastDiv d1(LT.n1), d2(LT.n2);
#pragma unroll
    for (int e = 0; e < NI; ++e) {
      const int t = threadIdx.x + e * COARSE_BS;
      if (t >= nt) continue;
      const int r = d1(t), k = d2(r);
      ut[e] = coarse_id<KIND>(LT, k, r - k * LT.n2, t - r * LT.n1);
      uv[e] = LT.u[ut[e]];
      sv[e] = LT.src[KIND == BC_PER ? t : ut[e]];
    }
    if constexpr (KIND == BC_MP) {
#pragma unroll
      for (int e = 0; e < NG; ++e) {
        const int q = threadIdx.x + e * COARSE_BS;
        gv[e] = q < gt ? 2.0 * LT.bcv[3 * q] : 0.0;
      }
#pragma unroll
      for (int l = 0; l < NL; ++l) {
        if (l >= top) break;
        const int nb = 3 * ghost_count(S.lv[l].n1, S.lv[l].n2, S.lv[l].n3);
#pragma unroll
        for (int e = 0; e < NG; ++e) {
          const int q = threadIdx.x + e * COARSE_BS;
          if (q < nb) bl[l][e] = S.lv[l].bcv[q];
        }
      }
    }
  }
  if (closed) return;
#pragma unroll
  for (int e = 0; e < NI; ++e) {
    const int t = threadIdx.x + e * COARSE_BS;
    if (t >= nt) continue;
    s[LT.lu + ut[e]] = uv[e];
    s[LT.ls + t] = sv[e];
  }
  if constexpr (KIND == BC_MP) {
#pragma unroll
    for (int l = 0; l < NL; ++l) {
      if (l >= top) break;
      const int nb = 3 * ghost_count(S.lv[l].n1, S.lv[l].n2, S.lv[l].n3);
#pragma unroll
      for (int e = 0; e < NG; ++e) {
        const int q = threadIdx.x + e * COARSE_BS;
        if (q < nb) s[S.lv[l].lb + q] = bl[l][e];
      }
    }
    for (int l = 0; l < top; ++l) {
      const int nb = 3 * ghost_count(S.lv[l].n1, S.lv[l].n2, S.lv[l].n3);
      for (int q = threadIdx.x + (l < NL ? NG * COARSE_BS : 0); q < nb; q += COARSE_BS)
        s[S.lv[l].lb + q] = S.lv[l].bcv[q];
    }
    __syncthreads();
  }
  if constexpr (KIND != BC_PER) {   // 2 phi_s into the face ghosts (the other ghosts are not read)
    for (int l = 0; l <= top; ++l) {
      const CoarseLevel<T> &L = S.lv[l];
      for (int q = threadIdx.x, e = 0; q < ghost_count(L.n1, L.n2, L.n3); q += COARSE_BS, ++e) {
        const GhostCell c = ghost_cell(L.n1, L.n2, L.n3, q);
        T face = T(0.0);
        if constexpr (KIND == BC_MP)
          face = l < top ? 2.0 * s[L.lb + 3 * q] : (e == 0 ? gv[0] : (e == 1 ? gv[1] : 2.0 * L.bcv[3 * q]));
        s[L.lu + BX(L.n1, L.n2, c.k, c.j, c.i)] = face;
      }
    }
  }
  __syncthreads();
  // boundary values of level l: in LDS below top (T is double with multipole values)
  auto bv = [&](int l) -> const double * {
    if constexpr (KIND == BC_MP) return l < top ? s + S.lv[l].lb : S.lv[l].bcv;
    else return nullptr;
  };
  for (int l = top; l > 0; --l) {
    if constexpr (KIND != BC_PER)
      if (l < fmglevel) coarse_fas<KIND>(S.lv[l], s, l < top ? s + S.lv[l].lo : S.lv[l].old, bv(l));
    if (!(first_sweep_done && l == top)) coarse_smooth<KIND>(S.lv[l], s, 0 ^ coffset, isix);
    coarse_smooth<KIND>(S.lv[l], s, 1 ^ coffset, isix);
    coarse_restrict<KIND>(S.lv[l], S.lv[l - 1], s);
  }
  if constexpr (KIND == BC_PER) {   // SolveCoarsestGrid of the one-cell root, multigrid_driver.cpp:781-787
    if (threadIdx.x == 0) s[S.lv[0].lu] = T(0.0);
    __syncthreads();
  } else {
    coarse_fas<KIND>(S.lv[0], s, 0 < top ? s + S.lv[0].lo : S.lv[0].old, bv(0));
    for (int it = 0; it < ni; ++it) {
      coarse_smooth<KIND>(S.lv[0], s, 0 ^ coffset, isix);
      coarse_smooth<KIND>(S.lv[0], s, 1 ^ coffset, isix);
    }
  }
  for (int l = 1; l <= top; ++l) {
    if constexpr (KIND != BC_PER) coarse_change<KIND>(S.lv[l - 1], s, bv(l - 1));
    coarse_prolong<KIND>(S.lv[l], S.lv[l - 1], s);
    coarse_smooth<KIND>(S.lv[l], s, 0 ^ coffset, isix);
    coarse_smooth<KIND>(S.lv[l], s, 1 ^ coffset, isix);
  }
  // u of every level (a later solve may start from it), with top's frame filled
  for (int l = 0; l <= top; ++l) {
    const CoarseLevel<T> &L = S.lv[l];
    const FastDiv d1(L.n1), d2(L.n2);
    for (int t = threadIdx.x; t < L.n1 * L.n2 * L.n3; t += COARSE_BS) {
      const int r = d1(t), k = d2(r), id = coarse_id<KIND>(L, k, r - k * L.n2, t - r * L.n1);
      L.u[id] = s[L.lu + id];
    }
  }
  if constexpr (KIND != BC_PER) {
    const CoarseLevel<T> &L = S.lv[top];
    const double *b = bv(top);
    for (int q = threadIdx.x; q < ghost_count(L.n1, L.n2, L.n3); q += COARSE_BS) {
      const GhostCell c = ghost_cell(L.n1, L.n2, L.n3, q);
      L.u[BX(L.n1, L.n2, c.k, c.j, c.i)] =
          chain_value<KIND>(s[L.lu + BX(L.n1, L.n2, c.kk, c.jj, c.ii)], c.depth, b + 3 * q);
    }
  }
}

// ================================================================ whole passes of a level
// k_mg_down does everything of one level on the way down (FAS right-hand side, both sweeps,
// restriction) and k_mg_up everything on the way up (prolongation and correction, both
// sweeps) in one launch each; the per-step form takes three to seven, every one of them a trip
// of the level through memory and, on small levels, 3.5 us of launch.  Every value is formed
// by the arithmetic of the per-step kernels, so the result equals theirs bit for bit.
//
// A workgroup owns TP_I x TP_J columns and kc planes.  A thread owns a pair of cells along i of
// the tile or of its ring (as wide as the steps reach) and walks the planes upwards with the
// steps staggered: red on plane q, black on q-1, the defect on q-2.  A colour's update is one
// cell of every pair, so no lane idles; its neighbours along k are the thread's own registers,
// those along i and j come from the plane in LDS, updated in place.  The steps of an iteration
// work on different planes, and one barrier a plane suffices.  256^3 FP64 periodic: 126 us down
// (two sweeps and the restriction: 238) and 130 us up (263), where the bytes of u and source
// alone take 80; 64^3 multipole: 14 us down and 12 up (29 and 32 with the ghost fills).  On
// large levels an iteration's instructions bound it (259 down and 198 up for a pair of cells,
// 44 of them floating point), on small ones their latency: loads two or three planes ahead and
// planes split by cell parity in LDS made it no faster.  A tile held whole in LDS takes the same
// time on small levels and 36 us instead of 34 at 128^3.
//
// Passes run out of place, u -> tmp on the way down and tmp -> u on the way up, as tiles read
// each other's old values.  Periodic levels wrap; framed levels hold 2 phi_s in their face
// ghosts, as k_mg_coarse does, and k_mg_up stores the frame that the next level's prolongation
// and the defect sum read, k_mg_down the frame of the FAS copy.
constexpr int TP_I = 32, TP_J = 16;

template <typename T>
struct PassArgs {
  const T *uin;          // u (down) or tmp (up)
  T *uout;               // tmp (down) or u (up)
  const T *src;
  T *rhs, *old;          // down with FAS: right-hand side and copy of u
  T *csrc, *cu;          // down: the coarse source and u
  const T *cc, *ccold;   // up: the coarse u and its FAS copy (framed levels)
  const double *bcv;     // boundary values of this level (BC_MP)
  int n1, n2, n3, kc;
  T dx2, idx2, isix;
  int c0;                // colour of the first sweep
  int first_sweep_done;  // down: the first sweep is in uin already
};

template <int KIND>
__device__ __forceinline__ int64_t pass_id(int n1, int n2, int k, int j, int i) {   // 0-based cell
  if constexpr (KIND == BC_PER) return LIX(n1, n2, k, j, i);
  else return (int64_t)BX(n1, n2, k + 1, j + 1, i + 1);
}

// ghost_cell's q of framed cell (k, j, i), one of its coordinates at least in the frame
__device__ __forceinline__ unsigned ghost_index(int n1, int n2, int n3, int k, int j, int i) {
  const unsigned w1 = n1 + 2, w2 = n2 + 2, np = 2 * w1 * w2, nr = 2 * n3 * w1;
  if (k == 0 || k == n3 + 1) return (k ? w1 * w2 : 0) + j * w1 + i;
  if (j == 0 || j == n2 + 1) return np + (2 * (k - 1) + (j ? 1 : 0)) * w1 + i;
  return np + nr + 2 * ((unsigned)(k - 1) * n2 + j - 1) + (i ? 1 : 0);
}

// the ghosts whose chain ends at boundary cell (k, j, i) (0-based; every extent at least 2)
template <int KIND, typename T>
__device__ __forceinline__ void push_frame(T *u, const double *bcv, int n1, int n2, int n3, int k, int j, int i, T v) {
  const int gk = k == 0 ? 0 : (k == n3 - 1 ? n3 + 1 : -1), gj = j == 0 ? 0 : (j == n2 - 1 ? n2 + 1 : -1),
            gi = i == 0 ? 0 : (i == n1 - 1 ? n1 + 1 : -1);
  if (gk < 0 && gj < 0 && gi < 0) return;
  for (int e = 1; e < 8; ++e) {
    if (((e & 4) && gk < 0) || ((e & 2) && gj < 0) || ((e & 1) && gi < 0)) continue;
    const int kk = (e & 4) ? gk : k + 1, jj = (e & 2) ? gj : j + 1, ii = (e & 1) ? gi : i + 1;
    const double *b = KIND == BC_MP ? bcv + 3 * (int64_t)ghost_index(n1, n2, n3, kk, jj, ii) : nullptr;
    u[BX(n1, n2, kk, jj, ii)] = chain_value<KIND>(v, __popc(e), b);
  }
}

// two neighbouring values, 8 bytes aligned in FP64: framed rows start at odd cells
template <typename T>
struct alignas(sizeof(T)) Pair {
  T x, y;
};

// A thread's pair of columns (i, i+1), j of a tile with a ring of 2 PR cells along i and RJ
// along j, and the plane steps on it
template <int KIND, int PR, int RJ, typename T>
struct PassColumn {
  static constexpr int NP = TP_I / 2 + 2 * PR, NJ = TP_J + 2 * RJ, W = 2 * NP, PL = NJ * W;
  static constexpr int NT = (NP * NJ + 63) / 64 * 64;
  const PassArgs<T> &a;
  int i0, j0, k0, ni, nj, k1;   // the tile: first cells, sizes, planes [k0, k1)
  int p, row, i, j;             // the pair's place in the region and its first cell
  bool in, upd, tile;           // inside the domain; a row that is updated (not the region's edge); in the tile
  int last;                     // cells 1 .. last of a row of the region are updated
  int near0;                    // the pair's place in LDS, its row kept off the region's edge
  int64_t base, sk;             // index of the pair in plane 0 (wrapped), plane stride
  __device__ __forceinline__ PassColumn(const PassArgs<T> &a_) : a(a_) {
    const int ti = (a.n1 + TP_I - 1) / TP_I, tj = (a.n2 + TP_J - 1) / TP_J;
    const int w = (int)xcd_slot(blockIdx.x, gridDim.x), r = w / ti;
    i0 = (w - r * ti) * TP_I; j0 = (r % tj) * TP_J; k0 = (r / tj) * a.kc;
    ni = min(TP_I, a.n1 - i0); nj = min(TP_J, a.n2 - j0); k1 = min(k0 + a.kc, a.n3);
    row = (int)threadIdx.x / NP; p = (int)threadIdx.x - row * NP;
    i = i0 - 2 * PR + 2 * p; j = j0 - RJ + row;
    const bool use = 2 * p < ni + 4 * PR && row < nj + 2 * RJ;
    in = use && (KIND == BC_PER || ((unsigned)j < (unsigned)a.n2 && (unsigned)i < (unsigned)a.n1));
    upd = in && row >= 1 && row < nj + 2 * RJ - 1;
    last = ni + 4 * PR - 2;
    near0 = min(max(row, 1), NJ - 2) * W + 2 * p;
    tile = use && p >= PR && 2 * p < ni + 2 * PR && row >= RJ && row < nj + RJ;
    const int wi = KIND == BC_PER ? wrap(i, a.n1) : i, wj = KIND == BC_PER ? wrap(j, a.n2) : j;
    base = pass_id<KIND>(a.n1, a.n2, 0, wj, wi);
    sk = KIND == BC_PER ? (int64_t)a.n1 * a.n2 : (int64_t)(a.n1 + 2) * (a.n2 + 2);
  }
  __device__ __forceinline__ int plane(int q) const { return KIND == BC_PER ? wrap(q, a.n3) : q; }
  __device__ __forceinline__ bool plane_in(int q) const { return KIND == BC_PER || (unsigned)q < (unsigned)a.n3; }
  // plane q of x, and half the value of face ghosts (scale doubles it where it is used)
  __device__ __forceinline__ Pair<T> load(const T *__restrict__ x, int q) const {
    Pair<T> v = {T(0.0), T(0.0)};
    if (in && plane_in(q)) {
      v = *reinterpret_cast<const Pair<T> *>(x + base + plane(q) * sk);
    } else if constexpr (KIND == BC_MP) {
      const bool jin = (unsigned)j < (unsigned)a.n2, iin = (unsigned)i < (unsigned)a.n1, kin = plane_in(q);
      const bool kg = q == -1 || q == a.n3, jg = j == -1 || j == a.n2;
      if ((kg && jin && iin) || (kin && jg && iin)) {
        const double *b = a.bcv + 3 * (int64_t)ghost_index(a.n1, a.n2, a.n3, q + 1, j + 1, i + 1);
        v.x = b[0];
        v.y = b[3];
      } else if (kin && jin && i == -2) {
        v.y = a.bcv[3 * (int64_t)ghost_index(a.n1, a.n2, a.n3, q + 1, j + 1, 0)];
      } else if (kin && jin && i == a.n1) {
        v.x = a.bcv[3 * (int64_t)ghost_index(a.n1, a.n2, a.n3, q + 1, j + 1, a.n1 + 1)];
      }
    }
    return v;
  }
  __device__ __forceinline__ T scale(int q) const { return (KIND == BC_MP && !(in && plane_in(q))) ? T(2.0) : T(1.0); }
  __device__ __forceinline__ Pair<T> load_src(const T *__restrict__ x, int q) const {
    Pair<T> v = {T(0.0), T(0.0)};
    if (in && plane_in(q)) v = *reinterpret_cast<const Pair<T> *>(x + base + plane(q) * sk);
    return v;
  }
  // The neighbours in LDS (the row of plane s) of the pair's first (odd = 0) or second cell.
  // Every thread reads, from a row inside the region, so that the reads of all the steps of an
  // iteration are in flight together; the values of edge threads go nowhere.
  struct Near {
    T jp, jm, e;   // e: the cell beyond the pair
  };
  // the cell of the pair that has this colour on plane q (tiles and pairs start at even cells)
  __device__ __forceinline__ int odd_of(int q, int color) const { return (color + q + j) & 1; }
  __device__ __forceinline__ Near near(const T *s, int odd) const {
    const T *t = s + near0 + odd;
    return {t[W], t[-W], s[near0 + (odd ? 2 : -1)]};
  }
  // the cross of that cell on plane q: values c, neighbours along k in kp and km
  __device__ __forceinline__ Cross<T> cross(const Near &n, const Pair<T> &c, const Pair<T> &kp, const Pair<T> &km, int q,
                                            int odd) const {
    Cross<T> x;
    x.c = odd ? c.y : c.x;
    x.kp = odd ? kp.y : kp.x;
    x.km = odd ? km.y : km.x;
    x.jp = n.jp;
    x.jm = n.jm;
    x.ip = odd ? n.e : c.y;
    x.im = odd ? c.x : n.e;
    if constexpr (KIND != BC_PER) {
      if (q == a.n3 - 1) x.kp -= x.c;
      if (q == 0) x.km -= x.c;
      if (j == a.n2 - 1) x.jp -= x.c;
      if (j == 0) x.jm -= x.c;
      if (i + odd == a.n1 - 1) x.ip -= x.c;
      if (i + odd == 0) x.im -= x.c;
    }
    return x;
  }
  // one colour on plane q, whose values are c here and s in LDS
  __device__ __forceinline__ void smooth(T *s, const Near &n, Pair<T> &c, const Pair<T> &kp, const Pair<T> &km,
                                         const Pair<T> &f, int q, int odd) const {
    const Cross<T> x = cross(n, c, kp, km, q, odd);
    const T v = gs_value(x.c, x.kp, x.jp, x.ip, x.km, x.jm, x.im, odd ? f.y : f.x, a.dx2, a.isix);
    const int e = 2 * p + odd;
    if (upd && e >= 1 && e <= last && plane_in(q)) {
      if (odd) c.y = v;
      else c.x = v;
      s[row * W + e] = v;
    }
  }
  __device__ __forceinline__ void put(T *s, const Pair<T> &v) const {
    if (row < NJ) {
      s[row * W + 2 * p] = v.x;
      s[row * W + 2 * p + 1] = v.y;
    }
  }
};

template <typename T, int KIND, bool FAS>
__global__ void __launch_bounds__((PassColumn<KIND, 2, 3, T>::NT))
k_mg_down(const int *__restrict__ gate, PassArgs<T> a) {
  const int closed = gate ? *gate : 0;   // a closed gate: the recorded V-cycle loop has ended
  using Col = PassColumn<KIND, 2, 3, T>;
  // planes in flight: the defect's q-2 .. q+1 (with FAS one more, as a plane's right-hand side is
  // formed from old values before its first colour changes), and the one being stored
  constexpr int AH = FAS ? 2 : 1, NB = 4 + AH;
  __shared__ T s_u[NB][Col::PL];
  __shared__ T s_d[2][TP_J][TP_I];
  const Col t(a);
  const int qa = t.k0 - 2, qe = t.k1 + 1;   // red planes
  int slot = 0;                             // of plane q
  auto buf = [&](int d) -> T * {            // plane q + d
    int z = slot + d;
    z = z < 0 ? z + NB : (z >= NB ? z - NB : z);
    return s_u[z];
  };
  // registers: u of planes q+AH .. q-3, the source of q+1 (FAS) .. q-2, and the loads ahead
  Pair<T> m1 = t.load(a.uin, qa - 1), c = t.load(a.uin, qa), p1 = t.load(a.uin, qa + 1), p2 = {};
  Pair<T> f0 = t.load_src(a.src, qa), f1 = {}, fm1 = {}, fm2 = {}, m2 = {}, m3 = {};
  if constexpr (FAS) { p2 = t.load(a.uin, qa + 2); f1 = t.load_src(a.src, qa + 1); }
  Pair<T> un = t.load(a.uin, qa + AH + 1), fn = t.load_src(a.src, qa + AH);
  if (closed) return;
  auto doubled = [&](Pair<T> &v, int q) {
    if constexpr (KIND == BC_MP) { v.x *= t.scale(q); v.y *= t.scale(q); }
  };
  doubled(m1, qa - 1); doubled(c, qa); doubled(p1, qa + 1);
  t.put(buf(-1), m1);
  t.put(buf(0), c);
  t.put(buf(1), p1);
  if constexpr (FAS) { doubled(p2, qa + 2); t.put(buf(2), p2); }
  __syncthreads();
  // FAS right-hand side of plane q (values v, neighbours up and lo) into f
  auto fas = [&](Pair<T> &f, const T *s, const Pair<T> &v, const Pair<T> &up, const Pair<T> &lo, int q) {
    const typename Col::Near n0 = t.near(s, 0), n1 = t.near(s, 1);
    const T fx = f.x - cross_lap(t.cross(n0, v, up, lo, q, 0)) * a.idx2;
    const T fy = f.y - cross_lap(t.cross(n1, v, up, lo, q, 1)) * a.idx2;
    if (!t.plane_in(q)) return;
    f.x = fx;
    f.y = fy;
    if (t.tile && q >= t.k0 && q < t.k1) {
      *reinterpret_cast<Pair<T> *>(a.rhs + t.base + q * t.sk) = f;
      *reinterpret_cast<Pair<T> *>(a.old + t.base + q * t.sk) = v;
      if constexpr (KIND != BC_PER) {
        push_frame<KIND>(a.old, a.bcv, a.n1, a.n2, a.n3, q, t.j, t.i, v.x);
        push_frame<KIND>(a.old, a.bcv, a.n1, a.n2, a.n3, q, t.j, t.i + 1, v.y);
      }
    }
  };
  if constexpr (FAS) {
    fas(f0, buf(0), c, p1, m1, qa);
    __syncthreads();   // red on plane qa changes what its neighbours' right-hand sides read
  }
  T acc = T(0.0), uacc = T(0.0);
  Pair<T> dl = {};   // the own pair's defects of the plane before
  const int dj = t.row - 3, di = 2 * t.p - 4;
  const bool even = t.tile && (dj & 1) == 0;
  const T *const so = &s_d[0][t.tile ? dj | 1 : 0][t.tile ? di : 0];
  for (int q = qa; q <= qe; ++q) {
    const int odd = t.odd_of(q, a.c0), kd = q - 2, kr = q - 3;   // black on q-1 is the same cell of the pair
    const T *s2 = buf(-2);
    const typename Col::Near nr = t.near(buf(0), odd), nb = t.near(buf(-1), odd), d0 = t.near(s2, 0), d1 = t.near(s2, 1);
    const Pair<T> o = {so[(kr & 1) * (TP_I * TP_J)], so[(kr & 1) * (TP_I * TP_J) + 1]};
    if constexpr (FAS) fas(f1, buf(1), p1, p2, c, q + 1);
    if (!a.first_sweep_done) t.smooth(buf(0), nr, c, p1, m1, f0, q, odd);
    if (q - 1 >= t.k0 - 1) t.smooth(buf(-1), nb, m1, c, m2, fm1, q - 1, odd);
    // restriction of plane q-3, whose defects all rows have stored; the sums run over the cells
    // in the order of k_mg_defect_restrict / k_mb_restrict
    acc = (kr & 1) ? acc + dl.x : dl.x;
    acc = acc + dl.y;
    acc = acc + o.x;
    acc = acc + o.y;
    if (even && kr >= t.k0 && (kr & 1)) {
      const int64_t id = pass_id<KIND>(a.n1 >> 1, a.n2 >> 1, kr >> 1, t.j >> 1, t.i >> 1);
      a.csrc[id] = T(0.125) * acc;
      a.cu[id] = KIND == BC_PER ? T(0.0) : T(0.125) * uacc;
    }
    dl.x = cross_lap(t.cross(d0, m2, m1, m3, kd, 0)) * a.idx2 + fm2.x;
    dl.y = cross_lap(t.cross(d1, m2, m1, m3, kd, 1)) * a.idx2 + fm2.y;
    if constexpr (KIND != BC_PER) {
      uacc = (kd & 1) ? uacc + m2.x : m2.x;
      uacc = uacc + m2.y;
      uacc = uacc + d0.jp;
      uacc = uacc + d1.jp;
    }
    if (t.tile && kd >= t.k0) {
      s_d[kd & 1][dj][di] = dl.x;
      s_d[kd & 1][dj][di + 1] = dl.y;
      *reinterpret_cast<Pair<T> *>(a.uout + t.base + kd * t.sk) = m2;
    }
    // the next plane: registers move down, the oldest slot takes plane q+AH+1
    const int qn = q + AH + 1;
    doubled(un, qn);
    m3 = m2; m2 = m1; m1 = c; c = p1;
    fm2 = fm1; fm1 = f0;
    if constexpr (FAS) { p1 = p2; p2 = un; f0 = f1; f1 = fn; }
    else { p1 = un; f0 = fn; }
    t.put(buf(AH + 1 - NB), un);
    un = t.load(a.uin, min(qn + 1, t.k1 + 2));
    fn = t.load_src(a.src, min(q + AH + 1, t.k1 + 1));
    slot = slot + 1 == NB ? 0 : slot + 1;
    __syncthreads();
  }
  if (even) {   // the last plane (odd)
    acc = acc + dl.x;
    acc = acc + dl.y;
    acc = acc + so[TP_I * TP_J];
    acc = acc + so[TP_I * TP_J + 1];
    const int64_t id = pass_id<KIND>(a.n1 >> 1, a.n2 >> 1, (t.k1 - 1) >> 1, t.j >> 1, t.i >> 1);
    a.csrc[id] = T(0.125) * acc;
    a.cu[id] = KIND == BC_PER ? T(0.0) : T(0.125) * uacc;
  }
}

template <typename T, int KIND>
__global__ void __launch_bounds__((PassColumn<KIND, 1, 2, T>::NT))
k_mg_up(const int *__restrict__ gate, PassArgs<T> a) {
  const int closed = gate ? *gate : 0;   // a closed gate: the recorded V-cycle loop has ended
  using Col = PassColumn<KIND, 1, 2, T>;
  constexpr int NB = 4, CI = TP_I / 2 + 4, CJ = TP_J / 2 + 4;   // coarse tile and two cells
  static_assert(CI * CJ <= Col::NT, "one coarse cell per thread");
  __shared__ T s_u[NB][Col::PL];
  __shared__ T s_c[4][CJ * CI];   // u - uold (framed) or u of coarse planes, slot = plane & 3
  const Col t(a);
  const int c1 = a.n1 >> 1, c2 = a.n2 >> 1, c3 = a.n3 >> 1;
  const int qa = t.k0 - 1, qe = t.k1;   // red planes
  int slot = 0;
  auto buf = [&](int d) -> T * {
    int z = slot + d;
    z = z < 0 ? z + NB : (z >= NB ? z - NB : z);
    return s_u[z];
  };
  // the coarse cell this thread carries into LDS
  const int cr = (int)threadIdx.x / CI, cj = (t.j0 >> 1) - 2 + cr, ci = (t.i0 >> 1) - 2 + (int)threadIdx.x - cr * CI;
  const bool cuse = cr < CJ && 2 * cr < t.nj + 8 && 2 * ((int)threadIdx.x - cr * CI) < t.ni + 8;
  auto cload = [&](int k, T &v, T &o) {
    v = o = T(0.0);
    if (!cuse) return;
    k = min(k, (t.k1 >> 1) + 1);   // the last that is read
    if constexpr (KIND == BC_PER) {
      v = a.cc[LIX(c1, c2, wrap(k, c3), wrap(cj, c2), wrap(ci, c1))];
    } else if (k >= -1 && k <= c3 && cj >= -1 && cj <= c2 && ci >= -1 && ci <= c1) {
      const unsigned id = BX(c1, c2, k + 1, cj + 1, ci + 1);
      v = a.cc[id];
      o = a.ccold[id];
    }
  };
  auto cput = [&](int k, const T &v, const T &o) {
    if (cr < CJ) s_c[k & 3][threadIdx.x] = KIND == BC_PER ? v : v - o;
  };
  // plane f of the corrected u; the low child of a coarse cell leans on the cell below, the high on
  // the one above (region parity is cell parity)
  const int cq = ((t.row >> 1) + 1) * CI + t.p + 1, cjo = (t.row & 1) ? CI : -CI;
  auto correct = [&](Pair<T> &v, int f) {
    if (!t.in || !t.plane_in(f)) return;
    const T *k0 = s_c[(f >> 1) & 3] + cq, *kn = s_c[((f >> 1) + ((f & 1) ? 1 : -1)) & 3] + cq;
    const T C0 = k0[0], Cj = k0[cjo], Ck = kn[0], Cjk = kn[cjo];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int d = h ? 1 : -1;
      const T Ci = k0[d], Cij = k0[cjo + d], Cik = kn[d], Cijk = kn[cjo + d];
      (h ? v.y : v.x) += T(0.015625) * (T(27.0) * C0 + Cijk + T(9.0) * (Ci + Cj + Ck) + T(3.0) * (Cjk + Cik + Cij));
    }
  };
  auto doubled = [&](Pair<T> &v, int q) {
    if constexpr (KIND == BC_MP) { v.x *= t.scale(q); v.y *= t.scale(q); }
  };
  // the first red plane qa = k0 - 1 is odd: fine planes qa-1 .. qa+1 lean on coarse planes
  // k0/2 - 2 .. k0/2, and later even planes f bring coarse plane f/2 + 1
  const int kc0 = (t.k0 >> 1) - 2;
  T cv[4], co[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) cload(kc0 + e, cv[e], co[e]);
  Pair<T> m1 = t.load(a.uin, qa - 1), c = t.load(a.uin, qa), p1 = t.load(a.uin, qa + 1), m2 = {}, fm1 = {};
  Pair<T> f0 = t.load_src(a.src, qa), un = t.load(a.uin, qa + 2), fn = t.load_src(a.src, qa + 1);
  if (closed) return;
#pragma unroll
  for (int e = 0; e < 4; ++e) cput(kc0 + e, cv[e], co[e]);
  __syncthreads();
  doubled(m1, qa - 1); correct(m1, qa - 1);
  doubled(c, qa); correct(c, qa);
  doubled(p1, qa + 1); correct(p1, qa + 1);
  t.put(buf(-1), m1);
  t.put(buf(0), c);
  t.put(buf(1), p1);
  T nv, no;   // the coarse plane after the newest
  cload(kc0 + 4, nv, no);
  __syncthreads();
  for (int q = qa; q <= qe; ++q) {
    // the plane that enters next, q+2, leans on coarse planes up to (q+3)/2, in LDS since the
    // last barrier
    const int f = q + 2, odd = t.odd_of(q, a.c0);
    const typename Col::Near nr = t.near(buf(0), odd), nb = t.near(buf(-1), odd);
    doubled(un, f);
    if (q < qe) correct(un, f);
    t.smooth(buf(0), nr, c, p1, m1, f0, q, odd);
    const int kb = q - 1;
    if (kb >= t.k0) {
      t.smooth(buf(-1), nb, m1, c, m2, fm1, kb, odd);
      if (t.tile) {
        *reinterpret_cast<Pair<T> *>(a.uout + t.base + kb * t.sk) = m1;
        if constexpr (KIND != BC_PER) {
          push_frame<KIND>(a.uout, a.bcv, a.n1, a.n2, a.n3, kb, t.j, t.i, m1.x);
          push_frame<KIND>(a.uout, a.bcv, a.n1, a.n2, a.n3, kb, t.j, t.i + 1, m1.y);
        }
      }
    }
    if (q == qe) break;
    t.put(buf(2), un);
    if ((f & 1) == 0) {   // the odd planes from f+1 on lean on coarse plane f/2 + 1
      cput((f >> 1) + 1, nv, no);
      cload((f >> 1) + 2, nv, no);
    }
    m2 = m1; m1 = c; c = p1; p1 = un;
    fm1 = f0; f0 = fn;
    un = t.load(a.uin, min(f + 1, t.k1 + 1));
    fn = t.load_src(a.src, min(q + 2, t.k1));
    slot = slot + 1 == NB ? 0 : slot + 1;
    __syncthreads();
  }
}

// FMGProlongate (multigrid.cpp:838-1048) from the framed coarse level
__global__ void __launch_bounds__(BS)
k_mb_fmg_prolong(const double *__restrict__ cu, double *__restrict__ fu, int n1, int n2, int n3) {
  const unsigned t = xcd_slot(blockIdx.x, gridDim.x) * BS + threadIdx.x;
  if (t >= (unsigned)n1 * n2 * n3) return;
  const int fi = 1 + t % n1, r = t / n1, fj = 1 + r % n2, fk = 1 + r / n2;
  const int c1 = n1 >> 1, c2 = n2 >> 1;
  const int i = (fi - 1) / 2 + 1, j = (fj - 1) / 2 + 1, k = (fk - 1) / 2 + 1;
  const double wlo[3] = {5.0, 30.0, -3.0}, whi[3] = {-3.0, 30.0, 5.0};
  const double *wk = ((fk - 1) & 1) ? whi : wlo;
  const double *wj = ((fj - 1) & 1) ? whi : wlo;
  const double *wi = ((fi - 1) & 1) ? whi : wlo;
  double acc = 0.0;
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b)
#pragma unroll
      for (int e = 0; e < 3; ++e) {
        const double term = (wk[a] * wj[b] * wi[e]) * cu[BX(c1, c2, k - 1 + a, j - 1 + b, i - 1 + e)];
        acc = (a == 0 && b == 0 && e == 0) ? term : acc + term;
      }
  fu[BX(n1, n2, fk, fj, fi)] = acc / 32768.0;
}

// RestrictFMGSource for a framed level (source only)
__global__ void __launch_bounds__(BS)
k_mb_restrict_src(const double *__restrict__ src, double *__restrict__ csrc, int n1, int n2, int n3) {
  const int c1 = n1 >> 1, c2 = n2 >> 1, c3 = n3 >> 1;
  const unsigned t = xcd_slot(blockIdx.x, gridDim.x) * BS + threadIdx.x;
  if (t >= (unsigned)c1 * c2 * c3) return;
  const int i = 1 + t % c1, r = t / c1, j = 1 + r % c2, k = 1 + r / c2;
  const int fi = 2 * i - 1, fj = 2 * j - 1, fk = 2 * k - 1;
#define S(kk, jj, ii) src[BX(n1, n2, kk, jj, ii)]
  csrc[BX(c1, c2, k, j, i)] = 0.125 * (S(fk, fj, fi) + S(fk, fj, fi + 1) + S(fk, fj + 1, fi) + S(fk, fj + 1, fi + 1) +
                                       S(fk + 1, fj, fi) + S(fk + 1, fj, fi + 1) + S(fk + 1, fj + 1, fi) +
                                       S(fk + 1, fj + 1, fi + 1));
#undef S
}

// squared defect of the framed finest level, partial sums per workgroup
__global__ void __launch_bounds__(BS)
k_mb_defect_partial(const int *__restrict__ gate,
                    const double *__restrict__ u, const double *__restrict__ src, int n1, int n2, int n3,
                    double idx2, double *__restrict__ part) {
  if (gate && *gate) return;   // a closed gate: the recorded V-cycle loop has ended
  __shared__ double sh[BS];
  unsigned t0, t1;
  wg_range((unsigned)n1 * n2 * n3, t0, t1);
  const unsigned sj = n1 + 2, sk = (unsigned)(n1 + 2) * (n2 + 2);
  double v = 0.0;
  for (unsigned t = t0 + threadIdx.x; t < t1; t += BS) {
    const int i = 1 + t % n1, r = t / n1, j = 1 + r % n2, k = 1 + r / n2;
    const double d = mb_defect(u, src, BX(n1, n2, k, j, i), sj, sk, idx2);
    v += d * d;
  }
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int s = BS / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

// Multipole moments of the finest source (Multigrid::CalculateMultipoleCoefficients,
// multigrid.cpp:1054-1264) or, with com, the centre-of-mass sums
// (Multigrid::CalculateCenterOfMass, multigrid.cpp:1270-1298); per-workgroup partials
// part[q * gridDim.x + w] for moment q.
constexpr int NMOM = 25;
__global__ void __launch_bounds__(BS)
k_mb_moments(const double *__restrict__ src, MPGeom G, const double *__restrict__ mp, int order, int com,
             double *__restrict__ part) {
  __shared__ double sh[BS];
  const int n1 = G.n1, n2 = G.n2, n3 = G.n3;
  unsigned t0, t1;
  wg_range((unsigned)n1 * n2 * n3, t0, t1);
  const double vol = (mp_face(G, 0, 2) - mp_face(G, 0, 1)) * (mp_face(G, 1, 2) - mp_face(G, 1, 1)) *
                     (mp_face(G, 2, 2) - mp_face(G, 2, 1));
  const double xo = com ? 0.0 : mp[0], yo = com ? 0.0 : mp[1], zo = com ? 0.0 : mp[2];
  const int nm = com ? 4 : (order == 4 ? 25 : 9);
  double m[NMOM];
#pragma unroll
  for (int q = 0; q < NMOM; ++q) m[q] = 0.0;
  for (unsigned t = t0 + threadIdx.x; t < t1; t += BS) {
    const int i = 1 + t % n1, r = t / n1, j = 1 + r % n2, k = 1 + r / n2;
    const double z = mp_centre(G, 2, k) - zo, y = mp_centre(G, 1, j) - yo, x = mp_centre(G, 0, i) - xo;
    const double s = src[BX(n1, n2, k, j, i)] * vol;
    m[0] += s;
    m[1] += s * y;
    m[2] += s * z;
    m[3] += s * x;
    if (com) continue;
    const double z2 = z * z, y2 = y * y, yz = y * z, x2 = x * x, xy = x * y, zx = z * x;
    const double r2 = x2 + y2 + z2;
    m[4] += s * xy;
    m[5] += s * yz;
    m[6] += s * (3.0 * z2 - r2);
    m[7] += s * zx;
    if (order == 2) {
      m[8] += s * 0.5 * (x2 - y2);
      continue;
    }
    const double hx2my2 = 0.5 * (x2 - y2), x2mty2 = x2 - 3.0 * y2, tx2my2 = 3.0 * x2 - y2;
    const double fz2mr2 = 5.0 * z2 - r2, sz2mr2 = 7.0 * z2 - r2, sz2mtr2 = 7.0 * z2 - 3.0 * r2;
    m[8] += s * hx2my2;
    m[9] += s * y * tx2my2;
    m[10] += s * xy * z;
    m[11] += s * y * fz2mr2;
    m[12] += s * z * (z2 - 3.0 * r2);
    m[13] += s * x * fz2mr2;
    m[14] += s * z * hx2my2;
    m[15] += s * x * x2mty2;
    m[16] += s * xy * hx2my2;
    m[17] += s * yz * tx2my2;
    m[18] += s * xy * sz2mr2;
    m[19] += s * yz * sz2mtr2;
    m[20] += s * (35.0 * z2 * z2 - 30.0 * z2 * r2 + 3.0 * r2 * r2);
    m[21] += s * zx * sz2mtr2;
    m[22] += s * hx2my2 * sz2mr2;
    m[23] += s * zx * x2mty2;
    m[24] += s * 0.125 * (x2 * x2mty2 - y2 * tx2my2);
  }
  for (int q = 0; q < nm; ++q) {
    sh[threadIdx.x] = m[q];
    __syncthreads();
    for (int st = BS / 2; st > 0; st >>= 1) {
      if (threadIdx.x < st) sh[threadIdx.x] += sh[threadIdx.x + st];
      __syncthreads();
    }
    if (threadIdx.x == 0) part[(unsigned)q * gridDim.x + blockIdx.x] = sh[0];
    __syncthreads();
  }
}

// Sums the partials in a fixed order; com: origin = (m3, m1, m2) / m0
// (MultigridDriver::CalculateCenterOfMass, multigrid_driver.cpp:1984-2015); otherwise
// the coefficients scaled as ScaleMultipoleCoefficients (multigrid_driver.cpp:1930-1981).
__global__ void __launch_bounds__(BS)
k_mb_moments_final(const double *__restrict__ part, int nwg, int order, int com, int nodipole,
                   double *__restrict__ mp) {
  __shared__ double sh[BS];
  const int nm = com ? 4 : (order == 4 ? 25 : 9);
  double acc[NMOM];
  for (int q = 0; q < nm; ++q) {
    double v = 0.0;
    for (int w = threadIdx.x; w < nwg; w += BS) v += part[q * nwg + w];
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int st = BS / 2; st > 0; st >>= 1) {
      if (threadIdx.x < st) sh[threadIdx.x] += sh[threadIdx.x + st];
      __syncthreads();
    }
    acc[q] = sh[0];
    __syncthreads();
  }
  if (threadIdx.x != 0) return;
  if (com) {
    const double im = 1.0 / acc[0];
    mp[0] = im * acc[3];
    mp[1] = im * acc[1];
    mp[2] = im * acc[2];
    return;
  }
  const double PI_ = 3.14159265358979323846;
  const double c0 = -0.25 / PI_, c1 = -0.25 / PI_, c2 = -0.0625 / PI_, c2a = -0.75 / PI_;
  const double c30 = -0.0625 / PI_, c31 = -0.0625 * 1.5 / PI_, c32 = -0.25 * 15.0 / PI_, c33 = -0.0625 * 2.5 / PI_;
  const double c40 = -0.0625 * 0.0625 / PI_, c41 = -0.0625 * 2.5 / PI_, c42 = -0.0625 * 5.0 / PI_,
               c43 = -0.0625 * 17.5 / PI_, c44 = -0.25 * 35.0 / PI_;
  const double sc[NMOM] = {c0, c1, c1, c1, c2a, c2a, c2, c2a, c2a, c33, c32, c31, c30,
                           c31, c32, c33, c44, c43, c42, c41, c40, c41, c42, c43, c44};
  if (nodipole) acc[1] = acc[2] = acc[3] = 0.0;   // nodipole: those sums are never formed
  for (int q = 0; q < NMOM; ++q) mp[3 + q] = (q < nm) ? acc[q] * sc[q] : 0.0;
}

// LoadSource (multigrid.cpp:194-231) into the framed finest level; MGI mode also loads
// u = phi (LoadFinestData, multigrid.cpp:160-180)
__global__ void __launch_bounds__(BS)
k_mb_load(Geo g, const double *__restrict__ u, const double *__restrict__ phi, double *__restrict__ src,
          double *__restrict__ mu, double fac, int load_phi, SrcMask mk) {
  const int N1 = g.nb1 * g.bx1, N2 = g.nb2 * g.bx2, N3 = g.nb3 * g.bx3;
  const unsigned t = xcd_slot(blockIdx.x, gridDim.x) * BS + threadIdx.x;
  if (t >= (unsigned)N1 * N2 * N3) return;
  const int I = t % N1, r = t / N1, J = r % N2, K = r / N2;
  const int b = ((K / g.bx3) * g.nb2 + (J / g.bx2)) * g.nb1 + (I / g.bx1);
  const int64_t id = IDX(g, K % g.bx3 + g.ng, J % g.bx2 + g.ng, I % g.bx1 + g.ng);
  const double v = u[(int64_t)b * NHYDRO * g.S + id];
  const unsigned f = BX(N1, N2, K + 1, J + 1, I + 1);
  src[f] = masked_out(mk, I, J, K) ? 0.0 : ((fac == 1.0) ? v : v * fac);
  if (load_phi) mu[f] = phi[(int64_t)b * g.S + id];
}

// RetrieveResult with one ghost layer (multigrid.cpp:269-288) from the framed finest level
__global__ void __launch_bounds__(BS)
k_mb_retrieve(Geo g, const double *__restrict__ mu, double *__restrict__ phi) {
  const int m1 = g.bx1 + 2, m2 = g.bx2 + 2, m3 = g.bx3 + 2;
  const unsigned t = xcd_slot(blockIdx.x, gridDim.x) * BS + threadIdx.x;
  if (t >= (unsigned)m1 * m2 * m3 * g.nb) return;
  const int li = t % m1;
  unsigned r = t / m1;
  const int lj = r % m2;
  r /= m2;
  const int lk = r % m3, b = r / m3;
  const int N1 = g.nb1 * g.bx1, N2 = g.nb2 * g.bx2;
  const int lx1 = b % g.nb1, lx2 = (b / g.nb1) % g.nb2, lx3 = b / (g.nb1 * g.nb2);
  const int I = lx1 * g.bx1 + li, J = lx2 * g.bx2 + lj, K = lx3 * g.bx3 + lk;   // framed: global + 1
  phi[(int64_t)b * g.S + IDX(g, lk - 1 + g.ng, lj - 1 + g.ng, li - 1 + g.ng)] = mu[BX(N1, N2, K, J, I)];
}

}  // namespace

namespace agx {

template <typename T>
static int64_t lcells(const MGLevelT<T> &L) { return (int64_t)L.n1 * L.n2 * L.n3; }
static int64_t pad32(int64_t n) { return (n + 63) / 64 * 64; }   // 64 elements: >= 256 B
static int64_t npart(int64_t n) { return std::min<int64_t>(grid1d(n, BS), NPART); }

static double finish_norm(agx_mesh *m);
static int iterate(agx_mesh *m, int stage, int &iters, double &def);
static void first_defect_sum(agx_mesh *m);
static void loop_step(agx_mesh *m);
static double mesh_volume(const agx_mesh_desc &d);
static double norm_dv(const agx_mesh *m) { return m->rdx_blk * m->rdy_blk * m->rdz_blk; }

// the nb partials in red summed into scal[slot]; slot 0 is the defect norm, which ends a gated
// pass and is checked there (k_mg_final_check)
static void final_sum(agx_mesh *m, int64_t nb, int slot) {
  if (m->gate && slot == 0)
    hipLaunchKernelGGL(k_mg_final_check, dim3(1), dim3(BS), 0, m->stream, m->red, nb, m->scal, m->gatedev, norm_dv(m),
                       mesh_volume(m->d), m->mg_eps);
  else
    hipLaunchKernelGGL(k_mg_final, dim3(1), dim3(BS), 0, m->stream, m->gate, m->red, nb, m->scal + slot);
}

// ---------------------------------------------------------------- multipole hierarchy
static int64_t bcells(const MGLevelB &L) { return (int64_t)(L.n1 + 2) * (L.n2 + 2) * (L.n3 + 2); }
static int64_t bghosts(const MGLevelB &L) { return bcells(L) - (int64_t)L.n1 * L.n2 * L.n3; }

// Framed levels with the same dimensions and smoother cell sizes as the periodic ones.
static int mp_create(agx_mesh *m) {
  const int L = m->ntotal;
  m->levb.resize(L);
  int64_t tot = 0;
  for (int l = 0; l < L; ++l) {
    MGLevelB &B = m->levb[l];
    B.n1 = m->lev[l].n1; B.n2 = m->lev[l].n2; B.n3 = m->lev[l].n3;
    B.dx = m->lev[l].dx;
    B.h[0] = (m->d.x1max - m->d.x1min) / B.n1;
    B.h[1] = (m->d.x2max - m->d.x2min) / B.n2;
    B.h[2] = (m->d.x3max - m->d.x3min) / B.n3;
    tot += (l < L - 1 ? 5 : 4) * pad32(bcells(B)) + pad32(3 * bghosts(B));
  }
  AGX_HIP(hipMalloc(&m->mgpoolb, tot * (int64_t)sizeof(double)));
  AGX_HIP(hipMemsetAsync(m->mgpoolb, 0, tot * sizeof(double), m->stream));
  m->mg_bytes += tot * (int64_t)sizeof(double);
  double *p = m->mgpoolb;
  for (int l = 0; l < L; ++l) {
    MGLevelB &B = m->levb[l];
    const int64_t n = pad32(bcells(B));
    B.u = p; p += n;
    B.src = p; p += n;
    B.uold = p; p += n;
    B.tmp = p; p += n;
    if (l < L - 1) { B.rhs = p; p += n; }
    B.bcv = p; p += pad32(3 * bghosts(B));
  }
  AGX_HIP(hipMalloc(&m->mpdev, sizeof(double) * (28 + NMOM * NPART)));
  AGX_HIP(hipMemsetAsync(m->mpdev, 0, sizeof(double) * (28 + NMOM * NPART), m->stream));
  m->mp_on = true;
  return 0;
}

static SrcMask src_mask(const agx_mesh *m) {
  SrcMask k;
  k.on = m->srcmask;
  const Geo &g = m->g;
  k.n[0] = g.nb1 * g.bx1; k.n[1] = g.nb2 * g.bx2; k.n[2] = g.nb3 * g.bx3;
  k.xmin[0] = m->d.x1min; k.xmin[1] = m->d.x2min; k.xmin[2] = m->d.x3min;
  k.xmax[0] = m->d.x1max; k.xmax[1] = m->d.x2max; k.xmax[2] = m->d.x3max;
  for (int d = 0; d < 3; ++d) k.c[d] = m->srcmask_c[d];
  k.r2 = m->srcmask_r2;
  return k;
}

static MPGeom mp_geom(const agx_mesh *m, const MGLevelB &B) {
  MPGeom G;
  G.n1 = B.n1; G.n2 = B.n2; G.n3 = B.n3;
  G.xmin[0] = m->d.x1min; G.xmin[1] = m->d.x2min; G.xmin[2] = m->d.x3min;
  G.xmax[0] = m->d.x1max; G.xmax[1] = m->d.x2max; G.xmax[2] = m->d.x3max;
  for (int d = 0; d < 3; ++d) G.h[d] = B.h[d];
  return G;
}

// ProlongateAndCorrect with FAS from the framed coarse level: the paired form where the
// fine rows have even length
template <typename T>
static void mb_prolong(agx_mesh *m, const T *cu, const T *cuold, T *fu, int n1, int n2, int n3) {
  if ((n1 & 1) == 0)
    hipLaunchKernelGGL(k_mb_prolong_pairs<T>, dim3(grid1d((int64_t)(n1 / 2) * n2 * n3, BS)), dim3(BS), 0,
                       m->stream, m->gate, cu, cuold, fu, n1, n2, n3);
  else
    hipLaunchKernelGGL(k_mb_prolong<T>, dim3(grid1d((int64_t)n1 * n2 * n3, BS)), dim3(BS), 0, m->stream,
                       m->gate, cu, cuold, fu, n1, n2, n3);
}

static void bc_b(agx_mesh *m, int l) {
  MGLevelB &B = m->levb[l];
  timer_begin(m, AGX_K_MG_OTHER);
  hipLaunchKernelGGL(k_mb_bc, dim3(grid1d(bghosts(B), BS)), dim3(BS), 0, m->stream, m->gate, B.u, mp_geom(m, B), B.bcv);
  timer_end(m);
}
static void smooth_b(agx_mesh *m, int l, int color) {
  MGLevelB &B = m->levb[l];
  const int64_t n = (int64_t)((B.n1 + 1) / 2) * B.n2 * B.n3;
  timer_begin(m, AGX_K_MG_SMOOTH);
  hipLaunchKernelGGL(k_mb_smooth<double>, dim3(grid1d(n, BS)), dim3(BS), 0, m->stream, m->gate,
                     B.u, B.src, B.n1, B.n2, B.n3,
                     B.dx * B.dx, 1.15 / 6.0, color ^ m->coffset);
  timer_end(m);
}
static void fas_b(agx_mesh *m, int l) {
  MGLevelB &B = m->levb[l];
  timer_begin(m, AGX_K_MG_OTHER);
  hipLaunchKernelGGL(k_mb_fas<double>, dim3(grid1d(bcells(B), BS)), dim3(BS), 0, m->stream, m->gate,
                     B.u, B.src, B.uold, B.n1,
                     B.n2, B.n3, 1.0 / (B.dx * B.dx));
  timer_end(m);
}

// Highest level k_mg_coarse takes: at most COARSE_CELLS interior cells, levels 0 .. top within
// its LDS; -1 if there is none.  N1 .. N3 from the level list, framed or not.
template <typename LV>
static int coarse_lds(const std::vector<LV> &H, int top, bool framed, bool bcv) {   // LDS elements
  int64_t n = 0;
  for (int l = 0; l <= top; ++l) {
    const LV &L = H[l];
    const int64_t c = (int64_t)L.n1 * L.n2 * L.n3, f = (int64_t)(L.n1 + 2) * (L.n2 + 2) * (L.n3 + 2);
    n += framed ? f + c : 2 * c;
    if (framed && l < top) n += f + (bcv ? 3 * (f - c) : 0);
  }
  return (int)std::min<int64_t>(n, INT32_MAX);
}
template <typename LV>
static int coarse_fit(const std::vector<LV> &H, bool framed, bool bcv) {
  int top = -1;
  while (top + 1 < (int)H.size() && top + 1 < MAXC &&
         (int64_t)H[top + 1].n1 * H[top + 1].n2 * H[top + 1].n3 <= COARSE_CELLS &&
         coarse_lds(H, top + 1, framed, bcv) <= COARSE_LDS)
    ++top;
  return top;
}
template <typename T, typename LV>
static CoarseSet<T> coarse_set(const std::vector<LV> &H, int top, bool framed, bool bcv) {
  CoarseSet<T> S = {};
  int o = 0;
  for (int l = 0; l <= top; ++l) {
    const LV &L = H[l];
    CoarseLevel<T> &c = S.lv[l];
    c.u = L.u;
    c.src = L.src;
    c.n1 = L.n1; c.n2 = L.n2; c.n3 = L.n3;
    c.dx2 = T(L.dx * L.dx);
    c.idx2 = T(1.0 / (L.dx * L.dx));
    const int n = L.n1 * L.n2 * L.n3, f = (L.n1 + 2) * (L.n2 + 2) * (L.n3 + 2);
    c.lu = o; o += framed ? f : n;
    c.ls = o; o += n;
    if (framed && l < top) {
      c.lo = o; o += f;
      if (bcv) { c.lb = o; o += 3 * (f - n); }
    }
  }
  return S;
}

static int coarse_top_b(const agx_mesh *m) { return m->mg_coarse ? coarse_fit(m->levb, true, true) : -1; }

static void coarse_b(agx_mesh *m, int top, int ni) {
  CoarseSet<double> c = coarse_set<double>(m->levb, top, true, true);
  for (int l = 0; l <= top; ++l) {
    c.lv[l].old = m->levb[l].uold;
    c.lv[l].bcv = m->levb[l].bcv;
  }
  timer_begin(m, AGX_K_MG_OTHER);
  hipLaunchKernelGGL((k_mg_coarse<double, BC_MP>), dim3(1), dim3(COARSE_BS), 0, m->stream, m->gate, c, top,
                     m->fmglevel, m->coffset, ni, 1.15 / 6.0, 0);
  timer_end(m);
}

// the same for the FP32 correction cycle (homogeneous boundary chain)
static void coarse_b32(agx_mesh *m, int top, int ni) {
  CoarseSet<float> c = coarse_set<float>(m->levb32, top, true, false);
  for (int l = 0; l <= top; ++l) c.lv[l].old = m->levb32[l].uold;
  timer_begin(m, AGX_K_MG_OTHER);
  hipLaunchKernelGGL((k_mg_coarse<float, BC_HOM>), dim3(1), dim3(COARSE_BS), 0, m->stream, m->gate, c, top,
                     m->fmglevel, m->coffset, ni, float(1.15 / 6.0), 0);
  timer_end(m);
}

// Levels that run as whole passes (k_mg_down, k_mg_up): those above the coarse kernel's.  Every
// extent above level 0 is even; a ring of four cells needs four to wrap once.
template <typename LV>
static bool pass_level(const LV &L) {
  return std::min(L.n1, std::min(L.n2, L.n3)) >= 4;
}
// Planes per workgroup: a chunk runs about six iterations more than it has planes, so the
// chunks are as long as 512 resident workgroups (two a CU) leave them.
template <typename LV>
static int pass_planes(const LV &L) {
  const int64_t tiles = (int64_t)((L.n1 + TP_I - 1) / TP_I) * ((L.n2 + TP_J - 1) / TP_J);
  int best = 2;
  int64_t least = INT64_MAX;
  for (int kc = 2; kc <= L.n3; kc += 2) {
    const int64_t t = (kc + 6) * ((tiles * ((L.n3 + kc - 1) / kc) + 511) / 512);
    if (t < least) { least = t; best = kc; }
  }
  return best;
}
template <typename T, typename LV>
static PassArgs<T> pass_args(const agx_mesh *m, const LV &L) {
  PassArgs<T> a = {};
  a.n1 = L.n1; a.n2 = L.n2; a.n3 = L.n3;
  a.kc = pass_planes(L);
  a.dx2 = T(L.dx * L.dx);
  a.idx2 = T(1.0 / (L.dx * L.dx));
  a.isix = T(1.15 / 6.0);
  a.c0 = m->coffset;
  a.src = L.src;
  return a;
}
template <typename T>
static dim3 pass_grid(const PassArgs<T> &a) {
  return dim3((unsigned)((a.n1 + TP_I - 1) / TP_I) * ((a.n2 + TP_J - 1) / TP_J) * ((a.n3 + a.kc - 1) / a.kc));
}
// framed level F of the multipole hierarchies (KIND BC_MP with FP64, BC_HOM with FP32);
// bcv is null for BC_HOM
template <typename T, int KIND, typename LV>
static void down_b(agx_mesh *m, LV &F, LV &C, const double *bcv, bool fas) {
  constexpr int NT = PassColumn<KIND, 2, 3, T>::NT;
  PassArgs<T> a = pass_args<T>(m, F);
  a.uin = F.u; a.uout = F.tmp;
  a.rhs = F.rhs; a.old = F.uold;
  a.csrc = C.src; a.cu = C.u;
  a.bcv = bcv;
  timer_begin(m, AGX_K_MG_SMOOTH);
  if (fas) hipLaunchKernelGGL((k_mg_down<T, KIND, true>), pass_grid(a), dim3(NT), 0, m->stream, m->gate, a);
  else hipLaunchKernelGGL((k_mg_down<T, KIND, false>), pass_grid(a), dim3(NT), 0, m->stream, m->gate, a);
  timer_end(m);
}
template <typename T, int KIND, typename LV>
static void up_b(agx_mesh *m, LV &F, LV &C, const double *bcv, bool fas) {
  PassArgs<T> a = pass_args<T>(m, F);
  a.uin = F.tmp; a.uout = F.u;
  if (fas) a.src = F.rhs;
  a.cc = C.u; a.ccold = C.uold;
  a.bcv = bcv;
  timer_begin(m, AGX_K_MG_SMOOTH);
  hipLaunchKernelGGL((k_mg_up<T, KIND>), pass_grid(a), dim3(PassColumn<KIND, 1, 2, T>::NT), 0, m->stream, m->gate, a);
  timer_end(m);
}

// SolveVCycle(1,1) (multigrid_driver.cpp:684-693) with the FAS steps of
// OneStepToCoarser / SolveCoarsestGrid / OneStepToFiner (:583-677, :778-819) and the
// MeshBlock task lists (mg_task_list.cpp:258-262, 287-510).  Boundaries are filled before
// every stencil step, as the reference's exchanges and ApplyPhysicalBoundaries are.
static void vcycle_b(agx_mesh *m) {
  int start = m->current;
  m->coffset ^= 1;
  const Geo &g0 = m->g;
  const int ct = coarse_top_b(m);
  if (ct >= 0) {
    // the levels above the coarse kernel's range as whole passes, or per step where they are flat; from level
    // min(start, ct) down to 0 and back, one launch
    while (m->current > ct) {
      const int l = m->current;
      MGLevelB &F = m->levb[l], &C = m->levb[l - 1];
      if (m->mg_coarse && pass_level(F)) {
        down_b<double, BC_MP>(m, F, C, F.bcv, l < m->fmglevel);
        m->current--;
        continue;
      }
      bc_b(m, l);
      if (l < m->fmglevel) fas_b(m, l);
      smooth_b(m, l, 0);
      bc_b(m, l);
      smooth_b(m, l, 1);
      bc_b(m, l);
      timer_begin(m, AGX_K_MG_RESTRICT);
      hipLaunchKernelGGL(k_mb_restrict<double>, dim3(grid1d((int64_t)C.n1 * C.n2 * C.n3, BS)), dim3(BS), 0, m->stream,
                         m->gate, F.u, F.src, C.src, C.u, F.n1, F.n2, F.n3, 1.0 / (F.dx * F.dx));
      timer_end(m);
      m->current--;
    }
    const int ni0 = std::max(g0.nb1, std::max(g0.nb2, g0.nb3)) >> (m->nrootlevel - 1);
    coarse_b(m, m->current, ni0);
    while (m->current < start) {
      const int l = m->current + 1;
      MGLevelB &F = m->levb[l], &C = m->levb[l - 1];
      if (m->mg_coarse && pass_level(F)) {   // the coarse frame is filled: by k_mg_coarse or by k_mg_up
        up_b<double, BC_MP>(m, F, C, F.bcv, l < m->fmglevel);
        m->current++;
        continue;
      }
      bc_b(m, l - 1);
      timer_begin(m, AGX_K_MG_PROLONG);
      mb_prolong(m, C.u, C.uold, F.u, F.n1, F.n2, F.n3);
      timer_end(m);
      bc_b(m, l);
      smooth_b(m, l, 0);
      bc_b(m, l);
      smooth_b(m, l, 1);
      bc_b(m, l);
      m->current++;
    }
    return;
  }
  while (m->current > 0) {
    const int l = m->current;
    MGLevelB &F = m->levb[l], &C = m->levb[l - 1];
    bc_b(m, l);
    if (l < m->fmglevel) fas_b(m, l);
    smooth_b(m, l, 0);
    bc_b(m, l);
    smooth_b(m, l, 1);
    bc_b(m, l);
    timer_begin(m, AGX_K_MG_RESTRICT);
    hipLaunchKernelGGL(k_mb_restrict<double>, dim3(grid1d((int64_t)C.n1 * C.n2 * C.n3, BS)), dim3(BS), 0, m->stream,
                       m->gate, F.u, F.src, C.src, C.u, F.n1, F.n2, F.n3, 1.0 / (F.dx * F.dx));
    timer_end(m);
    m->current--;
  }
  // SolveCoarsestGrid with FAS (no average subtraction): ni sweeps on the root level
  const Geo &g = m->g;
  int ni = std::max(g.nb1, std::max(g.nb2, g.nb3)) >> (m->nrootlevel - 1);
  bc_b(m, 0);
  fas_b(m, 0);
  for (int it = 0; it < ni; ++it) {
    smooth_b(m, 0, 0);
    bc_b(m, 0);
    smooth_b(m, 0, 1);
    bc_b(m, 0);
  }
  while (m->current < start) {
    const int l = m->current + 1;
    MGLevelB &F = m->levb[l], &C = m->levb[l - 1];
    bc_b(m, l - 1);
    timer_begin(m, AGX_K_MG_PROLONG);
    mb_prolong(m, C.u, C.uold, F.u, F.n1, F.n2, F.n3);
    timer_end(m);
    bc_b(m, l);
    smooth_b(m, l, 0);
    bc_b(m, l);
    smooth_b(m, l, 1);
    bc_b(m, l);
    m->current++;
  }
}

// SolveFMGCycle (multigrid_driver.cpp:700-714) after RestrictFMGSource
static void fmg_b(agx_mesh *m) {
  const int L = m->ntotal;
  for (int l = L - 1; l > 0; --l) {
    MGLevelB &F = m->levb[l], &C = m->levb[l - 1];
    hipLaunchKernelGGL(k_mb_restrict_src, dim3(grid1d((int64_t)C.n1 * C.n2 * C.n3, BS)), dim3(BS), 0, m->stream,
                       F.src, C.src, F.n1, F.n2, F.n3);
  }
  m->current = 0;
  for (m->fmglevel = 0; m->fmglevel < L; m->fmglevel++) {
    vcycle_b(m);
    if (m->fmglevel != L - 1) {   // FMGProlongate, multigrid_driver.cpp:553-575
      const int l = m->current + 1;
      MGLevelB &F = m->levb[l], &C = m->levb[l - 1];
      bc_b(m, l - 1);
      timer_begin(m, AGX_K_MG_PROLONG);
      hipLaunchKernelGGL(k_mb_fmg_prolong, dim3(grid1d((int64_t)F.n1 * F.n2 * F.n3, BS)), dim3(BS), 0, m->stream,
                         C.u, F.u, F.n1, F.n2, F.n3);
      timer_end(m);
      m->current++;
    }
  }
  m->fmglevel = L - 1;
}

// ---- mixed precision with multipole boundaries: FP32 V(1,1) cycles with FAS on the
// correction (ghosts by the homogeneous chain), inside the FP64 defect correction
static void bc_b32(agx_mesh *m, int l) {
  timer_begin(m, AGX_K_MG_OTHER);
  hipLaunchKernelGGL(k_mb_bc_hom, dim3(grid1d(bghosts(m->levb[l]), BS)), dim3(BS), 0, m->stream, m->gate,
                     m->levb32[l].u,
                     mp_geom(m, m->levb[l]));
  timer_end(m);
}
static void smooth_b32(agx_mesh *m, int l, int color) {
  MGLevelB32 &B = m->levb32[l];
  const int64_t n = (int64_t)((B.n1 + 1) / 2) * B.n2 * B.n3;
  timer_begin(m, AGX_K_MG_SMOOTH);
  hipLaunchKernelGGL(k_mb_smooth<float>, dim3(grid1d(n, BS)), dim3(BS), 0, m->stream, m->gate, B.u, B.src, B.n1, B.n2,
                     B.n3, float(B.dx * B.dx), float(1.15 / 6.0), color ^ m->coffset);
  timer_end(m);
}
static void fas_b32(agx_mesh *m, int l) {
  MGLevelB32 &B = m->levb32[l];
  timer_begin(m, AGX_K_MG_OTHER);
  hipLaunchKernelGGL(k_mb_fas<float>, dim3(grid1d(bcells(m->levb[l]), BS)), dim3(BS), 0, m->stream, m->gate, B.u, B.src,
                     B.uold, B.n1, B.n2, B.n3, float(1.0 / (B.dx * B.dx)));
  timer_end(m);
}
static void vcycle_b32(agx_mesh *m) {   // the per-level sequence of vcycle_b
  const int start = m->current;
  m->coffset ^= 1;
  const int ct = coarse_top_b(m);   // levels at or below it in one launch (coarse_b32)
  while (m->current > 0 && m->current > ct) {
    const int l = m->current;
    MGLevelB32 &F = m->levb32[l], &C = m->levb32[l - 1];
    if (m->mg_coarse && pass_level(F)) {
      down_b<float, BC_HOM>(m, F, C, nullptr, l < m->fmglevel);
      m->current--;
      continue;
    }
    bc_b32(m, l);
    if (l < m->fmglevel) fas_b32(m, l);
    smooth_b32(m, l, 0);
    bc_b32(m, l);
    smooth_b32(m, l, 1);
    bc_b32(m, l);
    timer_begin(m, AGX_K_MG_RESTRICT);
    hipLaunchKernelGGL(k_mb_restrict<float>, dim3(grid1d((int64_t)C.n1 * C.n2 * C.n3, BS)), dim3(BS), 0,
                       m->stream, m->gate, F.u, F.src, C.src, C.u, F.n1, F.n2, F.n3, float(1.0 / (F.dx * F.dx)));
    timer_end(m);
    m->current--;
  }
  const Geo &g = m->g;
  const int ni = std::max(g.nb1, std::max(g.nb2, g.nb3)) >> (m->nrootlevel - 1);
  if (ct >= 0) {
    coarse_b32(m, m->current, ni);
  } else {
    bc_b32(m, 0);
    fas_b32(m, 0);
    for (int it = 0; it < ni; ++it) {
      smooth_b32(m, 0, 0);
      bc_b32(m, 0);
      smooth_b32(m, 0, 1);
      bc_b32(m, 0);
    }
  }
  while (m->current < start) {
    const int l = m->current + 1;
    MGLevelB32 &F = m->levb32[l], &C = m->levb32[l - 1];
    if (m->mg_coarse && pass_level(F)) {
      up_b<float, BC_HOM>(m, F, C, nullptr, l < m->fmglevel);
      m->current++;
      continue;
    }
    bc_b32(m, l - 1);
    timer_begin(m, AGX_K_MG_PROLONG);
    mb_prolong(m, C.u, C.uold, F.u, F.n1, F.n2, F.n3);
    timer_end(m);
    bc_b32(m, l);
    smooth_b32(m, l, 0);
    bc_b32(m, l);
    smooth_b32(m, l, 1);
    bc_b32(m, l);
    m->current++;
  }
}

// One defect-correction step: ghosts of phi from the multipole expansion, d = defect in
// FP64, FP32 V(1,1) on the correction from zero, phi += e, ghosts again (the defect norm
// and the next step read them).
static void correction_step_b(agx_mesh *m) {
  const int L = m->ntotal;
  MGLevelB &F = m->levb[L - 1];
  MGLevelB32 &E = m->levb32[L - 1];
  bc_b(m, L - 1);
  timer_begin(m, AGX_K_MG_OTHER);
  hipLaunchKernelGGL(k_mb_defect32, dim3(grid1d(bcells(F), BS)), dim3(BS), 0, m->stream, m->gate, F.u, F.src, E.src,
                     E.u, F.n1, F.n2, F.n3, 1.0 / (F.dx * F.dx));
  timer_end(m);
  const int keep = m->fmglevel;
  m->current = L - 1;
  m->fmglevel = L - 1;
  vcycle_b32(m);
  m->fmglevel = keep;
  timer_begin(m, AGX_K_MG_OTHER);
  hipLaunchKernelGGL(k_mb_add32, dim3(grid1d(bcells(F), BS)), dim3(BS), 0, m->stream, m->gate, F.u, E.u, F.n1, F.n2,
                     F.n3);
  timer_end(m);
  bc_b(m, L - 1);
}

// squared sum of the framed finest level's defect into scal[0] (reads its ghost frame as
// it stands), and the defect norm from it
static void defect_sum_b(agx_mesh *m) {
  MGLevelB &F = m->levb[m->ntotal - 1];
  const int64_t nb = npart((int64_t)F.n1 * F.n2 * F.n3);
  hipLaunchKernelGGL(k_mb_defect_partial, dim3((unsigned)nb), dim3(BS), 0, m->stream, m->gate, F.u, F.src, F.n1,
                     F.n2, F.n3, 1.0 / (F.dx * F.dx), m->red);
  final_sum(m, nb, 0);
}
static double defect_norm_b(agx_mesh *m) {
  defect_sum_b(m);
  return finish_norm(m);
}

// origin of the expansion given in the input (<gravity>/mporigin_x1..x3, mg_gravity.cpp:116-118)
__global__ void k_mb_set_origin(double *mp, double x1, double x2, double x3) {
  if (threadIdx.x) return;
  mp[0] = x1;
  mp[1] = x2;
  mp[2] = x3;
}

// MultipoleCoefficients of the finest source (SetupMultigrid, multigrid_driver.cpp:441-445)
static void mp_coefficients(agx_mesh *m) {
  MGLevelB &F = m->levb[m->ntotal - 1];
  const int64_t nb = npart((int64_t)F.n1 * F.n2 * F.n3);
  const MPGeom G = mp_geom(m, F);
  double *part = m->mpdev + 28;
  if (m->d.mp_auto_origin) {
    hipLaunchKernelGGL(k_mb_moments, dim3((unsigned)nb), dim3(BS), 0, m->stream, F.src, G, m->mpdev,
                       m->d.mporder, 1, part);
    hipLaunchKernelGGL(k_mb_moments_final, dim3(1), dim3(BS), 0, m->stream, part, (int)nb, m->d.mporder, 1, 0,
                       m->mpdev);
  } else {   // the fixed origin is part of the mesh description: written by a kernel, so
             // that a recorded solve holds it
    hipLaunchKernelGGL(k_mb_set_origin, dim3(1), dim3(64), 0, m->stream, m->mpdev, m->d.mp_origin[0],
                       m->d.mp_origin[1], m->d.mp_origin[2]);
  }
  hipLaunchKernelGGL(k_mb_moments, dim3((unsigned)nb), dim3(BS), 0, m->stream, F.src, G, m->mpdev, m->d.mporder,
                     0, part);
  hipLaunchKernelGGL(k_mb_moments_final, dim3(1), dim3(BS), 0, m->stream, part, (int)nb, m->d.mporder, 0,
                     m->d.mp_nodipole ? 1 : 0, m->mpdev);
  // the boundary values of every level for this solve (the ghost fills then only gather)
  for (int l = 0; l < m->ntotal; ++l) {
    MGLevelB &B = m->levb[l];
    hipLaunchKernelGGL(k_mb_bc_fill, dim3(grid1d(bghosts(B), BS)), dim3(BS), 0, m->stream, B.bcv, mp_geom(m, B),
                       m->mpdev, m->d.mporder);
  }
}

// MGGravityDriver::Solve (mg_gravity.cpp:166-211) with multipole boundaries, up to the
// iteration: load, multipole coefficients, FMG
static void solve_load_b(agx_mesh *m) {
  const Geo &g = m->g;
  const int L = m->ntotal;
  MGLevelB &F = m->levb[L - 1];
  double **A = m->arr.a;
  hipLaunchKernelGGL(k_mb_load, dim3(grid1d((int64_t)F.n1 * F.n2 * F.n3, BS)), dim3(BS), 0, m->stream, g,
                     A[AGX_ARR_U], A[AGX_ARR_PHI], F.src, F.u, m->d.four_pi_G, m->mg_mode == 1 ? 1 : 0, src_mask(m));
  m->current = L - 1;
  m->fmglevel = L - 1;
  mp_coefficients(m);
  m->mp_solved = true;
  if (m->mg_mode == 0) fmg_b(m);
  m->current = L - 1;
}

static int retrieve_b(agx_mesh *m) {
  const Geo &g = m->g;
  MGLevelB &F = m->levb[m->ntotal - 1];
  const int64_t nret = (int64_t)(g.bx1 + 2) * (g.bx2 + 2) * (g.bx3 + 2) * g.nb;
  hipLaunchKernelGGL(k_mb_retrieve, dim3(grid1d(nret, BS)), dim3(BS), 0, m->stream, g, F.u, m->arr.a[AGX_ARR_PHI]);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_fail(e, "multipole mg_solve launches");
  return 0;
}

static int mg_solve_b(agx_mesh *m, int stage) {
  solve_load_b(m);
  int iters = 0;
  double def = 0.0;
  if (m->mg_eps >= 0.0) {   // SolveIterative, multigrid_driver.cpp:721-755
    int rc = iterate(m, stage, iters, def);
    if (rc) return rc;
    m->last_norm = def;
    if (stage >= 0 && stage <= 2) m->mg_kpred[stage] = iters;
  } else {   // SolveIterativeFixedTimes, multigrid_driver.cpp:762-771
    for (int n = 0; n < m->mg_niter; ++n) {
      if (m->mixed) correction_step_b(m);
      else vcycle_b(m);
      iters++;
    }
    m->last_norm = m->capturing ? NAN : defect_norm_b(m);   // diagnostic only, see mg_solve
  }
  m->last_iters = iters;
  return retrieve_b(m);
}

int mg_create(agx_mesh *m) {
  const agx_mesh_desc &d = m->d;
  const Geo &g = m->g;
  if (d.bnx1 != d.bnx2 || d.bnx1 != d.bnx3) {
    set_error("multigrid requires logically cubic MeshBlocks (multigrid.cpp:37-43)");
    return -20;
  }
  int nl = 0;
  for (int l = 0; l < 20; ++l)
    if ((1 << l) == d.bnx1) { nl = l + 1; break; }
  if (nl == 0) { set_error("MeshBlock size must be a power of two (multigrid.cpp:92-104)"); return -21; }
  int nrl = 0;
  for (int l = 0; l < 20; ++l)
    if (g.nb1 % (1 << l) == 0 && g.nb2 % (1 << l) == 0 && g.nb3 % (1 << l) == 0) nrl = l + 1;
  m->nmblevel = nl;
  m->nrootlevel = nrl;
  m->ntotal = nrl + nl - 1;
  m->mg_mode = d.mg_mode;
  m->mg_eps = d.mg_threshold;
  m->mg_niter = d.mg_niter;
  // cell sizes: block levels use the MeshBlock's rdx_/rdy_/rdz_, root levels the root
  // grid's (multigrid.cpp:61-63); taken from MeshBlock gid 0, whose upper corner is
  // UniformMeshGenerator(ComputeMeshGeneratorX(1, nb)) (mesh.cpp:1668-1760).
  auto blk0 = [](int nb, double xmin, double xmax) {
    if (nb == 1) return xmax;
    int64_t no = 1 - nb / 2, noc = 1 - (nb + 1) / 2;
    double rx = (double)(no + noc) / (2.0 * nb);
    return 0.5 * (xmin + xmax) + (rx * xmax - rx * xmin);
  };
  m->rdx_blk = (blk0(g.nb1, d.x1min, d.x1max) - d.x1min) / (double)d.bnx1;
  m->rdy_blk = (blk0(g.nb2, d.x2min, d.x2max) - d.x2min) / (double)d.bnx2;
  m->rdz_blk = (blk0(g.nb3, d.x3min, d.x3max) - d.x3min) / (double)d.bnx3;
  m->rdx_root = (d.x1max - d.x1min) / (double)g.nb1;
  m->rdy_root = (d.x2max - d.x2min) / (double)g.nb2;
  m->rdz_root = (d.x3max - d.x3min) / (double)g.nb3;
  int L = m->ntotal;
  m->lev.resize(L);
  int64_t tot = 0;
  for (int l = 0; l < L; ++l) {
    MGLevel &Lv = m->lev[l];
    int sh = L - 1 - l;
    Lv.n1 = d.nx1 >> sh;
    Lv.n2 = d.nx2 >> sh;
    Lv.n3 = d.nx3 >> sh;
    if (l >= nrl) Lv.dx = m->rdx_blk * (double)(1 << sh);
    else Lv.dx = m->rdx_root * (double)(1 << (nrl - 1 - l));
    tot += 3 * pad32(lcells(Lv));
  }
  m->mg_bytes = tot * (int64_t)sizeof(double);
  AGX_HIP(hipMalloc(&m->mgpool, m->mg_bytes));
  AGX_HIP(hipMemsetAsync(m->mgpool, 0, m->mg_bytes, m->stream));
  double *p = m->mgpool;
  for (int l = 0; l < L; ++l) {
    MGLevel &Lv = m->lev[l];
    int64_t n = pad32(lcells(Lv));   // every array 256-B aligned (vector loads of pairs)
    Lv.u = p; p += n;
    Lv.src = p; p += n;
    Lv.def = p; p += n;
  }
  if (m->mixed) {
    // FP32 hierarchy of the correction V-cycles: u (correction) and src per level
    m->lev32.resize(L);
    int64_t t32 = 0;
    for (int l = 0; l < L; ++l) t32 += 3 * pad32(lcells(m->lev[l]));
    AGX_HIP(hipMalloc(&m->mgpool32, t32 * (int64_t)sizeof(float)));
    AGX_HIP(hipMemsetAsync(m->mgpool32, 0, t32 * sizeof(float), m->stream));
    m->mg_bytes += t32 * (int64_t)sizeof(float);
    float *q = m->mgpool32;
    for (int l = 0; l < L; ++l) {
      MGLevel32 &Lv = m->lev32[l];
      Lv.n1 = m->lev[l].n1; Lv.n2 = m->lev[l].n2; Lv.n3 = m->lev[l].n3; Lv.dx = m->lev[l].dx;
      int64_t n = pad32(lcells(Lv));
      Lv.u = q; q += n;
      Lv.src = q; q += n;
      Lv.def = q; q += n;   // spare array (whole passes, the mixed correction)
    }
  }
  int64_t need = (lcells(m->lev[L - 1]) + BS - 1) / BS + 1;
  if (need > m->red_n) {
    if (m->red) AGX_HIP(hipFree(m->red));
    m->red_n = need;
    AGX_HIP(hipMalloc(&m->red, sizeof(double) * m->red_n));
  }
  if (d.mg_bc == 1) {
    int rc = mp_create(m);
    if (rc) return rc;
    if (m->mixed) {   // FP32 framed levels: correction, source, FAS copy
      m->levb32.resize(L);
      int64_t t32 = 0;
      for (int l = 0; l < L; ++l) t32 += (l < L - 1 ? 5 : 4) * pad32(bcells(m->levb[l]));
      AGX_HIP(hipMalloc(&m->mgpoolb32, t32 * (int64_t)sizeof(float)));
      AGX_HIP(hipMemsetAsync(m->mgpoolb32, 0, t32 * sizeof(float), m->stream));
      m->mg_bytes += t32 * (int64_t)sizeof(float);
      float *q = m->mgpoolb32;
      for (int l = 0; l < L; ++l) {
        MGLevelB32 &B = m->levb32[l];
        B.n1 = m->levb[l].n1; B.n2 = m->levb[l].n2; B.n3 = m->levb[l].n3; B.dx = m->levb[l].dx;
        const int64_t n = pad32(bcells(m->levb[l]));
        B.u = q; q += n;
        B.src = q; q += n;
        B.uold = q; q += n;
        B.tmp = q; q += n;
        if (l < L - 1) { B.rhs = q; q += n; }
      }
    }
  }
  if (!m->gatedev) AGX_HIP(hipMalloc(&m->gatedev, sizeof(MGGate)));
  if (!m->gatehost) AGX_HIP(hipHostMalloc(&m->gatehost, sizeof(MGGate)));
  AGX_HIP(hipStreamSynchronize(m->stream));
  m->mg_on = 1;
  return 0;
}

void mg_destroy(agx_mesh *m) {
  if (m->mgpoolb) hipFree(m->mgpoolb);
  if (m->mpdev) hipFree(m->mpdev);
  if (m->mgpoolb32) hipFree(m->mgpoolb32);
  m->mgpoolb = nullptr;
  m->mgpoolb32 = nullptr;
  m->mpdev = nullptr;
  m->levb.clear();
  m->levb32.clear();
  m->mp_on = false;
  if (m->mgpool) hipFree(m->mgpool);
  if (m->mgpool32) hipFree(m->mgpool32);
  m->mgpool = nullptr;
  m->mgpool32 = nullptr;
  m->lev.clear();
  m->lev32.clear();
  if (m->gatedev) hipFree(m->gatedev);
  if (m->gatehost) hipHostFree(m->gatehost);
  m->gatedev = nullptr;
  m->gatehost = nullptr;
  m->mg_on = 0;
}

// ---------------------------------------------------------------- level operations
// Each works on one hierarchy H: the FP64 levels, or the FP32 correction levels of the
// mixed-precision form.
template <typename T>
static void smooth(agx_mesh *m, std::vector<MGLevelT<T>> &H, int l, int color) {
  MGLevelT<T> &L = H[l];
  double dx2 = L.dx * L.dx;
  double isix = 1.15 / 6.0;
  int64_t n = (int64_t)((L.n1 + 1) / 2) * L.n2 * L.n3;
  auto odd = [](int q) { return (q & 1) && q > 1; };
  timer_begin(m, AGX_K_MG_SMOOTH);
  if (odd(L.n1) || odd(L.n2) || odd(L.n3)) {
    hipLaunchKernelGGL(k_mg_smooth_wrap<T>, dim3(grid1d(lcells(L), BS)), dim3(BS), 0, m->stream, m->gate, L.u, L.def,
                       L.src, L.n1, L.n2, L.n3, T(dx2), T(isix), color ^ m->coffset);
    std::swap(L.u, L.def);
  } else if ((L.n1 & 1) == 0)
    hipLaunchKernelGGL(k_mg_smooth_pairs<T>, dim3(grid1d(n, BS)), dim3(BS), 0, m->stream, m->gate, L.u, L.src, L.n1,
                       L.n2, L.n3, T(dx2), T(isix), color ^ m->coffset);
  else
    hipLaunchKernelGGL(k_mg_smooth<T>, dim3(grid1d(n, BS)), dim3(BS), 0, m->stream, m->gate, L.u, L.src, L.n1, L.n2,
                       L.n3, T(dx2), T(isix), color ^ m->coffset);
  timer_end(m);
}

template <typename T>
static void defect_restrict(agx_mesh *m, std::vector<MGLevelT<T>> &H, int l) {
  MGLevelT<T> &F = H[l], &C = H[l - 1];
  double idx2 = 1.0 / (F.dx * F.dx);
  timer_begin(m, AGX_K_MG_RESTRICT);
  hipLaunchKernelGGL(k_mg_defect_restrict<T>, dim3(grid1d(lcells(C), BS)), dim3(BS), 0, m->stream, m->gate, F.u,
                     F.src, C.src, C.u, F.n1, F.n2, F.n3, T(idx2));
  timer_end(m);
}

template <typename T>
static void prolong(agx_mesh *m, std::vector<MGLevelT<T>> &H, int l) {   // l-1 -> l
  MGLevelT<T> &F = H[l], &C = H[l - 1];
  timer_begin(m, AGX_K_MG_PROLONG);
  if ((F.n1 & 1) == 0)   // every level above the root: n1 = 2 * (coarse n1)
    hipLaunchKernelGGL(k_mg_prolong_pairs<T>, dim3(grid1d(lcells(F) / 2, BS)), dim3(BS), 0, m->stream, m->gate,
                       C.u, F.u,
                       F.n1, F.n2, F.n3);
  else
    hipLaunchKernelGGL(k_mg_prolong<T>, dim3(grid1d(lcells(F), BS)), dim3(BS), 0, m->stream, m->gate, C.u, F.u, F.n1,
                       F.n2, F.n3);
  timer_end(m);
}

template <typename T>
static void fmg_prolong(agx_mesh *m, std::vector<MGLevelT<T>> &H, int l) {   // l-1 -> l
  MGLevelT<T> &F = H[l], &C = H[l - 1];
  timer_begin(m, AGX_K_MG_PROLONG);
  hipLaunchKernelGGL(k_mg_fmg_prolong<T>, dim3(grid1d(lcells(F), BS)), dim3(BS), 0, m->stream, C.u, F.u,
                     F.n1, F.n2, F.n3);
  timer_end(m);
}

// device sum of a level array into scal[slot]
template <typename T>
static void array_sum(agx_mesh *m, const MGLevelT<T> &L, const T *a, int slot) {
  const int64_t nb = npart(lcells(L));
  hipLaunchKernelGGL(k_mg_partial<T>, dim3((unsigned)nb), dim3(BS), 0, m->stream, m->gate, a, (unsigned)lcells(L),
                     m->red);
  final_sum(m, nb, slot);
}
template <typename T>
static void level_sum(agx_mesh *m, std::vector<MGLevelT<T>> &H, int l, int slot) {
  timer_begin(m, AGX_K_MG_OTHER);
  array_sum(m, H[l], H[l].u, slot);
  timer_end(m);
}
// the finest FP64 level's squared defect into scal[0]
static void defect_sum(agx_mesh *m) {
  MGLevel &L = m->lev[m->ntotal - 1];
  const int64_t nb = npart(lcells(L) / 2);
  timer_begin(m, AGX_K_MG_OTHER);
  hipLaunchKernelGGL(k_mg_norm_pairs<double>, dim3((unsigned)nb), dim3(BS), 0, m->stream, m->gate, L.u, L.src, L.n1,
                     L.n2, L.n3, 1.0 / (L.dx * L.dx), m->red);
  final_sum(m, nb, 0);
  timer_end(m);
}

static double mesh_volume(const agx_mesh_desc &d) {
  return (d.x1max - d.x1min) * (d.x2max - d.x2min) * (d.x3max - d.x3min);
}

// MultigridDriver::SubtractAverage (multigrid_driver.cpp:305-330) on the finest FP64
// level: ave = sum * dx*dy*dz / volume, subtracted on the device without a host round
// trip.
static void subtract_average(agx_mesh *m, int type) {
  int l = m->ntotal - 1;
  MGLevel &L = m->lev[l];
  const agx_mesh_desc &d = m->d;
  double dv = m->rdx_blk * m->rdy_blk * m->rdz_blk;
  if (type == 0) array_sum(m, L, L.src, 1);
  else level_sum(m, m->lev, l, 1);
  double scale = dv / mesh_volume(d);
  hipLaunchKernelGGL(k_mg_add<double>, dim3(grid1d(lcells(L), BS)), dim3(BS), 0, m->stream, m->gate,
                     type ? L.u : L.src, lcells(L), m->scal + 1, scale);
}

template <typename T>
static void zero_level(agx_mesh *m, std::vector<MGLevelT<T>> &H, int l) {
  MGLevelT<T> &L = H[l];
  hipLaunchKernelGGL(k_mg_zero<T>, dim3(grid1d(lcells(L), BS)), dim3(BS), 0, m->stream, m->gate, L.u, lcells(L));
}

// SolveCoarsestGrid, multigrid_driver.cpp:778-819 (periodic: fsubtract_average_)
template <typename T>
static void solve_coarsest(agx_mesh *m, std::vector<MGLevelT<T>> &H) {
  const Geo &g = m->g;
  int ni = g.nb1 > g.nb2 ? g.nb1 : g.nb2;
  ni = ni > g.nb3 ? ni : g.nb3;
  ni >>= (m->nrootlevel - 1);
  if (ni == 1) {
    zero_level(m, H, 0);
    return;
  }
  // the root grid's average of level 0 is subtracted from the root grid's finest level
  // (Multigrid::CalculateTotal at the current level, SubtractAverage on u_[nlevel_-1],
  // multigrid.cpp:602-641)
  MGLevelT<T> &LR = H[m->nrootlevel - 1];
  int ll = m->nrootlevel - 1;
  double dxl = m->rdx_root * (double)(1 << ll), dyl = m->rdy_root * (double)(1 << ll),
         dzl = m->rdz_root * (double)(1 << ll);
  double scale = dxl * dyl * dzl / mesh_volume(m->d);
  for (int pass = 0; pass < 2; ++pass) {
    if (pass == 1) {
      for (int it = 0; it < ni; ++it) { smooth(m, H, 0, 0); smooth(m, H, 0, 1); }
    }
    level_sum(m, H, 0, 2);
    hipLaunchKernelGGL(k_mg_add<T>, dim3(grid1d(lcells(LR), BS)), dim3(BS), 0, m->stream, m->gate, LR.u, lcells(LR),
                       m->scal + 2, scale);
  }
}

// SolveVCycle(1,1), multigrid_driver.cpp:684-693 with OneStepToCoarser (:629-677) and
// OneStepToFiner (:583-622).  On the uniform periodic hierarchy every level step is:
// coarser = red sweep, black sweep, defect+restrict; finer = prolongate+correct, red,
// black.
// Highest level handled by k_mg_coarse, or -1 if the root grid is not a single cell.
template <typename T>
static int coarse_top(const std::vector<MGLevelT<T>> &H) {
  const MGLevelT<T> &L0 = H[0];
  return (L0.n1 == 1 && L0.n2 == 1 && L0.n3 == 1) ? coarse_fit(H, false, false) : -1;
}

template <typename T>
static void coarse_cycle(agx_mesh *m, std::vector<MGLevelT<T>> &H, int top, bool first_sweep_done) {
  timer_begin(m, AGX_K_MG_SMOOTH);
  hipLaunchKernelGGL((k_mg_coarse<T, BC_PER>), dim3(1), dim3(COARSE_BS), 0, m->stream, m->gate,
                     coarse_set<T>(H, top, false, false), top, 0, m->coffset, 0, T(1.15 / 6.0),
                     first_sweep_done ? 1 : 0);
  timer_end(m);
}

// A periodic level as whole passes; its spare array holds u between the way down and the way up.
template <typename T>
static void down_p(agx_mesh *m, MGLevelT<T> &F, MGLevelT<T> &C, bool first_sweep_done) {
  PassArgs<T> a = pass_args<T>(m, F);
  a.uin = F.u; a.uout = F.def;
  a.csrc = C.src; a.cu = C.u;
  a.first_sweep_done = first_sweep_done ? 1 : 0;
  timer_begin(m, AGX_K_MG_SMOOTH);
  hipLaunchKernelGGL((k_mg_down<T, BC_PER, false>), pass_grid(a), dim3(PassColumn<BC_PER, 2, 3, T>::NT), 0, m->stream,
                     m->gate, a);
  timer_end(m);
}
template <typename T>
static void up_p(agx_mesh *m, MGLevelT<T> &F, MGLevelT<T> &C) {
  PassArgs<T> a = pass_args<T>(m, F);
  a.uin = F.def; a.uout = F.u;
  a.cc = C.u;
  timer_begin(m, AGX_K_MG_SMOOTH);
  hipLaunchKernelGGL((k_mg_up<T, BC_PER>), pass_grid(a), dim3(PassColumn<BC_PER, 1, 2, T>::NT), 0, m->stream, m->gate,
                     a);
  timer_end(m);
}

template <typename T>
static void vcycle(agx_mesh *m, std::vector<MGLevelT<T>> &H, bool first_sweep_done = false) {
  int start = m->current;
  m->coffset ^= 1;
  const int ct = coarse_top(H);
  const bool passes = m->mg_fuse != 0;
  while (m->current > 0 && m->current > ct) {
    int l = m->current;
    const bool done = first_sweep_done && l == start;
    if (passes && pass_level(H[l])) {
      down_p(m, H[l], H[l - 1], done);
    } else {
      if (!done) smooth(m, H, l, 0);
      smooth(m, H, l, 1);
      defect_restrict(m, H, l);
    }
    m->current--;
  }
  if (ct >= 0) coarse_cycle(m, H, m->current, first_sweep_done && m->current == start);
  else solve_coarsest(m, H);
  while (m->current < start) {
    int l = m->current + 1;
    if (passes && pass_level(H[l])) {
      up_p(m, H[l], H[l - 1]);
    } else {
      prolong(m, H, l);
      smooth(m, H, l, 0);
      smooth(m, H, l, 1);
    }
    m->current++;
  }
}

// SolveFMGCycle, multigrid_driver.cpp:700-714, on the hierarchy H whose finest source
// is set; sources are restricted first (RestrictFMGSource, multigrid_driver.cpp:447-456).
template <typename T>
static void fmg(agx_mesh *m, std::vector<MGLevelT<T>> &H) {
  int L = m->ntotal;
  for (int l = L - 1; l > 0; --l) {
    MGLevelT<T> &Fl = H[l], &Cl = H[l - 1];
    hipLaunchKernelGGL(k_mg_restrict_src<T>, dim3(grid1d(lcells(Cl), BS)), dim3(BS), 0, m->stream, Fl.src,
                       Cl.src, Fl.n1, Fl.n2, Fl.n3);
  }
  m->current = 0;
  for (m->fmglevel = 0; m->fmglevel < L; m->fmglevel++) {
    vcycle(m, H);
    if (m->fmglevel != L - 1) {
      fmg_prolong(m, H, m->current + 1);
      m->current++;
    }
  }
  m->fmglevel = L - 1;
}

static double finish_norm(agx_mesh *m) {
  hipMemcpyAsync(m->scal_host, m->scal, sizeof(double), hipMemcpyDeviceToHost, m->stream);
  hipStreamSynchronize(m->stream);
  const agx_mesh_desc &d = m->d;
  double dv = m->rdx_blk * m->rdy_blk * m->rdz_blk;
  double norm = m->scal_host[0] * dv / mesh_volume(d);
  return std::sqrt(norm);
}

static double defect_norm(agx_mesh *m) {
  // MultigridDriver::CalculateDefectNorm (L2), multigrid_driver.cpp:826-858
  defect_sum(m);
  return finish_norm(m);
}

// Mixed precision: FP64 defect of the finest iterate into the FP32 finest source, its
// squared sum into scal[0], and the first sweep of the next correction V-cycle into the
// FP32 correction (k_mg_defect_to32).  With correct, phi += e of the cycle just run is
// applied in the same pass (into the spare array, then swapped).
static void defect_to32(agx_mesh *m, bool correct) {
  int l = m->ntotal - 1;
  MGLevel &F = m->lev[l];
  MGLevel32 &F32 = m->lev32[l];
  const int cred = 0 ^ (m->coffset ^ 1);   // colour of the next V-cycle's first sweep
  const bool tiled = F.n1 % DT_TI == 0 && F.n2 % DT_TJ == 0;
  const int64_t nb = tiled ? (int64_t)(F.n1 / DT_TI) * (F.n2 / DT_TJ) * ((F.n3 + DT_KC - 1) / DT_KC)
                           : npart(lcells(F));   // <= red_n (cells / BS + 1) either way
  const double idx2 = 1.0 / (F.dx * F.dx);
  const float dx2f = float(F32.dx * F32.dx), isixf = float(1.15 / 6.0);
  timer_begin(m, AGX_K_MG_OTHER);
  // e of the last cycle is read at neighbour cells, so the next cycle's start goes to the
  // spare FP32 array (then swapped), as the corrected phi goes to the FP64 one
  if (tiled && correct)
    hipLaunchKernelGGL(k_mg_defect_to32_t<true>, dim3((unsigned)nb), dim3(DT_TI * DT_TJ), 0, m->stream, m->gate, F.u,
                       F32.u, F.def, F.src, F32.src, F32.def, F.n1, F.n2, F.n3, idx2, dx2f, isixf, cred, m->red);
  else if (tiled)
    hipLaunchKernelGGL(k_mg_defect_to32_t<false>, dim3((unsigned)nb), dim3(DT_TI * DT_TJ), 0, m->stream, m->gate, F.u,
                       (const float *)nullptr, (double *)nullptr, F.src, F32.src, F32.def, F.n1, F.n2, F.n3, idx2,
                       dx2f, isixf, cred, m->red);
  else
    hipLaunchKernelGGL(k_mg_defect_to32, dim3((unsigned)nb), dim3(BS), 0, m->stream, m->gate, F.u,
                       correct ? F32.u : (const float *)nullptr, correct ? F.def : (double *)nullptr, F.src,
                       F32.src, F32.def, F.n1, F.n2, F.n3, idx2, dx2f, isixf, cred, m->red);
  final_sum(m, nb, 0);
  timer_end(m);
  if (correct) std::swap(F.u, F.def);
  std::swap(F32.u, F32.def);
}

// One defect-correction step: FP32 V(1,1) on L(e) = d from e = 0 (its first sweep
// already applied by defect_to32), then phi += e together with the next defect.  The
// FP32 source and correction must come from defect_to32.
static void correction_step(agx_mesh *m) {
  m->current = m->ntotal - 1;
  vcycle(m, m->lev32, true);
  defect_to32(m, true);
}

// MGGravityDriver::Solve (mg_gravity.cpp:166-211) on the periodic hierarchy, up to the
// iteration: load, mean subtraction, FMG
static void solve_load(agx_mesh *m) {
  const Geo &g = m->g;
  int L = m->ntotal;
  MGLevel &F = m->lev[L - 1];
  double **A = m->arr.a;
  hipLaunchKernelGGL(k_mg_load, dim3(grid1d(lcells(F), BS)), dim3(BS), 0, m->stream, g, A[AGX_ARR_U],
                     A[AGX_ARR_PHI], F.src, F.u, m->d.four_pi_G, m->mg_mode == 1 ? 1 : 0, src_mask(m));
  m->current = L - 1;
  m->fmglevel = L - 1;
  subtract_average(m, 0);   // SetupMultigrid, multigrid_driver.cpp:438-439
  if (m->mg_mode == 0) {
    if (!m->mixed) {
      fmg(m, m->lev);
    } else {
      // FMG in FP32 from the FP64 source; the result seeds the FP64 iterate
      MGLevel32 &F32 = m->lev32[L - 1];
      hipLaunchKernelGGL(k_mg_mix, dim3(grid1d(lcells(F), BS)), dim3(BS), 0, m->stream, F.src, F32.src,
                         lcells(F), 2);
      fmg(m, m->lev32);
      hipLaunchKernelGGL(k_mg_mix, dim3(grid1d(lcells(F), BS)), dim3(BS), 0, m->stream, F.u, F32.u,
                         lcells(F), 1);
    }
    m->current = L - 1;
    subtract_average(m, 1);
  }
}

static int retrieve(agx_mesh *m) {
  const Geo &g = m->g;
  int64_t nret = (int64_t)(g.bx1 + 2) * (g.bx2 + 2) * (g.bx3 + 2) * g.nb;
  hipLaunchKernelGGL(k_mg_retrieve, dim3(grid1d(nret, BS)), dim3(BS), 0, m->stream, g, m->lev[m->ntotal - 1].u,
                     m->arr.a[AGX_ARR_PHI]);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_fail(e, "mg_solve launches");
  return 0;
}

// SolveIterative (multigrid_driver.cpp:721-755): the finest defect's squared sum into
// scal[0] before the loop (the mixed form also writes the first correction cycle's
// inputs), and one pass of the loop with the new defect's squared sum into scal[0]
static void first_defect_sum(agx_mesh *m) {
  if (m->mp_on) defect_sum_b(m);
  else if (m->mixed) defect_to32(m, false);
  else defect_sum(m);
}
static void loop_step(agx_mesh *m) {
  if (m->mp_on) {
    if (m->mixed) correction_step_b(m);
    else vcycle_b(m);
    defect_sum_b(m);
  } else if (m->mixed) {
    correction_step(m);   // the defect comes with the correction
  } else {
    vcycle(m, m->lev);
    defect_sum(m);
  }
}

int mg_solve(agx_mesh *m, int stage) {
  if (m->mp_on) return mg_solve_b(m, stage);
  const bool mixed = m->mixed;
  solve_load(m);
  int iters = 0;
  double def = 0.0;
  if (m->mg_eps >= 0.0) {   // SolveIterative, multigrid_driver.cpp:721-755
    int rc = iterate(m, stage, iters, def);
    if (rc) return rc;
    m->last_norm = def;
    if (stage >= 0 && stage <= 2) m->mg_kpred[stage] = iters;
    subtract_average(m, 1);
  } else {   // SolveIterativeFixedTimes, multigrid_driver.cpp:762-771
    if (mixed && m->mg_niter > 0) defect_to32(m, false);
    for (int n = 0; n < m->mg_niter; ++n) {
      if (mixed) correction_step(m);
      else vcycle(m, m->lev);
      iters++;
    }
    subtract_average(m, 1);
    // the defect norm is only reported (agx_mg_last); a cycle being recorded into a graph
    // cannot read it back, so it is left out there
    m->last_norm = m->capturing ? NAN : defect_norm(m);
  }
  m->last_iters = iters;
  return retrieve(m);
}

// ---- a threshold solve recorded into a graph
//
// The loop's V-cycle count is only known on the device, so the recorded loop runs k
// passes whose kernels all take the gate: after each pass k_mg_final_check applies the
// loop's stopping rule to the new norm, and once it closes the gate the remaining passes
// return at once.  The host state a pass changes (red-black offset, swapped arrays) is
// captured after every recorded pass; mg_solve_settle reads how many passes ran and
// restores the state after that many, then runs any further passes eagerly as mg_solve
// would.  Every pass that runs is the same kernel sequence as mg_solve's, so the result
// is the eager one bit for bit.

MGSnap mg_snap(const agx_mesh *m) {
  MGSnap s;
  s.lev = m->lev;
  s.lev32 = m->lev32;
  s.coffset = m->coffset;
  s.current = m->current;
  s.fmglevel = m->fmglevel;
  return s;
}

void mg_restore(agx_mesh *m, const MGSnap &s) {
  m->lev = s.lev;
  m->lev32 = s.lev32;
  m->coffset = s.coffset;
  m->current = s.current;
  m->fmglevel = s.fmglevel;
}

std::vector<uintptr_t> mg_key(const agx_mesh *m) {
  std::vector<uintptr_t> k;
  for (const MGLevel &L : m->lev) { k.push_back((uintptr_t)L.u); k.push_back((uintptr_t)L.def); }
  for (const MGLevel32 &L : m->lev32) { k.push_back((uintptr_t)L.u); k.push_back((uintptr_t)L.def); }
  k.push_back((uintptr_t)m->coffset);
  k.push_back((uintptr_t)m->current);
  k.push_back((uintptr_t)m->fmglevel);
  return k;
}

int mg_solve_head(agx_mesh *m) {
  if (m->mp_on) solve_load_b(m);
  else solve_load(m);
  first_defect_sum(m);
  hipLaunchKernelGGL(k_mg_gate_open, dim3(1), dim3(64), 0, m->stream, m->gatedev, m->scal, norm_dv(m),
                     mesh_volume(m->d), m->mg_eps);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : hip_fail(e, "mg_solve_head launches");
}

void mg_solve_gated(agx_mesh *m, int k, std::vector<MGSnap> &snaps) {
  snaps.clear();
  snaps.push_back(mg_snap(m));
  m->gate = reinterpret_cast<const int *>(reinterpret_cast<const char *>(m->gatedev) + offsetof(MGGate, closed));
  for (int i = 0; i < k; ++i) {
    loop_step(m);   // ends with k_mg_final_check
    snaps.push_back(mg_snap(m));
  }
  m->gate = nullptr;
}

// SolveIterative's loop (multigrid_driver.cpp:733-753) from the iters-th V-cycle on, the host
// reading the norm after each
static void iterate_checked(agx_mesh *m, int &iters, double &def) {
  int n = iters;
  while (def > m->mg_eps) {
    loop_step(m);
    iters++;
    double olddef = def;
    def = finish_norm(m);
    if (def / olddef > 0.8) {
      if (m->mg_eps == 0.0) break;
    }
    if (n > 100) break;
    n++;
  }
}

// launches of one pass of the loop (loop_step)
static int pass_launches(const agx_mesh *m) {
  const bool mp = m->mp_on;
  const int ct = mp ? coarse_top_b(m) : coarse_top(m->lev);   // by the sizes alone: the FP32 levels' too
  const int ni = std::max(m->g.nb1, std::max(m->g.nb2, m->g.nb3)) >> (m->nrootlevel - 1);
  int n = 2 + (mp && m->mixed ? 4 : 0);   // the norm; correction_step_b's steps around its V-cycle
  if (ct >= 0) n += 1;
  else n += mp ? 2 + 4 * ni : (ni == 1 ? 1 : 6 + 2 * ni);
  for (int l = std::max(ct, 0) + 1; l < m->ntotal; ++l)
    n += ((mp ? m->mg_coarse != 0 : m->mg_fuse != 0) && pass_level(m->lev[l])) ? 2 : (mp ? 14 : 6);
  return n;
}

// SolveIterative (multigrid_driver.cpp:721-755) for an eager solve.  A norm that the host reads
// leaves the GPU idle for 25 to 35 us, so the host enqueues gated passes, as many as the norm's
// rate leaves whole V-cycles to the threshold (at most MG_AHEAD), and reads the gate after them.
// A pass behind the closed gate costs 2 us a launch, so
// - a solve reads the norm before the loop and after its first V-cycle, as it may need no more,
//   unless the stage's last solve took four or more (us a solve, 64^3: none needed 303 periodic FMG
//   and 69 from the last potential, with four passes enqueued unread 324 and 157);
// - passes of many launches keep the read after each (one a step with multipole boundaries, 100
//   launches: none needed 1130, with four passes unread 2460), and timed ones, whose launch counts
//   would hold the closed passes.
constexpr int MG_AHEAD = 16, MG_AHEAD_LAUNCHES = 56;
static int iterate(agx_mesh *m, int stage, int &iters, double &def) {
  first_defect_sum(m);
  iters = 0;
  const bool each = m->timer.enabled || pass_launches(m) > MG_AHEAD_LAUNCHES;
  int k = (!each && stage >= 0 && stage <= 2 && m->mg_kpred[stage] >= 4) ? 2 : 1;
  def = 0.0;   // not read yet
  if (k == 1) {
    def = finish_norm(m);
    if (!(def > m->mg_eps)) return 0;
    if (each) {
      iterate_checked(m, iters, def);
      return 0;
    }
  }
  hipLaunchKernelGGL(k_mg_gate_open, dim3(1), dim3(64), 0, m->stream, m->gatedev, m->scal, norm_dv(m),
                     mesh_volume(m->d), m->mg_eps);
  std::vector<MGSnap> snaps;
  for (;;) {
    mg_solve_gated(m, k, snaps);
    hipError_t e = hipMemcpyAsync(m->gatehost, m->gatedev, sizeof(MGGate), hipMemcpyDeviceToHost, m->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
    if (e != hipSuccess) return hip_fail(e, "mg_solve");
    const MGGate gs = *m->gatehost;
    const int ran = gs.iters - iters;
    if (ran < 0 || ran > k) {
      set_error("multigrid loop reports %d V-cycles of %d", ran, k);
      return -70;
    }
    mg_restore(m, snaps[ran]);
    const double before = iters ? def : gs.first;
    iters = gs.iters;
    def = gs.def;
    if (gs.closed) return 0;
    const double rate = std::pow(def / before, 1.0 / ran);   // an open gate: the whole chunk ran
    if (m->mg_eps == 0.0) k = 4;   // runs to the rounding floor, which no rate foretells
    else if (rate > 0.0 && rate < 1.0)
      k = (int)std::min<double>(MG_AHEAD, std::max(1.0, std::floor(std::log(m->mg_eps / def) / std::log(rate))));
    else k = 1;
  }
}

int mg_solve_settle(agx_mesh *m, int stage, const std::vector<MGSnap> &snaps) {
  hipError_t e = hipMemcpyAsync(m->gatehost, m->gatedev, sizeof(MGGate), hipMemcpyDeviceToHost, m->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
  if (e != hipSuccess) return hip_fail(e, "mg_solve_settle");
  const MGGate gs = *m->gatehost;
  if (gs.iters < 0 || gs.iters >= (int)snaps.size()) {
    set_error("recorded multigrid loop reports %d V-cycles of %d", gs.iters, (int)snaps.size() - 1);
    return -70;
  }
  mg_restore(m, snaps[gs.iters]);
  double def = gs.def;
  int iters = gs.iters;
  if (!gs.closed) iterate_checked(m, iters, def);   // the recorded passes ended before the loop did
  m->last_norm = def;
  m->last_iters = iters;
  if (stage >= 0 && stage <= 2) m->mg_kpred[stage] = iters;
  return 0;
}

int mg_solve_tail(agx_mesh *m) {
  if (m->mp_on) return retrieve_b(m);
  subtract_average(m, 1);
  return retrieve(m);
}

// Times V-cycles (on whatever the finest level holds; the next solve reloads it) with
// the levels as whole passes and as one launch per step, and keeps the faster.
int mg_autotune(agx_mesh *m) {
  if (!m->mg_on || m->mp_on) return 0;
  hipEvent_t e0, e1;
  AGX_HIP(hipEventCreate(&e0));
  AGX_HIP(hipEventCreate(&e1));
  const bool timing = m->timer.enabled;
  m->timer.enabled = false;
  float best = 0.f;
  int best_f = 0;
  int rc = 0;
  for (int f = 0; f <= 1 && rc == 0; ++f) {
    m->mg_fuse = f;
    rc = mg_vcycles(m, 1);   // warm-up
    if (rc) break;
    AGX_HIP(hipEventRecord(e0, m->stream));
    rc = mg_vcycles(m, 3);
    if (rc) break;
    AGX_HIP(hipEventRecord(e1, m->stream));
    AGX_HIP(hipEventSynchronize(e1));
    float ms = 0.f;
    AGX_HIP(hipEventElapsedTime(&ms, e0, e1));
    if (f == 0 || ms < best) { best = ms; best_f = f; }
  }
  m->timer.enabled = timing;
  hipEventDestroy(e0);
  hipEventDestroy(e1);
  m->mg_fuse = best_f;
  m->graph_gen++;
  return rc;
}

// n V(1,1) cycles on the current finest state; in the mixed form one cycle is one
// defect-correction step (FP64 defect, FP32 V-cycle, FP64 correction).
int mg_vcycles(agx_mesh *m, int n) {
  m->current = m->ntotal - 1;
  if (m->mp_on) {
    // the FAS levels, the boundary values and the source come from a solve
    if (!m->mp_solved) {
      set_error("agx_mg_vcycles: multipole boundaries need an agx_mg_solve first (it loads the source, "
                "the multipole boundary values and the FAS levels)");
      return -22;
    }
    for (int q = 0; q < n; ++q) {
      if (m->mixed) correction_step_b(m);
      else vcycle_b(m);
    }
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : hip_fail(e, "mg_vcycles launches");
  }
  if (m->mixed && n > 0) defect_to32(m, false);
  for (int q = 0; q < n; ++q) {
    if (m->mixed) correction_step(m);
    else vcycle(m, m->lev);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_fail(e, "mg_vcycles launches");
  return 0;
}

// ---------------------------------------------------------------- per-level steps
// The multigrid at the granularity of the reference's MultigridTaskList
// (multigrid/mg_task_list.cpp:183-280, 287-530) and MGGravity / Multigrid methods, on
// the FP64 hierarchy (every level of the whole mesh, finest = nlevels - 1), for callers
// that drive their own cycles.  Each value is formed by the arithmetic of agx_mg_solve's whole passes, so a V(1,1)
// cycle composed of them equals agx_mg_vcycles(1) bit for bit.
static int mg_level_check(agx_mesh *m, int level, int lo, const char *who) {
  if (!m) { set_error("%s: null mesh", who); return -1; }
  if (!m->mg_on) { set_error("%s: the mesh has no multigrid gravity", who); return -21; }
  if (level < lo || level >= m->ntotal) {
    set_error("%s: level %d not in [%d, %d]", who, level, lo, m->ntotal - 1);
    return -2;
  }
  return 0;
}

static int launches_ok(const char *who) {
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : hip_fail(e, who);
}

}  // namespace agx

using namespace agx;

// MGGravityDriver::Solve's set-up: Multigrid::LoadSource (src = 4 pi G rho, multigrid.cpp:
// 194-220), the source mask and MultigridDriver::SetupMultigrid (mean subtraction on
// periodic meshes; multipole coefficients and boundary values, multigrid_driver.cpp:
// 430-460), then RestrictFMGSource (:447-456) down to the root level.
extern "C" int agx_mg_setup(agx_mesh *m) {
  int rc = mg_level_check(m, 0, 0, "agx_mg_setup");
  if (rc) return rc;
  const Geo &g = m->g;
  const int L = m->ntotal;
  double **A = m->arr.a;
  if (m->mp_on) {
    MGLevelB &F = m->levb[L - 1];
    hipLaunchKernelGGL(k_mb_load, dim3(grid1d((int64_t)F.n1 * F.n2 * F.n3, BS)), dim3(BS), 0, m->stream, g,
                       A[AGX_ARR_U], A[AGX_ARR_PHI], F.src, F.u, m->d.four_pi_G, m->mg_mode == 1 ? 1 : 0,
                       src_mask(m));
    mp_coefficients(m);
    m->mp_solved = true;
    for (int l = L - 1; l > 0; --l) {
      MGLevelB &Fl = m->levb[l], &Cl = m->levb[l - 1];
      hipLaunchKernelGGL(k_mb_restrict_src, dim3(grid1d((int64_t)Cl.n1 * Cl.n2 * Cl.n3, BS)), dim3(BS), 0,
                         m->stream, Fl.src, Cl.src, Fl.n1, Fl.n2, Fl.n3);
    }
  } else {
    MGLevel &F = m->lev[L - 1];
    hipLaunchKernelGGL(k_mg_load, dim3(grid1d(lcells(F), BS)), dim3(BS), 0, m->stream, g, A[AGX_ARR_U],
                       A[AGX_ARR_PHI], F.src, F.u, m->d.four_pi_G, m->mg_mode == 1 ? 1 : 0, src_mask(m));
    subtract_average(m, 0);
    for (int l = L - 1; l > 0; --l) {
      MGLevel &Fl = m->lev[l], &Cl = m->lev[l - 1];
      hipLaunchKernelGGL(k_mg_restrict_src<double>, dim3(grid1d(lcells(Cl), BS)), dim3(BS), 0, m->stream, Fl.src,
                         Cl.src, Fl.n1, Fl.n2, Fl.n3);
    }
  }
  m->current = L - 1;
  m->fmglevel = L - 1;
  return launches_ok("agx_mg_setup");
}

// MGGravity::Smooth (mg_gravity.cpp:220-273): one colour of the red-black sweep on a level
// (multipole meshes: interior cells; fill the ghosts first, agx_mg_fill_ghost).  The colour
// is combined with the driver's colour offset (agx_mg_coffset) as mg_gravity.cpp:227,243 do.
extern "C" int agx_mg_smooth(agx_mesh *m, int32_t level, int32_t color) {
  int rc = mg_level_check(m, level, 0, "agx_mg_smooth");
  if (rc) return rc;
  if (color != 0 && color != 1) { set_error("agx_mg_smooth: colour must be 0 or 1"); return -3; }
  if (m->mp_on) smooth_b(m, level, color);
  else smooth(m, m->lev, level, color);
  return launches_ok("agx_mg_smooth");
}

// The ghost fill of a level before a stencil step (MGBoundaryValues, bvals_mg.cpp:321-370
// with MGMultipoleInnerX1..OuterX3, mgbval_multipole.cpp:28-426).  Periodic levels have no
// stored ghosts (neighbours are read through the periodic index wrap): nothing to do.
extern "C" int agx_mg_fill_ghost(agx_mesh *m, int32_t level) {
  int rc = mg_level_check(m, level, 0, "agx_mg_fill_ghost");
  if (rc) return rc;
  if (m->mp_on) bc_b(m, level);
  return launches_ok("agx_mg_fill_ghost");
}

// Multigrid::StoreOldData + MGGravity::CalculateFASRHS (multigrid.cpp:648-653,
// mg_gravity.cpp:324-351) on a level; multipole (FAS) meshes only.
extern "C" int agx_mg_fas(agx_mesh *m, int32_t level) {
  int rc = mg_level_check(m, level, 0, "agx_mg_fas");
  if (rc) return rc;
  if (!m->mp_on) { set_error("agx_mg_fas: FAS runs with multipole boundaries only (multigrid_driver.cpp:292-295)"); return -22; }
  fas_b(m, level);
  return launches_ok("agx_mg_fas");
}

// MGGravity::CalculateDefect + Multigrid::Restrict (mg_gravity.cpp:283-314,
// multigrid.cpp:684-724): the defect of `level` restricted into the source of level-1
// (with FAS also u), in one pass.
extern "C" int agx_mg_restrict(agx_mesh *m, int32_t level) {
  int rc = mg_level_check(m, level, 1, "agx_mg_restrict");
  if (rc) return rc;
  if (m->mp_on) {
    MGLevelB &F = m->levb[level], &C = m->levb[level - 1];
    hipLaunchKernelGGL(k_mb_restrict<double>, dim3(grid1d((int64_t)C.n1 * C.n2 * C.n3, BS)), dim3(BS), 0,
                       m->stream, m->gate, F.u, F.src, C.src, C.u, F.n1, F.n2, F.n3, 1.0 / (F.dx * F.dx));
  } else {
    defect_restrict(m, m->lev, level);
  }
  return launches_ok("agx_mg_restrict");
}

// Multigrid::ProlongateAndCorrect (multigrid.cpp:733-829): level-1 -> level.
extern "C" int agx_mg_prolong(agx_mesh *m, int32_t level) {
  int rc = mg_level_check(m, level, 1, "agx_mg_prolong");
  if (rc) return rc;
  if (m->mp_on) {
    MGLevelB &F = m->levb[level], &C = m->levb[level - 1];
    mb_prolong(m, C.u, C.uold, F.u, F.n1, F.n2, F.n3);
  } else {
    prolong(m, m->lev, level);
  }
  return launches_ok("agx_mg_prolong");
}

// Multigrid::FMGProlongate (multigrid.cpp:838-1048): level-1 -> level (multipole meshes:
// fill level-1's ghosts first, as SolveFMGCycle's exchange does).
extern "C" int agx_mg_fmg_prolong(agx_mesh *m, int32_t level) {
  int rc = mg_level_check(m, level, 1, "agx_mg_fmg_prolong");
  if (rc) return rc;
  if (m->mp_on) {
    MGLevelB &F = m->levb[level], &C = m->levb[level - 1];
    hipLaunchKernelGGL(k_mb_fmg_prolong, dim3(grid1d((int64_t)F.n1 * F.n2 * F.n3, BS)), dim3(BS), 0, m->stream, C.u,
                       F.u, F.n1, F.n2, F.n3);
  } else {
    fmg_prolong(m, m->lev, level);
  }
  return launches_ok("agx_mg_fmg_prolong");
}

// MultigridDriver::SolveCoarsestGrid (multigrid_driver.cpp:778-819) on level 0.
extern "C" int agx_mg_solve_coarsest(agx_mesh *m) {
  int rc = mg_level_check(m, 0, 0, "agx_mg_solve_coarsest");
  if (rc) return rc;
  if (m->mp_on) {
    const Geo &g = m->g;
    const int ni = std::max(g.nb1, std::max(g.nb2, g.nb3)) >> (m->nrootlevel - 1);
    bc_b(m, 0);
    fas_b(m, 0);
    for (int it = 0; it < ni; ++it) {
      smooth_b(m, 0, 0);
      bc_b(m, 0);
      smooth_b(m, 0, 1);
      bc_b(m, 0);
    }
  } else {
    solve_coarsest(m, m->lev);
  }
  return launches_ok("agx_mg_solve_coarsest");
}

// MultigridDriver::CalculateDefectNorm (L2, multigrid_driver.cpp:826-858) of the finest level.
extern "C" int agx_mg_defect_norm(agx_mesh *m, double *norm) {
  int rc = mg_level_check(m, 0, 0, "agx_mg_defect_norm");
  if (rc) return rc;
  if (!norm) { set_error("agx_mg_defect_norm: null output"); return -1; }
  *norm = m->mp_on ? defect_norm_b(m) : defect_norm(m);
  return launches_ok("agx_mg_defect_norm");
}

// Multigrid::RetrieveResult (multigrid.cpp:266-288): the finest u, with one ghost cell,
// into Gravity::phi; on periodic meshes after SubtractAverage of u, as
// MGGravityDriver::Solve does (multigrid_driver.cpp:755-771).
extern "C" int agx_mg_retrieve(agx_mesh *m) {
  int rc = mg_level_check(m, 0, 0, "agx_mg_retrieve");
  if (rc) return rc;
  const Geo &g = m->g;
  const int64_t nret = (int64_t)(g.bx1 + 2) * (g.bx2 + 2) * (g.bx3 + 2) * g.nb;
  if (m->mp_on) {
    hipLaunchKernelGGL(k_mb_retrieve, dim3(grid1d(nret, BS)), dim3(BS), 0, m->stream, g, m->levb[m->ntotal - 1].u,
                       m->arr.a[AGX_ARR_PHI]);
  } else {
    subtract_average(m, 1);
    hipLaunchKernelGGL(k_mg_retrieve, dim3(grid1d(nret, BS)), dim3(BS), 0, m->stream, g, m->lev[m->ntotal - 1].u,
                       m->arr.a[AGX_ARR_PHI]);
  }
  return launches_ok("agx_mg_retrieve");
}

// The red-black colour offset of the driver (MultigridDriver::coffset_, flipped at the
// start of every V-cycle, multigrid_driver.cpp:686); flip != 0 flips it first.
extern "C" int agx_mg_coffset(agx_mesh *m, int32_t flip, int32_t *value) {
  int rc = mg_level_check(m, 0, 0, "agx_mg_coffset");
  if (rc) return rc;
  if (flip) m->coffset ^= 1;
  if (value) *value = m->coffset;
  return 0;
}

// Levels of the hierarchy: n = nlevels; dims[3 l + d] = cells of level l along d.
extern "C" int agx_mg_levels(agx_mesh *m, int32_t *n, int32_t *dims, int32_t cap) {
  int rc = mg_level_check(m, 0, 0, "agx_mg_levels");
  if (rc) return rc;
  if (n) *n = m->ntotal;
  for (int l = 0; dims && l < m->ntotal && l < cap; ++l) {
    const int n1 = m->mp_on ? m->levb[l].n1 : m->lev[l].n1, n2 = m->mp_on ? m->levb[l].n2 : m->lev[l].n2,
              n3 = m->mp_on ? m->levb[l].n3 : m->lev[l].n3;
    dims[3 * l] = n1; dims[3 * l + 1] = n2; dims[3 * l + 2] = n3;
  }
  return 0;
}

extern "C" int agx_mg_set_source_mask_sphere(agx_mesh *m, double xc, double yc, double zc, double radius) {
  if (!m) { set_error("agx_mg_set_source_mask_sphere: null mesh"); return -1; }
  if (!m->mg_on) { set_error("agx_mg_set_source_mask_sphere: the mesh has no multigrid gravity"); return -21; }
  m->srcmask = radius > 0.0 ? 1 : 0;
  m->srcmask_c[0] = xc; m->srcmask_c[1] = yc; m->srcmask_c[2] = zc;
  m->srcmask_r2 = radius * radius;   // collapse.cpp:68: rc2 = rc*rc
  m->graph_gen++;
  return 0;
}

extern "C" int agx_set_mg_coarse(agx_mesh *m, int32_t on) {
  if (!m) { set_error("agx_set_mg_coarse: null mesh"); return -1; }
  m->mg_coarse = on ? 1 : 0;
  m->graph_gen++;
  return 0;
}
