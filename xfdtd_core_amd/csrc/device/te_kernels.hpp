// 2D (TE) grids whose Ex, Ey and Hz stay zero: a half-step (Ez, or Hx and Hy)
// with its CPML slabs, corrections and probes as one launch, as k_half does for
// 3D grids.  Small grids are bound by the launches (ten a step as separate
// ones, 4 us from one to the next), large ones by bytes.
//
// Lanes run along j, the contiguous axis of a 2D grid's layout; a wavefront is
// 64 points of one row i and marches `ichunk` rows, so membership in an x slab
// is uniform and a y slab takes some lanes.  Measured, kernel time
// per step, separate launches / this: 330 x 350 FP64 42 / 10.4 us, 2001 x 1501
// FP32 (54 MB of fields and class ids) 86 / 33 us, half of it from j being
// contiguous (k's two entries used to lie side by side).
#pragma once

#include "half_step.hpp"

namespace xfd {

constexpr int kTeRows = 4;  // wavefronts per work-group, one run of rows each

template <class T, class Coef, bool IsE>
__device__ __forceinline__ void teTile(const Grid& g, const FieldPtrs<T>& F, const Coef& C,
                                       const HalfSlabs<T>* __restrict__ HP, int bx, int by, int ichunk) {
#pragma clang fp contract(off)
  const HalfSlabs<T>& H = *HP;
  const int j = bx * 64 + static_cast<int>(threadIdx.x);
  const int i0 = (by * kTeRows + __builtin_amdgcn_readfirstlane(threadIdx.y)) * ichunk;
  const int i1 = min(i0 + ichunk, g.nx);
  if (j >= g.ny || i0 >= g.nx) return;
  const unsigned lane = static_cast<unsigned>(j);
  const int64_t pl = g.plane;
  T* __restrict__ ez = F.f[2];
  T* __restrict__ hx = F.f[3];
  T* __restrict__ hy = F.f[4];
  // psi boxes span both entries of k (nz + 1 = 2) and hold both components;
  // one of each moves
  const bool inY0 = H.n[1] > 0 && j >= H.s[1][0].lo && j < H.s[1][0].hi;
  const bool inY1 = H.n[1] > 1 && j >= H.s[1][1].lo && j < H.s[1][1].hi;
  const bool inY = inY0 || inY1;
  const AxisSlab<T>& Y0 = H.s[1][0];
  const AxisSlab<T>& Y1 = H.s[1][1];
  T yca = T(0), ycb = T(0);
  const T* yc = nullptr;
  T* yp = nullptr;
  int64_t ystep = 0;
  if (inY) {  // E: component A (Ez), H: component B (Hx)
    const int l = j - (inY1 ? Y1.lo : Y0.lo), n = inY1 ? Y1.hi - Y1.lo : Y0.hi - Y0.lo;
    yca = (inY1 ? Y1.ca : Y0.ca)[l];
    ycb = (inY1 ? Y1.cb : Y0.cb)[l];
    ystep = 4 * n;
    const int64_t y = i0 * ystep + 4 * l;
    yc = (inY1 ? Y1.c : Y0.c) + y + (IsE ? 0 : 1);
    yp = (inY1 ? Y1.psi : Y0.psi) + y + (IsE ? 0 : 1);
  }
  int64_t u = i0 * pl;
  // E: Hy of row i - 1; H: Ez of row i (carried along the march)
  T c = IsE ? (i0 > 0 ? (hy + (u - pl))[lane] : T(0)) : (ez + u)[lane];
  const unsigned jm = j >= 1 ? lane - 1 : lane;
  for (int i = i0; i < i1; ++i, u += pl) {
    const int xq = H.n[0] > 1 && i >= H.s[0][0].hi ? 1 : 0;
    const AxisSlab<T>& X = H.s[0][xq];
    const bool inX = H.n[0] > 0 && i >= X.lo && i < X.hi;
    T xca = T(0), xcb = T(0), xp = T(0), xc = T(0), yv = T(0), ycv = T(0);
    T* xpp = nullptr;
    // every load of the row first
    T s0, a0, b0, s1, a1, b1;
    typename Coef::Raw r0, r1;
    T o0, o1 = T(0), n0, n1;
    if (IsE) {
      r0 = C.template raw<false>(2, u + lane);
      o0 = (ez + u)[lane];
      n0 = (hx + u)[lane];
      n1 = (hy + u)[lane];
    } else {
      r0 = C.template raw<false>(3, u + lane);
      r1 = C.template raw<false>(4, u + lane);
      o0 = (hx + u)[lane];
      o1 = (hy + u)[lane];
      n0 = (ez + u)[lane + 1];
      n1 = (ez + (u + pl))[lane];
    }
    const T hxm = IsE ? (hx + u)[jm] : T(0);
    if (inX) {  // E: component B (Ez), H: component A (Hy)
      xca = X.ca[i - X.lo];
      xcb = X.cb[i - X.lo];
      const int64_t x = (static_cast<int64_t>(i - X.lo) * g.NY + j) * 4 + (IsE ? 1 : 0);
      xpp = X.psi + x;
      xp = *xpp;
      xc = X.c[x];
    }
    if (inY) {
      yv = *yp;
      ycv = *yc;
    }
    C.resolve(IsE ? 2 : 3, r0, s0, a0, b0);
    if (!IsE) C.resolve(4, r1, s1, a1, b1);
    // differences along x and y
    const T dx = n1 - c, dy = IsE ? n0 - hxm : n0 - c;
    if (inX) {
      xp = sumTwo(xcb, xp, xca, dx);
      *xpp = xp;
    }
    if (inY) {
      yv = sumTwo(ycb, yv, yca, dy);
      *yp = yv;
    }
    if (IsE) {
      T v = sumE(s0, o0, a0, dy, b0, dx);
      v = i >= 1 && j >= 1 ? v : o0;
      (ez + u)[lane] = addInOrder(v, xc, xp, ycv, yv, H.swap[2]);
    } else {
      (hx + u)[lane] = mulAdd(ycv, yv, sumTwo(s0, o0, b0, dy));
      (hy + u)[lane] = mulAdd(xc, xp, sumTwo(s1, o1, a1, dx));
    }
    c = n1;
    yc += ystep;
    yp += ystep;
  }
}

template <class T, class Coef, bool IsE>
__global__ __launch_bounds__(64 * kTeRows) void k_te_half(Grid g, FieldPtrs<T> F, Coef C, const HalfSlabs<T>* H,
                                                          HalfEvents<T> ev, int nbx, int ichunk, int64_t t) {
  const int bx = blockIdx.x % nbx, by = blockIdx.x / nbx;
  teTile<T, Coef, IsE>(g, F, C, H, bx, by, ichunk);
  halfEvents(F, ev, blockIdx.x, t);
}

template <class T>
struct TeLaunch {
  static void half(hipStream_t s, const Grid& g, const FieldPtrs<T>& F, const CoefPtrs<T>& C, const HalfArgs<T>& a,
                   bool is_e, int64_t t);
  static void half(hipStream_t s, const Grid& g, const FieldPtrs<T>& F, const ClassCoef<T>& C, const HalfArgs<T>& a,
                   bool is_e, int64_t t);
};

}  // namespace xfd
