// One Yee half-step as one launch: the update, every CPML slab, the TFSF and
// lumped corrections and (E) the point probes.
//
// All of them write a component from the other half's field and from itself
// only, so a half-step is point-wise and needs no order between points.  As
// launches of their own the three slab pairs, the records and the probes cost
// more than the update on boxes up to ~200 cells a side: they are short
// (2.5-6 us, 4 us from launch to launch) and read again what the update just
// held in registers.  Bound: HBM / cache bytes on large boxes, memory latency
// (wavefronts in flight) on small ones.
//
// Addressing: a work-group's tile has a uniform origin and a wavefront is one
// (j) row of 64 k, so every array is read at a scalar base plus the lane's own
// constant offset: no vector address arithmetic in the i-march.
//
// A point lies in at most one slab per axis.  Membership in an x slab is
// uniform over a plane and in a y slab over a wavefront's row (scalar
// branches); a z slab takes some lanes of a row.  psi and c_psi are loaded
// beside the field values, so slab points wait for memory as often as others.
// The far planes i = nx, j = ny, k = nz are left out: their slab corrections
// draw on each other only, so the zeros they start with stay.
//
// psi and c_psi hold both components of a point side by side: one access each
// where there were two, and half the lines of a z slab's short rows.
//
// Measured, us per step (kernel time), separate launches / this: 63^3 FP64 with
// a TFSF box 55 / 24, 100^3 FP32 66 / 35, 128^3 FP64 117 / 92, 203 x 181 x 225
// FP64 410 / 385, 384^3 FP32 1082 / 1041 (a half-step without its slabs: 435, so
// they cost 85 for 256 MB).  With the components apart: 100^3 37.1, 128^3 99.5,
// 203 x 181 x 225 407.  Rows padded to whole lines instead were slower (216 at
// 203 x 181 x 225, FP64), as were registers capped for one more wavefront per
// SIMD (spills: 384^3 690 a half-step).  Loading plane i + 1 during plane i was tried: no
// faster on small boxes and 2 % slower at 384^3 (fewer wavefronts per CU).
// HBM at 384^3: 3.15 GB a half-step (FP32) at 5.9 TB/s, 5.74 GB (FP64) at 5.7, 1.2
// times the compulsory bytes.
#pragma once

#include <climits>

#include "kernels.hpp"

namespace xfd {

// One CPML slab: layers [lo, hi) along its axis, the recursive-convolution
// coefficients per layer, and c_psi / psi of its components A = (axis+1)%3 and
// B = (axis+2)%3, a pair per point, in the slab's box layout (k fastest; the box
// spans N + 1 points along the other two axes).
template <class T>
struct AxisSlab {
  int lo, hi;
  const T* ca;
  const T* cb;
  const T* c;
  T* psi;
};

// The slabs of one half-step, per axis in position order.  Component q is
// corrected along axes (q+1)%3 and (q+2)%3; swap[q]: the latter comes first
// in boundary order.
template <class T>
struct HalfSlabs {
  AxisSlab<T> s[3][2];
  int n[3];
  int swap[3];
};

// A half-step's corrections and probes by tile: tile b owns the record
// segments seg_of[rec_off[b] .. rec_off[b + 1]) and the probes
// probe_of[probe_off[b] .. probe_off[b + 1]) (null: none in any tile).
template <class T>
struct HalfEvents {
  const int32_t* rec_off;
  const int32_t* seg_of;
  const Record* rec;
  const int64_t* seg;
  int64_t nseg;
  const double* pool;
  T* state;
  const int32_t* probe_off;
  const int32_t* probe_of;
  const Probe* probe;
  double* probe_out;
  int64_t probe_count;
};

template <class T>
struct SlabVals {
  T pA = T(0), pB = T(0), cA = T(0), cB = T(0);
};

// Both components of a point in one access.
template <class T>
struct alignas(2 * sizeof(T)) SlabPair {
  T a, b;
};

// u: uniform point offset in the box, e: the lane's
template <class T>
__device__ __forceinline__ SlabVals<T> slabLoad(const T* c, const T* psi, int64_t u, unsigned e) {
  const SlabPair<T> p = (reinterpret_cast<const SlabPair<T>*>(psi) + u)[e];
  const SlabPair<T> q = (reinterpret_cast<const SlabPair<T>*>(c) + u)[e];
  return SlabVals<T>{p.a, p.b, q.a, q.b};
}

// psi = b psi + a d for both components of a slab point, stored.
template <class T>
__device__ __forceinline__ void slabStore(T* psi, int64_t u, unsigned e, SlabVals<T>& v, T ca, T cb, T dA, T dB) {
  v.pA = sumTwo(cb, v.pA, ca, dA);
  v.pB = sumTwo(cb, v.pB, ca, dB);
  (reinterpret_cast<SlabPair<T>*>(psi) + u)[e] = SlabPair<T>{v.pA, v.pB};
}

// v + ca pa + cb pb, the latter first where the boundary's order swaps them.
template <class T>
__device__ __forceinline__ T addInOrder(T v, T ca, T pa, T cb, T pb, int swap) {
  return swap ? mulAdd(ca, pa, mulAdd(cb, pb, v)) : mulAdd(cb, pb, mulAdd(ca, pa, v));
}

// What one plane of a tile reads at (i, j, k): the other half's field d at the
// point and its neighbours, the half's own field f, the material id and the
// coefficients' raw data.
template <class T, class Coef>
struct HalfPlane {
  T a0;            // d0 at the point
  T b1, b2;        // d1, d2: E at the point, H one plane above
  T j0, j2;        // d0, d2 at the j neighbour
  T k0, k1;        // d0, d1 at the k neighbour
  T o0, o1, o2;    // f
  int m;
  typename Coef::Raw r0, r1, r2;
};

// One tile of a half-step: TK lanes along k, TJ rows along j, planes
// [i0, i0 + ichunk).  S: the dispersive scheme of the E half-step, or -1; P: the
// most poles whose currents a dispersive cell loads at once (its registers
// bound the wavefronts in flight: 160^3 FP32 with two poles, 133 us against 150 us
// with room for four).
template <class T, class Coef, bool IsE, int S, bool NT, int TK, int TJ, int P = kAdeFastPoles>
__device__ __forceinline__ void halfTile(const Grid g, const FieldPtrs<T> F, const Coef C, const AdeArgs<T> A,
                                         const HalfSlabs<T>* __restrict__ HP, int bx, int by, int bz, int ichunk) {
#pragma clang fp contract(off)
  static_assert(TK % 64 == 0, "a wavefront is part of one row");
  const HalfSlabs<T>& H = *HP;
  const unsigned lane = threadIdx.x;
  const int j = by * TJ + __builtin_amdgcn_readfirstlane(threadIdx.y);
  const int k0 = bx * TK, k = k0 + static_cast<int>(lane);
  const int i0 = bz * ichunk, i1 = min(i0 + ichunk, g.nx);
  if (k >= g.nz || j >= g.ny) return;
  const int64_t pz = g.pz, pl = g.plane;
  int64_t u = (static_cast<int64_t>(i0) * g.NY + j) * pz + k0;  // uniform; the lane's element is u + lane
  // slabs: the x slab of the march (re-picked where the march leaves it), the
  // row's y slab and the lane's z slab
  // The bounds that every plane tests are copies: memory that the stores below
  // might alias would be read again, a chain of scalar loads, in every plane.
  // The slabs' pointers stay in memory: as copies they cost registers (384^3
  // FP32 525 against 520 us a half-step).
  const int nx = H.n[0], ny = H.n[1], nz = H.n[2];
  const int swap0 = H.swap[0], swap1 = H.swap[1], swap2 = H.swap[2];
  const int xend = nx > 1 ? H.s[0][0].hi : INT_MAX;  // where the march passes to the far x slab
  bool second = i0 >= xend;
  const AxisSlab<T>* xs = &H.s[0][second ? 1 : 0];
  int xlo = nx > 0 ? xs->lo : INT_MAX, xhi = nx > 0 ? xs->hi : 0;
  const AxisSlab<T>&Z0 = H.s[2][0], &Z1 = H.s[2][1];
  const bool inY0 = ny > 0 && j >= H.s[1][0].lo && j < H.s[1][0].hi;
  const bool inY1 = ny > 1 && j >= H.s[1][1].lo && j < H.s[1][1].hi;
  const bool inY = inY0 || inY1;
  const AxisSlab<T>& Y = H.s[1][inY1 ? 1 : 0];
  T yca = T(0), ycb = T(0);
  int64_t yu = 0, yp = 0;
  if (inY) {
    yca = Y.ca[j - Y.lo];
    ycb = Y.cb[j - Y.lo];
    yp = static_cast<int64_t>(Y.hi - Y.lo) * (g.nz + 1);
    yu = i0 * yp + static_cast<int64_t>(j - Y.lo) * (g.nz + 1) + k0;
  }
  const bool inZ0 = nz > 0 && k >= Z0.lo && k < Z0.hi;
  const bool inZ1 = nz > 1 && k >= Z1.lo && k < Z1.hi;
  T zca = T(0), zcb = T(0);
  unsigned ze = 0;
  int64_t zu0 = 0, zu1 = 0, zp0 = 0, zp1 = 0;
  if (inZ0) {
    ze = static_cast<unsigned>(k - Z0.lo);
    zca = Z0.ca[ze];
    zcb = Z0.cb[ze];
  }
  if (inZ1) {
    ze = static_cast<unsigned>(k - Z1.lo);
    zca = Z1.ca[ze];
    zcb = Z1.cb[ze];
  }
  if (nz > 0) {
    const int n0 = Z0.hi - Z0.lo;
    zp0 = static_cast<int64_t>(g.NY) * n0;
    zu0 = i0 * zp0 + static_cast<int64_t>(j) * n0;
  }
  if (nz > 1) {
    const int n1 = Z1.hi - Z1.lo;
    zp1 = static_cast<int64_t>(g.NY) * n1;
    zu1 = i0 * zp1 + static_cast<int64_t>(j) * n1;
  }
  // the half's own fields f and the other half's d (x, y, z components)
  T* __restrict__ f0 = F.f[IsE ? 0 : 3];
  T* __restrict__ f1 = F.f[IsE ? 1 : 4];
  T* __restrict__ f2 = F.f[IsE ? 2 : 5];
  const T* __restrict__ d0 = F.f[IsE ? 3 : 0];
  const T* __restrict__ d1 = F.f[IsE ? 4 : 1];
  const T* __restrict__ d2 = F.f[IsE ? 5 : 2];
  constexpr int q0 = IsE ? 0 : 3;
  // E: the duals of plane i - 1; H: of plane i (carried along the march)
  T c1, c2;
  if (IsE) {
    c1 = i0 > 0 ? (d1 + (u - pl))[lane] : T(0);
    c2 = i0 > 0 ? (d2 + (u - pl))[lane] : T(0);
  } else {
    c1 = (d1 + u)[lane];
    c2 = (d2 + u)[lane];
  }
  const bool jk = j >= 1 && k >= 1;
  const int64_t dj = IsE ? (j >= 1 ? -pz : 0) : pz;   // the j neighbour
  // the k neighbour: one element up, or (E) down; on the k = 0 face the point itself
  const int64_t uk = IsE ? -1 : 1;
  const unsigned ek = lane + (IsE && k == 0 ? 1u : 0u);
  auto load = [&](int64_t w) {
    HalfPlane<T, Coef> p;
    p.r0 = C.template rawAt<NT>(q0, w, lane);
    p.r1 = C.template rawAt<NT>(q0 + 1, w, lane);
    p.r2 = C.template rawAt<NT>(q0 + 2, w, lane);
    p.m = S >= 0 ? ldOwn<NT>((A.mat + w) + lane) : -1;
    p.a0 = (d0 + w)[lane];
    p.b1 = (d1 + (IsE ? w : w + pl))[lane];
    p.b2 = (d2 + (IsE ? w : w + pl))[lane];
    p.j0 = (d0 + (w + dj))[lane];
    p.j2 = (d2 + (w + dj))[lane];
    p.k0 = (d0 + (w + uk))[ek];
    p.k1 = (d1 + (w + uk))[ek];
    p.o0 = ldOwn<NT>((f0 + w) + lane);
    p.o1 = ldOwn<NT>((f1 + w) + lane);
    p.o2 = ldOwn<NT>((f2 + w) + lane);
    return p;
  };
  for (int i = i0; i < i1; ++i, u += pl) {
    const HalfPlane<T, Coef> L = load(u);  // every load of the plane first
    T s0, p0, r0, s1, p1, r1, s2, p2, r2;
    C.resolveAt(q0, L.r0, s0, p0, r0);
    C.resolveAt(q0 + 1, L.r1, s1, p1, r1);
    C.resolveAt(q0 + 2, L.r2, s2, p2, r2);
    if (i >= xend && !second) {
      second = true;
      xs = &H.s[0][1];
      xlo = xs->lo;
      xhi = xs->hi;
    }
    const AxisSlab<T>& X = *xs;
    const bool inX = i >= xlo && i < xhi;
    SlabVals<T> sx, sy, sz;
    T xca = T(0), xcb = T(0);
    int64_t xu = 0;
    if (inX) {
      xca = X.ca[i - X.lo];
      xcb = X.cb[i - X.lo];
      xu = (static_cast<int64_t>(i - X.lo) * g.NY + j) * (g.nz + 1) + k0;
      sx = slabLoad<T>(X.c, X.psi, xu, lane);
    }
    if (inY) sy = slabLoad<T>(Y.c, Y.psi, yu, lane);
    if (inZ0) sz = slabLoad<T>(Z0.c, Z0.psi, zu0, ze);
    if (inZ1) sz = slabLoad<T>(Z1.c, Z1.psi, zu1, ze);
    const int m = L.m;
    const T a0 = L.a0, o0 = L.o0, o1 = L.o1, o2 = L.o2;
    // differences of dual component q along axis x, y, z
    const T x1 = L.b1 - c1, x2 = L.b2 - c2;
    const T b1 = IsE ? L.b1 : c1, b2 = IsE ? L.b2 : c2;
    const T y0 = IsE ? a0 - L.j0 : L.j0 - a0, y2 = IsE ? b2 - L.j2 : L.j2 - b2;
    const T z0 = IsE ? a0 - L.k0 : L.k0 - a0, z1 = IsE ? b1 - L.k1 : L.k1 - b1;
    // component 0: d1 along z, d2 along y; 1: d2 along x, d0 along z; 2: d0 along y, d1 along x
    const T w0 = IsE ? sumE(s0, o0, p0, z1, r0, y2) : sumH(s0, o0, p0, z1, r0, y2);
    const T w1 = IsE ? sumE(s1, o1, p1, x2, r1, z0) : sumH(s1, o1, p1, x2, r1, z0);
    const T w2 = IsE ? sumE(s2, o2, p2, y0, r2, x1) : sumH(s2, o2, p2, y0, r2, x1);
    T v0 = w0, v1 = w1, v2 = w2;
    if (IsE) {
      const bool r[3] = {jk, i >= 1 && k >= 1, i >= 1 && j >= 1};
      if (S < 0 || m < 0) {
        v0 = r[0] ? w0 : o0;
        v1 = r[1] ? w1 : o1;
        v2 = r[2] ? w2 : o2;
      } else {
        const T cur[3] = {o0, o1, o2}, en[3] = {w0, w1, w2};
        T v[3];
        if (A.poles <= P) {
          adeCell<T, S < 0 ? 0 : S, P>(A, m, u + lane, r, cur, en, v);
        } else {
#pragma unroll
          for (int q = 0; q < 3; ++q) v[q] = r[q] ? adeUpdate<T, S < 0 ? 0 : S>(A, m, q, u + lane, cur[q], en[q]) : cur[q];
        }
        v0 = v[0];
        v1 = v[1];
        v2 = v[2];
      }
    }
    // x: components 1 (dual 2) and 2 (dual 1); y: 2 (dual 0) and 0 (dual 2);
    // z: 0 (dual 1) and 1 (dual 0)
    if (inX) slabStore(X.psi, xu, lane, sx, xca, xcb, x2, x1);
    if (inY) slabStore(Y.psi, yu, lane, sy, yca, ycb, y0, y2);
    if (inZ0) slabStore(Z0.psi, zu0, ze, sz, zca, zcb, z1, z0);
    if (inZ1) slabStore(Z1.psi, zu1, ze, sz, zca, zcb, z1, z0);
    v0 = addInOrder(v0, sy.cB, sy.pB, sz.cA, sz.pA, swap0);
    v1 = addInOrder(v1, sz.cB, sz.pB, sx.cA, sx.pA, swap1);
    v2 = addInOrder(v2, sx.cB, sx.pB, sy.cA, sy.pA, swap2);
    stOwn<NT>((f0 + u) + lane, v0);
    stOwn<NT>((f1 + u) + lane, v1);
    stOwn<NT>((f2 + u) + lane, v2);
    c1 = L.b1;
    c2 = L.b2;
    yu += yp;
    zu0 += zp0;
    zu1 += zp1;
  }
}

// The tile's corrections, then its probes: on points that the tile's own
// work-group stored, so a work-group barrier orders them after the update.
// No record lands in a slab (the context's choice of this path), so the
// order of records and slabs does not matter.
template <class T>
__device__ __forceinline__ void halfEvents(const FieldPtrs<T>& F, const HalfEvents<T>& ev, int64_t tile, int64_t t) {
  const int tid = threadIdx.y * blockDim.x + threadIdx.x, threads = blockDim.x * blockDim.y;
  if (ev.rec_off) {
    const int r0 = ev.rec_off[tile], r1 = ev.rec_off[tile + 1];
    if (r1 > r0) {
      __syncthreads();
      for (int r = r0 + tid; r < r1; r += threads)
        recordSeg(F, ev.rec, ev.seg, ev.nseg, ev.pool, ev.state, ev.seg_of[r], t);
    }
  }
  if (ev.probe_off && t < ev.probe_count) {
    const int p0 = ev.probe_off[tile], p1 = ev.probe_off[tile + 1];
    if (p1 > p0) {
      __syncthreads();
      for (int r = p0 + tid; r < p1; r += threads) {
        const int q = ev.probe_of[r];
        const Probe P = ev.probe[q];
        ev.probe_out[q * ev.probe_count + t] = static_cast<double>(F.f[P.field][P.idx]);
      }
    }
  }
}

template <class T, class Coef, bool IsE, int S, bool NT, int TK, int TJ, int P = kAdeFastPoles>
__global__ __launch_bounds__(TK * TJ) void k_half(Grid g, FieldPtrs<T> F, Coef C, AdeArgs<T> A, const HalfSlabs<T>* H,
                                                  HalfEvents<T> ev, SweepMap M, int ichunk, int64_t t) {
  int bx, by, bz;
  M.coords(bx, by, bz);
  halfTile<T, Coef, IsE, S, NT, TK, TJ, P>(g, F, C, A, H, bx, by, bz, ichunk);
  halfEvents(F, ev, (static_cast<int64_t>(bz) * M.nby + by) * M.nbx + bx, t);
}

// Everything of one half-step's launch but the fields, coefficients and step.
template <class T>
struct HalfArgs {
  const HalfSlabs<T>* slabs;  // device memory: as kernel arguments the six slabs' pointers spill scalar registers
  HalfEvents<T> events;
  AdeArgs<T> ade;
  int scheme;  // AdeScheme of the E half-step, or -1
  int tk, tj;  // tile: 64 x 4 or 128 x 2
  int ichunk;
  bool stream;  // non-temporal hint on data read and written once per launch
};

template <class T>
struct HalfLaunch {
  static void half(hipStream_t s, const Grid& g, const FieldPtrs<T>& F, const CoefPtrs<T>& C, const HalfArgs<T>& a,
                   bool is_e, int64_t t);
  static void half(hipStream_t s, const Grid& g, const FieldPtrs<T>& F, const ClassCoef<T>& C, const HalfArgs<T>& a,
                   bool is_e, int64_t t);
  static void half(hipStream_t s, const Grid& g, const FieldPtrs<T>& F, const WideCoef<T>& C, const HalfArgs<T>& a,
                   bool is_e, int64_t t);
};

}  // namespace xfd
