// 1D (TEM) grids: many steps in one launch of one work-group.
//
// A 1D step is a few hundred to a few thousand cells, so as seven launches a
// step it was bound by the launches (4 us each from one to the next).  Here
// Ex and Hy live in LDS for the whole stretch of steps, each work-item keeps
// its cells' coefficients and Hz in registers, and a step costs two barriers.
// What bounds it is the serial chain of a step: LDS reads, the update, the
// write and the barrier.  Measured, 320 cells, FP64, TFSF and two probes, us a
// step: separate launches 28, this 0.69 (2.5 with the source tables read inside
// the step, 2.1 with their first record alone ahead of it).
//
// Only Ex, Hy and Hz of the column (0, 0) move, and the few points of the
// column (0, 1) that a TFSF face corrects (no update or slab reaches those);
// Ey, Ez, Hx and everything else stay zero.
#pragma once

#include "half_step.hpp"

namespace xfd {

constexpr int kLineThreads = 1024;
constexpr int kLineCells = 8;        // cells per work-item at most
constexpr int kLineSlabCells = 512;  // CPML cells of both ends held in LDS
constexpr int64_t kLineSteps = 4096; // steps per launch at most
constexpr int kLineSegments = 32;    // record segments per half whose addends are computed ahead
constexpr int kLineAhead = 64;       // steps whose addends LDS holds
constexpr int kLineExtra = 64;       // corrected points of the column (0, 1), per field, held in LDS

// The z slab's component on the line, Ex (Hy) corrected from Hy (Ex): every
// other value of the slab's c_psi and psi.
template <class T>
struct LineSlab {
  int lo, n;
  const T* c;   // c_psi
  T* psi;
  const T* ca;
  const T* cb;
};

// One half-step's record segments by work-item (cell k belongs to work-item
// k % threads): work-item w owns of[off[w] .. off[w + 1]) (null: none).  loc:
// a segment's point in the LDS array, from nz + 1 on in the column (0, 1).
template <class T>
struct LineEvents {
  const int32_t *off, *of, *loc;
  const Record* rec;
  const int64_t* seg;
  int64_t nseg;
  int held;         // segments with addends: nseg or 0
  double* addends;  // k_line_addends, or null
};

template <class T>
struct LineArgs {
  int nz, threads;
  int extra_e, extra_h;               // corrected points of the column (0, 1)
  const int32_t* extra_cell;          // and the cells of Ex's
  T* ex;
  T* hy;
  T* hz;
  LineSlab<T> e[2], h[2];
  int slabs;
  LineEvents<T> re, rh;
  const double* pool;
  T* state;
  const int32_t *probe_off, *probe_of;
  const Probe* probe;
  double* probe_out;
  int64_t probe_count;
};

// True where a segment is one TFSF or waveform record: its addend does not
// depend on the fields.  The part without the record's coefficient is computed
// ahead, so that the sum at the point rounds as recordRun's.
__device__ __forceinline__ bool plainSegment(const Record* rec, const int64_t* seg, int64_t s) {
  return seg[s + 1] - seg[s] == 1 && rec[seg[s]].kind != 2;
}

// The addends of every plain segment, without their coefficients, for steps [t0,
// t0 + n), in step order:
// out[s * kLineSteps + t - t0].  The tables hold a step's row kilobytes from
// the next one's, so read inside the step they cost trips to memory that the
// whole line waits for; k_line takes the addends through LDS, kLineAhead steps
// at a time.
template <class T>
__global__ __launch_bounds__(256) void k_line_addends(const Record* __restrict__ rec,
                                                      const int64_t* __restrict__ seg, int64_t nseg,
                                                      const double* __restrict__ pool, int64_t t0, int64_t n,
                                                      double* __restrict__ out) {
  const int64_t q = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t s = blockIdx.y;
  if (q >= n || !plainSegment(rec, seg, s)) return;
  const Record R = rec[seg[s]];
  const double* row = pool + R.pool + (t0 + q) * R.row;
  out[s * kLineSteps + q] = R.kind == 0 ? recordInc<T>(R, row) : row[0];
}

// A work-item's records of one half-step; the first one, where plain, without
// a global access.
struct LineRecords {
  int r0, r1, at, plain;  // plain: the first segment, or -1
  double coef;            // its coefficient

  template <class T>
  __device__ __forceinline__ void init(const LineEvents<T>& e) {
    r0 = e.off ? e.off[threadIdx.x] : 0;
    r1 = e.off ? e.off[threadIdx.x + 1] : 0;
    at = 0;
    plain = -1;
    coef = 0;
    if (r0 < r1 && e.addends) {
      const int s = e.of[r0];
      at = e.loc[s];
      if (plainSegment(e.rec, e.seg, s)) {
        plain = s;
        coef = e.rec[e.seg[s]].coef;
      }
    }
  }
  // corrects the work-item's points of f (LDS) for step t; add: the addends (LDS) of step t
  template <class T>
  __device__ __forceinline__ void apply(T* f, const LineEvents<T>& e, const double* add, const double* pool,
                                        T* state, int64_t t) {
    int r = r0;
    if (plain >= 0) {
      f[at] = static_cast<T>(recordAdd<T>(add[plain * kLineAhead], coef, static_cast<double>(f[at])));
      ++r;
    }
    for (; r < r1; ++r) {
      const int s = e.of[r];
      f[e.loc[s]] = recordRun<T>(f[e.loc[s]], e.rec, e.seg[s], e.seg[s + 1], pool, state, t);
    }
  }
};

// A work-group barrier over LDS alone: global loads and stores stay in flight
// (the recordings' stores, which __syncthreads would wait for in every step).
__device__ __forceinline__ void ldsBarrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <class T, class Coef, int C>
__global__ __launch_bounds__(kLineThreads) void k_line(Coef K, LineArgs<T> a, int64_t t0, int n) {
#pragma clang fp contract(off)
  extern __shared__ unsigned char lds[];
  double* add_e = reinterpret_cast<double*>(lds);
  double* add_h = add_e + a.re.held * kLineAhead;
  T* ex = reinterpret_cast<T*>(add_h + a.rh.held * kLineAhead);
  T* hy = ex + a.nz + 1 + a.extra_e;
  T* slab = hy + a.nz + 1 + a.extra_h;  // per half, per slab cell: psi, c_psi, a, b
  const int tid = threadIdx.x, nth = a.threads, nz = a.nz;
  T se[C], ae[C], sh[C], bh[C], sz[C], az[C], hz[C];
  int ex1[C];  // the cell's Ex of the column (0, 1) in LDS, or -1: zero
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int k = tid + c * nth;
    if (k <= nz) {
      T u0, u1;
      ex1[c] = -1;
      ex[k] = a.ex[k];
      hy[k] = k < nz ? a.hy[k] : T(0);
      hz[c] = T(0);
      se[c] = T(1);
      ae[c] = T(0);
      if (k >= 1 && k < nz) K.get(0, k, se[c], ae[c], u0);
      if (k < nz) {
        K.get(4, k, sh[c], u0, bh[c]);
        K.get(5, k, sz[c], az[c], u1);
        hz[c] = a.hz[k];
      }
    }
  }
  const int m0 = a.slabs > 0 ? a.e[0].n : 0, m1 = a.slabs > 1 ? a.e[1].n : 0, cells = m0 + m1;
  for (int q = tid; q < cells; q += nth) {
    const LineSlab<T>& E = a.e[q < m0 ? 0 : 1];
    const LineSlab<T>& H = a.h[q < m0 ? 0 : 1];
    const int w = q < m0 ? q : q - m0;
    T* se4 = slab + 4 * q;
    T* sh4 = slab + 4 * (cells + q);
    se4[0] = E.psi[2 * w];
    se4[1] = E.c[2 * w];
    se4[2] = E.ca[w];
    se4[3] = E.cb[w];
    sh4[0] = H.psi[2 * w];
    sh4[1] = H.c[2 * w];
    sh4[2] = H.ca[w];
    sh4[3] = H.cb[w];
  }
  LineRecords RE, RH;
  RE.init(a.re);
  RH.init(a.rh);
  for (int r = RE.r0; r < RE.r1; ++r) {
    const int at = a.re.loc[a.re.of[r]];
    if (at > nz) ex[at] = a.ex[a.re.rec[a.re.seg[a.re.of[r]]].target];
  }
  for (int r = RH.r0; r < RH.r1; ++r) {
    const int at = a.rh.loc[a.rh.of[r]];
    if (at > nz) hy[at] = a.hy[a.rh.rec[a.rh.seg[a.rh.of[r]]].target];
  }
  for (int x = 0; x < a.extra_e; ++x)
#pragma unroll
    for (int c = 0; c < C; ++c)
      if (a.extra_cell[x] == tid + c * nth) ex1[c] = nz + 1 + x;
  const int p0 = a.probe_off ? a.probe_off[tid] : 0, p1 = a.probe_off ? a.probe_off[tid + 1] : 0;
  const T* probed = ex;  // the first probe's value and series
  double* out = nullptr;
  if (p0 < p1) {
    const int q = a.probe_of[p0];
    const Probe P = a.probe[q];
    probed = (P.field == 0 ? ex : hy) + P.idx;
    out = a.probe_out + q * a.probe_count;
  }
  // the first cell of each slab that this work-item owns
  int ke[2], kh[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    ke[q] = a.e[q].lo + (tid - a.e[q].lo % nth + nth) % nth;
    kh[q] = a.h[q].lo + (tid - a.h[q].lo % nth + nth) % nth;
  }
  auto slabs = [&](const LineSlab<T>* S, const int* k0, T* base, T* f, const T* d, int dk) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int lo = S[q].lo, hi = q < a.slabs ? lo + S[q].n : 0;
      for (int k = k0[q]; k < hi; k += nth) {
        T* v = base + 4 * ((q ? m0 : 0) + k - lo);
        const T diff = dk < 0 ? d[k] - d[k - 1] : d[k + 1] - d[k];
        const T psi = sumTwo(v[3], v[0], v[2], diff);
        v[0] = psi;
        f[k] = mulAdd(v[1], psi, f[k]);
      }
    }
  };
  __syncthreads();
  for (int step = 0; step < n; ++step) {
    const int64_t t = t0 + step;
    const int ahead = step % kLineAhead;
    if (ahead == 0 && a.re.held + a.rh.held > 0) {
      for (int x = tid; x < (a.re.held + a.rh.held) * kLineAhead; x += nth) {
        const bool is_e = x < a.re.held * kLineAhead;
        const int y = is_e ? x : x - a.re.held * kLineAhead;
        if (step + y % kLineAhead < n)
          add_e[x] = (is_e ? a.re : a.rh).addends[y / kLineAhead * kLineSteps + step + y % kLineAhead];
      }
      ldsBarrier();
    }
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int k = tid + c * nth;
      if (k < nz) {
        const T e0 = ex[k];
        hy[k] = mulAdd(bh[c], ex[k + 1] - e0, sh[c] * hy[k]);
        hz[c] = mulAdd(az[c], (ex1[c] < 0 ? T(0) : ex[ex1[c]]) - e0, sz[c] * hz[c]);
      }
    }
    if (RH.r0 < RH.r1) RH.apply(hy, a.rh, add_h + ahead, a.pool, a.state, t);
    slabs(a.h, kh, slab + 4 * cells, hy, ex, 1);
    ldsBarrier();
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int k = tid + c * nth;
      if (k >= 1 && k < nz) ex[k] = sumTwo(se[c], ex[k], ae[c], hy[k] - hy[k - 1]);
    }
    if (RE.r0 < RE.r1) RE.apply(ex, a.re, add_e + ahead, a.pool, a.state, t);
    slabs(a.e, ke, slab, ex, hy, -1);
    if (p0 < p1 && t < a.probe_count) {  // of this work-item's own cells
      out[t] = static_cast<double>(*probed);
      for (int p = p0 + 1; p < p1; ++p) {
        const int q = a.probe_of[p];
        const Probe P = a.probe[q];
        a.probe_out[q * a.probe_count + t] = static_cast<double>(P.field == 0 ? ex[P.idx] : hy[P.idx]);
      }
    }
    ldsBarrier();
  }
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int k = tid + c * nth;
    if (k <= nz) a.ex[k] = ex[k];
    if (k < nz) {
      a.hy[k] = hy[k];
      a.hz[k] = hz[c];
    }
  }
  for (int r = RE.r0; r < RE.r1; ++r) {
    const int at = a.re.loc[a.re.of[r]];
    if (at > nz) a.ex[a.re.rec[a.re.seg[a.re.of[r]]].target] = ex[at];
  }
  for (int r = RH.r0; r < RH.r1; ++r) {
    const int at = a.rh.loc[a.rh.of[r]];
    if (at > nz) a.hy[a.rh.rec[a.rh.seg[a.rh.of[r]]].target] = hy[at];
  }
  for (int q = tid; q < cells; q += nth) {
    const int w = q < m0 ? q : q - m0;
    a.e[q < m0 ? 0 : 1].psi[2 * w] = slab[4 * q];
    a.h[q < m0 ? 0 : 1].psi[2 * w] = slab[4 * (cells + q)];
  }
}

template <class T>
struct LineLaunch {
  static size_t ldsBytes(int nz, int extra, int slab_cells, int held) {
    return held * static_cast<size_t>(kLineAhead) * sizeof(double) +
           (2 * (static_cast<size_t>(nz) + 1) + extra + 8 * static_cast<size_t>(slab_cells)) * sizeof(T);
  }
  static void steps(hipStream_t s, const CoefPtrs<T>& C, const LineArgs<T>& a, int64_t t0, int64_t n);
  static void steps(hipStream_t s, const ClassCoef<T>& C, const LineArgs<T>& a, int64_t t0, int64_t n);
};

}  // namespace xfd
