// Per-wrapper kernels: the native launchers beneath the drop-in replacements
// of the reference's kbench/core/kernels/*.py wrappers (declarations and the
// reference function each replaces: include/kbench_ops.h).
//
// Design (MI355X):
//  * one workgroup per row (item row, clade row, split or split side), the
//    smallest of a list of shapes (64 to 1024 threads of 1 to 8 positions, powers
//    of two) that holds the row;
//    global row accesses are coalesced (column t + k * threads), and the kernels
//    that sum over the tree move the row to preorder positions in LDS, thread t
//    owning positions t*CPT + k;
//  * the species tree is described once by preorder positions (kb_tree);
//    ancestors-or-self path sums are a preorder scan less a postorder scan and
//    subtree sums differences of one preorder scan, in registers with one
//    exchange per scan, independent of the tree depth (but for estep_row_log,
//    which follows the parents);
//  * the E-step kernels (O(S) work) run in float64;
//  * no atomics: cross-row accumulations are written as rows and summed in a
//    fixed order by kb_rows_scatter_add / kb_rows_sum_into.
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>

#include <algorithm>
#include <cstdint>
#include <mutex>
#include <type_traits>
#include <vector>

#include "kb_ops_common.hpp"

namespace kbo {

// ---- E-step -------------------------------------------------------------------

template <typename T>
struct EsArgs {
  int G, S, mode, use_col, max_iter;
  double tol;
  const T *E, *pS, *pD, *pL, *mt, *col;
  T *E_out, *Es1, *Es2, *Ebar, *max_diff;
  int* n_iter;
};

// Largest value over a BT-thread workgroup; ends with a barrier (red: BT / 64).
template <int BT, typename V>
__device__ __forceinline__ V wg_max_of(V x, V* red) {
  x = wave_max(x);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
  __syncthreads();
  V m = red[0];
  for (int i = 1; i < BT / 64; ++i) m = tmax(m, red[i]);
  __syncthreads();
  return m;
}
template <int BT, typename V>
__device__ __forceinline__ V wg_sum_of(V x, V* red) {
  x = wave_sum(x);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
  __syncthreads();
  V m = red[0];
  for (int i = 1; i < BT / 64; ++i) m += red[i];
  __syncthreads();
  return m;
}

// One row of estep_kernel term by term in log space (column order, Ev and X:
// LDS rows), for values that linear float64 might not hold: the path sums by
// following the parents.
template <typename T, int BT, int CPT>
__device__ void estep_row_log(const OpsTree& t, const EsArgs<T>& a, size_t base, double* Ev, double* X, double* red) {
  const int S = t.S, tid = threadIdx.x;
  const double NI = -__builtin_inf();
  for (int s = tid; s < S; s += BT) Ev[s] = (double)a.E[base + s];
  __syncthreads();
  double M = NI;
  // X[s] = the others' sum of 2^(E + col - M); M the row's maximum
  auto others = [&]() {
    double lm = NI, ls = 0.0, den[CPT];
    for (int s = tid; s < S; s += BT) lm = fmax(lm, Ev[s] + (a.use_col ? (double)a.col[s] : 0.0));
    M = wg_max_of<BT>(lm, red);
    const double Ms = M == NI ? 0.0 : M;
    for (int s = tid; s < S; s += BT) {
      X[s] = exp2(Ev[s] + (a.use_col ? (double)a.col[s] : 0.0) - Ms);
      ls += X[s];
    }
    const double tot = wg_sum_of<BT>(ls, red);
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      den[k] = tot;
      const int s = tid + k * BT;
      if (s < S) {
        double ps = 0.0;
        for (int n = s; n >= 0; n = t.par[n]) ps += X[n];
        den[k] = tot - ps;
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < CPT; ++k)
      if (tid + k * BT < S) X[tid + k * BT] = den[k];
  };
  auto ebar_of = [&](int s) { return X[s] > 0.0 ? log2(X[s]) + M + (double)a.mt[base + s] : NI; };
  auto step_of = [&](int s) {
    const size_t i = base + s;
    const double E = Ev[s];
    const double t0 = (double)a.pS[i] + (t.c1[s] >= 0 ? Ev[t.c1[s]] : NI) + (t.c2[s] >= 0 ? Ev[t.c2[s]] : NI);
    const double t1 = (double)a.pD[i] + 2.0 * E;
    const double t2 = E + ebar_of(s);
    const double t3 = (double)a.pL[i];
    const double m = fmax(fmax(t0, t1), fmax(t2, t3));
    const double ms = m == NI ? 0.0 : m;
    return log2(exp2(t0 - ms) + exp2(t1 - ms) + exp2(t2 - ms) + exp2(t3 - ms)) + m;
  };
  auto child = [&](int c) { return c >= 0 ? Ev[c] : NI; };
  if (a.mode == 0) {
    others();
    double ld = 0.0;
#pragma unroll 1
    for (int s = tid; s < S; s += BT) {
      const T en = (T)step_of(s);
      a.E_out[base + s] = en;
      a.Es1[base + s] = (T)child(t.c1[s]);
      a.Es2[base + s] = (T)child(t.c2[s]);
      a.Ebar[base + s] = (T)ebar_of(s);
      const T d = en - (T)Ev[s];  // (E may have been E_out)
      ld = fmax(ld, (double)(d < T(0) ? -d : d));
    }
    const double md = wg_max_of<BT>(ld, red);
    if (a.max_diff && tid == 0) a.max_diff[blockIdx.x] = (T)md;
    return;
  }
  for (int it = 1;; ++it) {
    others();
    double ld = 0.0;
#pragma unroll 1
    for (int s = tid; s < S; s += BT) {
      const double en = step_of(s), d = en - Ev[s];
      if (!(fabs(d) < a.tol) && !(en == Ev[s])) ld = fmax(ld, d != d ? __builtin_inf() : fabs(d));
      X[s] = en;
    }
    const double md = wg_max_of<BT>(ld, red);
    for (int s = tid; s < S; s += BT) Ev[s] = X[s];
    __syncthreads();
    if (md < a.tol || it >= a.max_iter) {
      if (a.n_iter && tid == 0) a.n_iter[blockIdx.x] = it;
      break;
    }
  }
  others();
#pragma unroll 1
  for (int s = tid; s < S; s += BT) {
    a.E_out[base + s] = (T)Ev[s];
    a.Es1[base + s] = (T)child(t.c1[s]);
    a.Es2[base + s] = (T)child(t.c2[s]);
    a.Ebar[base + s] = (T)ebar_of(s);
  }
}

// One E step (mode 0) or the E fixed point (mode 1) of an item row, in linear
// float64 at preorder positions as kb_estep.hip's estep_pre_kernel: e = 2^E,
//   e' = 2^pS e[c1] e[c2] + 2^pD e^2 + e 2^mt (rowsum - ps) + 2^pL,
// path sums from an inclusive preorder and an exclusive postorder register
// scan, two barriers per step, and no exponential or logarithm inside the
// iteration.  Rows with a parameter or start outside [-400, 200] (log2) are
// evaluated in log space: a step multiplies up to four of these values, and what
// falls below the smallest double vanishes next to 2^pL.  A row whose iterates
// outgrow float64 (which then stay infinite or NaN) starts again there.
// Bound by one row's latency (two barriers and two scans a step).  100 rows of
// 1023 states: 16 iterations and one step 290 -> 39 us (against a 1024-thread
// workgroup summing by tree levels, with eight transcendentals an entry and
// iteration), one VJP 23 -> 12 us.
template <typename T, int BT, int CPT, bool WEIGHTED>
__global__ __launch_bounds__(BT) void estep_kernel(OpsTree t, EsArgs<T> a) {
  constexpr int MAXS = BT * CPT, BW = BT / 64, ZERO = MAXS, SEG = 64 * CPT;
  extern __shared__ __align__(16) unsigned char smraw[];
  double* X = reinterpret_cast<double*>(smraw);  // e at preorder positions
  double* Q = X + MAXS + 64;                     // wavefront-local exclusive postorder scan
  __shared__ double wP[BW], wQ[BW], red[BW];
  __shared__ int wok[BW];
  const int S = t.S;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const size_t base = (size_t)blockIdx.x * S;
  const double NI = -__builtin_inf();
  int colk[CPT], c2p[CPT], nex[CPT], qp[CPT];
  bool h1[CPT], linear = true;
  double e[CPT], kS[CPT], kD[CPT], kL[CPT], kM[CPT], w[WEIGHTED ? CPT : 1], wq[WEIGHTED ? CPT : 1];
  auto in_range = [&](double x) { linear = linear && x >= -400.0 && x <= 200.0; };
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const int i = tid * CPT + k;
    colk[k] = -1;
    c2p[k] = qp[k] = ZERO;
    nex[k] = 0;
    h1[k] = false;
    e[k] = kS[k] = kD[k] = kL[k] = kM[k] = 0.0;
    if constexpr (WEIGHTED) w[k] = wq[k] = 0.0;
    if (i < S) {
      const int s = colk[k] = t.pcol[i];
      const int c2 = t.pc2[i];
      c2p[k] = c2 >= 0 ? c2 : ZERO;
      h1[k] = t.pc1[i] >= 0;  // child1 of i is i + 1
      nex[k] = t.pnex[i];
      qp[k] = t.ppost[i];
      const double E = a.E[base + s], ps = a.pS[base + s], pd = a.pD[base + s], pl = a.pL[base + s], mt = a.mt[base + s];
      in_range(E);
      in_range(ps);
      in_range(pd);
      in_range(pl);
      in_range(mt);
      e[k] = exp2(E);
      // (a missing child is the probability 0)
      kS[k] = h1[k] && c2 >= 0 ? exp2(ps) : 0.0;
      kD[k] = exp2(pd);
      kL[k] = exp2(pl);
      kM[k] = exp2(mt);
      if constexpr (WEIGHTED) {
        const double c = a.col[s];
        in_range(c);
        w[k] = exp2(c);
        wq[k] = exp2((double)a.col[t.pcol[qp[k]]]);
      }
    }
  }
  if (tid < 64) X[MAXS + tid] = Q[MAXS + tid] = 0.0;
  linear = __syncthreads_and(linear);
  const double hi = exp2(a.tol), lo = exp2(-a.tol);
  bool ok = true;  // the last update moved the own positions by less than tol
  double e1[CPT], e2[CPT], ps[CPT], tot = 0.0;
  int it = 0;
  if (linear) for (;;) {
    double sp[CPT], ta = 0.0;
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      ta += WEIGHTED ? w[WEIGHTED ? k : 0] * e[k] : e[k];
      sp[k] = ta;
    }
    const double wa = wscan(ta);
    own_store<CPT>(X, e);
    const bool wave_ok = __ballot(!ok) == 0;
    if (lane == 63) {
      wP[wv] = wa;
      wok[wv] = wave_ok ? 1 : 0;
    }
    __syncthreads();
    const int fl = kb::lds_wave_values<BW>(wok, lane, 1);
    const bool stop = it > 0 && (a.mode == 0 || __ballot(fl == 0) == 0 || it >= a.max_iter);
    const double tp = kb::lds_wave_values<BW>(wP, lane, 0.0);
    double yq[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      yq[k] = X[qp[k]];
      if constexpr (WEIGHTED) yq[k] *= wq[k];
      e2[k] = X[c2p[k]];
    }
    const double e1last = X[tid * CPT + CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) e1[k] = k + 1 < CPT ? e[k + 1 < CPT ? k + 1 : k] : e1last;
    const double ip = wscan_first<BW>(tp);
    tot = lane_of(ip, BW - 1);
    const double offp = lane_of(ip - tp, wv) + (wa - ta);
    double sq[CPT], tb = 0.0;
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      sq[k] = tb;
      tb += yq[k];
    }
    const double wb = wscan(tb);
#pragma unroll
    for (int k = 0; k < CPT; ++k) sq[k] += wb - tb;
    own_store<CPT>(Q, sq);
    if (lane == 63) wQ[wv] = wb;
    __syncthreads();
    const double tq = kb::lds_wave_values<BW>(wQ, lane, 0.0);
    const double eq = wscan_first<BW>(tq) - tq;
#pragma unroll
    for (int k = 0; k < CPT; ++k) ps[k] = (sp[k] + offp) - (Q[nex[k]] + (BW > 1 ? shfl_of(eq, nex[k] / SEG) : 0.0));
    // (mode 0 stops after one step; its outputs are those of the point before it)
    if (stop) break;
    if (a.mode == 0) {
      double ld = 0.0;
      // E itself for the children (X's readers have passed a barrier); all of it is
      // read before any of E_out, which may be E, is written
      double E0[CPT];
#pragma unroll
      for (int k = 0; k < CPT; ++k) E0[k] = colk[k] >= 0 ? (double)a.E[base + colk[k]] : NI;
      own_store<CPT>(X, E0);
      __syncthreads();
      const double E1last = X[tid * CPT + CPT];
#pragma unroll
      for (int k = 0; k < CPT; ++k)
        if (colk[k] >= 0) {
          const size_t o = base + colk[k];
          const double na = tot - ps[k];
          const double en = kS[k] * e1[k] * e2[k] + kD[k] * e[k] * e[k] + (na > 0.0 ? e[k] * kM[k] * na : 0.0) + kL[k];
          const T En = (T)log2(en);
          a.E_out[o] = En;
          a.Ebar[o] = (T)(na > 0.0 ? log2(na) + (double)a.mt[o] : NI);
          a.Es1[o] = (T)(h1[k] ? (k + 1 < CPT ? E0[k + 1 < CPT ? k + 1 : k] : E1last) : NI);
          a.Es2[o] = (T)(c2p[k] != ZERO ? X[c2p[k]] : NI);
          const T d = En - (T)E0[k];
          ld = fmax(ld, (double)(d < T(0) ? -d : d));
        }
      if (a.max_diff) {
        const double md = wg_max_of<BT>(ld, red);
        if (tid == 0) a.max_diff[blockIdx.x] = (T)md;
      }
      return;
    }
    ok = true;
#pragma unroll
    for (int k = 0; k < CPT; ++k)
      if (colk[k] >= 0) {
        const double na = tot - ps[k];
        const double eb = na > 0.0 ? kM[k] * na : 0.0;
        const double en = kS[k] * e1[k] * e2[k] + kD[k] * e[k] * e[k] + e[k] * eb + kL[k];
        // |log2(en / e)| < tol without a logarithm (e > 0)
        if (!(en < e[k] * hi && en > e[k] * lo) && en != e[k]) ok = false;
        e[k] = en;
      }
    ++it;
  }
  // (the total of every thread; no weight is 0, so one infinite or NaN e makes it so)
  if (!(linear && tot < __builtin_inf())) {
    estep_row_log<T, BT, CPT>(t, a, base, X, Q, red);
    return;
  }
#pragma unroll
  for (int k = 0; k < CPT; ++k)
    if (colk[k] >= 0) {
      const size_t o = base + colk[k];
      const double na = tot - ps[k];
      a.E_out[o] = (T)log2(e[k]);
      a.Es1[o] = (T)(h1[k] ? log2(e1[k]) : NI);
      a.Es2[o] = (T)(c2p[k] != ZERO ? log2(e2[k]) : NI);
      a.Ebar[o] = (T)(na > 0.0 ? log2(na) + (double)a.mt[o] : NI);
    }
  if (a.n_iter && tid == 0) a.n_iter[blockIdx.x] = it;
}

template <typename T>
struct EvArgs {
  int G, S, use_col;
  const T *E, *En, *Es1, *Es2, *Ebar, *pS, *pD, *pL, *col, *gN, *g1, *g2, *gB;
  T *gE, *gpS, *gpD, *gpL, *gmt;
  double* work;  // [G, S] per-row contribution to grad_col
};

// VJP of one E step of an item row, float64 at preorder positions: the path
// sums as in estep_kernel, the subtree sums of u from one preorder scan, and
// each parent hands its children their terms through LDS.
template <typename T, int BT, int CPT>
__global__ __launch_bounds__(BT) void estep_vjp_kernel(OpsTree t, EvArgs<T> a) {
  constexpr int MAXS = BT * CPT, BW = BT / 64, ZERO = MAXS, SEG = 64 * CPT;
  extern __shared__ __align__(16) unsigned char smraw[];
  double* X = reinterpret_cast<double*>(smraw);  // r, then what each position gets from its parent
  double* Q = X + MAXS + 64;                     // postorder scan, then the preorder scan of u
  __shared__ double wP[BW], wQ[BW], red[BW];
  const int S = t.S;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const size_t base = (size_t)blockIdx.x * S;
  const double NI = -__builtin_inf();
  int colk[CPT], c2p[CPT], nex[CPT], qp[CPT], endm1[CPT];
  bool h1[CPT];
  double r[CPT], lm = NI;
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const int i = tid * CPT + k;
    colk[k] = -1;
    c2p[k] = qp[k] = endm1[k] = ZERO;
    nex[k] = 0;
    h1[k] = false;
    r[k] = NI;
    if (i < S) {
      const int s = colk[k] = t.pcol[i];
      const int c2 = t.pc2[i];
      c2p[k] = c2 >= 0 ? c2 : ZERO;
      h1[k] = t.pc1[i] >= 0;
      nex[k] = t.pnex[i];
      qp[k] = t.ppost[i];
      endm1[k] = t.pend[s] - 1;
      r[k] = (double)a.E[base + s] + (a.use_col ? (double)a.col[s] : 0.0);
      lm = fmax(lm, r[k]);
    }
  }
  if (tid < 64) X[MAXS + tid] = Q[MAXS + tid] = 0.0;
  const double M = wg_max_of<BT>(lm, red);
  const double Ms = M == NI ? 0.0 : M;
  // path sums of r
  double sp[CPT], ta = 0.0;
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    r[k] = colk[k] >= 0 ? exp2(r[k] - Ms) : 0.0;
    ta += r[k];
    sp[k] = ta;
  }
  const double wa = wscan(ta);
  own_store<CPT>(X, r);
  if (lane == 63) wP[wv] = wa;
  __syncthreads();
  const double tp = kb::lds_wave_values<BW>(wP, lane, 0.0);
  const double ip = wscan_first<BW>(tp);
  const double rowsum = lane_of(ip, BW - 1);
  const double offp = lane_of(ip - tp, wv) + (wa - ta);
  double sq[CPT], tb = 0.0;
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    sq[k] = tb;
    tb += X[qp[k]];
  }
  const double wb = wscan(tb);
#pragma unroll
  for (int k = 0; k < CPT; ++k) sq[k] += wb - tb;
  own_store<CPT>(Q, sq);
  if (lane == 63) wQ[wv] = wb;
  __syncthreads();
  const double tq = kb::lds_wave_values<BW>(wQ, lane, 0.0);
  const double eq = wscan_first<BW>(tq) - tq;
  double ge[CPT], u[CPT], tu = 0.0;
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    ge[k] = u[k] = 0.0;
    const double off = BW > 1 ? shfl_of(eq, nex[k] / SEG) : 0.0;
    if (colk[k] >= 0) {
      const size_t i = base + colk[k];
      const double En = a.En[i], E = a.E[i];
      const double gN = a.gN[i];
      const double t0 = (double)a.pS[i] + (double)a.Es1[i] + (double)a.Es2[i];
      const double t1 = (double)a.pD[i] + 2.0 * E;
      const double t2 = E + (double)a.Ebar[i];
      const double t3 = (double)a.pL[i];
      const double q0 = gN * exp2(t0 - En), q1 = gN * exp2(t1 - En);
      const double q2 = gN * exp2(t2 - En), q3 = gN * exp2(t3 - En);
      const double wbar = q2 + (double)a.gB[i];
      a.gpS[i] = (T)q0;
      a.gpD[i] = (T)q1;
      a.gpL[i] = (T)q3;
      a.gmt[i] = (T)wbar;
      ge[k] = 2.0 * q1 + q2;
      if (h1[k]) X[tid * CPT + k + 1] = q0 + (double)a.g1[i];
      if (c2p[k] != ZERO) X[c2p[k]] = q0 + (double)a.g2[i];
      const double denom = rowsum - ((sp[k] + offp) - (Q[nex[k]] + off));
      u[k] = denom > 0.0 ? wbar / denom : 0.0;
    }
    tu += u[k];
    sp[k] = tu;
  }
  const double wu = wscan(tu);
#pragma unroll
  for (int k = 0; k < CPT; ++k) sp[k] += wu - tu;  // wavefront-local inclusive scan of u
  __syncthreads();  // Q was read
  own_store<CPT>(Q, sp);
  if (lane == 63) wP[wv] = wu;
  __syncthreads();
  const double tv = kb::lds_wave_values<BW>(wP, lane, 0.0);
  const double iv = wscan_first<BW>(tv);
  const double ev = iv - tv;
  const double total = lane_of(iv, BW - 1), offv = lane_of(ev, wv);
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const double oe = BW > 1 ? shfl_of(ev, min(endm1[k], MAXS - 1) / SEG) : 0.0;
    if (colk[k] >= 0) {
      const int i = tid * CPT + k;
      const double before = (sp[k] + offv) - u[k];
      const double pv = r[k] * (before + (total - (Q[endm1[k]] + oe)));
      a.gE[base + colk[k]] = (T)(ge[k] + (i > 0 ? X[i] : 0.0) + pv);
      a.work[base + colk[k]] = pv;
    }
  }
}

// ---- wave rows ------------------------------------------------------------------

template <typename T>
struct WsArgs {
  int S, W, use_col, use_leaf, store_final, n_sweeps;
  long long ws, pi_ws, cstride;
  const T* Pi_in;
  T *Pi_out, *Pibar, *rowmax;
  float* resid;
  const T *dts, *mt, *DL, *Ebar, *E, *SL1, *SL2, *col;
  const int64_t *item, *leaf_state;
  const T* leaf_logp;
};

// hardware exponential and logarithm for float (arguments that keep clear of
// denormals, or whose denormal results vanish next to the sums they enter)
__device__ __forceinline__ float fexp2(float x) { return kb::exp2_hw(x); }
__device__ __forceinline__ double fexp2(double x) { return exp2(x); }
__device__ __forceinline__ float flog2(float x) { return kb::log2_hw(x); }
__device__ __forceinline__ double flog2(double x) { return log2(x); }

// z = mantissa * 2^exponent, mantissa in [1/2, 1)
__device__ __forceinline__ float mantissa(float z) { return __builtin_amdgcn_frexp_mantf(z); }
__device__ __forceinline__ double mantissa(double z) { return __builtin_amdgcn_frexp_mant(z); }
__device__ __forceinline__ int exponent(float z) { return __builtin_amdgcn_frexp_expf(z); }
__device__ __forceinline__ int exponent(double z) { return __builtin_amdgcn_frexp_exp(z); }
__device__ __forceinline__ float xceil(float x) { return ceilf(x); }
__device__ __forceinline__ double xceil(double x) { return ceil(x); }

// float rows of two positions per thread: six wavefronts per SIMD (at most 80
// VGPRs; eight spill, and the spills cost more than the wavefronts give)
template <typename T>
constexpr int step_min_waves(int cpt) { return std::is_same_v<T, float> && cpt == 2 ? 6 : 1; }

// see wave_step_kernel: four rows of constants in LDS
template <typename T>
__host__ __device__ constexpr bool step_consts_in_lds(int maxs) { return 4 * maxs * (int)sizeof(T) <= 64 * 1024; }

// One sweep of rows [ws, ws + W) (float64: n_sweeps of them), one workgroup
// per row in flight.  Threads own preorder positions: the path sums are an
// inclusive preorder scan minus an exclusive postorder scan, both in registers
// (two barriers), and the row passes through LDS once each way between column
// and preorder order.
//
// A sweep is evaluated in linear space relative to the row's largest entry,
// 2^-M y' = a x + emc (rowsum - ps) + k1 x[c1] + k2 x[c2] + (leaf + dts) 2^-M,
// so an entry takes one exponential per input and one logarithm instead of
// seven and two.  The smallest product that a sum may consist of is the row's
// smallest entry times the smallest constant (for the transfer term, times the
// smallest weight): a row is swept in linear space where that lies at most RANGE
// binary orders below its largest entry, a few above the smallest normal number.
// Any other row, and one with a NaN or +inf, is evaluated term by term in log
// space, where nothing underflows: both forms in one kernel, chosen per row.
//
// A workgroup walks its rows with the position tables in registers and the linear
// constants in LDS (step_consts_in_lds; else in registers), formed again when the
// item changes.  A row is loaded when it begins: its latency is hidden by the
// other rows of the CU.  Measured: see launch_wave_step.
template <typename T, int BT, int CPT, bool WEIGHTED>
__global__ __launch_bounds__(BT, step_min_waves<T>(CPT)) void wave_step_kernel(OpsTree t, WsArgs<T> a) {
  constexpr int MAXS = BT * CPT, BW = BT / 64, ZERO = MAXS, SEG = 64 * CPT, LD = MAXS + 64;
  constexpr int NONE = 0xffff;
  constexpr bool CHAINS = !std::is_same_v<T, float>;  // (float chains: wave_step_lin_kernel)
  // the constants are formed only for a row whose span leaves room for them (inside
  // the loop of a chain that would cost registers: doubles 84 -> 116 us a sweep)
  constexpr bool LAZY = !CHAINS;
  constexpr T RANGE = std::is_same_v<T, float> ? T(120) : T(1000);
  constexpr T HIGH = std::is_same_v<T, float> ? T(60) : T(400);  // the largest constant (log2)
  extern __shared__ __align__(16) unsigned char smraw[];
  T* X = reinterpret_cast<T*>(smraw);  // the row's values at preorder positions; [ZERO] stays 0
  T* Q = X + LD;                       // the split term, then the postorder scan
  // the linear constants of the own positions: in LDS where they fit in 64 KB,
  // which leaves registers for more rows per CU
  constexpr bool KC = step_consts_in_lds<T>(MAXS);
  T* Kc = Q + LD;
  __shared__ T wP[BW], wQ[BW], wA[BW], wB[BW];
  const int S = t.S;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const T NI = ninf<T>();
  // Tables of the own positions i = tid*CPT + k, two 16-bit entries a word:
  // child2's position and the position at postorder slot i (ZERO: none);
  // tin(i) - i and the preorder position of column tid + k*BT (NONE: past the
  // row).  Child1 of i is i + 1.
  unsigned cq[CPT], np[CPT];
  auto load_tables = [&]() {
    int c2[CPT], q[CPT], nex[CPT];
    kb::gld_own<CPT>(t.pc2, S, c2, -1);
    kb::gld_own<CPT>(t.ppost, S, q, ZERO);
    kb::gld_own<CPT>(t.pnex, S, nex, 0);
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      cq[k] = (unsigned)(c2[k] >= 0 ? c2[k] : ZERO) | ((unsigned)q[k] << 16);
      const int sc = tid + k * BT;
      np[k] = (unsigned)nex[k] | ((unsigned)(sc < S ? t.ppos[sc] : NONE) << 16);
    }
  };
  load_tables();
  auto own = [&](int k) { return kb::own_pos_c<BT, CPT>(k); };
  if (tid < 64) {
    X[MAXS + tid] = T(0);
    Q[MAXS + tid] = T(0);
  }
  // the largest value over the workgroup (two barriers)
  auto wg_max = [&](T x) {
    x = wmax63(x);
    __syncthreads();
    if (lane == 63) wA[wv] = x;
    __syncthreads();
    return wmax_first<BW>(wA, lane);
  };
  // Binary orders by which a factor 2^lg may lower what it multiplies, at least
  // 0; +inf if it is NaN or larger than HIGH.
  auto depth = [&](T lg) { return lg == NI ? T(0) : lg <= HIGH ? tmax(-lg, T(0)) : -NI; };
  T cw[WEIGHTED ? CPT : 1], cwq[WEIGHTED ? CPT : 1];
  T wdepth = T(0), whigh = T(0);  // of the weights: the largest depth, the largest log2 above 0
  if constexpr (WEIGHTED) {
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      cw[k] = cwq[k] = T(0);
      if (own(k) < S) {
        const T c = a.col[t.pcol[own(k)]];
        wdepth = tmax(wdepth, depth(c));
        whigh = tmax(whigh, c);
        cw[k] = xexp2(c);
        cwq[k] = xexp2(a.col[t.pcol[cq[k] >> 16]]);
      }
    }
    wdepth = wg_max(wdepth);
    whigh = wg_max(tmax(whigh, T(0)));
  }
  T kr[4][KC ? 1 : CPT];
  // The constants at cb, read in column order (coalesced) and moved to the own
  // positions through LDS (X and Q free); returns the largest depth of their
  // products.  Against reads at preorder positions: one item 35 -> 31 us a sweep
  // (2140 rows of 2047 floats), another item with every row 62 -> 41 us (650 of
  // 8191 191 -> 134 us).
  if constexpr (KC) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      for (int i = S + tid; i < MAXS; i += BT) Kc[j * MAXS + i] = T(0);
  }
  auto load_consts = [&](size_t cb) {
    T deep = wdepth;
    T ca[CPT], ce[CPT], ck1[CPT], ck2[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int sc = tid + k * BT;
      ca[k] = ce[k] = ck1[k] = ck2[k] = T(0);
      if (sc < S) {
        const size_t ci = cb + sc;
        const T dl = a.DL[ci], eb = a.Ebar[ci], em = a.E[ci] + a.mt[ci], s1 = a.SL1[ci], s2 = a.SL2[ci];
        ca[k] = xexp2(dl) + xexp2(eb);
        ce[k] = xexp2(em);
        // (of the sum dl and eb the larger one counts; dl > eb fails for a NaN)
        deep = tmax(deep, dl != dl ? -NI : depth(dl > eb ? dl : eb));
        deep = tmax(deep, em + whigh <= HIGH ? depth(em) + (em == NI ? T(0) : wdepth) : -NI);
        if (t.c1[sc] >= 0) {
          ck1[k] = xexp2(s1);
          deep = tmax(deep, depth(s1));
        }
        if (t.c2[sc] >= 0) {
          ck2[k] = xexp2(s2);
          deep = tmax(deep, depth(s2));
        }
      }
    }
    auto put = [&](T* dst, const T (&v)[CPT]) {
#pragma unroll
      for (int k = 0; k < CPT; ++k)
        if (tid + k * BT < S) dst[np[k] >> 16] = v[k];
    };
    if constexpr (KC) {
      put(Kc, ca);
      put(Kc + MAXS, ce);
      put(Kc + 2 * MAXS, ck1);
      put(Kc + 3 * MAXS, ck2);
    } else {
      auto get = [&](const T* src, T (&v)[CPT]) {
        own_load<CPT>(src, v);
#pragma unroll
        for (int k = 0; k < CPT; ++k)
          if (own(k) >= S) v[k] = T(0);
      };
      __syncthreads();  // the row was read from X and Q
      put(X, ca);
      put(Q, ce);
      __syncthreads();
      get(X, kr[0]);
      get(Q, kr[1]);
      __syncthreads();
      put(X, ck1);
      put(Q, ck2);
      __syncthreads();
      get(X, kr[2]);
      get(Q, kr[3]);
    }
    return wg_max(deep);  // (its barriers: Kc is written, X and Q are free)
  };
  auto konst = [&](int j, T (&v)[CPT]) {
    if constexpr (KC) {
      own_load<CPT>(Kc + j * MAXS, v);
    } else {
#pragma unroll
      for (int k = 0; k < CPT; ++k) v[k] = kr[j][k];
    }
  };
  // Publishes v (own positions; with WGT its sums are column-weighted) and
  // returns the ancestors-or-self sums and the total; with WGT or an unweighted
  // sweep (KIDS) also the children's values.
  auto path_sums = [&](auto wgt_, auto kids_, const T (&v)[CPT], T (&ps)[CPT], T& total, T (&x2)[CPT], T& x1last) {
    constexpr bool WGT = decltype(wgt_)::value && WEIGHTED, KIDS = decltype(kids_)::value;
    T sp[CPT], ta = T(0);
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      ta += WGT ? cw[WGT ? k : 0] * v[k] : v[k];
      sp[k] = ta;
    }
    const T wa = wscan(ta);
    own_store<CPT>(X, v);
    if (lane == 63) wP[wv] = wa;
    __syncthreads();
    const T tp = kb::lds_wave_values<BW>(wP, lane, T(0));
    T yq[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      yq[k] = X[cq[k] >> 16];
      if constexpr (KIDS) x2[k] = X[cq[k] & 0xffff];
    }
    if constexpr (KIDS) x1last = X[tid * CPT + CPT];
    const T ip = wscan_first<BW>(tp);
    total = lane_of(ip, BW - 1);
    const T offp = lane_of(ip - tp, wv) + (wa - ta);
    T sq[CPT], tb = T(0);
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      sq[k] = tb;
      tb += WGT ? cwq[WGT ? k : 0] * yq[k] : yq[k];
    }
    const T wb = wscan(tb);
#pragma unroll
    for (int k = 0; k < CPT; ++k) sq[k] += wb - tb;
    own_store<CPT>(Q, sq);
    if (lane == 63) wQ[wv] = wb;
    __syncthreads();
    const T tq = kb::lds_wave_values<BW>(wQ, lane, T(0));
    const T eq = wscan_first<BW>(tq) - tq;
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int n = np[k] & 0xffff;
      ps[k] = (sp[k] + offp) - (Q[n] + (BW > 1 ? shfl_of(eq, n / SEG) : T(0)));
    }
  };
  long long citem = -1;
  T deep = T(0);
  for (int w = blockIdx.x; w < a.W; w += gridDim.x) {
    // (opaque in every row: the LDS addresses formed from the packed tables
    // would otherwise be kept in registers through the loop)
#pragma unroll
    for (int k = 0; k < CPT; ++k) asm("" : "+v"(cq[k]), "+v"(np[k]));
    const long long grow = a.ws + w;
    const long long item = a.item[grow];
    const size_t cb = (size_t)(item * a.cstride);
    const T* in = a.Pi_in + (size_t)(a.pi_ws + w) * S;
    const T* dt = a.dts ? a.dts + (size_t)w * S : nullptr;
    T vin[CPT], vdt[CPT];  // columns tid + j*BT
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      const int sc = tid + j * BT;
      vin[j] = sc < S ? kb::ldg(in, sc) : NI;
      vdt[j] = dt && sc < S ? kb::ldg(dt, sc) : NI;
    }
    if constexpr (!LAZY) {
      if (citem < 0 || (a.cstride != 0 && item != citem)) deep = load_consts(cb);
      citem = item;
    }
    const long long lstate = a.use_leaf ? a.leaf_state[grow] : -1;
    const bool has_leaf = lstate >= 0 && lstate < S;
    const int lpos = has_leaf ? t.ppos[lstate] : -1;
    const T lval = has_leaf ? a.leaf_logp[(size_t)item * S + lstate] : NI;
    T* out = a.Pi_out + (size_t)grow * S;
    // Largest and (negated) smallest finite input.  tmax may drop a NaN but never
    // a +inf: a NaN is kept as +inf in lo, a +inf in hi.
    T hi = NI, lo = NI;
    auto span = [&](T x) {
      hi = tmax(hi, x);
      lo = tmax(lo, x == NI ? NI : x == x ? -x : -NI);
    };
    auto publish_span = [&]() {
      span(lval);
      hi = wmax63(hi);
      lo = wmax63(lo);
      if (lane == 63) {
        wA[wv] = hi;
        wB[wv] = lo;
      }
      __syncthreads();
      hi = wmax_first<BW>(wA, lane);
      lo = wmax_first<BW>(wB, lane);
    };
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      span(vin[j]);
      span(vdt[j]);
      const unsigned i = np[j] >> 16;
      if (i != NONE) {
        X[i] = vin[j];
        Q[i] = vdt[j];
      }
    }
    publish_span();
    T pr[CPT], dd[CPT], res[CPT];
    own_load<CPT>(X, pr);
    own_load<CPT>(Q, dd);
#pragma unroll
    for (int k = 0; k < CPT; ++k)
      if (own(k) >= S) pr[k] = dd[k] = NI;
    for (int sweep = 0;; ++sweep) {
      if constexpr (LAZY) {
        if (hi + lo <= RANGE && (citem < 0 || (a.cstride != 0 && item != citem))) {
          deep = load_consts(cb);
          citem = item;
        }
      }
      // (-inf for a row of -inf; +inf or NaN, which fail the test, for a row or
      // constants with a NaN or +inf)
      if (hi + lo <= RANGE && hi + lo + deep <= RANGE) {
        // an integer reference: Pi - Ms and the exponent of the result are exact,
        // and the result is rounded once
        const T Ms = xceil(msafe(hi));
        T x[CPT], x2[CPT], ps[CPT], tot, x1last;
#pragma unroll
        for (int k = 0; k < CPT; ++k) x[k] = fexp2(pr[k] - Ms);  // 0 at padding positions
        path_sums(std::true_type{}, std::true_type{}, x, ps, tot, x2, x1last);
        T ca[CPT], ce[CPT], ck1[CPT], ck2[CPT];
        konst(0, ca);
        konst(1, ce);
        konst(2, ck1);
        konst(3, ck2);
#pragma unroll
        for (int k = 0; k < CPT; ++k) {
          T z = ca[k] * x[k];
          z += ck1[k] * (k + 1 < CPT ? x[k + 1 < CPT ? k + 1 : k] : x1last);
          z += ck2[k] * x2[k];
          z += ce[k] * tmax(tot - ps[k], T(0));
          z += fexp2(dd[k] - Ms);
          if (own(k) == lpos) z += fexp2(lval - Ms);
          // (0 at padding positions)
          res[k] = z > T(0) ? flog2(mantissa(z)) + (Ms + (T)exponent(z)) : NI;
        }
      } else {
        // Term by term in log space: the others' sums from the same scans over
        // 2^(col + Pi - M).  Then they go to Q and Pi to X in column order, so that
        // the entries are evaluated with coalesced reads of the constants, each
        // result in the place of its sum in Q.  Rows of this kind only, against
        // sums by following the parents entry by entry and reads at preorder
        // positions: 2140 rows of 2047 floats over 200 orders 226 -> 46 us, 650 of
        // 8191 543 -> 115 us, 600 of 2047 on a tree of depth 1023 981 -> 20 us.
        {
          T lm = NI, x[CPT], x2[CPT], ps[CPT], tot, x1last;
#pragma unroll
          for (int k = 0; k < CPT; ++k) {
            x[k] = WEIGHTED && own(k) < S ? a.col[t.pcol[own(k)]] + pr[k] : pr[k];
            lm = tmax(lm, x[k]);
          }
          const T M = wg_max(lm);
          const T Mw = msafe(M);
#pragma unroll
          for (int k = 0; k < CPT; ++k) x[k] = own(k) < S ? xexp2(x[k] - Mw) : T(0);
          path_sums(std::false_type{}, std::false_type{}, x, ps, tot, x2, x1last);
          __syncthreads();  // X and Q were read
#pragma unroll
          for (int k = 0; k < CPT; ++k) {
            ps[k] = tot - ps[k];
            if (own(k) < S) X[t.pcol[own(k)]] = pr[k];
          }
          own_store<CPT>(Q, ps);
          __syncthreads();
#pragma unroll 1
          for (int sc = tid; sc < S; sc += BT) {
            const size_t ci = cb + sc;
            const int i = t.ppos[sc], c1 = t.c1[sc], c2 = t.c2[sc];
            const T denom = Q[i], p = X[sc];
            const T d = a.dts ? a.dts[(size_t)w * S + sc] : NI;
            const T pibar = denom > T(0) ? xlog2(denom) + M + a.mt[ci] : NI;
            const T t0 = a.DL[ci] + p;
            const T t1 = p + a.Ebar[ci];
            const T t2 = pibar + a.E[ci];
            const T t3 = a.SL1[ci] + (c1 >= 0 ? X[c1] : NI);
            const T t4 = a.SL2[ci] + (c2 >= 0 ? X[c2] : NI);
            const T t5 = i == lpos ? lval : NI;
            const T m = tmax(tmax(tmax(tmax(t0, t1), tmax(t2, t3)), tmax(t4, t5)), d);
            const T ms = msafe(m);
            T sum = xexp2(t0 - ms) + xexp2(t1 - ms) + xexp2(t2 - ms) + xexp2(t3 - ms) + xexp2(t4 - ms) + xexp2(t5 - ms);
            if (a.dts) sum += xexp2(d - ms);
            Q[i] = xlog2(sum) + m;
          }
          __syncthreads();
          own_load<CPT>(Q, res);
#pragma unroll
          for (int k = 0; k < CPT; ++k)
            if (own(k) >= S) res[k] = NI;
        }
        // (where registers are short the tables are read again, so that this branch
        // does not hold them)
        if constexpr (step_min_waves<T>(CPT) > 1 || CPT == 8) load_tables();
      }
      if (a.resid && sweep + 1 >= a.n_sweeps) {
        T ldiff = T(0);
        bool nan = false;
#pragma unroll
        for (int k = 0; k < CPT; ++k)
          if (res[k] != NI && pr[k] != NI) {
            const T df = res[k] - pr[k];
            nan = nan || df != df;
            ldiff = df == df ? tmax(ldiff, df < T(0) ? -df : df) : ldiff;
          }
        ldiff = wg_max(ldiff);
        if (__syncthreads_or(nan)) ldiff = __builtin_nanf("");
        if (tid == 0) a.resid[grow] = (float)ldiff;
      }
      if (!CHAINS || sweep + 1 >= a.n_sweeps) break;
      hi = lo = NI;
#pragma unroll
      for (int k = 0; k < CPT; ++k) {
        pr[k] = res[k];
        span(pr[k]);
        span(dd[k]);
      }
      publish_span();
    }
    if (a.store_final) {
      T lm = NI, x[CPT], x2[CPT], ps[CPT], tot, x1last;
#pragma unroll
      for (int k = 0; k < CPT; ++k) {
        x[k] = WEIGHTED && own(k) < S ? a.col[t.pcol[own(k)]] + res[k] : res[k];
        lm = tmax(lm, x[k]);
      }
      const T M = wg_max(lm);  // (its barriers: every earlier read of X and Q is done)
      const T Mw = msafe(M);
#pragma unroll
      for (int k = 0; k < CPT; ++k) x[k] = own(k) < S ? fexp2(x[k] - Mw) : T(0);
      path_sums(std::false_type{}, std::false_type{}, x, ps, tot, x2, x1last);
      __syncthreads();  // Q is written again
#pragma unroll
      for (int k = 0; k < CPT; ++k) {
        const T denom = tot - ps[k];
        x[k] = own(k) < S && denom > T(0) ? flog2(denom) + M + a.mt[cb + t.pcol[own(k)]] : NI;
      }
      own_store<CPT>(Q, x);
      if (tid == 0) a.rowmax[grow] = M;
    }
    own_store<CPT>(X, res);
    __syncthreads();
    T* pbo = a.store_final ? a.Pibar + (size_t)grow * S : nullptr;
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      const unsigned i = np[j] >> 16;
      if (i != NONE) {
        const int sc = tid + j * BT;
        kb::stg(out, sc, X[i]);
        if (pbo) kb::stg(pbo, sc, Q[i]);
      }
    }
    __syncthreads();  // X and Q are free for the next row
  }
}

// Sweep chains (n_sweeps > 1) of float32 rows in linear space, as the
// whole-pass forward row kernel runs its sweeps: x = 2^(Pi - M) with a row
// exponent M renormalised by an exact power of two every sweep, so a sweep is
//   y' = a y + emc (rowsum - ps) + k1 y[c1] + k2 y[c2] + (leaf | dts) 2^-M
// with a = 2^DL + 2^Ebar, emc = 2^(E + mt), k1 = 2^SL1, k2 = 2^SL2 formed
// once per launch, and no exponential or logarithm inside the chain.  The
// path sums come from an inclusive preorder scan and an exclusive postorder
// scan (two barriers per sweep).  The outputs equal the log-space sweeps to
// float32 rounding.
template <int CPT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(kb::pre_waves_per_eu(CPT)))) void wave_step_lin_kernel(OpsTree t, WsArgs<float> a) {
  constexpr int MAXS = NT * CPT;
  constexpr int LD = MAXS + 64;
  constexpr int ZERO = MAXS;     // padding slot: 0 in X
  constexpr int SEG = 64 * CPT;  // postorder slots per wavefront
  extern __shared__ __align__(16) unsigned char smraw[];
  float* X = reinterpret_cast<float*>(smraw);  // y of the sweep at preorder positions
  float* Q = X + LD;                           // exclusive postorder scan
  float* O = Q + LD;                           // the input row, then the outputs, at preorder positions
  __shared__ float wP[NW], wQ[NW], wM[NW];
  const int S = t.S;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int w = blockIdx.x;
  const long long grow = a.ws + w;
  const float NI = -__builtin_inff();
  const long long item = a.item[grow];
  const size_t cb = (size_t)(item * a.cstride);
  const float* in = a.Pi_in + (size_t)(a.pi_ws + w) * S;
  const long long lstate = a.use_leaf ? a.leaf_state[grow] : -1;
#pragma unroll
  for (int j = 0; j < CPT; ++j) {
    const int sc = tid + j * NT;
    if (sc < S) O[t.ppos[sc]] = in[sc];
  }
  if (tid < 64) {
    X[MAXS + tid] = 0.0f;
    Q[MAXS + tid] = 0.0f;
  }
  // own positions: tables, the linear constants, and the log2 terms of the outputs
  int c1p[CPT], c2p[CPT], nex[CPT], qp[CPT];
  bool okp[CPT];
  float ca[CPT], ce[CPT], ck1[CPT], ck2[CPT], cw[CPT], cwq[CPT], kmt[CPT], kcol[CPT], klf[CPT], kd[CPT];
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const int i = kb::own_pos_c<NT, CPT>(k);
    okp[k] = i < S;
    c1p[k] = c2p[k] = ZERO;
    nex[k] = 0;
    qp[k] = ZERO;
    ca[k] = ce[k] = ck1[k] = ck2[k] = kmt[k] = kcol[k] = 0.0f;
    cw[k] = cwq[k] = a.use_col ? 0.0f : 1.0f;
    klf[k] = kd[k] = NI;
    if (okp[k]) {
      const int col = t.pcol[i];
      const size_t ci = cb + col;
      const int c1 = t.pc1[i], c2 = t.pc2[i];
      c1p[k] = c1 >= 0 ? c1 : ZERO;
      c2p[k] = c2 >= 0 ? c2 : ZERO;
      nex[k] = t.pnex[i];
      qp[k] = t.ppost[i];
      ca[k] = (float)(exp2((double)a.DL[ci]) + exp2((double)a.Ebar[ci]));
      ce[k] = (float)exp2((double)a.E[ci] + (double)a.mt[ci]);
      ck1[k] = c1 >= 0 ? (float)exp2((double)a.SL1[ci]) : 0.0f;
      ck2[k] = c2 >= 0 ? (float)exp2((double)a.SL2[ci]) : 0.0f;
      kmt[k] = a.mt[ci];
      if (a.use_col) {
        kcol[k] = a.col[col];
        cw[k] = exp2f(kcol[k]);
        cwq[k] = exp2f(a.col[t.pcol[qp[k]]]);
      }
      if (lstate == col) klf[k] = a.leaf_logp[(size_t)item * S + col];
      if (a.dts) kd[k] = a.dts[(size_t)w * S + col];
    }
  }
  __syncthreads();
  float pr[CPT];
  kb::lds_load_own<CPT>(O, pr);
  float lm = NI;
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    if (!okp[k]) pr[k] = NI;
    lm = fmaxf(lm, pr[k]);
  }
  // linear space relative to the input's row maximum Ms
  const float Ms = kb::fsafe(kb::block_max1<NT>(lm, wM));
  float y[CPT], dl[CPT];
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    y[k] = okp[k] ? exp2f(pr[k] - Ms) : 0.0f;
    dl[k] = (klf[k] != NI ? exp2f(klf[k] - Ms) : 0.0f) + (kd[k] != NI ? exp2f(kd[k] - Ms) : 0.0f);
  }
  int kexp = 0, kexp_prev = 0;
  float ps[CPT], yprev[CPT], rowsum = 0.0f, tsum = 0.0f, f = 1.0f;
#pragma unroll
  for (int k = 0; k < CPT; ++k) yprev[k] = y[k];
  for (int sweep = 0;; ++sweep) {
    // phase A: publish y; inclusive (column-weighted) preorder scan in registers
    float sp[CPT], ta = 0.0f;
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      ta += cw[k] * y[k];
      sp[k] = ta;
    }
    const float wa = kb::wave_scan_incl(ta);
    kb::lds_store_own<CPT>(X, y);
    if (lane == 63) wP[wv] = wa;
    __syncthreads();
    // phase B: row sum (renormalised by an exact power of two), the postorder
    // values and children (read before the next barrier), exclusive postorder scan
    const float tp = kb::lds_wave_values<NW>(wP, lane, 0.0f);
    float yq[CPT], x1[CPT], x2[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      yq[k] = X[qp[k]];
      x1[k] = X[c1p[k]];
      x2[k] = X[c2p[k]];
    }
    const float ip = kb::wave_scan_first<NW>(tp);
    tsum = kb::lane_value(ip, NW - 1);
    const float offp = kb::lane_value(ip - tp, wv) + (wa - ta);
    float sq[CPT], tb = 0.0f;
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      sq[k] = tb;
      tb += cwq[k] * yq[k];
    }
    const float wb = kb::wave_scan_incl(tb);
#pragma unroll
    for (int k = 0; k < CPT; ++k) sq[k] += wb - tb;
    kb::lds_store_own<CPT>(Q, sq);
    if (lane == 63) wQ[wv] = wb;
    const int e = tsum > 0.0f ? __builtin_amdgcn_frexp_expf(tsum) : 0;
    f = __builtin_amdgcn_ldexpf(1.0f, -e);
    kexp += e;
    rowsum = tsum * f;
    __syncthreads();
    // phase C: path sums ps(i) = Pre(i) - PostEx(tin(i) - i)
    const float tq = kb::lds_wave_values<NW>(wQ, lane, 0.0f);
    const float eq = kb::wave_scan_first<NW>(tq) - tq;
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int n = nex[k];
      ps[k] = (sp[k] + offp) - (Q[n] + __shfl(eq, n / SEG, 64));
    }
    if (sweep == a.n_sweeps) break;
    if (sweep == a.n_sweeps - 1) {  // the row before the last sweep, for the residual
#pragma unroll
      for (int k = 0; k < CPT; ++k) yprev[k] = y[k];
      kexp_prev = kexp - e;
    }
    const float scale = __builtin_amdgcn_ldexpf(1.0f, -kexp);
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      float z = ca[k] * y[k];
      z += ck1[k] * x1[k];
      z += ck2[k] * x2[k];
      z += ce[k] * fmaxf(tsum - ps[k], 0.0f);
      y[k] = z * f + dl[k] * scale;
    }
  }
  // ---- outputs: Pi, the residual of the last sweep, Pibar and the row max
  const float M = Ms + (float)kexp;  // relative exponent of x = y f
  float po[CPT], pb[CPT];
  float ldiff = 0.0f, lmax = NI;
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    po[k] = pb[k] = NI;
    if (okp[k]) {
      const float x = y[k] * f;
      po[k] = x > 0.0f ? log2f(x) + M : NI;
      const float prev = yprev[k] > 0.0f ? log2f(yprev[k]) + (Ms + (float)kexp_prev) : NI;
      if (po[k] != NI && prev != NI) ldiff = fmaxf(ldiff, fabsf(po[k] - prev));
      const float na = rowsum - ps[k] * f;
      pb[k] = na > 0.0f ? log2f(na) + M + kmt[k] : NI;
      lmax = fmaxf(lmax, kcol[k] + po[k]);
    }
  }
  // O (the input) was last read before the first sweep's barrier; X's readers
  // finished before the last pass's second barrier
  kb::lds_store_own<CPT>(O, po);
  kb::lds_store_own<CPT>(X, pb);
  __syncthreads();
  float* out = a.Pi_out + (size_t)grow * S;
  float* pbo = a.store_final ? a.Pibar + (size_t)grow * S : nullptr;
#pragma unroll
  for (int j = 0; j < CPT; ++j) {
    const int sc = tid + j * NT;
    if (sc < S) {
      const int i = t.ppos[sc];
      out[sc] = O[i];
      if (pbo) pbo[sc] = X[i];
    }
  }
  if (a.resid) {
    const float md = kb::block_max1<NT>(ldiff, wM);
    if (tid == 0) a.resid[grow] = md;
  }
  if (a.store_final) {
    const float rmax = kb::block_max1<NT>(lmax, wP);
    if (tid == 0) a.rowmax[grow] = rmax;
  }
}

template <typename T>
struct LiArgs {
  int S, W, use_col;
  long long ws, cstride;
  T* Pi_out;
  const T *mt, *DL, *Ebar, *E, *SL1, *SL2, *col;
  const int64_t *sub_start, *sub_end, *item, *leaf_state, *c1, *c2;
  const T* leaf_logp;
};

template <typename T>
__global__ __launch_bounds__(256) void leaf_init_kernel(LiArgs<T> a) {
  const int w = blockIdx.x;
  const int s = blockIdx.y * 256 + threadIdx.x;
  const int S = a.S;
  if (s >= S) return;
  const T NI = ninf<T>();
  const long long grow = a.ws + w;
  const long long item = a.item[grow];
  const size_t ci = (size_t)(item * a.cstride) + s;
  const long long leaf = a.leaf_state[grow];
  const bool valid_leaf = leaf >= 0 && leaf < S;
  const long long ls = valid_leaf ? a.sub_start[leaf] : 0, le = valid_leaf ? a.sub_end[leaf] : 0;
  const long long st = a.sub_start[s];
  const bool desc = valid_leaf && st >= ls && st < le;
  const bool hit = s == leaf;
  const T lcol = (a.use_col && valid_leaf) ? a.col[leaf] : T(0);
  const T obs = valid_leaf ? a.leaf_logp[(size_t)item * S + leaf] : NI;
  const T pi_w = hit ? obs : NI;
  const T pibar_w = desc ? NI : a.mt[ci] + lcol + obs;
  const int c1 = child_at(a.c1, s, S), c2 = child_at(a.c2, s, S);
  const T ps1 = (c1 >= 0 && c1 == leaf) ? obs : NI;
  const T ps2 = (c2 >= 0 && c2 == leaf) ? obs : NI;
  const T t0 = a.DL[ci] + pi_w;
  const T t1 = pi_w + a.Ebar[ci];
  const T t2 = pibar_w + a.E[ci];
  const T t3 = a.SL1[ci] + ps1;
  const T t4 = a.SL2[ci] + ps2;
  const T t5 = hit ? a.leaf_logp[(size_t)item * S + s] : NI;
  const T m = tmax(tmax(tmax(t0, t1), tmax(t2, t3)), tmax(t4, t5));
  const T ms = msafe(m);
  const T sum = xexp2(t0 - ms) + xexp2(t1 - ms) + xexp2(t2 - ms) + xexp2(t3 - ms) + xexp2(t4 - ms) + xexp2(t5 - ms);
  a.Pi_out[(size_t)grow * S + s] = xlog2(sum) + m;
}

// ---- split reduction --------------------------------------------------------------

template <typename T>
struct DtsArgs {
  int S, W, by_state;
  long long item_offset, prow;
  const T *Pi, *Pibar, *lsp, *pD, *pS;
  const int64_t *sl, *sr, *item, *c1, *c2;
  const int *ptr, *order;
  const uint8_t* active;
  T* out;
};

template <typename T, int CPT>
__global__ __launch_bounds__(NT) void dts_kernel(DtsArgs<T> a) {
  const int S = a.S;
  const int w = blockIdx.x;
  const T NI = ninf<T>();
  T* out = a.out + (size_t)w * S;
  const int b = a.ptr[w], e = a.ptr[w + 1];
  if ((a.active && !a.active[w]) || b == e) {
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int s = threadIdx.x + k * NT;
      if (s < S) out[s] = NI;
    }
    return;
  }
  const long long item = a.item[a.item_offset + w];
  const size_t pb = (size_t)(item * a.prow);
  T m[CPT], acc[CPT];
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    m[k] = NI;
    acc[k] = 0;
  }
  for (int j = b; j < e; ++j) {
    const int si = a.order[j];
    const T* Pl = a.Pi + (size_t)a.sl[si] * S;
    const T* Pr = a.Pi + (size_t)a.sr[si] * S;
    const T* Bl = a.Pibar + (size_t)a.sl[si] * S;
    const T* Br = a.Pibar + (size_t)a.sr[si] * S;
    const T lsp = a.lsp[si];
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int s = threadIdx.x + k * NT;
      if (s < S) {
        const T d = a.by_state ? a.pD[pb + s] : a.pD[pb];
        const T sp = a.by_state ? a.pS[pb + s] : a.pS[pb];
        const T pl = Pl[s], pr = Pr[s];
        const int c1 = child_at(a.c1, s, S), c2 = child_at(a.c2, s, S);
        const T l1 = c1 >= 0 ? Pl[c1] : NI, r1 = c1 >= 0 ? Pr[c1] : NI;
        const T l2 = c2 >= 0 ? Pl[c2] : NI, r2 = c2 >= 0 ? Pr[c2] : NI;
        const T v0 = lsp + d + pl + pr;
        const T v1 = lsp + pl + Br[s];
        const T v2 = lsp + pr + Bl[s];
        const T v3 = lsp + sp + l1 + r2;
        const T v4 = lsp + sp + r1 + l2;
        const T sm = tmax(tmax(tmax(v0, v1), tmax(v2, v3)), v4);
        const T sms = msafe(sm);
        const T ss = xexp2(v0 - sms) + xexp2(v1 - sms) + xexp2(v2 - sms) + xexp2(v3 - sms) + xexp2(v4 - sms);
        const T nm = tmax(m[k], sm);
        const T nms = msafe(nm);
        acc[k] = (m[k] != NI ? acc[k] * xexp2(m[k] - nms) : T(0)) + ss * xexp2(sms - nms);
        m[k] = nm;
      }
    }
  }
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const int s = threadIdx.x + k * NT;
    if (s < S) out[s] = xlog2(acc[k]) + m[k];
  }
}

// ---- active mask ------------------------------------------------------------------------

__device__ __forceinline__ float absval(float x) { return fabsf(x); }
__device__ __forceinline__ double absval(double x) { return fabs(x); }

template <typename T>
__device__ __forceinline__ double as_double(T x) {
  return (double)x;
}
template <>
__device__ __forceinline__ double as_double<__hip_bfloat16>(__hip_bfloat16 x) {
  return (double)__bfloat162float(x);
}

template <typename T>
__global__ __launch_bounds__(256) void active_kernel(int S, long long stride, const T* rhs, float thr, int strict,
                                                     uint8_t* active) {
  __shared__ double red[4];
  const T* row = rhs + (size_t)blockIdx.x * stride;
  double m = 0.0;
  for (int s = threadIdx.x; s < S; s += 256) {
    const double v = fabs(as_double(row[s]));
    m = v > m || v != v ? v : m;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const double y = __shfl_xor(m, o, 64);
    m = y > m || y != y ? y : m;
  }
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    double r = red[0];
    for (int i = 1; i < 4; ++i) r = red[i] > r || red[i] != red[i] ? red[i] : r;
    // compare in the row's precision against the float32 threshold, as a
    // Triton kernel does with a Python float argument
    const double th = (double)thr;
    active[blockIdx.x] = strict ? (r > th) : (r >= th);
  }
}

// ---- self-loop adjoint ---------------------------------------------------------------------

template <typename T>
struct WbArgs {
  int S, W, n_terms, clayout, leaf_mode, use_leaf, use_col;
  long long ws;
  const T *Pi, *Pibar, *rowmax, *dts, *rhs, *v0;
  const uint8_t* active;
  const T *mt, *DL, *Ebar, *E, *SL1, *SL2, *col;
  const int64_t *item, *leaf_state;
  const T *leaf_logp, *leaf_term;
  T *v, *aw0, *aw1, *aw2, *aw345, *aw3, *aw4, *col_rows;
  float* relres;
};

template <typename T, int CPT>
__global__ __launch_bounds__(NT) void wave_bwd_kernel(OpsTree t, WbArgs<T> a) {
  extern __shared__ unsigned char smraw[];
  T* X = reinterpret_cast<T*>(smraw);  // p', then path sums
  T* Ed = X + t.S;                     // edge weight into each column from its parent
  T* Tm = Ed + t.S;                    // current Neumann term (column order)
  T* Up = Tm + t.S;                    // preorder scan of u; Tm..Up double as the 2S Euler scan
  __shared__ T red[NW];
  const int S = a.S;
  const int w = blockIdx.x;
  const long long grow = a.ws + w;
  const size_t ob = (size_t)w * S;
  const T NI = ninf<T>();
  const bool act = a.active ? a.active[w] != 0 : true;
  if (!act) {
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int s = threadIdx.x + k * NT;
      if (s < S) {
        a.v[ob + s] = 0;
        a.aw0[ob + s] = 0;
        a.aw1[ob + s] = 0;
        a.aw2[ob + s] = 0;
        a.aw345[ob + s] = 0;
        a.aw3[ob + s] = 0;
        a.aw4[ob + s] = 0;
        a.col_rows[ob + s] = 0;
      }
    }
    if (a.relres && threadIdx.x == 0) a.relres[w] = 0.0f;
    return;
  }
  const long long item = a.item ? a.item[grow] : 0;
  const size_t cb = a.clayout == 1 ? ob : (a.clayout == 2 ? (size_t)item * S : 0);
  const T* pirow = a.Pi + (size_t)grow * S;
  const T* pbrow = a.Pibar + (size_t)grow * S;
  const T rms = msafe(a.rowmax[grow]);
  // p' and its row sum
  T pp[CPT];
  T ls = 0;
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const int s = threadIdx.x + k * NT;
    pp[k] = 0;
    if (s < S) {
      pp[k] = xexp2((a.use_col ? a.col[s] + pirow[s] : pirow[s]) - rms);
      X[s] = pp[k];
      Ed[s] = 0;
      ls += pp[k];
    }
  }
  const T row_sum = block_sum(ls, red);
  path_sums(t, X, Tm, X, red);
  const long long lstate = a.use_leaf ? a.leaf_state[grow] : -1;
  T diag[CPT], pcoef[CPT], wl[CPT], e0[CPT], e1[CPT], e2[CPT], e3[CPT], e4[CPT], e5[CPT], isum[CPT];
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const int s = threadIdx.x + k * NT;
    diag[k] = pcoef[k] = wl[k] = 0;
    e0[k] = e1[k] = e2[k] = e3[k] = e4[k] = e5[k] = isum[k] = 0;
    if (s < S) {
      const size_t ci = cb + s;
      const T pi = pirow[s];
      const int c1 = t.c1[s], c2 = t.c2[s];
      const T ps1 = c1 >= 0 ? pirow[c1] : NI;
      const T ps2 = c2 >= 0 ? pirow[c2] : NI;
      const T t0 = a.DL[ci] + pi;
      const T t1 = pi + a.Ebar[ci];
      const T t2 = pbrow[s] + a.E[ci];
      const T t3 = a.SL1[ci] + ps1;
      const T t4 = a.SL2[ci] + ps2;
      T t5 = NI;
      if (a.use_leaf) {
        if (lstate == s) {
          if (a.leaf_mode == 3) t5 = a.leaf_logp[0];
          else if (a.leaf_mode == 1) t5 = a.leaf_logp[item];
          else if (a.leaf_mode == 2) t5 = a.leaf_logp[(size_t)item * S + s];
          else t5 = a.leaf_logp[s];
        }
      } else if (a.leaf_term) {
        t5 = a.leaf_term[ob + s];
      }
      const T m = tmax(tmax(tmax(t0, t1), tmax(t2, t3)), tmax(t4, t5));
      const T ms = msafe(m);
      e0[k] = xexp2(t0 - ms);
      e1[k] = xexp2(t1 - ms);
      e2[k] = xexp2(t2 - ms);
      e3[k] = xexp2(t3 - ms);
      e4[k] = xexp2(t4 - ms);
      e5[k] = xexp2(t5 - ms);
      const T sum = e0[k] + e1[k] + e2[k] + e3[k] + e4[k] + e5[k];
      isum[k] = sum > T(0) ? T(1) / sum : T(0);
      wl[k] = 1;
      if (a.dts) {
        const T dl = xlog2(sum) + m;
        const T dr = a.dts[ob + s];
        const T pm = tmax(dl, dr);
        const T pms = msafe(pm);
        const T pnew = xlog2(xexp2(dl - pms) + xexp2(dr - pms)) + pm;
        wl[k] = dl != NI ? xexp2(dl - pnew) : T(0);
      }
      const T denom = row_sum - X[s];
      const T idn = denom > T(0) ? T(1) / denom : T(0);
      diag[k] = wl[k] * (e0[k] + e1[k]) * isum[k];
      pcoef[k] = wl[k] * e2[k] * isum[k] * idn;
      if (c1 >= 0) Ed[c1] = wl[k] * e3[k] * isum[k];
      if (c2 >= 0) Ed[c2] = wl[k] * e4[k] * isum[k];
    }
  }
  __syncthreads();
  T edge[CPT], term[CPT], v[CPT], rh[CPT];
  int par[CPT];
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const int s = threadIdx.x + k * NT;
    edge[k] = s < S ? Ed[s] : T(0);
    par[k] = s < S ? t.par[s] : -1;
    rh[k] = s < S ? a.rhs[ob + s] : T(0);
    // Neumann: term_0 = rhs; fixed point from initial_v: the term is v itself
    v[k] = a.v0 ? (s < S ? a.v0[ob + s] : T(0)) : rh[k];
    term[k] = v[k];
  }
  // Neumann series v = sum_{n <= N} (J^T)^n rhs, or N steps of v <- rhs + J^T v
  for (int n = 0; n < a.n_terms; ++n) {
    T lu = 0;
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int s = threadIdx.x + k * NT;
      if (s < S) {
        Tm[s] = term[k];
        const T u = term[k] * pcoef[k];
        X[s] = u;
        lu += u;
      }
    }
    __syncthreads();
    subtree_scan(t, X, Up, red);
    const T A = Up[S - 1];
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int s = threadIdx.x + k * NT;
      if (s < S) {
        const T nt = term[k] * diag[k] + pp[k] * complement_of(t, Up, s, A) + (par[k] >= 0 ? Tm[par[k]] : T(0)) * edge[k];
        if (a.v0) {
          v[k] = rh[k] + nt;
          term[k] = v[k];
        } else {
          term[k] = nt;
          v[k] += nt;
        }
      }
    }
    __syncthreads();
  }
  // column gradient p' (A - subtree(v pcoef)) and the parameter contributions
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const int s = threadIdx.x + k * NT;
    if (s < S) X[s] = v[k] * pcoef[k];
  }
  __syncthreads();
  subtree_scan(t, X, Up, red);
  const T A = Up[S - 1];
  T ln = 0, lv = 0;
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const int s = threadIdx.x + k * NT;
    if (s < S) {
      a.col_rows[ob + s] = pp[k] * complement_of(t, Up, s, A);
      const T al = v[k] * wl[k] * isum[k];
      const T a3 = al * e3[k], a4 = al * e4[k], a5 = al * e5[k];
      a.v[ob + s] = v[k];
      a.aw0[ob + s] = al * e0[k];
      a.aw1[ob + s] = al * e1[k];
      a.aw2[ob + s] = al * e2[k];
      a.aw3[ob + s] = a3;
      a.aw4[ob + s] = a4;
      a.aw345[ob + s] = a3 + a4 + a5;
      const float tf = (float)term[k], vf = (float)v[k];
      ln += (T)(tf * tf);
      lv += (T)(vf * vf);
    }
  }
  if (a.relres) {
    const T n2 = block_sum(ln, red);
    const T v2 = block_sum(lv, red);
    if (threadIdx.x == 0) {
      const float tiny = 1.17549435e-38f;
      const float den = fmaxf(sqrtf((float)v2), tiny);
      a.relres[w] = a.n_terms > 0 ? sqrtf((float)n2) / den : 0.0f;
    }
  }
}

// Rows at preorder ownership (thread t owns positions t*CPT + k, as the
// whole-pass backward row kernel): the root-path sums of p' from an inclusive
// preorder and an exclusive postorder scan, one barrier per Neumann term
// (wavefront-local scans published, the readers add the wavefront offsets),
// and the [W, S] outputs written back in column order through LDS.  Same
// mathematics as wave_bwd_kernel.  Shapes and figures: launch_wave_bwd.
template <typename T>
constexpr int wave_bwd_waves(int cpt) { return cpt > 2 ? 1 : std::is_same_v<T, float> ? 8 : 4; }

template <typename T, int BT, int CPT>
__global__ __launch_bounds__(BT) __attribute__((amdgpu_waves_per_eu(wave_bwd_waves<T>(CPT)))) void wave_bwd_pre_kernel(OpsTree t, WbArgs<T> a) {
  constexpr int BW = BT / 64;
  constexpr int MAXS = BT * CPT;
  constexpr int LD = MAXS + 64;  // [MAXS] is the padding slot, kept at 0
  constexpr int ZERO = MAXS;
  constexpr int SEG = 64 * CPT;  // postorder slots per wavefront
  extern __shared__ __align__(16) unsigned char smraw[];
  T* L0 = reinterpret_cast<T*>(smraw);
  T* L1 = L0 + LD;
  T* L2 = L1 + LD;
  T* L3 = L2 + LD;
  __shared__ T wA[BW], wB[BW];
  const int S = a.S;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int w = blockIdx.x;
  const long long grow = a.ws + w;
  const size_t ob = (size_t)w * S;
  const T NI = ninf<T>();
  const bool act = a.active ? a.active[w] != 0 : true;
  if (!act) {
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int s = tid + k * BT;
      if (s < S) {
        a.v[ob + s] = 0;
        a.aw0[ob + s] = 0;
        a.aw1[ob + s] = 0;
        a.aw2[ob + s] = 0;
        a.aw345[ob + s] = 0;
        a.aw3[ob + s] = 0;
        a.aw4[ob + s] = 0;
        a.col_rows[ob + s] = 0;
      }
    }
    if (a.relres && tid == 0) a.relres[w] = T(0.0);
    return;
  }
  const long long item = a.item ? a.item[grow] : 0;
  const size_t cb = a.clayout == 1 ? ob : (a.clayout == 2 ? (size_t)item * S : 0);
  const T* pirow = a.Pi + (size_t)grow * S;
  const T* pbrow = a.Pibar + (size_t)grow * S;
  const T rms = msafe(a.rowmax[grow]);
  // Pi and Pibar to their preorder positions (coalesced column reads)
#pragma unroll
  for (int j = 0; j < CPT; ++j) {
    const int sc = tid + j * BT;
    if (sc < S) {
      const int p = t.ppos[sc];
      L0[p] = pirow[sc];
      L1[p] = pbrow[sc];
    }
  }
  if (tid < 64) {
    L0[MAXS + tid] = T(0.0);
    L1[MAXS + tid] = T(0.0);
    L2[MAXS + tid] = T(0.0);
    L3[MAXS + tid] = T(0.0);
  }
  // own positions: column, children, parent, subtree end - 1, postorder slot, tin - i
  int colk[CPT], c1p[CPT], c2p[CPT], ppar[CPT], endm1[CPT], wend[CPT], qp[CPT], nex[CPT];
  bool okp[CPT];
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const int i = kb::own_pos_c<BT, CPT>(k);
    okp[k] = i < S;
    colk[k] = okp[k] ? t.pcol[i] : 0;
    c1p[k] = okp[k] ? t.pc1[i] : -1;
    c2p[k] = okp[k] ? t.pc2[i] : -1;
    const int par = okp[k] ? t.par[colk[k]] : -1;
    ppar[k] = par >= 0 ? t.ppos[par] : ZERO;
    endm1[k] = okp[k] ? t.pend[colk[k]] - 1 : ZERO;
    wend[k] = endm1[k] < ZERO ? endm1[k] / SEG : 0;
    qp[k] = okp[k] ? t.ppost[i] : ZERO;
    nex[k] = okp[k] ? t.pnex[i] : 0;
  }
  __syncthreads();
  T piv[CPT], pbv[CPT];
  own_load<CPT>(L0, piv);
  own_load<CPT>(L1, pbv);
  // p' = 2^(col + Pi - rowmax) and its root-path sums ps(i) = Pre(i) - PostEx(tin(i) - i)
  T pp[CPT], sp[CPT], ta = T(0.0);
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    pp[k] = okp[k] ? xexp2((a.use_col ? a.col[colk[k]] + piv[k] : piv[k]) - rms) : T(0.0);
    ta += pp[k];
    sp[k] = ta;
  }
  const T wa = wscan(ta);
  own_store<CPT>(L2, pp);
  if (lane == 63) wA[wv] = wa;
  __syncthreads();
  T ps[CPT], ch1[CPT], ch2[CPT], row_sum;
  {
    const T tp = kb::lds_wave_values<BW>(wA, lane, T(0));
    T yq[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      yq[k] = L2[qp[k]];
      ch1[k] = c1p[k] >= 0 ? L0[c1p[k]] : NI;
      ch2[k] = c2p[k] >= 0 ? L0[c2p[k]] : NI;
    }
    const T ip = wscan_first<BW>(tp);
    row_sum = lane_of(ip, BW - 1);
    const T offp = lane_of(ip - tp, wv) + (wa - ta);
    T sq[CPT], tb = T(0.0);
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      sq[k] = tb;
      tb += yq[k];
    }
    const T wb = wscan(tb);
#pragma unroll
    for (int k = 0; k < CPT; ++k) sq[k] += wb - tb;
    own_store<CPT>(L3, sq);
    if (lane == 63) wB[wv] = wb;
    __syncthreads();
    const T tq = kb::lds_wave_values<BW>(wB, lane, T(0.0));
    const T eq = wscan_first<BW>(tq) - tq;
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int n = nex[k];
      ps[k] = (sp[k] + offp) - (L3[n] + shfl_of(eq, n / SEG));
    }
  }
  // J^T coefficients; the child-edge weights (q3 into child1, q4 into child2)
  // scattered by the parent's owner into L1; the rhs and initial rows staged
  // into L2 / L0 (free since the scans above), all under one barrier
  const long long lstate = a.use_leaf ? a.leaf_state[grow] : -1;
  T diag[CPT], pcoef[CPT], q[6][CPT];
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    diag[k] = pcoef[k] = T(0.0);
#pragma unroll
    for (int j = 0; j < 6; ++j) q[j][k] = T(0.0);
    if (okp[k]) {
      const int s = colk[k];
      const size_t ci = cb + s;
      const T pi = piv[k];
      const T t0 = a.DL[ci] + pi;
      const T t1 = pi + a.Ebar[ci];
      const T t2 = pbv[k] + a.E[ci];
      const T t3 = a.SL1[ci] + ch1[k];
      const T t4 = a.SL2[ci] + ch2[k];
      T t5 = NI;
      if (a.use_leaf) {
        if (lstate == s) {
          if (a.leaf_mode == 3) t5 = a.leaf_logp[0];
          else if (a.leaf_mode == 1) t5 = a.leaf_logp[item];
          else if (a.leaf_mode == 2) t5 = a.leaf_logp[(size_t)item * S + s];
          else t5 = a.leaf_logp[s];
        }
      } else if (a.leaf_term) {
        t5 = a.leaf_term[ob + s];
      }
      const T m = tmax(tmax(tmax(t0, t1), tmax(t2, t3)), tmax(t4, t5));
      const T ms = msafe(m);
      const T e0 = xexp2(t0 - ms), e1 = xexp2(t1 - ms), e2 = xexp2(t2 - ms);
      const T e3 = xexp2(t3 - ms), e4 = xexp2(t4 - ms), e5 = xexp2(t5 - ms);
      const T sum = e0 + e1 + e2 + e3 + e4 + e5;
      const T isum = sum > T(0.0) ? T(1.0) / sum : T(0.0);
      T wl = T(1.0);
      if (a.dts) {
        const T dl = xlog2(sum) + m;
        const T dr = a.dts[ob + s];
        const T pm = tmax(dl, dr);
        const T pms = msafe(pm);
        const T pnew = xlog2(xexp2(dl - pms) + xexp2(dr - pms)) + pm;
        wl = dl != NI ? xexp2(dl - pnew) : T(0.0);
      }
      const T denom = row_sum - ps[k];
      const T idn = denom > T(0.0) ? T(1.0) / denom : T(0.0);
      diag[k] = wl * (e0 + e1) * isum;
      pcoef[k] = wl * e2 * isum * idn;
      const T c = wl * isum;
      q[0][k] = c * e0;
      q[1][k] = c * e1;
      q[2][k] = c * e2;
      q[3][k] = c * e3;
      q[4][k] = c * e4;
      q[5][k] = c * e5;
      if (c1p[k] >= 0) L1[c1p[k]] = wl * e3 * isum;
      if (c2p[k] >= 0) L1[c2p[k]] = wl * e4 * isum;
    }
  }
#pragma unroll
  for (int j = 0; j < CPT; ++j) {
    const int sc = tid + j * BT;
    if (sc < S) {
      const int p = t.ppos[sc];
      L2[p] = a.rhs[ob + sc];
      if (a.v0) L0[p] = a.v0[ob + sc];
    }
  }
  __syncthreads();
  T edge[CPT], rh[CPT], v[CPT], term[CPT];
  own_load<CPT>(L1, edge);
  own_load<CPT>(L2, rh);
  if (a.v0) own_load<CPT>(L0, v);
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    edge[k] = ppar[k] != ZERO ? edge[k] : T(0.0);
    if (!okp[k]) rh[k] = T(0.0);
    // Neumann: term_0 = rhs; fixed point from initial_v: the term is v itself
    v[k] = a.v0 ? (okp[k] ? v[k] : T(0.0)) : rh[k];
    term[k] = v[k];
  }
  // Neumann series v = sum_{n <= N} (J^T)^n rhs, or N steps of v <- rhs + J^T v.
  // Buffers alternate by parity: (Tb, Lb) = (L0, L2) for even terms, (L1, L3)
  // for odd ones; every thread read its own L0..L2 entries above, and the
  // other threads' entries are read only after each term's barrier.
  // the scan of u at the own positions, wavefront-local, published in Lb / wt
  auto publish_scan = [&](const T (&u)[CPT], T (&sc)[CPT], T* Lb, T* wt) {
#pragma unroll
    for (int k = 0; k < CPT; ++k) sc[k] = u[k] + (k > 0 ? sc[k > 0 ? k - 1 : 0] : T(0));
    const T tsum = sc[CPT - 1];
    const T ws = wscan(tsum);
    if (lane == 63) wt[wv] = ws;
#pragma unroll
    for (int k = 0; k < CPT; ++k) sc[k] += ws - tsum;
    own_store<CPT>(Lb, sc);
  };
  // after a barrier: the sum of u outside each own position's subtree
  auto outside = [&](const T (&sc)[CPT], const T* Lb, const T* wt, T (&x)[CPT]) {
    T le[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) le[k] = Lb[endm1[k]];
    const T wtot = kb::lds_wave_values<BW>(wt, lane, T(0));
    const T wincl = wscan_first<BW>(wtot);
    const T wexcl = wincl - wtot;
    const T A = lane_of(wincl, BW - 1);
    const T woff = lane_of(wexcl, wv);
    const T p0 = prev_lane(sc[CPT - 1]) + woff;
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const T pm1 = k == 0 ? p0 : sc[k > 0 ? k - 1 : 0] + woff;
      x[k] = pm1 + (A - (le[k] + (BW > 1 ? shfl_of(wexcl, wend[k]) : T(0))));
    }
  };
  auto neumann_term = [&](T* Tb, T* Lb, T* wt) {
    T u[CPT], sc[CPT], tpar[CPT], x[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) u[k] = term[k] * pcoef[k];
    publish_scan(u, sc, Lb, wt);
    own_store<CPT>(Tb, term);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < CPT; ++k) tpar[k] = Tb[ppar[k]];
    outside(sc, Lb, wt, x);
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const T nt = term[k] * diag[k] + pp[k] * x[k] + tpar[k] * edge[k];
      if (a.v0) {
        v[k] = rh[k] + nt;
        term[k] = v[k];
      } else {
        term[k] = nt;
        v[k] += nt;
      }
    }
  };
  {
    int n = 0;
    for (; n + 2 <= a.n_terms; n += 2) {
      neumann_term(L0, L2, wA);
      neumann_term(L1, L3, wB);
    }
    if (n < a.n_terms) neumann_term(L0, L2, wA);
  }
  // column gradient p' (A - subtree(v pcoef)), in the next parity's buffers
  T colg[CPT];
  {
    const int n = a.n_terms;
    T* Pb = (n & 1) ? L3 : L2;
    T* wt = (n & 1) ? wB : wA;
    T u[CPT], sc[CPT], x[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) u[k] = v[k] * pcoef[k];
    publish_scan(u, sc, Pb, wt);
    __syncthreads();
    outside(sc, Pb, wt, x);
#pragma unroll
    for (int k = 0; k < CPT; ++k) colg[k] = okp[k] ? pp[k] * x[k] : T(0);
  }
  // outputs in column order, four rows at a time through L0..L3
  T* const outs[8] = {a.v, a.aw0, a.aw1, a.aw2, a.aw3, a.aw4, a.aw345, a.col_rows};
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    __syncthreads();  // the previous readers of L0..L3 are done
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int o = 4 * half + r;
      T x[CPT];
#pragma unroll
      for (int k = 0; k < CPT; ++k) {
        if (o == 0) x[k] = v[k];
        else if (o == 7) x[k] = colg[k];
        else if (o == 6) x[k] = v[k] * (q[3][k] + q[4][k] + q[5][k]);
        else x[k] = v[k] * q[o - 1][k];
      }
      own_store<CPT>(L0 + r * LD, x);
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      T* dst = outs[4 * half + r] + ob;
#pragma unroll
      for (int j = 0; j < CPT; ++j) {
        const int sc = tid + j * BT;
        if (sc < S) dst[sc] = L0[r * LD + t.ppos[sc]];
      }
    }
  }
  if (a.relres) {
    T ln = T(0), lv = T(0);
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const float tf = (float)term[k], vf = (float)v[k];
      ln += (T)(tf * tf);
      lv += (T)(vf * vf);
    }
    const T n2 = wg_sum_of<BT>(ln, wA);
    const T v2 = wg_sum_of<BT>(lv, wB);
    if (tid == 0) {
      const float tiny = 1.17549435e-38f;
      const float den = fmaxf(sqrtf((float)v2), tiny);
      a.relres[w] = a.n_terms > 0 ? sqrtf((float)n2) / den : 0.0f;
    }
  }
}

// ---- cross-wave split adjoint ----------------------------------------------------------------

template <typename T>
struct DcArgs {
  int S, playout, mlayout, output_ud, skip_zero;
  long long N, ws;
  double side_thr;
  const T *Pi, *Pibar, *v;
  const uint8_t* active;
  const int64_t *sl, *sr, *red_idx, *item, *c1, *c2;
  const T *wlsp, *pD, *pS, *mt, *rowmax;
  T *side_rows, *ud, *A;
  uint8_t* side_active;
  T *gPl, *gPr, *prow, *psum, *mrow;
};

// One split per workgroup of the smallest shape that holds a row; memory-bound
// (six rows read, two to eight written), so what counts is how many splits a CU
// has in flight: up to 2048 threads of them instead of two 1024-thread
// workgroups.  The up to six row sums share one exchange (each took two
// barriers).  Measured against 1024 threads for every row: 2047 states 81 -> 76
// us a wave, 1023 states (18 mostly narrow waves) 211 -> 166 us.
template <typename T, int BT, int CPT>
__global__ __launch_bounds__(BT) void dts_cross_kernel(DcArgs<T> a) {
  constexpr int BW = BT / 64;
  extern __shared__ __align__(16) unsigned char smraw[];
  T* Lr = reinterpret_cast<T*>(smraw);
  T* Rr = Lr + a.S;
  __shared__ T red[6][BW];
  const int S = a.S;
  const long long i = blockIdx.x;
  const long long N = a.N;
  const T NI = ninf<T>();
  const long long pw = a.red_idx[i];
  const bool act = a.active ? a.active[pw] != 0 : true;
  T* sideL = a.side_rows + (size_t)i * S;
  T* sideR = a.side_rows + (size_t)(N + i) * S;
  if (!act) {
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int s = threadIdx.x + k * BT;
      if (s < S) {
        sideL[s] = 0;
        sideR[s] = 0;
        if (a.prow) {
          a.prow[(size_t)i * S + s] = 0;
          a.prow[(size_t)(N + i) * S + s] = 0;
        }
        if (a.mrow) {
          a.mrow[(size_t)i * S + s] = 0;
          a.mrow[(size_t)(N + i) * S + s] = 0;
        }
        if (a.output_ud) {
          if (!a.skip_zero) {
            a.ud[(size_t)i * S + s] = 0;
            a.ud[(size_t)(N + i) * S + s] = 0;
          }
        } else {
          a.gPl[(size_t)i * S + s] = 0;
          a.gPr[(size_t)i * S + s] = 0;
        }
      }
    }
    if (threadIdx.x == 0) {
      if (a.psum) {
        a.psum[i] = 0;
        a.psum[N + i] = 0;
      }
      if (a.output_ud) {
        if (a.side_active) {
          a.side_active[i] = 0;
          a.side_active[N + i] = 0;
        }
        if (!a.skip_zero) {
          a.A[i] = 0;
          a.A[N + i] = 0;
        }
      }
    }
    return;
  }
  const long long l = a.sl[i], r = a.sr[i];
  const long long prow_g = a.ws + pw;
  const long long pitem = a.item ? a.item[prow_g] : 0;
  const long long il = (a.item && a.mlayout == 1) ? a.item[l] : 0;
  const long long ir = (a.item && a.mlayout == 1) ? a.item[r] : 0;
  const T wlsp = a.wlsp[i];
  const T* Pl = a.Pi + (size_t)l * S;
  const T* Prr = a.Pi + (size_t)r * S;
  const T* Bl = a.Pibar + (size_t)l * S;
  const T* Br = a.Pibar + (size_t)r * S;
  const T* Pp = a.Pi + (size_t)prow_g * S;
  const T* vr = a.v + (size_t)pw * S;
  T vd3[CPT], vd4[CPT];
  int c1v[CPT], c2v[CPT];
  T sd = 0, ss = 0, sul = 0, sur = 0, bl = 0, br = 0;
  T rml = 0, rmr = 0;
  if (a.output_ud) {
    rml = a.rowmax[l];
    rmr = a.rowmax[r];
  }
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const int s = threadIdx.x + k * BT;
    vd3[k] = vd4[k] = 0;
    c1v[k] = c2v[k] = -1;
    if (s < S) {
      T d, sp;
      if (a.playout == 0) {
        d = a.pD[0];
        sp = a.pS[0];
      } else if (a.playout == 1) {
        d = a.pD[s];
        sp = a.pS[s];
      } else if (a.playout == 2) {
        d = a.pD[pitem];
        sp = a.pS[pitem];
      } else {
        d = a.pD[(size_t)pitem * S + s];
        sp = a.pS[(size_t)pitem * S + s];
      }
      const T pil = Pl[s], pir = Prr[s];
      const int c1 = child_at(a.c1, s, S), c2 = child_at(a.c2, s, S);
      c1v[k] = c1;
      c2v[k] = c2;
      const T l1 = c1 >= 0 ? Pl[c1] : NI, r1 = c1 >= 0 ? Prr[c1] : NI;
      const T l2 = c2 >= 0 ? Pl[c2] : NI, r2 = c2 >= 0 ? Prr[c2] : NI;
      const T d0 = d + pil + pir;
      const T d1 = pil + Br[s];
      const T d2 = pir + Bl[s];
      const T d3 = sp + l1 + r2;
      const T d4 = sp + r1 + l2;
      const T pp = Pp[s];
      const bool pv = pp != NI;
      const T vv = vr[s];
      const T vd0 = pv ? vv * xexp2(wlsp + d0 - pp) : T(0);
      const T vd1 = pv ? vv * xexp2(wlsp + d1 - pp) : T(0);
      const T vd2 = pv ? vv * xexp2(wlsp + d2 - pp) : T(0);
      vd3[k] = pv ? vv * xexp2(wlsp + d3 - pp) : T(0);
      vd4[k] = pv ? vv * xexp2(wlsp + d4 - pp) : T(0);
      Lr[s] = vd0 + vd1;
      Rr[s] = vd0 + vd2;
      sd += vd0;
      ss += vd3[k] + vd4[k];
      if (a.prow) {
        a.prow[(size_t)i * S + s] = vd0;
        a.prow[(size_t)(N + i) * S + s] = vd3[k] + vd4[k];
      }
      if (a.mrow) {
        a.mrow[(size_t)i * S + s] = vd2;
        a.mrow[(size_t)(N + i) * S + s] = vd1;
      }
      if (a.output_ud) {
        const T mtl = a.mlayout == 1 ? a.mt[(size_t)il * S + s] : a.mt[s];
        const T mtr = a.mlayout == 1 ? a.mt[(size_t)ir * S + s] : a.mt[s];
        const T pbl = Bl[s], pbr = Br[s];
        const T invl = pbl != NI ? xexp2(rml + mtl - pbl) : T(0);
        const T invr = pbr != NI ? xexp2(rmr + mtr - pbr) : T(0);
        const T udl = vd2 * invl, udr = vd1 * invr;
        a.ud[(size_t)i * S + s] = udl;
        a.ud[(size_t)(N + i) * S + s] = udr;
        sul += udl;
        sur += udr;
        if (a.side_thr > 0.0) {
          bl += udl < T(0) ? -udl : udl;
          br += udr < T(0) ? -udr : udr;
        } else {
          bl = tmax(bl, udl < T(0) ? -udl : udl);
          br = tmax(br, udr < T(0) ? -udr : udr);
        }
      } else {
        a.gPl[(size_t)i * S + s] = vd2;
        a.gPr[(size_t)i * S + s] = vd1;
      }
    }
  }
  {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    auto put = [&](int j, T x) {
      if (lane == 63) red[j][wv] = x;
    };
    if (a.psum) {
      put(0, wscan(sd));
      put(1, wscan(ss));
    }
    if (a.output_ud) {
      put(2, wscan(sul));
      put(3, wscan(sur));
      put(4, a.side_thr > 0.0 ? wscan(bl) : wmax63(bl));
      put(5, a.side_thr > 0.0 ? wscan(br) : wmax63(br));
    }
  }
  __syncthreads();
  // speciation terms land in the children's columns (each column has one parent)
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    if (c1v[k] >= 0) {
      Lr[c1v[k]] += vd3[k];
      Rr[c1v[k]] += vd4[k];
    }
    if (c2v[k] >= 0) {
      Rr[c2v[k]] += vd3[k];
      Lr[c2v[k]] += vd4[k];
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const int s = threadIdx.x + k * BT;
    if (s < S) {
      sideL[s] = Lr[s];
      sideR[s] = Rr[s];
    }
  }
  if (threadIdx.x == 0) {
    auto sum = [&](int j) {
      T x = red[j][0];
#pragma unroll
      for (int w = 1; w < BW; ++w) x += red[j][w];
      return x;
    };
    auto top = [&](int j) {
      T x = red[j][0];
#pragma unroll
      for (int w = 1; w < BW; ++w) x = tmax(x, red[j][w]);
      return x;
    };
    if (a.psum) {
      a.psum[i] = sum(0);
      a.psum[N + i] = sum(1);
    }
    if (a.output_ud) {
      a.A[i] = sum(2);
      a.A[N + i] = sum(3);
      if (a.side_active) {
        if (a.side_thr > 0.0) {
          a.side_active[i] = (double)sum(4) > a.side_thr;
          a.side_active[N + i] = (double)sum(5) > a.side_thr;
        } else {
          a.side_active[i] = top(4) != T(0);
          a.side_active[N + i] = top(5) != T(0);
        }
      }
    }
  }
}

// ---- Pibar VJP through the subtree sums ----------------------------------------------------------

template <typename T>
struct PvArgs {
  int S, use_col;
  long long N;
  const T *Pi, *col, *A, *rowmax;
  T* ud;
  const uint8_t *side_active, *active;
  const int64_t *sl, *sr, *red_idx;
  T* contrib;
};

// One side per workgroup of the smallest shape that holds a row.  The row's ud
// goes to its preorder positions in LDS, is scanned in registers (thread t owns
// positions t*CPT + k, one wavefront scan, published with the wavefront totals
// under one barrier), and each column reads its two prefix values back: two
// barriers in all, and the Pi row is loaded ahead of them.  Measured against an
// LDS block scan on 1024 threads: 2047 states 57 -> 34 us a wave, 1023 states
// (18 waves) 144 -> 105 us.
template <typename T, int BT, int CPT>
__global__ __launch_bounds__(BT) void pibar_vjp_kernel(OpsTree t, PvArgs<T> a) {
  constexpr int BW = BT / 64;
  constexpr int MAXS = BT * CPT;
  constexpr int SEG = 64 * CPT;  // positions per wavefront
  extern __shared__ __align__(16) unsigned char smraw[];
  T* L = reinterpret_cast<T*>(smraw);
  __shared__ T wA[BW];
  const int S = a.S;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const long long row = blockIdx.x;
  const long long si = row < a.N ? row : row - a.N;
  T* crow = a.contrib + (size_t)row * S;
  bool go = a.side_active ? a.side_active[row] != 0 : true;
  if (go && a.active) go = a.active[a.red_idx[si]] != 0;
  if (!go) {
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int s = tid + k * BT;
      if (s < S) crow[s] = 0;
    }
    return;
  }
  const long long child = row < a.N ? a.sl[si] : a.sr[si];
  T* udr = a.ud + (size_t)row * S;
  const T* pr = a.Pi + (size_t)child * S;
  int pos[CPT], end[CPT];
  T pic[CPT];
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const int s = tid + k * BT;
    pos[k] = 0;
    end[k] = 1;
    pic[k] = T(0);
    if (s < S) {
      pos[k] = t.ppos[s];
      end[k] = t.pend[s];
      pic[k] = a.use_col ? a.col[s] + pr[s] : pr[s];
      L[pos[k]] = udr[s];
    }
  }
  for (int i = S + tid; i < MAXS; i += BT) L[i] = T(0);
  __syncthreads();
  T sc[CPT], run = T(0);
  own_load<CPT>(L, sc);
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    run += sc[k];
    sc[k] = run;
  }
  const T ws = wscan(run);
#pragma unroll
  for (int k = 0; k < CPT; ++k) sc[k] += ws - run;
  own_store<CPT>(L, sc);
  if (lane == 63) wA[wv] = ws;
  __syncthreads();
  const T wt = kb::lds_wave_values<BW>(wA, lane, T(0));
  const T wex = wscan_first<BW>(wt) - wt;  // lane x < BW: offset of wavefront x
  const T A = a.A[row];
  const T rms = msafe(a.rowmax[child]);
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const int s = tid + k * BT;
    const int q = pos[k] > 0 ? pos[k] - 1 : 0, e = end[k] - 1;
    const T pq = L[q] + shfl_of(wex, q / SEG), pe = L[e] + shfl_of(wex, e / SEG);
    if (s < S) {
      const T pm1 = pos[k] > 0 ? pq : T(0);
      udr[s] = pe - pm1;
      crow[s] = xexp2(pic[k] - rms) * (pm1 + (A - pe));
    }
  }
}

// ---- fixed-order row accumulation -------------------------------------------------------

// Workgroup x takes the runs that start at sorted entries SCAT_K x .. SCAT_K x +
// SCAT_K - 1.  Mostly a run is one row (a child row has one parent): those are
// loaded and added together; longer runs are summed in order first.  One entry
// per workgroup waited out a chain of four loads for 1 KB of data: 34 us per wave
// of 2047 states against 26 us (1023-state waves of a few rows 5.2 against 5.4).
constexpr int SCAT_K = 4;

template <typename T>
__global__ __launch_bounds__(256) void scatter_add_kernel(int S, long long n, const T* src, const int* order,
                                                          const int64_t* keys, T* dst, long long dst_stride) {
  const long long k0 = (long long)blockIdx.x * SCAT_K;
  const int s = blockIdx.y * 256 + threadIdx.x;
  if (s >= S) return;
  long long key[SCAT_K];
  bool one[SCAT_K], run[SCAT_K];  // the entry is a run of one row / starts a longer run
  T x[SCAT_K], d[SCAT_K];
#pragma unroll
  for (int u = 0; u < SCAT_K; ++u) {
    const long long k = k0 + u;
    key[u] = k < n ? keys[k] : -1;
    const bool first = key[u] >= 0 && (k == 0 || keys[k - 1] != key[u]);
    const bool more = first && k + 1 < n && keys[k + 1] == key[u];
    one[u] = first && !more;
    run[u] = more;
    x[u] = d[u] = T(0);
    if (one[u]) {
      x[u] = src[(size_t)order[k] * S + s];
      d[u] = dst[(size_t)(key[u] * dst_stride) + s];
    }
  }
#pragma unroll
  for (int u = 0; u < SCAT_K; ++u)
    if (one[u]) dst[(size_t)(key[u] * dst_stride) + s] = d[u] + x[u];
#pragma unroll
  for (int u = 0; u < SCAT_K; ++u) {
    if (!run[u]) continue;
    const long long k = k0 + u;
    long long e = k + 2;  // end of the run of this key (the same for every thread)
    while (e < n && keys[e] == key[u]) ++e;
    // the run's rows added in order; the loads of eight rows are issued before their adds
    T acc = 0;
    long long j = k;
    for (; j + 8 <= e; j += 8) {
      T y[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) y[i] = src[(size_t)order[j + i] * S + s];
#pragma unroll
      for (int i = 0; i < 8; ++i) acc += y[i];
    }
    for (; j < e; ++j) acc += src[(size_t)order[j] * S + s];
    dst[(size_t)(key[u] * dst_stride) + s] += acc;
  }
}

// Column sums of row blocks: a workgroup of SUM_G wavefronts takes 64 columns
// of a chunk of SUM_CHUNK rows, each wavefront an equal range of the chunk's
// rows (added in row order), and the wavefronts' sums are added in order.  The
// partition depends on the row count only.  The waves of a pass have tens to
// hundreds of rows: one launch for up to SUM_CHUNK of them, each thread waiting
// for a sixteenth of the rows (before, 256 columns a workgroup and 64 rows a
// thread, and a second launch past 64 rows): the Hessian product of 1023 states
// 433 -> 398 launches, 2.80 -> 2.75 ms.
constexpr int SUM_CHUNK = 1024;
constexpr int SUM_G = 16;

// sum(r0, r1) over this workgroup's rows; valid in wavefront 0
template <typename F>
__device__ __forceinline__ double chunk_rows(long long r0, long long r1, bool col_ok, F&& sum) {
  __shared__ double red[SUM_G][64];
  const int g = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const long long q = (r1 - r0 + SUM_G - 1) / SUM_G;
  const long long a = r0 + g * q, b = min(r1, a + q);
  red[g][lane] = col_ok && a < b ? sum(a, b) : 0.0;
  __syncthreads();
  double acc = 0.0;
  if (g == 0) {
#pragma unroll
    for (int i = 0; i < SUM_G; ++i) acc += red[i][lane];
  }
  return acc;
}

// Sum over rows r0 <= r < r1 of column s of a row-major block with S columns,
// added in row order in float64 (with a second block B, each row's A + B is
// formed first).  The loads of eight rows are issued before their adds: the
// adds keep their order, so the sum is the one of the plain loop.
template <typename T>
__device__ __forceinline__ double col_sum(const T* A, const T* B, int S, long long r0, long long r1, int s) {
  double acc = 0.0;
  long long r = r0;
  for (; r + 8 <= r1; r += 8) {
    T x[8], y[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = A[(size_t)(r + i) * S + s];
    if (B) {
#pragma unroll
      for (int i = 0; i < 8; ++i) y[i] = B[(size_t)(r + i) * S + s];
#pragma unroll
      for (int i = 0; i < 8; ++i) acc += (double)x[i] + (double)y[i];
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) acc += (double)x[i];
    }
  }
  for (; r < r1; ++r) {
    double x = (double)A[(size_t)r * S + s];
    if (B) x += (double)B[(size_t)r * S + s];
    acc += x;
  }
  return acc;
}

// Sum over chunks c < n of work[c * S + s], in chunk order, eight loads ahead.
__device__ __forceinline__ double chunk_sum(const double* work, int S, int n, int s) {
  double acc = 0.0;
  int c = 0;
  for (; c + 8 <= n; c += 8) {
    double x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = work[(size_t)(c + i) * S + s];
#pragma unroll
    for (int i = 0; i < 8; ++i) acc += x[i];
  }
  for (; c < n; ++c) acc += work[(size_t)c * S + s];
  return acc;
}

// One chunk: added to dst; more: their partials to work.
template <typename T>
__global__ __launch_bounds__(64 * SUM_G) void rows_sum_stage1(int S, long long n, const T* src, double* work, T* dst) {
  const int s = blockIdx.x * 64 + (threadIdx.x & 63);
  const long long r0 = (long long)blockIdx.y * SUM_CHUNK;
  const double acc = chunk_rows(r0, min(n, r0 + SUM_CHUNK), s < S,
                                [&](long long a, long long b) { return col_sum<T>(src, nullptr, S, a, b, s); });
  if (threadIdx.x >= 64 || s >= S) return;
  if (gridDim.y == 1)
    dst[s] = (T)((double)dst[s] + acc);
  else
    work[(size_t)blockIdx.y * S + s] = acc;
}

// Column sums of up to 8 row blocks in one launch (grid z = block): row chunk
// y of block j, summed in float64 (chunk_rows); one chunk writes the result,
// more write partials that rows_sum_multi_stage2 adds in chunk order.
struct RsmArgs {
  int S, m, chunks;
  long long n;
  const void* a[8];
  const void* b[8];  // optional second addend of each block
};

template <typename T>
__global__ __launch_bounds__(64 * SUM_G) void rows_sum_multi_stage1(RsmArgs p, double* work, T* out) {
  const int s = blockIdx.x * 64 + (threadIdx.x & 63);
  const int j = blockIdx.z, c = blockIdx.y;
  const T* A = static_cast<const T*>(p.a[j]);
  const T* B = static_cast<const T*>(p.b[j]);
  const long long r0 = (long long)c * SUM_CHUNK;
  const double acc = chunk_rows(r0, min(p.n, r0 + SUM_CHUNK), s < p.S,
                                [&](long long a, long long b) { return col_sum<T>(A, B, p.S, a, b, s); });
  if (threadIdx.x >= 64 || s >= p.S) return;
  if (p.chunks == 1)
    out[(size_t)j * p.S + s] = (T)acc;
  else
    work[((size_t)j * p.chunks + c) * p.S + s] = acc;
}

template <typename T>
__global__ __launch_bounds__(256) void rows_sum_multi_stage2(RsmArgs p, const double* work, T* out) {
  const int s = blockIdx.x * 256 + threadIdx.x;
  if (s >= p.S) return;
  const int j = blockIdx.z;
  out[(size_t)j * p.S + s] = (T)chunk_sum(work + (size_t)j * p.chunks * p.S, p.S, p.chunks, s);
}

// Column sums of up to 8 row blocks, each added into its own accumulator row:
// block j has n[j] rows of k[j] <= 4 addends (each row's addends summed first,
// in order), summed in float64 (chunk_rows).  Blocks of one chunk add into
// their accumulator in stage 1 when no block has more (one launch); otherwise
// stage 1 writes every block's chunk partials and stage 2 adds them in chunk
// order, so each accumulator gets dst + sum, as rows_sum_stage1 /
// rows_sum_stage2 form it.
struct RsaArgs {
  int S, m, chunks;  // chunks: the most any block has
  long long n[8];
  int k[8];
  const void* a[8][4];
  void* dst[8];
};

template <typename T>
__device__ __forceinline__ double col_sum_k(const RsaArgs& p, int j, long long r0, long long r1, int s) {
  const int S = p.S;
  const T* A0 = static_cast<const T*>(p.a[j][0]);
  if (p.k[j] == 1) return col_sum<T>(A0, nullptr, S, r0, r1, s);
  if (p.k[j] == 2) return col_sum<T>(A0, static_cast<const T*>(p.a[j][1]), S, r0, r1, s);
  const T* A1 = static_cast<const T*>(p.a[j][1]);
  const T* A2 = static_cast<const T*>(p.a[j][2]);
  const T* A3 = p.k[j] > 3 ? static_cast<const T*>(p.a[j][3]) : nullptr;
  double acc = 0.0;
  long long r = r0;
  for (; r + 4 <= r1; r += 4) {
    T x[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const size_t o = (size_t)(r + i) * S + s;
      x[i][0] = A0[o];
      x[i][1] = A1[o];
      x[i][2] = A2[o];
      x[i][3] = A3 ? A3[o] : T(0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      double v = (double)x[i][0] + (double)x[i][1] + (double)x[i][2];
      if (A3) v += (double)x[i][3];
      acc += v;
    }
  }
  for (; r < r1; ++r) {
    const size_t o = (size_t)r * S + s;
    double v = (double)A0[o] + (double)A1[o] + (double)A2[o];
    if (A3) v += (double)A3[o];
    acc += v;
  }
  return acc;
}

template <typename T>
__global__ __launch_bounds__(64 * SUM_G) void rows_sum_accum_stage1(RsaArgs p, double* work) {
  const int s = blockIdx.x * 64 + (threadIdx.x & 63);
  const int j = blockIdx.z, c = blockIdx.y;
  const long long r0 = (long long)c * SUM_CHUNK;
  if (r0 >= p.n[j] && p.chunks > 1) return;
  const double acc = chunk_rows(r0, min(p.n[j], r0 + SUM_CHUNK), s < p.S,
                                [&](long long a, long long b) { return col_sum_k<T>(p, j, a, b, s); });
  if (threadIdx.x >= 64 || s >= p.S) return;
  if (p.chunks == 1) {
    T* D = static_cast<T*>(p.dst[j]);
    D[s] = (T)((double)D[s] + acc);
  } else {
    work[((size_t)j * p.chunks + c) * p.S + s] = acc;
  }
}

template <typename T>
__global__ __launch_bounds__(256) void rows_sum_accum_stage2(RsaArgs p, const double* work) {
  const int s = blockIdx.x * 256 + threadIdx.x;
  const int j = blockIdx.z;
  if (s >= p.S || p.n[j] <= 0) return;
  const int nc = (int)((p.n[j] + SUM_CHUNK - 1) / SUM_CHUNK);
  T* D = static_cast<T*>(p.dst[j]);
  D[s] = (T)((double)D[s] + chunk_sum(work + (size_t)j * p.chunks * p.S, p.S, nc, s));
}

template <typename T>
__global__ __launch_bounds__(256) void rows_sum_stage2(int S, int n_chunks, const double* work, T* dst) {
  const int s = blockIdx.x * 256 + threadIdx.x;
  if (s >= S) return;
  const double acc = chunk_sum(work, S, n_chunks, s);
  dst[s] = (T)((double)dst[s] + acc);
}

}  // namespace kbo

// Device scratch of kb_estep_vjp_noalloc: the [G, S] float64 grad_col
// contributions.  Each GPU holds its own copy for the life of the process; in
// host code its name is only a symbol handle, so the address used in launches
// comes from hipGetSymbolAddress (scratch_on_current_device below).
static __device__ __align__(256) double scratch[KB_ESTEP_VJP_NOALLOC_MAX];

// =====================================================================================
// host side
// =====================================================================================

// The smallest workgroup whose BT * CPT positions hold a row (see estep_kernel,
// dts_cross_kernel, pibar_vjp_kernel).
#define KBO_SHAPE(S, ...)                                                      \
  do {                                                                               \
    if ((S) <= 128) { constexpr int BT = 64, CPT = 2; __VA_ARGS__; }                 \
    else if ((S) <= 256) { constexpr int BT = 128, CPT = 2; __VA_ARGS__; }           \
    else if ((S) <= 512) { constexpr int BT = 256, CPT = 2; __VA_ARGS__; }           \
    else if ((S) <= 1024) { constexpr int BT = 512, CPT = 2; __VA_ARGS__; }          \
    else if ((S) <= 2048) { constexpr int BT = 512, CPT = 4; __VA_ARGS__; }          \
    else if ((S) <= 4096) { constexpr int BT = 1024, CPT = 4; __VA_ARGS__; }         \
    else { constexpr int BT = 1024, CPT = 8; __VA_ARGS__; }                          \
  } while (0)

// Dispatch over the element type.
#define KBO_TYPE(DTYPE, S, ...)                                                      \
  do {                                                                               \
    if (cpt_for(S) == 0) return kb::set_error(KB_ERR_ARG, "S=%d exceeds 8192", S);   \
    if ((DTYPE) == KB_F64) { using T = double; __VA_ARGS__; }                        \
    else { using T = float; __VA_ARGS__; }                                           \
  } while (0)

namespace {

using namespace kbo_host;

// Address of `scratch` on the current device, looked up once per device.
int scratch_on_current_device(double** out) {
  static std::mutex mu;
  static std::vector<double*> addr;  // by device ordinal; nullptr until looked up
  int dev = -1;
  KBO_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(mu);
  if ((int)addr.size() <= dev) addr.resize(dev + 1, nullptr);
  if (!addr[dev]) {
    void* p = nullptr;
    KBO_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    addr[dev] = static_cast<double*>(p);
  }
  *out = addr[dev];
  return 0;
}


int put(int** dst, const std::vector<int>& v) {
  *dst = nullptr;
  KBO_HIP(hipMalloc((void**)dst, std::max<size_t>(1, v.size()) * sizeof(int)));
  if (!v.empty()) KBO_HIP(hipMemcpy(*dst, v.data(), v.size() * sizeof(int), hipMemcpyHostToDevice));
  return 0;
}

}  // namespace

extern "C" {

int kb_tree_create(int32_t S, const int64_t* parent, const int64_t* child1, const int64_t* child2, kb_tree** out) {
  if (!out || !parent || !child1 || !child2) return kb::set_error(KB_ERR_ARG, "null argument");
  *out = nullptr;
  if (S < 1 || S > 8192) return kb::set_error(KB_ERR_ARG, "S=%d outside [1, 8192]", S);
  std::vector<int> par(S), c1(S), c2(S);
  int root = -1;
  for (int s = 0; s < S; ++s) {
    const int64_t p = parent[s];
    if (p < 0 || p >= S) {
      if (root >= 0) return kb::set_error(KB_ERR_ARG, "node_parent has more than one root (%d, %d)", root, s);
      root = s;
      par[s] = -1;
    } else {
      par[s] = (int)p;
    }
    c1[s] = (child1[s] >= 0 && child1[s] < S) ? (int)child1[s] : -1;
    c2[s] = (child2[s] >= 0 && child2[s] < S) ? (int)child2[s] : -1;
  }
  if (root < 0) return kb::set_error(KB_ERR_ARG, "node_parent has no root");
  for (int s = 0; s < S; ++s) {
    for (int c : {c1[s], c2[s]})
      if (c >= 0 && par[c] != s)
        return kb::set_error(KB_ERR_ARG, "node_child of %d is %d but node_parent[%d] = %d", s, c, c, par[c]);
    if (par[s] >= 0 && c1[par[s]] != s && c2[par[s]] != s)
      return kb::set_error(KB_ERR_ARG, "node %d is not a child of its parent %d", s, par[s]);
  }
  // preorder DFS (child1 first), Euler tour
  std::vector<int> pcol, ppos(S, -1), pend(S, 0), tin(S, 0), ev;
  pcol.reserve(S);
  ev.reserve(2 * S);
  std::vector<std::pair<int, int>> stack;  // (node, state) 0: enter, 1: exit
  stack.push_back({root, 0});
  while (!stack.empty()) {
    auto [n, state] = stack.back();
    stack.pop_back();
    if (state == 0) {
      if (ppos[n] >= 0) return kb::set_error(KB_ERR_ARG, "species tree has a cycle at node %d", n);
      ppos[n] = (int)pcol.size();
      pcol.push_back(n);
      tin[n] = (int)ev.size();
      ev.push_back(n << 1);
      stack.push_back({n, 1});
      if (c2[n] >= 0) stack.push_back({c2[n], 0});
      if (c1[n] >= 0) stack.push_back({c1[n], 0});
    } else {
      pend[n] = (int)pcol.size();
      ev.push_back((n << 1) | 1);
    }
  }
  if ((int)pcol.size() != S)
    return kb::set_error(KB_ERR_ARG, "species tree is not connected (%zu of %d nodes reachable)", pcol.size(), S);
  // preorder-position tables of the contiguous-ownership sweeps
  std::vector<int> pc1(S), pc2(S), pnex(S), ppost;
  ppost.reserve(S);
  for (int i = 0; i < S; ++i) {
    const int n = pcol[i];
    pc1[i] = c1[n] >= 0 ? ppos[c1[n]] : -1;
    pc2[i] = c2[n] >= 0 ? ppos[c2[n]] : -1;
    pnex[i] = tin[n] - i;
  }
  for (int e : ev)
    if (e & 1) ppost.push_back(ppos[e >> 1]);
  kb_tree* t = new kb_tree();
  t->S = S;
  int rc = 0;
  rc |= put(&t->par, par);
  rc |= put(&t->c1, c1);
  rc |= put(&t->c2, c2);
  rc |= put(&t->ev, ev);
  rc |= put(&t->tin, tin);
  rc |= put(&t->pcol, pcol);
  rc |= put(&t->ppos, ppos);
  rc |= put(&t->pend, pend);
  rc |= put(&t->pc1, pc1);
  rc |= put(&t->pc2, pc2);
  rc |= put(&t->pnex, pnex);
  rc |= put(&t->ppost, ppost);
  if (rc) {
    kb_tree_destroy(t);
    return KB_ERR_HIP;
  }
  *out = t;
  return 0;
}

void kb_tree_destroy(kb_tree* t) {
  if (!t) return;
  for (int* p : {t->par, t->c1, t->c2, t->ev, t->tin, t->pcol, t->ppos, t->pend, t->pc1,
                 t->pc2, t->pnex, t->ppost})
    if (p) (void)hipFree(p);
  delete t;
}

int kb_ops_max_states(int dtype) {
  // wave_step / wave_backward use 4 S elements of LDS per row
  const size_t per = 4 * elem_size(dtype);
  size_t s = LDS_BYTES / per;
  return (int)std::min<size_t>(8192, s);
}

}  // extern "C"

template <typename T>
static int launch_estep_rows(const kbo::OpsTree& t, const kbo::EsArgs<T>& a, hipStream_t st) {
  KBO_SHAPE(t.S, {
    const size_t lds = (size_t)2 * (BT * CPT + 64) * sizeof(double);
    auto k = a.use_col ? kbo::estep_kernel<T, BT, CPT, true> : kbo::estep_kernel<T, BT, CPT, false>;
    if (int rc = set_lds(k, lds)) return rc;
    hipLaunchKernelGGL(k, dim3(a.G), dim3(BT), lds, st, t, a);
  });
  return 0;
}
template <typename T>
static int launch_estep_vjp_rows(const kbo::OpsTree& t, const kbo::EvArgs<T>& a, hipStream_t st) {
  KBO_SHAPE(t.S, {
    const size_t lds = (size_t)2 * (BT * CPT + 64) * sizeof(double);
    auto k = kbo::estep_vjp_kernel<T, BT, CPT>;
    if (int rc = set_lds(k, lds)) return rc;
    hipLaunchKernelGGL(k, dim3(a.G), dim3(BT), lds, st, t, a);
  });
  return 0;
}

extern "C" {

int kb_estep(const kb_tree* tr, const kb_estep_io* io, void* stream) {
  if (!tr || !io) return kb::set_error(KB_ERR_ARG, "null argument");
  if (int rc = dtype_ok(io->dtype)) return rc;
  if (io->G < 0) return kb::set_error(KB_ERR_ARG, "G must be non-negative");
  if (io->mode == 1 && (io->max_iter < 1 || !(io->tol > 0.0)))
    return kb::set_error(KB_ERR_ARG, "max_iter must be >= 1 and tol > 0");
  if (io->G == 0) return 0;
  const int S = tr->S;
  const kbo::OpsTree t = tr->dev();
  KBO_DISPATCH(io->dtype, S, {
    kbo::EsArgs<T> a{io->G, S, io->mode, io->use_col_weights, io->max_iter, io->tol,
                     (const T*)io->E, (const T*)io->log_pS, (const T*)io->log_pD, (const T*)io->log_pL,
                     (const T*)io->max_coupling, (const T*)io->col_log_probs,
                     (T*)io->E_out, (T*)io->E_s1, (T*)io->E_s2, (T*)io->Ebar, (T*)io->max_diff, io->n_iter};
    if (int rc = launch_estep_rows<T>(t, a, st_of(stream))) return rc;
  });
  KBO_HIP(hipGetLastError());
  return 0;
}

}  // extern "C"

namespace {

// The E-step VJP launches with `work` ([G, S] float64) as the grad_col staging rows.
int estep_vjp_launch(const kb_tree* tr, const kb_estep_vjp_io* io, double* work, void* stream) {
  const int S = tr->S;
  const kbo::OpsTree t = tr->dev();
  KBO_DISPATCH(io->dtype, S, {
    kbo::EvArgs<T> a{io->G, S, io->use_col_weights,
                     (const T*)io->E, (const T*)io->E_new, (const T*)io->E_s1, (const T*)io->E_s2, (const T*)io->Ebar,
                     (const T*)io->log_pS, (const T*)io->log_pD, (const T*)io->log_pL, (const T*)io->col_log_probs,
                     (const T*)io->g_E_new, (const T*)io->g_E_s1, (const T*)io->g_E_s2, (const T*)io->g_Ebar,
                     (T*)io->grad_E, (T*)io->grad_log_pS, (T*)io->grad_log_pD, (T*)io->grad_log_pL,
                     (T*)io->grad_max_coupling, work};
    if (int rc = launch_estep_vjp_rows<T>(t, a, st_of(stream))) return rc;
    // grad_col += sum over item rows of the per-row contributions (fixed row order)
    hipLaunchKernelGGL((kbo::rows_sum_stage2<T>), dim3((S + 255) / 256), dim3(256), 0, st_of(stream), S, io->G,
                       (const double*)work, (T*)io->grad_col_log_probs);
  });
  KBO_HIP(hipGetLastError());
  return 0;
}

}  // namespace

namespace {
// Chains of float sweeps run the linear-space preorder-ownership kernel, which
// keeps the row in linear space between sweeps (three LDS rows of NT * CPT + 64
// floats); single sweeps and float64 rows wave_step_kernel.  A chain agrees
// with the same sweeps launched one at a time to float32 rounding.
template <typename T, int BT, int CPT>
int launch_step(const kbo::OpsTree& t, const kbo::WsArgs<T>& a, int W, hipStream_t st) {
  constexpr int MAXS = BT * CPT;
  const size_t lds = (2 * (MAXS + 64) + (kbo::step_consts_in_lds<T>(MAXS) ? 4 * MAXS : 0)) * sizeof(T);
  auto k = a.use_col ? kbo::wave_step_kernel<T, BT, CPT, true> : kbo::wave_step_kernel<T, BT, CPT, false>;
  if (int rc = set_lds(k, lds)) return rc;
  hipLaunchKernelGGL(k, dim3(std::min(W, resident_blocks(k, BT, lds))), dim3(BT), lds, st, t, a);
  return 0;
}

template <typename T, int CPT>
int launch_wave_step(const kbo::OpsTree& t, const kbo::WsArgs<T>& a, int W, hipStream_t st) {
  if constexpr (std::is_same_v<T, float>) {
    if (a.n_sweeps > 1) {
      const size_t lds_lin = (size_t)3 * (kbo::NT * CPT + 64) * sizeof(float);
      auto k = kbo::wave_step_lin_kernel<CPT>;
      if (int rc = set_lds(k, lds_lin)) return rc;
      hipLaunchKernelGGL(k, dim3(W), dim3(kbo::NT), lds_lin, st, t, a);
      return 0;
    }
  }
  // The smallest shape that holds the row.  Times of the 15 sweeps and the split
  // term of a wave through the wrappers, against one 1024-thread workgroup per
  // row with an Euler-tour scan and log-space sums: 127 states, 5015 rows 1240 ->
  // 243 us; 1023 states, 2386 rows 817 -> 285 us; 2047 states, 2140 rows 1047 ->
  // 441 us (weighted 1057 -> 492 us); 4095 states, 721 rows 650 -> 364 us; 7999
  // states, 515 rows 2300 -> 1360 us.  float64: 511 states, 2550 rows 1289 -> 403
  // us, 1023 states 1667 -> 687 us, 2047 states 3434 -> 1220 us.  (Other shapes
  // for one size: 2047 floats on 1024 x 2 an eighth slower than on 512 x 4, 1023
  // on 256 x 4 an eighth slower than on 512 x 2; doubles of 2047 on 1024 x 2 spill,
  // a quarter slower, of 1023 on 512 x 2 a fifth.)  A sweep of 2140 x 2047 floats
  // moves 53 MB (10 us at 5.3 TB/s) in about 28 us: barriers and the LDS round
  // trips of a row, with two to three rows per CU.
  const int S = t.S;
  constexpr bool F32 = std::is_same_v<T, float>;
  if (S <= 128) return launch_step<T, 64, 2>(t, a, W, st);
  if (S <= 256) return launch_step<T, 128, 2>(t, a, W, st);
  if (S <= 512) return launch_step<T, 256, 2>(t, a, W, st);
  if (S <= 1024) return launch_step<T, F32 ? 512 : 256, F32 ? 2 : 4>(t, a, W, st);
  if (S <= 2048) return launch_step<T, 512, 4>(t, a, W, st);
  if (S <= 4096) return launch_step<T, 1024, 4>(t, a, W, st);
  return launch_step<T, 1024, 8>(t, a, W, st);
}

template <typename T, int BT, int CPT>
int launch_bwd(const kbo::OpsTree& t, const kbo::WbArgs<T>& a, int W, hipStream_t st) {
  const size_t lds = (size_t)4 * (BT * CPT + 64) * sizeof(T);
  auto k = kbo::wave_bwd_pre_kernel<T, BT, CPT>;
  if (int rc = set_lds(k, lds)) return rc;
  hipLaunchKernelGGL(k, dim3(W), dim3(BT), lds, st, t, a);
  return 0;
}

// The preorder-ownership kernel on the smallest shape that holds the row (floats
// of 513..1024 states on 1024 x 1: 19.1 us a narrow wave against 20.9 on 512 x
// 2); its four padded LDS rows do not hold doubles past 4096 states, where the
// column-order kernel (four rows of S) goes on.  Doubles against that kernel:
// 1500 rows of 599 states 228 -> 79 us.
template <typename T>
int launch_wave_bwd(const kbo::OpsTree& t, const kbo::WbArgs<T>& a, int W, size_t lds, hipStream_t st) {
  constexpr bool F32 = std::is_same_v<T, float>;
  const int S = t.S;
  if (S <= 128) return launch_bwd<T, 64, 2>(t, a, W, st);
  if (S <= 256) return launch_bwd<T, 128, 2>(t, a, W, st);
  if (S <= 512) return launch_bwd<T, 256, 2>(t, a, W, st);
  if (S <= 1024) return launch_bwd<T, F32 ? 1024 : 512, F32 ? 1 : 2>(t, a, W, st);
  if (S <= 2048) return launch_bwd<T, 1024, 2>(t, a, W, st);
  if (S <= 4096) return launch_bwd<T, 1024, 4>(t, a, W, st);
  if constexpr (F32) return launch_bwd<T, 1024, 8>(t, a, W, st);
  auto k = kbo::wave_bwd_kernel<T, 8>;
  if (int rc = set_lds(k, lds)) return rc;
  hipLaunchKernelGGL(k, dim3(W), dim3(kbo::NT), lds, st, t, a);
  return 0;
}

}  // namespace

extern "C" {

int kb_estep_vjp(const kb_tree* tr, const kb_estep_vjp_io* io, void* stream) {
  if (!tr || !io || !io->work) return kb::set_error(KB_ERR_ARG, "null argument");
  if (int rc = dtype_ok(io->dtype)) return rc;
  if (io->G <= 0) return kb::set_error(KB_ERR_ARG, "G must be positive");
  return estep_vjp_launch(tr, io, io->work, stream);
}

int kb_estep_vjp_noalloc(const kb_tree* tr, const kb_estep_vjp_io* io, void* stream) {
  if (!tr || !io) return kb::set_error(KB_ERR_ARG, "null argument");
  if (io->work) return kb::set_error(KB_ERR_ARG, "kb_estep_vjp_noalloc takes no work buffer (io->work must be NULL)");
  if (int rc = dtype_ok(io->dtype)) return rc;
  if (io->G <= 0) return kb::set_error(KB_ERR_ARG, "G must be positive");
  if ((int64_t)io->G * tr->S > (int64_t)KB_ESTEP_VJP_NOALLOC_MAX)
    return kb::set_error(KB_ERR_ARG, "kb_estep_vjp_noalloc: G * S = %lld exceeds its scratch of %d doubles",
                         (long long)io->G * tr->S, (int)KB_ESTEP_VJP_NOALLOC_MAX);
  double* work = nullptr;
  if (int rc = scratch_on_current_device(&work)) return rc;
  return estep_vjp_launch(tr, io, work, stream);
}

int kb_wave_step(const kb_tree* tr, const kb_wave_step_io* io, void* stream) {
  if (!tr || !io) return kb::set_error(KB_ERR_ARG, "null argument");
  if (int rc = dtype_ok(io->dtype)) return rc;
  if (io->S != tr->S) return kb::set_error(KB_ERR_ARG, "S=%d does not match the tree (%d)", io->S, tr->S);
  if (io->W <= 0) return 0;
  const int S = io->S;
  const size_t lds = (size_t)4 * S * elem_size(io->dtype);
  if (int rc = check_lds(lds, S, io->dtype)) return rc;
  const kbo::OpsTree t = tr->dev();
  KBO_DISPATCH(io->dtype, S, {
    kbo::WsArgs<T> a{S, io->W, io->use_col_weights, io->use_leaf_index, io->store_final_pibar,
                     io->n_sweeps > 1 ? io->n_sweeps : 1, io->ws, io->pi_ws,
                     io->const_stride, (const T*)io->Pi_in, (T*)io->Pi_out, (T*)io->Pibar, (T*)io->pibar_row_max,
                     io->pi_residual, (const T*)io->dts, (const T*)io->max_coupling, (const T*)io->DL,
                     (const T*)io->Ebar, (const T*)io->E, (const T*)io->SL1, (const T*)io->SL2,
                     (const T*)io->col_log_probs, io->item_idx, io->leaf_state, (const T*)io->leaf_logp};
    if (int rc = launch_wave_step<T, CPT>(t, a, io->W, st_of(stream))) return rc;
  });
  KBO_HIP(hipGetLastError());
  return 0;
}

int kb_leaf_init(const kb_leaf_init_io* io, void* stream) {
  if (!io) return kb::set_error(KB_ERR_ARG, "null argument");
  if (int rc = dtype_ok(io->dtype)) return rc;
  if (io->W <= 0) return 0;
  if (!io->node_child1 || !io->node_child2) return kb::set_error(KB_ERR_ARG, "node_child1/2 are required");
  dim3 g(io->W, (io->S + 255) / 256);
  if (io->dtype == KB_F64) {
    using T = double;
    kbo::LiArgs<T> a{io->S, io->W, io->use_col_weights, io->ws, io->const_stride, (T*)io->Pi_out,
                     (const T*)io->max_coupling, (const T*)io->DL, (const T*)io->Ebar, (const T*)io->E,
                     (const T*)io->SL1, (const T*)io->SL2, (const T*)io->col_log_probs, io->subtree_start,
                     io->subtree_end, io->item_idx, io->leaf_state, io->node_child1, io->node_child2,
                     (const T*)io->leaf_logp};
    hipLaunchKernelGGL(kbo::leaf_init_kernel<T>, g, dim3(256), 0, st_of(stream), a);
  } else {
    using T = float;
    kbo::LiArgs<T> a{io->S, io->W, io->use_col_weights, io->ws, io->const_stride, (T*)io->Pi_out,
                     (const T*)io->max_coupling, (const T*)io->DL, (const T*)io->Ebar, (const T*)io->E,
                     (const T*)io->SL1, (const T*)io->SL2, (const T*)io->col_log_probs, io->subtree_start,
                     io->subtree_end, io->item_idx, io->leaf_state, io->node_child1, io->node_child2,
                     (const T*)io->leaf_logp};
    hipLaunchKernelGGL(kbo::leaf_init_kernel<T>, g, dim3(256), 0, st_of(stream), a);
  }
  KBO_HIP(hipGetLastError());
  return 0;
}

int kb_dts_forward(const kb_dts_io* io, void* stream) {
  if (!io) return kb::set_error(KB_ERR_ARG, "null argument");
  if (int rc = dtype_ok(io->dtype)) return rc;
  if (io->W <= 0) return 0;
  if (!io->node_child1 || !io->node_child2) return kb::set_error(KB_ERR_ARG, "node_child1/2 are required");
  const int S = io->S;
  KBO_DISPATCH(io->dtype, S, {
    kbo::DtsArgs<T> a{S, io->W, io->param_by_state, io->item_offset, io->param_row_stride, (const T*)io->Pi,
                      (const T*)io->Pibar, (const T*)io->log_split_probs, (const T*)io->log_pD,
                      (const T*)io->log_pS, io->sl, io->sr, io->item_idx, io->node_child1, io->node_child2,
                      io->split_ptr, io->split_order, io->active, (T*)io->out};
    hipLaunchKernelGGL((kbo::dts_kernel<T, CPT>), dim3(io->W), dim3(kbo::NT), 0, st_of(stream), a);
  });
  KBO_HIP(hipGetLastError());
  return 0;
}

int kb_active_mask(int32_t dtype, int32_t W, int32_t S, int64_t row_stride, const void* rhs, float threshold,
                   int32_t strict, uint8_t* active, void* stream) {
  if (W < 0 || S < 0) return kb::set_error(KB_ERR_ARG, "bad sizes");
  if (W == 0) return 0;
  if (!rhs || !active) return kb::set_error(KB_ERR_ARG, "null argument");
  if (dtype == KB_F64)
    hipLaunchKernelGGL(kbo::active_kernel<double>, dim3(W), dim3(256), 0, st_of(stream), S, (long long)row_stride,
                       (const double*)rhs, threshold, strict, active);
  else if (dtype == KB_BF16)
    hipLaunchKernelGGL(kbo::active_kernel<__hip_bfloat16>, dim3(W), dim3(256), 0, st_of(stream), S,
                       (long long)row_stride, (const __hip_bfloat16*)rhs, threshold, strict, active);
  else if (dtype == KB_F32)
    hipLaunchKernelGGL(kbo::active_kernel<float>, dim3(W), dim3(256), 0, st_of(stream), S, (long long)row_stride,
                       (const float*)rhs, threshold, strict, active);
  else
    return kb::set_error(KB_ERR_ARG, "active mask supports float32, float64 and bfloat16");
  KBO_HIP(hipGetLastError());
  return 0;
}

int kb_wave_backward(const kb_tree* tr, const kb_wave_bwd_io* io, void* stream) {
  if (!tr || !io) return kb::set_error(KB_ERR_ARG, "null argument");
  if (int rc = dtype_ok(io->dtype)) return rc;
  if (io->S != tr->S) return kb::set_error(KB_ERR_ARG, "S=%d does not match the tree (%d)", io->S, tr->S);
  if (io->n_terms < 0) return kb::set_error(KB_ERR_ARG, "neumann_terms must be non-negative");
  if (io->W <= 0) return 0;
  const int S = io->S;
  const size_t lds = (size_t)4 * S * elem_size(io->dtype);
  if (int rc = check_lds(lds, S, io->dtype)) return rc;
  const kbo::OpsTree t = tr->dev();
  KBO_DISPATCH(io->dtype, S, {
    kbo::WbArgs<T> a{S, io->W, io->n_terms, io->const_layout, io->leaf_mode, io->use_leaf_index,
                     io->use_col_weights, io->ws, (const T*)io->Pi, (const T*)io->Pibar, (const T*)io->pibar_row_max,
                     (const T*)io->dts, (const T*)io->rhs, (const T*)io->initial_v, io->active, (const T*)io->max_coupling, (const T*)io->DL,
                     (const T*)io->Ebar, (const T*)io->E, (const T*)io->SL1, (const T*)io->SL2,
                     (const T*)io->col_log_probs, io->item_idx, io->leaf_state, (const T*)io->leaf_logp,
                     (const T*)io->leaf_term, (T*)io->v, (T*)io->aw0, (T*)io->aw1, (T*)io->aw2, (T*)io->aw345,
                     (T*)io->aw3, (T*)io->aw4, (T*)io->col_rows, io->relres};
    if (int rc = launch_wave_bwd<T>(t, a, io->W, lds, st_of(stream))) return rc;
  });
  KBO_HIP(hipGetLastError());
  return 0;
}

int kb_dts_cross_backward(const kb_dts_cross_io* io, void* stream) {
  if (!io) return kb::set_error(KB_ERR_ARG, "null argument");
  if (int rc = dtype_ok(io->dtype)) return rc;
  if (io->N <= 0) return 0;
  if (!io->node_child1 || !io->node_child2) return kb::set_error(KB_ERR_ARG, "node_child1/2 are required");
  if (!io->side_rows) return kb::set_error(KB_ERR_ARG, "side_rows is required");
  if (io->output_ud && (!io->ud || !io->A || !io->mt || !io->pibar_row_max))
    return kb::set_error(KB_ERR_ARG, "output_ud needs ud, A, mt and pibar_row_max");
  if (!io->output_ud && (!io->grad_Pibar_l || !io->grad_Pibar_r))
    return kb::set_error(KB_ERR_ARG, "grad_Pibar_l / grad_Pibar_r are required without output_ud");
  if ((io->param_layout >= 2 || io->mt_layout == 1) && !io->item_idx)
    return kb::set_error(KB_ERR_ARG, "item-indexed layouts need item_idx");
  const int S = io->S;
  const size_t lds = (size_t)2 * S * elem_size(io->dtype);
  if (int rc = check_lds(lds, S, io->dtype)) return rc;
  KBO_TYPE(io->dtype, S, {
    kbo::DcArgs<T> a{S, io->param_layout, io->mt_layout, io->output_ud, io->skip_inactive_ud_zero, io->N, io->ws,
                     io->side_threshold, (const T*)io->Pi, (const T*)io->Pibar, (const T*)io->v, io->active, io->sl,
                     io->sr, io->reduce_idx, io->item_idx, io->node_child1, io->node_child2, (const T*)io->wlsp, (const T*)io->log_pD,
                     (const T*)io->log_pS, (const T*)io->mt, (const T*)io->pibar_row_max, (T*)io->side_rows,
                     (T*)io->ud, (T*)io->A, io->side_active, (T*)io->grad_Pibar_l, (T*)io->grad_Pibar_r,
                     (T*)io->param_rows, (T*)io->param_sums, (T*)io->mt_rows};
    KBO_SHAPE(S, {
      auto k = kbo::dts_cross_kernel<T, BT, CPT>;
      if (int rc = set_lds(k, lds)) return rc;
      hipLaunchKernelGGL(k, dim3((unsigned)io->N), dim3(BT), lds, st_of(stream), a);
    });
  });
  KBO_HIP(hipGetLastError());
  return 0;
}

int kb_pibar_vjp(const kb_tree* tr, const kb_pibar_vjp_io* io, void* stream) {
  if (!tr || !io) return kb::set_error(KB_ERR_ARG, "null argument");
  if (int rc = dtype_ok(io->dtype)) return rc;
  if (io->S != tr->S) return kb::set_error(KB_ERR_ARG, "S=%d does not match the tree (%d)", io->S, tr->S);
  if (io->N <= 0) return 0;
  if (io->active && !io->reduce_idx) return kb::set_error(KB_ERR_ARG, "reduce_idx is required with active");
  const int S = io->S;
  const size_t lds = (size_t)2 * S * elem_size(io->dtype);
  if (int rc = check_lds(lds, S, io->dtype)) return rc;
  const kbo::OpsTree t = tr->dev();
  KBO_TYPE(io->dtype, S, {
    kbo::PvArgs<T> a{S, io->use_col_weights, io->N, (const T*)io->Pi, (const T*)io->col_log_probs, (const T*)io->A,
                     (const T*)io->pibar_row_max, (T*)io->ud, io->side_active, io->active, io->sl, io->sr,
                     io->reduce_idx, (T*)io->contrib};
    KBO_SHAPE(S, {
      const size_t bytes = (size_t)BT * CPT * sizeof(T);
      auto k = kbo::pibar_vjp_kernel<T, BT, CPT>;
      if (int rc = set_lds(k, bytes)) return rc;
      hipLaunchKernelGGL(k, dim3((unsigned)(2 * io->N)), dim3(BT), bytes, st_of(stream), t, a);
    });
  });
  KBO_HIP(hipGetLastError());
  return 0;
}

int kb_rows_scatter_add(int32_t dtype, int32_t S, int64_t n, const void* src, const int32_t* order,
                        const int64_t* keys_sorted, void* dst, int64_t dst_stride, void* stream) {
  if (n <= 0 || S <= 0) return 0;
  if (!src || !order || !keys_sorted || !dst) return kb::set_error(KB_ERR_ARG, "null argument");
  if (int rc = dtype_ok(dtype)) return rc;
  dim3 g((unsigned)((n + kbo::SCAT_K - 1) / kbo::SCAT_K), (S + 255) / 256);
  if (dtype == KB_F64)
    hipLaunchKernelGGL(kbo::scatter_add_kernel<double>, g, dim3(256), 0, st_of(stream), S, (long long)n,
                       (const double*)src, order, keys_sorted, (double*)dst, (long long)dst_stride);
  else
    hipLaunchKernelGGL(kbo::scatter_add_kernel<float>, g, dim3(256), 0, st_of(stream), S, (long long)n,
                       (const float*)src, order, keys_sorted, (float*)dst, (long long)dst_stride);
  KBO_HIP(hipGetLastError());
  return 0;
}

int kb_rows_sum_multi(int32_t dtype, int32_t S, int64_t n, int32_t m, const void* const* a, const void* const* b,
                      void* out, double* work, void* stream) {
  if (S <= 0 || m <= 0) return 0;
  if (m > 8) return kb::set_error(KB_ERR_ARG, "at most 8 row blocks per call (m=%d)", m);
  if (!a || !out) return kb::set_error(KB_ERR_ARG, "null argument");
  if (int rc = dtype_ok(dtype)) return rc;
  kbo::RsmArgs p{};
  p.S = S;
  p.m = m;
  p.n = n;
  p.chunks = (int)std::max<int64_t>(1, (n + kbo::SUM_CHUNK - 1) / kbo::SUM_CHUNK);
  for (int j = 0; j < m; ++j) {
    if (!a[j] && n > 0) return kb::set_error(KB_ERR_ARG, "row block %d is null", j);
    p.a[j] = a[j];
    p.b[j] = b ? b[j] : nullptr;
  }
  if (n > 64 && !work) return kb::set_error(KB_ERR_ARG, "work is required for more than 64 rows");
  const dim3 g1((S + 63) / 64, p.chunks, m), g2((S + 255) / 256, 1, m), b1(64 * kbo::SUM_G);
  if (dtype == KB_F64) {
    hipLaunchKernelGGL(kbo::rows_sum_multi_stage1<double>, g1, b1, 0, st_of(stream), p, work, (double*)out);
    if (p.chunks > 1)
      hipLaunchKernelGGL(kbo::rows_sum_multi_stage2<double>, g2, dim3(256), 0, st_of(stream), p, work, (double*)out);
  } else {
    hipLaunchKernelGGL(kbo::rows_sum_multi_stage1<float>, g1, b1, 0, st_of(stream), p, work, (float*)out);
    if (p.chunks > 1)
      hipLaunchKernelGGL(kbo::rows_sum_multi_stage2<float>, g2, dim3(256), 0, st_of(stream), p, work, (float*)out);
  }
  KBO_HIP(hipGetLastError());
  return 0;
}

int kb_rows_sum_accum(int32_t dtype, int32_t S, int32_t m, const int64_t* n, const int32_t* k, const void* const* a,
                      void* const* dst, double* work, void* stream) {
  if (S <= 0 || m <= 0) return 0;
  if (m > 8) return kb::set_error(KB_ERR_ARG, "at most 8 row blocks per call (m=%d)", m);
  if (!n || !k || !a || !dst) return kb::set_error(KB_ERR_ARG, "null argument");
  if (int rc = dtype_ok(dtype)) return rc;
  kbo::RsaArgs p{};
  p.S = S;
  p.m = m;
  p.chunks = 1;
  int64_t most = 0;
  for (int j = 0; j < m; ++j) {
    if (n[j] < 0) return kb::set_error(KB_ERR_ARG, "row block %d has %lld rows", j, (long long)n[j]);
    if (k[j] < 1 || k[j] > 4) return kb::set_error(KB_ERR_ARG, "row block %d has %d addends (1..4)", j, k[j]);
    if (!dst[j]) return kb::set_error(KB_ERR_ARG, "row block %d has no accumulator", j);
    for (int i = 0; i < j; ++i)
      if (dst[i] == dst[j]) return kb::set_error(KB_ERR_ARG, "row blocks %d and %d share an accumulator", i, j);
    p.n[j] = n[j];
    p.k[j] = k[j];
    p.dst[j] = dst[j];
    for (int i = 0; i < k[j]; ++i) {
      if (!a[4 * j + i] && n[j] > 0) return kb::set_error(KB_ERR_ARG, "row block %d addend %d is null", j, i);
      p.a[j][i] = a[4 * j + i];
    }
    p.chunks = (int)std::max<int64_t>(p.chunks, (n[j] + kbo::SUM_CHUNK - 1) / kbo::SUM_CHUNK);
    most = std::max(most, n[j]);
  }
  if (most > 64 && !work) return kb::set_error(KB_ERR_ARG, "work is required for blocks of more than 64 rows");
  const dim3 g1((S + 63) / 64, p.chunks, m), g2((S + 255) / 256, 1, m), b1(64 * kbo::SUM_G);
  if (dtype == KB_F64) {
    hipLaunchKernelGGL(kbo::rows_sum_accum_stage1<double>, g1, b1, 0, st_of(stream), p, work);
    if (p.chunks > 1)
      hipLaunchKernelGGL(kbo::rows_sum_accum_stage2<double>, g2, dim3(256), 0, st_of(stream), p, (const double*)work);
  } else {
    hipLaunchKernelGGL(kbo::rows_sum_accum_stage1<float>, g1, b1, 0, st_of(stream), p, work);
    if (p.chunks > 1)
      hipLaunchKernelGGL(kbo::rows_sum_accum_stage2<float>, g2, dim3(256), 0, st_of(stream), p, (const double*)work);
  }
  KBO_HIP(hipGetLastError());
  return 0;
}

int kb_rows_sum_into(int32_t dtype, int32_t S, int64_t n, const void* src, void* dst, double* work, void* stream) {
  if (n <= 0 || S <= 0) return 0;
  if (!src || !dst || !work) return kb::set_error(KB_ERR_ARG, "null argument");
  if (int rc = dtype_ok(dtype)) return rc;
  const int chunks = (int)((n + kbo::SUM_CHUNK - 1) / kbo::SUM_CHUNK);
  const dim3 g1((S + 63) / 64, chunks), g2((S + 255) / 256), b1(64 * kbo::SUM_G);
  if (dtype == KB_F64) {
    hipLaunchKernelGGL(kbo::rows_sum_stage1<double>, g1, b1, 0, st_of(stream), S, (long long)n, (const double*)src, work,
                       (double*)dst);
    if (chunks > 1)
      hipLaunchKernelGGL(kbo::rows_sum_stage2<double>, g2, dim3(256), 0, st_of(stream), S, chunks, (const double*)work,
                         (double*)dst);
  } else {
    hipLaunchKernelGGL(kbo::rows_sum_stage1<float>, g1, b1, 0, st_of(stream), S, (long long)n, (const float*)src, work,
                       (float*)dst);
    if (chunks > 1)
      hipLaunchKernelGGL(kbo::rows_sum_stage2<float>, g2, dim3(256), 0, st_of(stream), S, chunks, (const double*)work,
                         (float*)dst);
  }
  KBO_HIP(hipGetLastError());
  return 0;
}

}  // extern "C"
