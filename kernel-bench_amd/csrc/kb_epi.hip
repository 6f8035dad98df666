// Backward epilogue: E adjoint and the theta / column VJP, one workgroup, float64.
//
// Reference: kbench/api/_implicit_grad.py:373-475 (_e_adjoint_and_theta_vjp)
// with _bicgstab (_implicit_grad.py:28-94) and the E-step VJP kernels
// (pristine e_step.py:102-241), then autograd through
// extract_parameters_weighted_cols (extract_parameters.py:68-93).
//
// The E-step VJP is linear in its cotangents once E* is fixed, so the
// weights 2^(t_k - E_new), r = 2^(E - rowmax) and 1/denom are computed once;
// each BiCGSTAB mat-vec is then a child gather plus one subtree sum.
#include "kb_device.hpp"
#include "kb_kernels.hpp"

namespace kb {

// Every [S] vector lives in registers at preorder positions (thread t owns
// positions t*CPT + k; past 2048 positions the compiler keeps part of them in
// scratch memory), and the sums over the tree are register scans (DPP float64)
// with one LDS exchange:
//   * one E-step VJP (each parent hands its children their terms, and one
//     subtree sum): one barrier;
//   * one or two dot products: one barrier;
//   * ancestors-or-self sums, Pre(i) - PostEx(tin(i) - i): two barriers.
// Two LDS rows: 132 KB at 8192 positions.
//
// One workgroup, so its latency is the call's: the launch takes the smallest
// shape that holds the tree.
// Measured per call (4 BiCGSTAB steps): 127 nodes 37 -> 21 us (64 x 2 instead of
// 512 x 4), 511 nodes 38 -> 25 us, 2047 nodes 55 us; 3001 nodes 330 -> 128 us
// and 8191 nodes 630 -> 419 us (against LDS / global vectors with sums by levels).
template <int NT, int CPT>
__global__ __launch_bounds__(NT) void epilogue_pre_kernel(EpiParams P) {
  constexpr int MAXS = NT * CPT;
  constexpr int NW = NT / 64;
  constexpr int ZERO = MAXS;     // padding slot: 0 in every buffer
  constexpr int SEG = 64 * CPT;  // positions / postorder slots per wavefront
  // VJP: what each position gets from its parent (the root's stays 0);
  // path sums and child gathers: values at positions
  __shared__ __align__(16) double Xp[MAXS + 64];
  // VJP: wavefront-local inclusive preorder scan; path sums: wavefront-local
  // exclusive postorder scan
  __shared__ __align__(16) double Lv[MAXS + 64];
  __shared__ double wV[NW], wP[NW], wQ[NW], mred[NW];
  __shared__ double red[2][2 * NW];
  const PreDev& T = P.pd;
  const int S = P.S;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const double NINF = -__builtin_inf();
  const double TINY = 2.2250738585072014e-308;
  const double LN2 = 0.6931471805599453;

  int colk[CPT], c2p[CPT], nex[CPT], qp[CPT], endm1[CPT];
  bool okp[CPT], h1[CPT];
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const int i = tid * CPT + k;
    okp[k] = i < S;
    colk[k] = okp[k] ? T.col[i] : 0;
    const int a = okp[k] ? T.c1pos[i] : -1, b = okp[k] ? T.c2pos[i] : -1;
    h1[k] = a >= 0;  // child1 of i is i + 1 (preorder, child1 first)
    c2p[k] = b >= 0 ? b : ZERO;
    nex[k] = okp[k] ? T.tin[i] - i : 0;
    qp[k] = okp[k] ? T.post[i] : ZERO;
    endm1[k] = okp[k] ? T.endpos[i] - 1 : ZERO;
  }
  const int c1last = h1[CPT - 1] ? tid * CPT + CPT : ZERO;
  if (tid < 64) {
    Xp[MAXS + tid] = 0.0;
    Lv[MAXS + tid] = 0.0;
  }
  __syncthreads();

  // sums over all positions of a and b (fixed order), one barrier
  int rbuf = 0;
  auto sum2 = [&](double a, double b, double& ra, double& rb) {
    const double sa = lane_value_f64(wave_scan_incl_f64(a), 63);
    const double sb = lane_value_f64(wave_scan_incl_f64(b), 63);
    double* R = red[rbuf];
    rbuf ^= 1;
    if (lane == 0) {
      R[wv] = sa;
      R[NW + wv] = sb;
    }
    __syncthreads();
    ra = 0.0;
    rb = 0.0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      ra += R[w];
      rb += R[NW + w];
    }
  };
  auto dot = [&](const double (&a)[CPT], const double (&b)[CPT]) {
    double l = 0.0, r0, r1;
#pragma unroll
    for (int k = 0; k < CPT; ++k) l += a[k] * b[k];
    sum2(l, 0.0, r0, r1);
    return r0;
  };

  // ancestors-or-self sums of x and the total (two barriers)
  auto path_sums = [&](const double (&x)[CPT], double (&ps)[CPT], double& total) {
    double sp[CPT], ta = 0.0;
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      ta += x[k];
      sp[k] = ta;
    }
    const double wa = wave_scan_incl_f64(ta);
    lds_store_own_f64<CPT>(Xp, x);
    if (lane == 63) wP[wv] = wa;
    __syncthreads();
    const double tp = lds_wave_values<NW>(wP, lane, 0.0);
    double yq[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) yq[k] = Xp[qp[k]];
    const double ip = wave_scan_first_f64<NW>(tp);
    total = lane_value_f64(ip, NW - 1);
    const double offp = lane_value_f64(ip - tp, wv) + (wa - ta);
    double sq[CPT], tb = 0.0;
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      sq[k] = tb;
      tb += yq[k];
    }
    const double wb = wave_scan_incl_f64(tb);
#pragma unroll
    for (int k = 0; k < CPT; ++k) sq[k] += wb - tb;
    lds_store_own_f64<CPT>(Lv, sq);
    if (lane == 63) wQ[wv] = wb;
    __syncthreads();
    const double tq = lds_wave_values<NW>(wQ, lane, 0.0);
    const double iq = wave_scan_first_f64<NW>(tq);
    const double eq = iq - tq;
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int n = nex[k];
      ps[k] = (sp[k] + offp) - (Lv[n] + shfl_f64(eq, n / SEG));
    }
  };

  // subtree (descendants-or-self) sums of u after the caller's scan setup:
  // sc = wavefront-local inclusive scan (published in Lv with the wavefront
  // totals in wV before the caller's barrier); returns the total
  auto subtree_finish = [&](const double (&sc)[CPT], double (&sub)[CPT]) {
    double le[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) le[k] = Lv[endm1[k]];
    const double tv = lds_wave_values<NW>(wV, lane, 0.0);
    const double iv = wave_scan_first_f64<NW>(tv);
    const double ev = iv - tv;
    const double tot = lane_value_f64(iv, NW - 1);
    const double offv = lane_value_f64(ev, wv);
    const double pm0 = wave_prev_lane_f64(sc[CPT - 1]) + offv;  // P[i - 1] of slot 0
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const double pm1 = k == 0 ? pm0 : sc[k - 1] + offv;
      sub[k] = (le[k] + shfl_f64(ev, endm1[k] / SEG)) - pm1;
    }
    return tot;
  };

  // ---- E-step linearisation at E* (fp64 recomputation of pristine e_step.py:42-91)
  double Ev[CPT], R[CPT], ID[CPT], W0[CPT], W1[CPT], W2[CPT], W3[CPT];
  double lm = NINF;
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    Ev[k] = okp[k] ? (double)P.E[colk[k]] : 0.0;
    if (okp[k]) lm = fmax(lm, P.use_col ? (double)P.col[colk[k]] + Ev[k] : Ev[k]);
  }
  lds_store_own_f64<CPT>(Xp, Ev);  // for the child gathers (published by the barriers of the maximum)
  const double rmax = block_max<NT>(lm, mred);
  const double rms = rmax == NINF ? 0.0 : rmax;
  const double e1last = Xp[c1last];
  double Ec2[CPT];
#pragma unroll
  for (int k = 0; k < CPT; ++k) Ec2[k] = Xp[c2p[k]];
  __syncthreads();  // Xp is written again below
#pragma unroll
  for (int k = 0; k < CPT; ++k)
    R[k] = okp[k] ? exp2((P.use_col ? (double)P.col[colk[k]] + Ev[k] : Ev[k]) - rms) : 0.0;
  double Upath[CPT], rowsum;
  path_sums(R, Upath, rowsum);
  {
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      W0[k] = W1[k] = W2[k] = W3[k] = ID[k] = 0.0;
      if (!okp[k]) continue;
      const int s = colk[k];
      const double E = Ev[k];
      const double Es1 = h1[k] ? (k + 1 < CPT ? Ev[k + 1] : e1last) : NINF;
      const double Es2 = c2p[k] != ZERO ? Ec2[k] : NINF;
      const double denom = rowsum - Upath[k];
      const double Ebar = denom > 0.0 ? log2(denom) + rmax + (double)P.mt[s] : NINF;
      ID[k] = denom > 0.0 ? 1.0 / denom : 0.0;
      const double pS = P.log_pS[P.statewise ? s : 0], pD = P.log_pD[P.statewise ? s : 0];
      const double pL = P.log_pL[P.statewise ? s : 0];
      const double t0 = pS + Es1 + Es2, t1 = pD + 2.0 * E, t2 = E + Ebar, t3 = pL;
      const double m = fmax(fmax(t0, t1), fmax(t2, t3));
      const double ms = m == NINF ? 0.0 : m;
      const double En = log2(exp2(t0 - ms) + exp2(t1 - ms) + exp2(t2 - ms) + exp2(t3 - ms)) + m;
      auto wgt = [&](double t) {
        double w = exp2(t - En);
        return (w == w) ? w : 0.0;  // NaN (both -inf) -> 0
      };
      W0[k] = wgt(t0);
      W1[k] = wgt(t1);
      W2[k] = wgt(t2);
      W3[k] = wgt(t3);
    }
  }

  // E-step VJP (pristine e_step.py:164-241) at the own positions, one barrier:
  //   q_j = g W_j, wbar = q2 + gebar, tot = sum wbar ID,
  //   gE = 2 q1 + q2 + (parent's q0 + gs1 if child1, else q0 + gs2) + R (tot - subtree(wbar ID)).
  // gs1 / gs2 / gebar are column-indexed (may be null); pv = R (tot - subtree).
  auto vjp = [&](const double (&g)[CPT], const double* gs1, const double* gs2, const double* gebar,
                 double (&gE)[CPT], double (&wbar)[CPT], double (&pv)[CPT]) {
    double sc[CPT], ta = 0.0;
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int s = colk[k];
      const double q0 = g[k] * W0[k];
      if (h1[k]) Xp[tid * CPT + k + 1] = q0 + (gs1 ? gs1[s] : 0.0);
      if (c2p[k] != ZERO) Xp[c2p[k]] = q0 + (gs2 ? gs2[s] : 0.0);
      wbar[k] = g[k] * W2[k] + ((gebar && okp[k]) ? gebar[s] : 0.0);
      ta += wbar[k] * ID[k];
      sc[k] = ta;
    }
    const double wa = wave_scan_incl_f64(ta);
#pragma unroll
    for (int k = 0; k < CPT; ++k) sc[k] += wa - ta;
    lds_store_own_f64<CPT>(Lv, sc);
    if (lane == 63) wV[wv] = wa;
    __syncthreads();
    double par[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) par[k] = okp[k] && tid * CPT + k > 0 ? Xp[tid * CPT + k] : 0.0;  // position 0 is the root
    double sub[CPT];
    const double tot = subtree_finish(sc, sub);
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const double q1 = g[k] * W1[k], q2 = g[k] * W2[k];
      double acc = 2.0 * q1 + q2;
      acc += par[k];
      const double p = R[k] * (tot - sub[k]);
      gE[k] = acc + p;
      pv[k] = p;
    }
  };
  // y = x - J^T x
  auto ag = [&](const double (&xv)[CPT], double (&y)[CPT]) {
    double gE[CPT], wb[CPT], pv[CPT];
    vjp(xv, nullptr, nullptr, nullptr, gE, wb, pv);
#pragma unroll
    for (int k = 0; k < CPT; ++k) y[k] = xv[k] - gE[k];
  };

  const double* acc = P.acc;
  const double* a_pD = acc + 0 * (size_t)S;
  const double* a_pS = acc + 1 * (size_t)S;
  const double* a_E = acc + 2 * (size_t)S;
  const double* a_Ebar = acc + 3 * (size_t)S;
  const double* a_Es1 = acc + 4 * (size_t)S;
  const double* a_Es2 = acc + 5 * (size_t)S;
  const double* a_mt = acc + 6 * (size_t)S;
  const double* a_col = acc + 7 * (size_t)S;

  // ---- q_E = grad_E + d/dE [n_fam log2(norm) + <E_s1,gEs1> + <E_s2,gEs2> + <Ebar,gEbar>]
  double qE[CPT];
  {
    double le = 0.0, r0, r1;
#pragma unroll
    for (int k = 0; k < CPT; ++k)
      if (okp[k]) le += exp2(Ev[k]);
    sum2(le, 0.0, r0, r1);
    const double mean = r0 / (double)S;
    const double norm = 1.0 - mean;
    const double scale = (P.n_items_rows == P.n_fam) ? 1.0 : (double)P.n_fam;
    double zero[CPT], gE[CPT], wb[CPT], pv[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) zero[k] = 0.0;
    vjp(zero, a_Es1, a_Es2, a_Ebar, gE, wb, pv);
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const double dd = (!P.no_norm && norm >= TINY) ? -scale * exp2(Ev[k]) / ((double)S * norm) : 0.0;
      const double qx = (okp[k] && P.q_extra) ? P.q_extra[colk[k]] : 0.0;
      qE[k] = okp[k] ? a_E[colk[k]] + gE[k] + dd + qx : 0.0;
    }
  }

  // ---- BiCGSTAB on (I - J^T) w = q_E (_implicit_grad.py:28-94, same stopping rules).
  // A x with x = 0 is exactly 0, so r = q_E.
  double x[CPT], r[CPT], xs[CPT];
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    x[k] = 0.0;
    r[k] = qE[k];
  }
  const double qq = dot(qE, qE);
  const double bnorm = fmax(sqrt(qq), 1.0);
  double rel = sqrt(qq) / bnorm;
  int kit = 0;
  int done = rel <= P.tol;
  int failed = 0;
  bool use_xs = false;
  if (!done) {
    double rh[CPT], vv[CPT], pp[CPT], sv[CPT], tv[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      rh[k] = r[k];
      vv[k] = 0.0;
      pp[k] = 0.0;
    }
    double rho_old = 1.0, alpha = 1.0, omega = 1.0, rho_next = 0.0;
    for (kit = 1; kit <= P.max_iter; ++kit) {
      const double rho = kit == 1 ? dot(rh, r) : rho_next;
      if (fabs(rho) <= P.breakdown) break;
      const double beta = (rho / rho_old) * (alpha / omega);
#pragma unroll
      for (int k = 0; k < CPT; ++k) pp[k] = r[k] + beta * (pp[k] - omega * vv[k]);
      ag(pp, vv);
      const double den = dot(rh, vv);
      if (fabs(den) <= P.breakdown) break;
      alpha = rho / den;
#pragma unroll
      for (int k = 0; k < CPT; ++k) sv[k] = r[k] - alpha * vv[k];
      if (sqrt(dot(sv, sv)) / bnorm <= P.tol) {
#pragma unroll
        for (int k = 0; k < CPT; ++k) xs[k] = x[k] + alpha * pp[k];
        use_xs = true;
        done = 1;
        break;
      }
      ag(sv, tv);
      double tt, ts;
      {
        double lt = 0.0, ls = 0.0;
#pragma unroll
        for (int k = 0; k < CPT; ++k) {
          lt += tv[k] * tv[k];
          ls += tv[k] * sv[k];
        }
        sum2(lt, ls, tt, ts);
      }
      if (fabs(tt) <= P.breakdown) break;
      omega = ts / tt;
#pragma unroll
      for (int k = 0; k < CPT; ++k) {
        x[k] = x[k] + alpha * pp[k] + omega * sv[k];
        r[k] = sv[k] - omega * tv[k];
      }
      double rr;
      {
        double lr = 0.0, lh = 0.0;
#pragma unroll
        for (int k = 0; k < CPT; ++k) {
          lr += r[k] * r[k];
          lh += rh[k] * r[k];
        }
        sum2(lr, lh, rr, rho_next);
      }
      rel = sqrt(rr) / bnorm;
      if (rel <= P.tol) {
        done = 1;
        break;
      }
      if (fabs(omega) <= P.breakdown) break;
      rho_old = rho;
    }
    if (!done) failed = 1;
    if (kit > P.max_iter) kit = P.max_iter;
  }
  if (tid == 0) {
    P.status[0] = kit;
    P.status[1] = failed;
  }

  // ---- parameter cotangents: param_loss + E-step(E*, params) with (wE, g_Ebar)
  double G_pS[CPT], G_pD[CPT], G_pL[CPT], G_mt[CPT], G_col[CPT];
  {
    double ws[CPT], gE[CPT], wb[CPT], pv[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) ws[k] = use_xs ? xs[k] : x[k];
    vjp(ws, nullptr, nullptr, a_Ebar, gE, wb, pv);
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int s = colk[k];
      G_pS[k] = okp[k] ? ws[k] * W0[k] + a_pS[s] : 0.0;
      G_pD[k] = okp[k] ? ws[k] * W1[k] + a_pD[s] : 0.0;
      G_pL[k] = okp[k] ? ws[k] * W3[k] : 0.0;
      G_mt[k] = okp[k] ? wb[k] + a_mt[s] : 0.0;
      G_col[k] = okp[k] ? pv[k] + a_col[s] : 0.0;
    }
    if (P.g_out) {  // E adjoint and per-state parameter cotangents only
#pragma unroll
      for (int k = 0; k < CPT; ++k) {
        if (!okp[k]) continue;
        const int s = colk[k];
        P.g_out[s] = G_pS[k];
        P.g_out[(size_t)S + s] = G_pD[k];
        P.g_out[2 * (size_t)S + s] = G_pL[k];
        P.g_out[3 * (size_t)S + s] = G_mt[k];
        P.g_out[4 * (size_t)S + s] = G_col[k];
        if (P.w_out) P.w_out[s] = ws[k];
      }
      return;
    }
  }

  // theta VJP through log2-softmax of [0, theta] (extract_parameters.py:71-74)
  if (P.statewise) {
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      if (!okp[k]) continue;
      const int s = colk[k];
      const float* th = P.theta + 3 * (size_t)s;
      const double l0 = 0.0, l1 = th[0], l2 = th[1], l3 = th[2];
      const double mx = fmax(fmax(l0, l1), fmax(l2, l3));
      const double z = exp2(l0 - mx) + exp2(l1 - mx) + exp2(l2 - mx) + exp2(l3 - mx);
      const double gs = G_pS[k] + G_pD[k] + G_pL[k] + G_mt[k];
      P.grad_theta[3 * (size_t)s + 0] = (float)(G_pD[k] - exp2(l1 - mx) / z * gs);
      P.grad_theta[3 * (size_t)s + 1] = (float)(G_pL[k] - exp2(l2 - mx) / z * gs);
      P.grad_theta[3 * (size_t)s + 2] = (float)(G_mt[k] - exp2(l3 - mx) / z * gs);
    }
  } else {
    double a = 0.0, b = 0.0, d = 0.0, e = 0.0;
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      a += G_pS[k];
      b += G_pD[k];
      d += G_pL[k];
      e += G_mt[k];
    }
    sum2(a, b, a, b);
    sum2(d, e, d, e);
    if (tid == 0) {
      const double l0 = 0.0, l1 = P.theta[0], l2 = P.theta[1], l3 = P.theta[2];
      const double mx = fmax(fmax(l0, l1), fmax(l2, l3));
      const double z = exp2(l0 - mx) + exp2(l1 - mx) + exp2(l2 - mx) + exp2(l3 - mx);
      const double gs = a + b + d + e;
      P.grad_theta[0] = (float)(b - exp2(l1 - mx) / z * gs);
      P.grad_theta[1] = (float)(d - exp2(l2 - mx) / z * gs);
      P.grad_theta[2] = (float)(e - exp2(l3 - mx) / z * gs);
    }
  }

  // column VJP: col_log_probs = log_softmax(w)/ln2, col_norm = -log2(1 - pathsum(2^cl))
  double lmx = NINF;
#pragma unroll
  for (int k = 0; k < CPT; ++k)
    if (okp[k]) lmx = fmax(lmx, (double)P.col_weights[colk[k]]);
  const double wmax = block_max<NT>(lmx, mred);
  double lz = 0.0;
#pragma unroll
  for (int k = 0; k < CPT; ++k)
    if (okp[k]) lz += exp((double)P.col_weights[colk[k]] - wmax);
  double zsum, unused;
  sum2(lz, 0.0, zsum, unused);
  const double logz = wmax + log(zsum);
  double pc[CPT], pcs[CPT], ptot;
#pragma unroll
  for (int k = 0; k < CPT; ++k) pc[k] = okp[k] ? exp2(((double)P.col_weights[colk[k]] - logz) / LN2) : 0.0;
  path_sums(pc, pcs, ptot);
  double sc[CPT], ta = 0.0;
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    const double valid = 1.0 - pcs[k];
    const double xv = (okp[k] && valid > 0.0 && valid >= TINY) ? G_mt[k] / valid : 0.0;
    ta += xv;
    sc[k] = ta;
  }
  const double wa = wave_scan_incl_f64(ta);
#pragma unroll
  for (int k = 0; k < CPT; ++k) sc[k] += wa - ta;
  __syncthreads();  // the path sums above are still reading Lv
  lds_store_own_f64<CPT>(Lv, sc);
  if (lane == 63) wV[wv] = wa;
  __syncthreads();
  double sub[CPT];
  subtree_finish(sc, sub);
  double g[CPT], lg = 0.0;
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    g[k] = okp[k] ? G_col[k] + pc[k] * sub[k] : 0.0;
    lg += g[k];
  }
  double gsum;
  sum2(lg, 0.0, gsum, unused);
#pragma unroll
  for (int k = 0; k < CPT; ++k) {
    if (!okp[k]) continue;
    const int s = colk[k];
    const double qn = exp((double)P.col_weights[s] - logz);
    P.grad_col[s] = (float)((g[k] - qn * gsum) / LN2);
  }
}

#define KB_EPI_CASE(NT_, CPT_)                                                                \
  if (P.S <= NT_ * CPT_) {                                                                    \
    hipLaunchKernelGGL((epilogue_pre_kernel<NT_, CPT_>), dim3(1), dim3(NT_), 0, st, P);       \
    return;                                                                                   \
  }

void launch_epilogue(const EpiParams& P, hipStream_t st) {
  KB_EPI_CASE(64, 2)
  KB_EPI_CASE(128, 2)
  KB_EPI_CASE(256, 2)
  KB_EPI_CASE(256, 4)
  KB_EPI_CASE(512, 4)  // 512 x 4: fewer wavefronts, less per-wavefront scan overhead than 1024 x 2
  KB_EPI_CASE(1024, 4)
  KB_EPI_CASE(1024, 8)
}

}  // namespace kb
