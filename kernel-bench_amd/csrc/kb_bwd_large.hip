// Backward row kernel for species trees of 2049 to 8192 nodes (of 1025 to 8192
// with KB_BWD_LARGE=2).
//
// Same per-row mathematics as bwd_row_kernel (kb_bwd.hip; reference
// kbench/api/_implicit_grad.py:97-370 driving pristine wave_backward.py):
// adjoint gather or root seed, active mask, split term at Pi*, J^T
// coefficients, Neumann series, self-loop column gradient and parameter
// buckets, split adjoints into the children's staging rows.
//
// At these sizes a row needs 1024 threads owning 4 or 8 preorder positions
// each, and 16 wavefronts per workgroup leave 128 VGPRs per thread: per-position
// tables, six coefficient rows and eight bucket rows do not fit beside the
// Neumann series.  So a row is solved and its gradient buckets are summed in
// two kernels:
//  * bwd_row_large_kernel solves the rows of one level: adjoint, coefficients,
//    Neumann series, split adjoints into the children's staging rows.  It keeps
//    across phases only what the series needs, writes the row's v, and adds the
//    column-gradient bucket (the one that needs the row's scans) to this
//    workgroup's slot in memory;
//  * bwd_buckets_large_kernel runs once, after the last level, over all rows:
//    it recomputes q_0..q_5 and the split shares (same code, same values) from
//    v, Pi*, Pibar* and the split term, and holds the seven other bucket rows in
//    registers over every row of its workgroup.
// One kernel for both read and wrote the eight bucket rows of its slot (0.5 MB,
// 0.75 MB for a split row, of 8191 positions) on every row, more than L2 holds
// for 256 workgroups.  Measured per whole solve, with the vector row accesses of
// both: 8191 states 10.85 -> 9.3 ms (row kernels 7.1 -> 4.8 ms, buckets 0.73
// ms), 3001 weighted states 2.58 -> 2.37 ms.
// v takes the staging row of the row's first child side (only this row reads
// it, and has by then), an extra staging row for a family root, and the class's
// adjoint row for a class of level-0 rows.
#include "kb_device.hpp"
#include "kb_kernels.hpp"
#include "kb_rowops.hpp"

namespace kb {

namespace {

// the per-position constants the coefficients read
struct CoefK {
  float DL, Ebar, E, SL1, SL2, pS;
};

// q_0..q_5 of own position i: the self-loop terms' shares of the row's
// log-sum (wave_backward.py:264-416), with the split mixing weight folded into
// the normaliser, q_j = e_j / (sum_j e_j + 2^(dts - m)).
struct Coef6 {
  float q[6];
};

__device__ __forceinline__ Coef6 coef_at(const CoefK& K, float piv, float pbv, float dts, float pc1, float pc2,
                                         bool leaf_row, bool is_leaf_pos) {
  const float t0 = K.DL + piv;
  const float t1 = piv + K.Ebar;
  const float t2 = pbv + K.E;
  const float t3 = K.SL1 + pc1;
  const float t4 = K.SL2 + pc2;
  const float t5 = is_leaf_pos ? K.pS : KB_NEG_INF;
  const float m = fmaxf(fmaxf(fmaxf(t0, t1), fmaxf(t2, t3)), fmaxf(t4, t5));
  const float msf = fsafe(m);
  Coef6 c;
  c.q[0] = exp2_hw(t0 - msf);
  c.q[1] = exp2_hw(t1 - msf);
  c.q[2] = exp2_hw(t2 - msf);
  c.q[3] = exp2_hw(t3 - msf);
  c.q[4] = exp2_hw(t4 - msf);
  c.q[5] = exp2_hw(t5 - msf);
  const float sum = c.q[0] + c.q[1] + c.q[2] + c.q[3] + c.q[4] + c.q[5];
  const float den = sum + (leaf_row ? 0.0f : exp2_hw(dts - msf));
  const float inv = sum > 0.0f ? rcp_hw(den) : 0.0f;
#pragma unroll
  for (int j = 0; j < 6; ++j) c.q[j] *= inv;
  return c;
}

}  // namespace

// a workgroup-uniform value, in a scalar register
__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

// Where a solved row's v is kept for bwd_buckets_large_kernel: the staging row
// of its first child side s0, the extra staging row of a family root, or none.
__device__ __forceinline__ float* bwd_v_row(const BwdParams& P, int s0, int fam) {
  if (s0 < 0 && fam < 0) return nullptr;
  return P.staging + (s0 >= 0 ? (size_t)s0 : (size_t)2 * P.n_splits + fam) * kb_stage_ld(P.S);
}

template <int N>
__device__ __forceinline__ void vld(const float* p, float (&x)[N]) {
#pragma unroll
  for (int k = 0; k < N; k += 4) {
    const float4 q = *reinterpret_cast<const float4*>(p + k);
    x[k] = q.x;
    x[k + 1] = q.y;
    x[k + 2] = q.z;
    x[k + 3] = q.w;
  }
}

template <int N>
__device__ __forceinline__ void vst(float* p, const float (&x)[N]) {
#pragma unroll
  for (int k = 0; k < N; k += 4) *reinterpret_cast<float4*>(p + k) = make_float4(x[k], x[k + 1], x[k + 2], x[k + 3]);
}

__device__ __forceinline__ float4 ld4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float f4(const float4& v, int j) { return j == 0 ? v.x : j == 1 ? v.y : j == 2 ? v.z : v.w; }
// NT threads (1024, or 512 for rows of at most 2048 states) own CPT positions
// each; at most 128 VGPRs, so 16 wavefronts per CU are resident (two
// workgroups of 512).
// EARLY: the Neumann series may stop early (P.rtol > 0), as in bwd_row_kernel
template <int NT, int CPT, bool WEIGHTED, bool EARLY>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4)))
void bwd_row_large_kernel(BwdParams P, int first, int n_rows, int poff) {
  constexpr int MAXS = NT * CPT;
  constexpr int LD = MAXS + 64;  // [MAXS] is the padding slot, kept at 0
  constexpr int NW = NT / 64;
  constexpr int ZERO = MAXS;
  constexpr int SEGSH = CPT == 4 ? 8 : 9;  // log2 of the positions per wavefront
  constexpr int NG = CPT / 4;              // groups of four own positions
  static_assert(CPT == 4 || CPT == 8, "4 or 8 positions per thread");
  static_assert(NT == 512 || NT == 1024, "512 or 1024 threads");
  __shared__ float L[4 * LD];
  __shared__ float wA[2 * NW], wB[2 * NW];
  __shared__ float wMk[NW];
  float* R0 = L;
  float* R1 = L + LD;
  float* R2 = L + 2 * LD;
  float* R3 = L + 3 * LD;

  const PreDev& T = P.pre;
  const int S = P.S;
  const int tid = threadIdx.x;
  const int wv = tid >> 6, lane = tid & 63;
  if (tid < 64) {
    R0[MAXS + tid] = 0.0f;
    R1[MAXS + tid] = 0.0f;
    R2[MAXS + tid] = 0.0f;
    R3[MAXS + tid] = 0.0f;
  }
  // this workgroup's slot (KB_LARGE_SLOT_ROWS rows of MAXS floats, preorder
  // positions): the eight bucket rows, then the current row's Pi*.  srow(j) is
  // this thread's first own position of row j.
  float* const slot = P.contrib + (size_t)(poff + (int)blockIdx.x) * KB_LARGE_SLOT_ROWS * MAXS;
  int ep = 0;  // epoch of the current phase (see fresh)
  auto srow = [&](int j) {
    return reinterpret_cast<float*>(reinterpret_cast<char*>(fresh(slot + (size_t)j * MAXS, ep)) +
                                    (unsigned)(tid * CPT) * 4u);
  };
  enum { SL_COL = 7, SL_PI = 8 };
  // own position k; with 8 positions per thread recomputed where it is used
  // (the positions and the LDS addresses derived from them would otherwise be
  // held across the row loop)
  auto pos = [&](int k) {
    int b = tid * CPT;
    if constexpr (CPT > 4) asm("; %1" : "+v"(b) : "s"(ep));
    return b + k;
  };
  // Column tid + j*NT of a row: with 4 positions per thread columns past the
  // row read and store its last one again (no branches); with 8 the loads all
  // in flight at once would spill, and the guarded form measured faster.
  constexpr bool CLAMP = CPT == 4;
  auto column = [&](int j) { return CLAMP ? min(tid + j * NT, S - 1) : tid + j * NT; };
  // two global rows in column order -> LDS at preorder positions (coalesced reads)
  auto stage2 = [&](float* d0, const float* s0, float* d1, const float* s1) {
    int sp[CPT];
    float x[CPT], y[CPT];
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      const int s = column(j);
      sp[j] = CLAMP || s < S ? ldg(fresh(T.pre, ep), s) : -1;
      x[j] = CLAMP || s < S ? ldg(fresh(s0, ep), s) : 0.0f;
      y[j] = CLAMP || s < S ? ldg(fresh(s1, ep), s) : 0.0f;
    }
#pragma unroll
    for (int j = 0; j < CPT; ++j)
      if (CLAMP || sp[j] >= 0) {
        d0[sp[j]] = x[j];
        d1[sp[j]] = y[j];
      }
  };
  auto field = [](int rec, int f) { return __builtin_amdgcn_readlane(rec, f); };
  // row j of the owner-major tables / constants at own position k (one
  // contiguous read per wavefront)
  const int om0 = (tid >> 6) * 64 * CPT + (tid & 63);  // kb_om_index(tid * CPT, CPT)
  auto omi = [&](int j, int k) { return ldg(fresh(P.om_tab + (size_t)j * MAXS, ep) + k * 64, om0); };
  auto omf = [&](int j, int k) { return ldg(fresh(P.om_const + (size_t)j * MAXS, ep) + k * 64, om0); };
  auto coef_k = [&](int k) {
    return CoefK{omf(OMC_DL, k), omf(OMC_EBAR, k), omf(OMC_E, k), omf(OMC_SL1, k), omf(OMC_SL2, k), omf(OMC_PS, k)};
  };
  // subtree-sum offsets of a scan published by local_scan_publish: the block
  // total A, this wavefront's offset, and lane x < NW holding wavefront x's
  auto scan_offsets = [&](const float* wt, float& A, float& woff, float& wexcl) {
    const float wtot = lds_wave_values<NW>(wt, lane, 0.0f);
    const float wincl = wave_scan_first<NW>(wtot);
    wexcl = wincl - wtot;
    A = lane_value(wincl, NW - 1);
    woff = lane_value(wexcl, wv);
  };

  for (int rr = blockIdx.x; rr < n_rows; rr += gridDim.x) {
    __syncthreads();  // LDS of the previous row is no longer read
    ep = rr * 16 + 1;
    const int cm = P.class_mode;
    const int rec = cm ? 0 : P.bslot[(size_t)KB_BREC * (first + rr) + (tid & (KB_BREC - 1))];
    const int f_row = field(rec, BR_ROW), f_leaf = field(rec, BR_LEAF), f_sb = field(rec, BR_SB);
    const int f_se = field(rec, BR_SE), f_fam = field(rec, BR_FAM), f_s0 = field(rec, BR_S0);
    const int f_s1 = field(rec, BR_S1), f_lpos = field(rec, BR_LPOS), f_rep = field(rec, BR_REP);
    const int row = cm ? uniform(P.cls_rows[P.cls_ptr[rr]]) : f_row;
    const bool leaf_row = (cm ? P.row_kind[row] : f_leaf) != 0;
    const int sb = cm ? P.split_ptr[row] : f_sb, se = cm ? P.split_ptr[row + 1] : f_se;
    const int fam = cm ? -1 : f_fam;
    const size_t rb = (size_t)row * S;

    // ---- 1. adjoint: the class's summed adjoint, the root seed (below), or the
    // fixed-order gather of the live staging rows of the row's child sides.
    // The row's loads are issued together: Pi* / Pibar* (columns tid + j*NT,
    // to LDS below), the first two child sides' flags and staging rows (added
    // when live), and the stored split term.
    float nPi[CPT], nPb[CPT];
    int spre[CPT];
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      const int s = column(j);
      spre[j] = CLAMP || s < S ? ldg(fresh(T.pre, ep), s) : -1;
      nPi[j] = CLAMP || s < S ? ldg(fresh(P.pi + rb, ep), s) : 0.0f;
      nPb[j] = CLAMP || s < S ? ldg(fresh(P.pibar + rb, ep), s) : 0.0f;
    }
    float rhs[CPT], dts[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) dts[k] = KB_NEG_INF;
    if (!leaf_row && P.dts_in)
      gld_own<CPT>(fresh(P.dts_in + (size_t)(cm ? P.rep_of[row] : f_rep) * kb_stage_ld(S), ep), S, dts, KB_NEG_INF);
    bool any_active = false;
    float row_amax = 0.0f;  // max |adjoint| of the row
    if (cm) {
      any_active = P.cls_active[rr] != 0;
      gld_own<CPT>(fresh(P.rhsc + (size_t)rr * kb_stage_ld(S), ep), S, rhs, 0.0f);
    } else {
      const int s1 = f_s1 < 0 ? -1 : (f_s1 & ((1 << 30) - 1));
      const bool on0 = f_s0 >= 0 && P.split_on[f_s0 >> 1];
      const bool on1 = s1 >= 0 && P.split_on[s1 >> 1];
      const float* st0 = P.staging + (size_t)(f_s0 >= 0 ? f_s0 : 0) * kb_stage_ld(S);
      const float* st1 = P.staging + (size_t)(s1 >= 0 ? s1 : 0) * kb_stage_ld(S);
      float a0[CPT], a1[CPT];
      gld_own<CPT>(fresh(st0, ep), f_s0 >= 0 ? S : 0, a0, 0.0f);
      gld_own<CPT>(fresh(st1, ep), s1 >= 0 ? S : 0, a1, 0.0f);
#pragma unroll
      for (int k = 0; k < CPT; ++k) {
        rhs[k] = 0.0f;
        if (on0) rhs[k] += a0[k];
        if (on1) rhs[k] += a1[k];
      }
      const int n2 = (f_s1 >= 0 && (f_s1 >> 30) != 0) ? P.child_ptr[row + 1] - P.child_ptr[row] - 2 : 0;
      for (int j = 0; j < n2; ++j) {
        const int side = P.child_in[P.child_ptr[row] + 2 + j];
        if (!P.split_on[side >> 1]) continue;
        float a[CPT];
        gld_own<CPT>(fresh(P.staging + (size_t)side * kb_stage_ld(S), ep), S, a, 0.0f);
#pragma unroll
        for (int k = 0; k < CPT; ++k) rhs[k] += a[k];
      }
    }
    const bool mask_early = !cm && fam < 0;
    // (class rows publish them too when the Neumann series may stop early: its
    // threshold is relative to the row's largest adjoint entry)
    if (mask_early || (EARLY && cm)) {
      float am = 0.0f;
#pragma unroll
      for (int k = 0; k < CPT; ++k) am = fmaxf(am, fabsf(rhs[k]));
      const float wm = wave_reduce_max(am);
      if (lane == 0) wMk[wv] = wm;
    }
#pragma unroll
    for (int j = 0; j < CPT; ++j)
      if (CLAMP || spre[j] >= 0) {
        R0[spre[j]] = nPi[j];
        R1[spre[j]] = nPb[j];
      }
    __syncthreads();
    float piv[CPT];
    lds_load_own<CPT>(R0, piv);
#pragma unroll
    for (int k = 0; k < CPT; ++k)
      if (pos(k) >= S) piv[k] = KB_NEG_INF;
    if (EARLY && cm) {
#pragma unroll
      for (int w = 0; w < NW; ++w) row_amax = fmaxf(row_amax, wMk[w]);
    }
    if (!cm) {
      if (fam >= 0) {
        // logsumexp2 (logspace.py:11-16) and _safe_exp2_ratio (_implicit_grad.py:21-25)
        float lm = KB_NEG_INF;
#pragma unroll
        for (int k = 0; k < CPT; ++k) lm = fmaxf(lm, piv[k]);
        const float rmax = block_max1<NT>(lm, wA);
        const float rmx = fsafe(rmax);
        float ls = 0.0f;
#pragma unroll
        for (int k = 0; k < CPT; ++k) ls += pos(k) < S ? exp2f(piv[k] - rmx) : 0.0f;
        const float tot = block_sum1<NT>(ls, wB);
        const float lse = (tot > 0.0f ? log2f(tot) : KB_NEG_INF) + rmax;
        const float lses = fsafe(lse);
#pragma unroll
        for (int k = 0; k < CPT; ++k) rhs[k] = (piv[k] == KB_NEG_INF) ? 0.0f : -exp2f(piv[k] - lses);
      }
      // ---- 2. active mask (the reference's rule, wave_backward.py:150-163)
      float amax;
      if (mask_early) {
        amax = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; ++w) amax = fmaxf(amax, wMk[w]);
      } else {
        float am = 0.0f;
#pragma unroll
        for (int k = 0; k < CPT; ++k) am = fmaxf(am, fabsf(rhs[k]));
        amax = block_max1<NT>(am, wA);
      }
      any_active = P.use_pruning ? (amax >= P.thr) : (amax > P.thr);
      if (tid == 0) P.mask[row] = any_active ? 1 : 0;
      row_amax = amax;
    }
    if (!any_active) {
      for (int i = sb + tid; i < se; i += NT) P.split_on[i] = 0;
      continue;
    }
    const float rms = fsafe(P.rowmax[row]);
    const int lpos = cm ? (leaf_row ? T.pre[P.leaf_state[row]] : -1) : f_lpos;
    // Pibar* at the own positions (each thread reads its own positions only,
    // before any thread restages R1); Pi* kept in the slot for the split adjoints
    float pbv[CPT];
    lds_load_own<CPT>(R1, pbv);
#pragma unroll
    for (int k = 0; k < CPT; ++k)
      if (pos(k) >= S) pbv[k] = KB_NEG_INF;
    if (se > sb) vst<CPT>(srow(SL_PI), piv);
    // the reductions above reused scratch, and the split term below restages
    // R0..R3 when it is not stored
    if (fam >= 0 || (!leaf_row && !P.dts_in)) __syncthreads();

    // ---- 3. split term at Pi* (split rows)
    // (a stored split term was loaded with the row)
    ep = rr * 16 + 3;
    if (!leaf_row && !P.dts_in) {
      float acc[CPT];
#pragma unroll
      for (int k = 0; k < CPT; ++k) acc[k] = 0.0f;
      for (int si = sb; si < se; ++si) {
        const size_t l = (size_t)uniform(P.split_l[si]) * S, r = (size_t)uniform(P.split_r[si]) * S;
        const float lsp = P.split_lsp[si];
        stage2(R0, P.pi + l, R1, P.pi + r);
        stage2(R2, P.pibar + l, R3, P.pibar + r);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < CPT; ++k) {
          const int i = pos(k);
          if (i < S) {
            const int c1 = omi(OMT_C1, k), c2 = omi(OMT_C2, k);
            const float pl = R0[i], pr = R1[i];
            const float l1 = c1 >= 0 ? R0[c1] : KB_NEG_INF, r1 = c1 >= 0 ? R1[c1] : KB_NEG_INF;
            const float l2 = c2 >= 0 ? R0[c2] : KB_NEG_INF, r2 = c2 >= 0 ? R1[c2] : KB_NEG_INF;
            const float t0 = lsp + omf(OMC_PD, k) + pl + pr;
            const float t1 = lsp + pl + R3[i];
            const float t2 = lsp + pr + R2[i];
            const float sp = omf(OMC_PS, k);
            const float t3 = lsp + sp + l1 + r2;
            const float t4 = lsp + sp + r1 + l2;
            const float m5 = fmaxf(fmaxf(fmaxf(t0, t1), fmaxf(t2, t3)), t4);
            const float ms = fsafe(m5);
            const float s5 = exp2f(t0 - ms) + exp2f(t1 - ms) + exp2f(t2 - ms) + exp2f(t3 - ms) + exp2f(t4 - ms);
            lse_merge(dts[k], acc[k], m5, s5);
          }
        }
        __syncthreads();
      }
#pragma unroll
      for (int k = 0; k < CPT; ++k) dts[k] = log2f(acc[k]) + dts[k];
    }

    // ---- 4. J^T coefficients at Pi* (wave_backward.py:264-416)
    ep = rr * 16 + 4;
    // p' = 2^(col + Pi* - rowmax).  The Pibar coefficient's denominator,
    // rowsum - pathsum(i) = the sum of p' over the non-ancestors of i (the
    // reference's ancestor chase, wave_backward.py:364-389), is the row's own
    // Pibar* in linear units, 2^(Pibar*_i - mt_i - rowmax): the forward's last
    // sweep wrote Pibar* from the same Pi*, so no scan is needed.  Pi* is in
    // R0 at preorder positions (the child gathers) since the row's staging,
    // unless the split term above restaged R0.
    float pp[CPT], pcoef[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int i = pos(k);
      pp[k] = i < S ? exp2_hw((WEIGHTED ? omf(OMC_COL, k) : 0.0f) + piv[k] - rms) : 0.0f;
      const float denom = i < S ? exp2_hw(pbv[k] - omf(OMC_MT, k) - rms) : 0.0f;
      pcoef[k] = denom > 0.0f ? rcp_hw(denom) : 0.0f;  // 1 / (rowsum - ps) for now
    }
    if (!leaf_row && !P.dts_in) {
      lds_store_own<CPT>(R0, piv);  // padding positions: -inf
      __syncthreads();
    }
    // diag = q0 + q1, pcoef = q2 / (rowsum - ps); child-edge weights into
    // position i from its parent (q3 if i is child1, else q4) scattered by the
    // parent's owner into R1 (Pibar* was read above), then read back.  The
    // barrier also ends the reads of R2 / R3, which become scan buffers.
    float diag[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      const int i = pos(k);
      diag[k] = 0.0f;
      if (i < S) {
        const int c1 = omi(OMT_C1, k), c2 = omi(OMT_C2, k);
        const Coef6 c = coef_at(coef_k(k), piv[k], pbv[k], dts[k], c1 >= 0 ? R0[c1] : KB_NEG_INF,
                                c2 >= 0 ? R0[c2] : KB_NEG_INF, leaf_row, i == lpos);
        diag[k] = c.q[0] + c.q[1];
        pcoef[k] = c.q[2] * pcoef[k];
        if (c1 >= 0) R1[c1] = c.q[3];
        if (c2 >= 0) R1[c2] = c.q[4];
      } else {
        pcoef[k] = 0.0f;
      }
    }
    __syncthreads();
    // parent position, subtree end - 1 and child-1 flag of each own position,
    // packed (OMT_PK)
    float edge[CPT];
    int pk[CPT];
    lds_load_own<CPT>(R1, edge);
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      pk[k] = omi(OMT_PK, k);
      edge[k] = (pk[k] & 0xffff) != ZERO ? edge[k] : 0.0f;
    }
    // pk as values the optimiser cannot hoist out of the loops below (the LDS
    // addresses derived from it would otherwise stay live across them)
    auto pk_now = [&](int (&o)[CPT], int epoch) {
#pragma unroll
      for (int k = 0; k < CPT; ++k) {
        o[k] = pk[k];
        if constexpr (CPT > 4) asm("; %1" : "+v"(o[k]) : "s"(epoch));
      }
    };
    auto ppos_of = [](int x) { return x & 0xffff; };
    auto endm1_of = [](int x) { return (x >> 16) & 0x3fff; };
    auto wend_of = [](int x) { return (x >> (16 + SEGSH)) & (NW - 1); };  // ZERO -> wavefront 0

    // ---- 5. Neumann series v = sum_{n<=N} (J^T)^n rhs with the row on chip:
    // one barrier per term, buffers alternating by parity, and with EARLY the
    // same early stop as bwd_row_kernel (the series ends at the first term
    // with every entry at most rtol * max|rhs|; the wavefronts' votes travel
    // with their scan totals, in wt[NW + w])
    float v[CPT], term[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
      v[k] = rhs[k];
      term[k] = rhs[k];
    }
    const float tau = P.rtol * row_amax;
    auto neumann_term = [&](float* Tb, float* Lb, float* wt, int n_term) -> bool {
      // the LDS addresses come from the packed tables in every term: held
      // across the loop they would take 3 x CPT registers
      int pkt[CPT];
      pk_now(pkt, n_term);
      float sc[CPT];
#pragma unroll
      for (int k = 0; k < CPT; ++k) sc[k] = term[k] * pcoef[k] + (k > 0 ? sc[k - 1] : 0.0f);
      const float tsum = sc[CPT - 1];
      const float ws = wave_scan_incl(tsum);
      if (lane == 63) wt[wv] = ws;
      if constexpr (EARLY) {
        bool small = true;
#pragma unroll
        for (int k = 0; k < CPT; ++k) small = small && fabsf(term[k]) <= tau;
        const bool all_small = __all(small);
        if (lane == 63) wt[NW + wv] = all_small ? 1.0f : 0.0f;
      }
#pragma unroll
      for (int k = 0; k < CPT; ++k) sc[k] += ws - tsum;
      lds_store_own<CPT>(Lb, sc);
      lds_store_own<CPT>(Tb, term);
      __syncthreads();
      if constexpr (EARLY) {
        const float f = lane < NW ? wt[NW + lane] : 1.0f;
        if (__all(f != 0.0f)) return true;
      }
      float le[CPT], tpar[CPT];
#pragma unroll
      for (int k = 0; k < CPT; ++k) {
        le[k] = Lb[endm1_of(pkt[k])];
        tpar[k] = Tb[ppos_of(pkt[k])];
      }
      float A, woff, wexcl;
      scan_offsets(wt, A, woff, wexcl);
      const float p0 = wave_prev_lane(sc[CPT - 1]) + woff;
#pragma unroll
      for (int k = 0; k < CPT; ++k) {
        const float pm1 = k == 0 ? p0 : sc[k - 1] + woff;
        const int we = wend_of(pkt[k]);
        const float nt = term[k] * diag[k] + pp[k] * (pm1 + (A - (le[k] + __shfl(wexcl, we, 64)))) + tpar[k] * edge[k];
        term[k] = nt;
        v[k] += nt;
      }
      return false;
    };
    // calls: terms whose buffers were written (the stopping term included)
    int calls = 0;
    {
      bool stopped = false;
      for (; calls + 2 <= P.n_terms; calls += 2) {
        if (neumann_term(R0, R2, wA, calls)) {
          calls += 1;
          stopped = true;
          break;
        }
        if (neumann_term(R1, R3, wB, calls + 1)) {
          calls += 2;
          stopped = true;
          break;
        }
      }
      if (!stopped && calls < P.n_terms) {
        stopped = neumann_term(R0, R2, wA, calls);
        calls += 1;
      }
      if (P.terms_out && tid == 0) P.terms_out[row] = (unsigned char)min(stopped ? calls - 1 : calls, 255);
    }

    ep = rr * 16 + 6;
    // ---- 6. v for the bucket kernel, and the self-loop's column gradient (the
    // scan of u = v * pcoef in the Lb buffer of the next term's parity)
    {
      float* vr = cm ? P.rhsc + (size_t)rr * kb_stage_ld(S) : bwd_v_row(P, f_s0, fam);
      if (vr) gst_own<CPT>(vr, S, v);
    }
    float gcol[CPT];
    {
      // the buffers the last term did not write (its readers may still be
      // reading its own)
      float* Pb = (calls & 1) ? R3 : R2;
      float* wt = (calls & 1) ? wB : wA;
      float x[CPT], sc[CPT];
#pragma unroll
      for (int k = 0; k < CPT; ++k) x[k] = v[k] * pcoef[k];
      local_scan_publish<NT, CPT>(sc, x, Pb, wt);
      __syncthreads();
      float A, woff, wexcl;
      scan_offsets(wt, A, woff, wexcl);
      const float p0 = wave_prev_lane(sc[CPT - 1]) + woff;
      int pkt[CPT];
      pk_now(pkt, ep);
      // p' (P(i-1) + A - P(end(i)-1))
#pragma unroll
      for (int k = 0; k < CPT; ++k) {
        const float pm1 = k == 0 ? p0 : sc[k - 1] + woff;
        const float rest = A - (Pb[endm1_of(pkt[k])] + __shfl(wexcl, wend_of(pkt[k]), 64));
        gcol[k] = pos(k) < S ? pp[k] * (pm1 + rest) : 0.0f;
      }
    }

    // ---- 7. split adjoints into the child rows (staging, preorder layout)
    for (int si = sb; si < se; ++si) {
      const int lrow = uniform(P.split_l[si]), rrow = uniform(P.split_r[si]);
      const size_t l = (size_t)lrow * S, r = (size_t)rrow * S;
      const float lsp = P.split_lsp[si];
      const float rml = P.rowmax[lrow], rmr = P.rowmax[rrow];
      const float rmsl = fsafe(rml), rmsr = fsafe(rmr);
      ep = -4 * si - 1;
      __syncthreads();  // previous readers of R0..R3 are done
      stage2(R0, P.pi + l, R1, P.pi + r);
      stage2(R2, P.pibar + l, R3, P.pibar + r);
      __syncthreads();
      ep = -4 * si - 2;
      // pass 1 (own positions, four at a time): the five split-term shares
      // vd_j; vd3 / vd4 replace the own positions of the children's Pibar
      // rows (R2 / R3, read only at own positions) for the child positions'
      // parent reads
      float av[CPT], bv[CPT], udl[CPT], udr[CPT], ppl[CPT], ppr[CPT];
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        float pv4[4];
        vld<4>(srow(SL_PI) + 4 * g, pv4);
        // own positions of the four staged child rows (vector LDS reads)
        const float4 pl4 = ld4(R0 + tid * CPT + 4 * g), pr4 = ld4(R1 + tid * CPT + 4 * g);
        const float4 bl4 = ld4(R2 + tid * CPT + 4 * g), br4 = ld4(R3 + tid * CPT + 4 * g);
        float d3[4], d4[4];
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
          const int k = 4 * g + kk;
          const int i = pos(k);
          float vd0 = 0.0f, vd1 = 0.0f, vd2 = 0.0f, vd3 = 0.0f, vd4 = 0.0f;
          udl[k] = udr[k] = ppl[k] = ppr[k] = 0.0f;
          if (i < S) {
            const int c1 = omi(OMT_C1, k), c2 = omi(OMT_C2, k);
            const float pl = f4(pl4, kk), pr = f4(pr4, kk), bl = f4(bl4, kk), br = f4(br4, kk);
            const float l1 = c1 >= 0 ? R0[c1] : KB_NEG_INF, r1 = c1 >= 0 ? R1[c1] : KB_NEG_INF;
            const float l2 = c2 >= 0 ? R0[c2] : KB_NEG_INF, r2 = c2 >= 0 ? R1[c2] : KB_NEG_INF;
            const float d = omf(OMC_PD, k), sp = omf(OMC_PS, k);
            const bool pv = pv4[kk] != KB_NEG_INF;
            const float base = pv ? lsp - pv4[kk] : 0.0f;
            vd0 = pv ? v[k] * exp2_hw(base + (d + pl + pr)) : 0.0f;
            vd1 = pv ? v[k] * exp2_hw(base + (pl + br)) : 0.0f;
            vd2 = pv ? v[k] * exp2_hw(base + (pr + bl)) : 0.0f;
            vd3 = pv ? v[k] * exp2_hw(base + (sp + l1 + r2)) : 0.0f;
            vd4 = pv ? v[k] * exp2_hw(base + (sp + r1 + l2)) : 0.0f;
            const float mts = omf(OMC_MT, k);
            const float inv_l = bl != KB_NEG_INF ? exp2_hw(rml + mts - bl) : 0.0f;
            const float inv_r = br != KB_NEG_INF ? exp2_hw(rmr + mts - br) : 0.0f;
            udl[k] = vd2 * inv_l;
            udr[k] = vd1 * inv_r;
            const float cw = WEIGHTED ? omf(OMC_COL, k) : 0.0f;
            ppl[k] = exp2_hw(cw + pl - rmsl);
            ppr[k] = exp2_hw(cw + pr - rmsr);
          }
          av[k] = vd0 + vd1;
          bv[k] = vd0 + vd2;
          d3[kk] = vd3;
          d4[kk] = vd4;
        }
        *reinterpret_cast<float4*>(R2 + tid * CPT + 4 * g) = make_float4(d3[0], d3[1], d3[2], d3[3]);
        *reinterpret_cast<float4*>(R3 + tid * CPT + 4 * g) = make_float4(d4[0], d4[1], d4[2], d4[3]);
      }
      __syncthreads();  // the staged children (R0, R1) fully read; vd3 / vd4 published
      float scl[CPT], scr[CPT];
      local_scan_publish<NT, CPT>(scl, udl, R0, wA);
      local_scan_publish<NT, CPT>(scr, udr, R1, wA + NW);
      __syncthreads();
      float Al, woffl, wexl, Ar, woffr, wexr;
      scan_offsets(wA, Al, woffl, wexl);
      scan_offsets(wA + NW, Ar, woffr, wexr);
      const float p0l = wave_prev_lane(scl[CPT - 1]) + woffl;
      const float p0r = wave_prev_lane(scr[CPT - 1]) + woffr;
      ep = -4 * si - 3;
      float* stl = P.staging + (size_t)(2 * si) * kb_stage_ld(S);
      float* str = P.staging + (size_t)(2 * si + 1) * kb_stage_ld(S);
      int pkt[CPT];
      pk_now(pkt, ep);
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        float yl[4], yr[4];
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
          const int k = 4 * g + kk;
          const int i = pos(k);
          const int e1 = endm1_of(pkt[k]), we = wend_of(pkt[k]);
          const float pml = k == 0 ? p0l : scl[k - 1] + woffl;
          const float pmr = k == 0 ? p0r : scr[k - 1] + woffr;
          yl[kk] = yr[kk] = 0.0f;
          const float rsl = Al - (R0[e1] + __shfl(wexl, we, 64));
          const float rsr = Ar - (R1[e1] + __shfl(wexr, we, 64));
          if (i < S) {
            const float tl = ppl[k] * (pml + rsl);
            const float tr = ppr[k] * (pmr + rsr);
            const int pa = ppos_of(pkt[k]);
            const bool first_child = (pkt[k] >> 30) & 1;
            const float sh3 = R2[pa], sh4 = R3[pa];  // padding slot holds 0
            const float shl = first_child ? sh3 : sh4;
            const float shr = first_child ? sh4 : sh3;
            yl[kk] = av[k] + shl + tl;
            yr[kk] = bv[k] + shr + tr;
            gcol[k] += tl + tr;
          }
        }
        // (rows are a multiple of four floats long: the tail goes to padding)
        if (pos(4 * g) < S) {
          *reinterpret_cast<float4*>(stl + pos(4 * g)) = make_float4(yl[0], yl[1], yl[2], yl[3]);
          *reinterpret_cast<float4*>(str + pos(4 * g)) = make_float4(yr[0], yr[1], yr[2], yr[3]);
        }
      }
      if (tid == 0) P.split_on[si] = 1;
    }
    float old[CPT];
    vld<CPT>(srow(SL_COL), old);
#pragma unroll
    for (int k = 0; k < CPT; ++k) old[k] += gcol[k];
    vst<CPT>(srow(SL_COL), old);
  }  // rows
}

// The seven other bucket rows of all solved rows: levels 1 and up (schedule
// slots first .. first + n_rows) and the n_cls classes of level 0, workgroup b
// taking items b, b + gridDim.x, ... in order into slot b, whose rows 0..6 it
// writes once.
//
// One row is in flight per CU (four LDS rows), so the row's loads are issued
// together ahead of its arithmetic: record and mask one row early, then v, the
// split term, Pi*, Pibar* and the first split's children's Pi; the children's
// Pibar while the coefficients are computed (with 8 positions per thread the
// children are loaded in the split loop instead: the loads ahead spilled, 731 us
// against 1305).  128 VGPRs hold 7 * CPT sums and the position tables packed 16
// bits each.  Against one load per position, tables from memory and no loads
// ahead: 11000 rows of 8191 states 953 -> 731 us, 5500 of 3001 186 -> 144 us.
template <int NT, int CPT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4)))
void bwd_buckets_large_kernel(BwdParams P, int first, int n_rows, int n_cls) {
  constexpr int MAXS = NT * CPT;
  constexpr int LD = MAXS + 64;
  constexpr int ZERO = MAXS;
  constexpr int NG = CPT / 4;
  constexpr bool PREF = CPT == 4;
  static_assert(CPT == 4 || CPT == 8, "4 or 8 positions per thread");
  static_assert(MAXS <= 8192, "positions in 16 bits");
  __shared__ __align__(16) float L[4 * LD];
  float* R0 = L;
  float* R1 = L + LD;
  float* R2 = L + 2 * LD;
  float* R3 = L + 3 * LD;
  const PreDev& T = P.pre;
  const int S = P.S;
  const int tid = threadIdx.x;
  int ep = 0;
  auto pos = [&](int k) {
    int b = tid * CPT;
    if constexpr (CPT > 4) asm("; %1" : "+v"(b) : "s"(ep));
    return b + k;
  };
  auto field = [](int rec, int f) { return __builtin_amdgcn_readlane(rec, f); };
  const int om0 = (tid >> 6) * 64 * CPT + (tid & 63);  // kb_om_index(tid * CPT, CPT)
  auto omf = [&](int j, int k) { return ldg(fresh(P.om_const + (size_t)j * MAXS, ep) + k * 64, om0); };
  auto coef_k = [&](int k) {
    return CoefK{omf(OMC_DL, k), omf(OMC_EBAR, k), omf(OMC_E, k), omf(OMC_SL1, k), omf(OMC_SL2, k), omf(OMC_PS, k)};
  };
  // preorder position of column tid + j*NT, child2 (ZERO: none) of own position
  // k, two to a register; bit k of has1: own position k has a child1 (k + 1)
  unsigned pre2[CPT / 2], c22[CPT / 2], has1 = 0;
#pragma unroll
  for (int k = 0; k < CPT; k += 2) {
    auto pre_of = [&](int s) { return (unsigned)T.pre[min(s, S - 1)]; };
    auto c2_at = [&](int j) {
      const int c2 = P.om_tab[(size_t)OMT_C2 * MAXS + j * 64 + om0];
      return c2 >= 0 ? (unsigned)c2 : (unsigned)ZERO;
    };
    pre2[k / 2] = pre_of(tid + k * NT) | pre_of(tid + (k + 1) * NT) << 16;
    c22[k / 2] = c2_at(k) | c2_at(k + 1) << 16;
  }
#pragma unroll
  for (int k = 0; k < CPT; ++k) has1 |= P.om_tab[(size_t)OMT_C1 * MAXS + k * 64 + om0] >= 0 ? 1u << k : 0u;
  auto opaque = [&]() {  // unpacked where they are used, not held unpacked
#pragma unroll
    for (int k = 0; k < CPT / 2; ++k) {
      asm("; %1" : "+v"(pre2[k]) : "s"(ep));
      asm("; %1" : "+v"(c22[k]) : "s"(ep));
    }
  };
  auto half = [](const unsigned (&x)[CPT / 2], int k) { return (int)((k & 1) ? x[k / 2] >> 16 : x[k / 2] & 0xffffu); };
  auto load_row = [&](const float* src, float (&x)[CPT]) {  // columns tid + j*NT (the last one past the row)
#pragma unroll
    for (int j = 0; j < CPT; ++j) x[j] = ldg(fresh(src, ep), min(tid + j * NT, S - 1));
  };
  auto put_row = [&](float* dst, const float (&x)[CPT]) {
#pragma unroll
    for (int j = 0; j < CPT; ++j) dst[half(pre2, j)] = x[j];
  };
  // child1 / child2 of own position k = 4g + kk in the staged row Rw (-inf: none);
  // q: the row's own positions 4g .. 4g+3
  auto child1 = [&](const float* Rw, const float4& q, int k) {
    return (has1 >> k) & 1 ? ((k & 3) < 3 ? f4(q, (k & 3) + 1) : Rw[pos(k) + 1]) : KB_NEG_INF;
  };
  auto child2 = [&](const float* Rw, int k) {
    const int c2 = half(c22, k);
    return c2 != ZERO ? Rw[c2] : KB_NEG_INF;
  };
  enum { B_PD, B_PS, B_E, B_EBAR, B_SL2, B_SL1, B_MT, NB };
  float acc[NB][CPT];
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int k = 0; k < CPT; ++k) acc[j][k] = 0.0f;

  // the sums as single registers: as vectors of four the compiler spills them
  auto pin = [&]() {
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int k = 0; k < CPT; ++k) asm("" : "+v"(acc[j][k]));
  };
  const int n_items = n_rows + n_cls;
  auto load_rec = [&](int it) {
    return it < n_rows ? P.bslot[(size_t)KB_BREC * (first + it) + (tid & (KB_BREC - 1))] : 0;
  };
  auto load_on = [&](int it, int rec) {
    return it >= n_items ? 0 : it >= n_rows ? (int)P.cls_active[it - n_rows] : (int)P.mask[field(rec, BR_ROW)];
  };
  int nrec = load_rec(blockIdx.x), non = load_on(blockIdx.x, nrec);
  for (int it = blockIdx.x; it < n_items; it += gridDim.x) {
    const int rec = nrec, on = __builtin_amdgcn_readfirstlane(non);
    const int nit = it + (int)gridDim.x;
    nrec = load_rec(nit);
    const bool cm = it >= n_rows;
    const int c = it - n_rows;
    // (no row: neither a root nor anyone's child, v = 0)
    const float* vr = cm ? P.rhsc + (size_t)c * kb_stage_ld(S) : bwd_v_row(P, field(rec, BR_S0), field(rec, BR_FAM));
    if (!on || !vr) {
      non = load_on(nit, nrec);
      continue;
    }
    const int row = cm ? uniform(P.cls_rows[P.cls_ptr[c]]) : field(rec, BR_ROW);
    const bool leaf_row = (cm ? P.row_kind[row] : field(rec, BR_LEAF)) != 0;
    const int lpos = cm ? (leaf_row ? T.pre[P.leaf_state[row]] : -1) : field(rec, BR_LPOS);
    const int sb = cm ? P.split_ptr[row] : field(rec, BR_SB), se = cm ? P.split_ptr[row + 1] : field(rec, BR_SE);
    const bool split = se > sb;
    const size_t l0 = split ? (size_t)(cm ? uniform(P.split_l[sb]) : field(rec, BR_L0)) * S : 0;
    const size_t r0 = split ? (size_t)(cm ? uniform(P.split_r[sb]) : field(rec, BR_R0)) * S : 0;
    const float lsp0 = split ? (cm ? P.split_lsp[sb] : __int_as_float(field(rec, BR_LSP0))) : 0.0f;
    ep = 8 * it + 1;
    opaque();
    float v[CPT], dts[CPT];
#pragma unroll
    for (int k = 0; k < CPT; ++k) dts[k] = KB_NEG_INF;
    if (!leaf_row) {
      if (P.dts_in) {
        gld_own<CPT>(fresh(P.dts_in + (size_t)(cm ? P.rep_of[row] : field(rec, BR_REP)) * kb_stage_ld(S), ep), S, dts,
                     KB_NEG_INF);
      } else {
        // the split term at Pi*, as in bwd_row_large_kernel
        float sum[CPT];
#pragma unroll
        for (int k = 0; k < CPT; ++k) sum[k] = 0.0f;
        for (int si = sb; si < se; ++si) {
          const size_t l = (size_t)uniform(P.split_l[si]) * S, r = (size_t)uniform(P.split_r[si]) * S;
          const float lsp = P.split_lsp[si];
          __syncthreads();
          float x[CPT], y[CPT];
          load_row(P.pi + l, x);
          load_row(P.pi + r, y);
          put_row(R0, x);
          put_row(R1, y);
          load_row(P.pibar + l, x);
          load_row(P.pibar + r, y);
          put_row(R2, x);
          put_row(R3, y);
          __syncthreads();
#pragma unroll
          for (int g = 0; g < NG; ++g) {
            const float4 pl4 = ld4(R0 + tid * CPT + 4 * g), pr4 = ld4(R1 + tid * CPT + 4 * g);
            const float4 bl4 = ld4(R2 + tid * CPT + 4 * g), br4 = ld4(R3 + tid * CPT + 4 * g);
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
              const int k = 4 * g + kk;
              if (pos(k) < S) {
                const float pl = f4(pl4, kk), pr = f4(pr4, kk);
                const float l1 = child1(R0, pl4, k), r1 = child1(R1, pr4, k), l2 = child2(R0, k), r2 = child2(R1, k);
                const float t0 = lsp + omf(OMC_PD, k) + pl + pr;
                const float t1 = lsp + pl + f4(br4, kk);
                const float t2 = lsp + pr + f4(bl4, kk);
                const float sp = omf(OMC_PS, k);
                const float t3 = lsp + sp + l1 + r2;
                const float t4 = lsp + sp + r1 + l2;
                const float m5 = fmaxf(fmaxf(fmaxf(t0, t1), fmaxf(t2, t3)), t4);
                const float ms = fsafe(m5);
                const float s5 = exp2f(t0 - ms) + exp2f(t1 - ms) + exp2f(t2 - ms) + exp2f(t3 - ms) + exp2f(t4 - ms);
                lse_merge(dts[k], sum[k], m5, s5);
              }
            }
          }
        }
#pragma unroll
        for (int k = 0; k < CPT; ++k) dts[k] = log2f(sum[k]) + dts[k];
      }
    }
    gld_own<CPT>(fresh(vr, ep), S, v, 0.0f);
    {
      float a[CPT], b[CPT], x[CPT], y[CPT];
      load_row(P.pi + (size_t)row * S, a);
      load_row(P.pibar + (size_t)row * S, b);
      if (PREF && split) {
        load_row(P.pi + l0, x);
        load_row(P.pi + r0, y);
      }
      __syncthreads();  // LDS of the previous row or split is no longer read
      put_row(R0, a);
      put_row(R1, b);
      if (PREF && split) {
        put_row(R2, x);
        put_row(R3, y);
      }
    }
    __syncthreads();
    non = load_on(nit, nrec);
    ep = 8 * it + 2;
    opaque();
    float bx[CPT], by[CPT];  // the first split's children's Pibar, in flight below
    if (PREF && split) {
      load_row(P.pibar + l0, bx);
      load_row(P.pibar + r0, by);
    }
    float piv[CPT];
    lds_load_own<CPT>(R0, piv);
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const float4 pi4 = make_float4(piv[4 * g], piv[4 * g + 1], piv[4 * g + 2], piv[4 * g + 3]);
      const float4 pb4 = ld4(R1 + tid * CPT + 4 * g);
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        const int k = 4 * g + kk;
        const int i = pos(k);
        if (i < S) {
          const Coef6 q = coef_at(coef_k(k), piv[k], f4(pb4, kk), dts[k], child1(R0, pi4, k), child2(R0, k), leaf_row,
                                  i == lpos);
          const float aw0 = v[k] * q.q[0], aw1 = v[k] * q.q[1], aw2 = v[k] * q.q[2];
          const float aw3 = v[k] * q.q[3], aw4 = v[k] * q.q[4], aw5 = v[k] * q.q[5];
          acc[B_PD][k] += aw0;
          acc[B_PS][k] += aw3 + aw4 + aw5;
          acc[B_E][k] += aw0 + aw2;
          acc[B_EBAR][k] += aw1;
          acc[B_SL2][k] += aw4;
          acc[B_SL1][k] += aw3;
          acc[B_MT][k] += aw2;
        }
      }
    }
    pin();
    for (int si = sb; si < se; ++si) {
      float lsp = lsp0;
      __syncthreads();
      ep = -4 * si - 1;
      opaque();
      if (!PREF || si > sb) {
        const size_t l = (size_t)uniform(P.split_l[si]) * S, r = (size_t)uniform(P.split_r[si]) * S;
        lsp = P.split_lsp[si];
        float x[CPT], y[CPT];
        load_row(P.pi + l, x);
        load_row(P.pi + r, y);
        if (PREF) {
          load_row(P.pibar + l, bx);
          load_row(P.pibar + r, by);
        }
        put_row(R2, x);
        put_row(R3, y);
        if (!PREF) {
          load_row(P.pibar + l, bx);
          load_row(P.pibar + r, by);
        }
      }
      put_row(R0, bx);
      put_row(R1, by);
      __syncthreads();
      ep = -4 * si - 2;
      opaque();
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const float4 pl4 = ld4(R2 + tid * CPT + 4 * g), pr4 = ld4(R3 + tid * CPT + 4 * g);
        const float4 bl4 = ld4(R0 + tid * CPT + 4 * g), br4 = ld4(R1 + tid * CPT + 4 * g);
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
          const int k = 4 * g + kk;
          if (pos(k) < S && piv[k] != KB_NEG_INF) {
            const float pl = f4(pl4, kk), pr = f4(pr4, kk), bl = f4(bl4, kk), br = f4(br4, kk);
            const float l1 = child1(R2, pl4, k), r1 = child1(R3, pr4, k), l2 = child2(R2, k), r2 = child2(R3, k);
            const float d = omf(OMC_PD, k), sp = omf(OMC_PS, k);
            const float base = lsp - piv[k];
            const float vd0 = v[k] * exp2_hw(base + (d + pl + pr));
            const float vd1 = v[k] * exp2_hw(base + (pl + br));
            const float vd2 = v[k] * exp2_hw(base + (pr + bl));
            const float vd3 = v[k] * exp2_hw(base + (sp + l1 + r2));
            const float vd4 = v[k] * exp2_hw(base + (sp + r1 + l2));
            acc[B_PD][k] += vd0;
            acc[B_PS][k] += vd3 + vd4;
            acc[B_MT][k] += vd1 + vd2;
          }
        }
      }
      pin();
    }
  }
  float* const slot = P.contrib + (size_t)blockIdx.x * KB_LARGE_SLOT_ROWS * MAXS + tid * CPT;
#pragma unroll
  for (int j = 0; j < NB; ++j) vst<CPT>(slot + (size_t)j * MAXS, acc[j]);
}

#define KB_BWD_LARGE_CASE(NT_, CPT_)                                                                           \
  if (S <= NT_ * CPT_) {                                                                                       \
    const bool early = P.rtol > 0.0f;                                                                          \
    if (P.use_col && early)                                                                                    \
      hipLaunchKernelGGL((bwd_row_large_kernel<NT_, CPT_, true, true>), dim3(nb), dim3(NT_), 0, st, P, first, W, poff);   \
    else if (P.use_col)                                                                                        \
      hipLaunchKernelGGL((bwd_row_large_kernel<NT_, CPT_, true, false>), dim3(nb), dim3(NT_), 0, st, P, first, W, poff);  \
    else if (early)                                                                                            \
      hipLaunchKernelGGL((bwd_row_large_kernel<NT_, CPT_, false, true>), dim3(nb), dim3(NT_), 0, st, P, first, W, poff);  \
    else                                                                                                       \
      hipLaunchKernelGGL((bwd_row_large_kernel<NT_, CPT_, false, false>), dim3(nb), dim3(NT_), 0, st, P, first, W, poff); \
    return true;                                                                                               \
  }

bool launch_bwd_large(const BwdParams& P, int first, int W, int nb, int poff, hipStream_t st) {
  const int S = P.S;
  if (!kb_use_large(S, P.large)) return false;
  // the shape kb_large_nt / kb_large_ld give the owner-major tables
  if (kb_large_nt(S) == 512) {
    KB_BWD_LARGE_CASE(512, 4)
  }
  KB_BWD_LARGE_CASE(1024, 4)
  KB_BWD_LARGE_CASE(1024, 8)
  return false;
}

void launch_bwd_buckets_large(const BwdParams& P, int first, int n_rows, int n_cls, int nb, hipStream_t st) {
  const int S = P.S;
  if (!kb_use_large(S, P.large) || n_rows + n_cls <= 0) return;
  const dim3 g(std::min(nb, n_rows + n_cls));
  if (kb_large_nt(S) == 512)
    hipLaunchKernelGGL((bwd_buckets_large_kernel<512, 4>), g, dim3(512), 0, st, P, first, n_rows, n_cls);
  else if (S <= 4096)
    hipLaunchKernelGGL((bwd_buckets_large_kernel<1024, 4>), g, dim3(1024), 0, st, P, first, n_rows, n_cls);
  else
    hipLaunchKernelGGL((bwd_buckets_large_kernel<1024, 8>), g, dim3(1024), 0, st, P, first, n_rows, n_cls);
}

int bwd_large_blocks_per_cu(int S, int use_col) {
  int n = 0;
  auto occ = [&](auto kernel, int nt) { (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, nt, 0); };
  if (kb_large_nt(S) == 512)
    use_col ? occ(bwd_row_large_kernel<512, 4, true, false>, 512) : occ(bwd_row_large_kernel<512, 4, false, false>, 512);
  else if (S <= 4096)
    use_col ? occ(bwd_row_large_kernel<1024, 4, true, false>, 1024) : occ(bwd_row_large_kernel<1024, 4, false, false>, 1024);
  else
    use_col ? occ(bwd_row_large_kernel<1024, 8, true, false>, 1024) : occ(bwd_row_large_kernel<1024, 8, false, false>, 1024);
  return n > 0 ? n : 1;
}

}  // namespace kb
