// Model evaluation, stop-test partials and the KKT residual on the matrix
// cores, for the tanh model with stage-invariant A, W, B, Q, R (FP32, n <= 48,
// m <= 16): one wave takes 16 consecutive stages t < N of one instance, in the
// layout of k_linearize_mma (k_lin_mma.h): stage vectors are columns of
// B-operand tiles, matrices A-operand tiles, rows 16 i + 4 g + v of stage c in
// lane (g, c).  Entries past a vector's end are read as 0 (not as the next
// stage's: a NaN there stays in its stage).  The transposed products of the residual, A'V and
// W'(sech^2 V), read the matrices' columns (64 contiguous bytes per row).  The
// block after the last takes the terminal stage (eval_stage; a launch of its own
// made the smallest evaluations, bound by their launches, slower than the thread
// per row they replaced: 12 x 12 x 25, B = 1, evaluation and residual 42 us there, 50
// with a launch more each, 43 now).  Bound by its loads: at B = 1024, 36 x 12 x 50, p
// = 8 the model evaluation takes 22 us and the residual 47; the row form
// (k_eval_rows), which reads every matrix once per stage, took 180 and 286.
#pragma once
#include "k_eval.h"
#include "k_lin_mma.h"

namespace mpxk {

// A-operand tiles of M' (M row-major, rows x cols): lane (g, c) of tile (i, k)
// holds M[16 k + 4 g + s][16 i + c]
template <int KT, int IT>
__device__ __forceinline__ void load_aop_t(f4 (&out)[IT][KT], const float* M, int rows, int cols, int g, int c) {
  const rsrc_t r = make_rsrc(M, rows * cols);
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int off = 16 * i + c < cols ? (4 * g * cols + 16 * i + c) * 4 : kOOB;
#pragma unroll
    for (int k = 0; k < KT; ++k)
#pragma unroll
      for (int s = 0; s < 4; ++s) out[i][k][s] = rload(r, off + (16 * k + s) * cols * 4);
  }
}

template <int NT, bool WIDE, int WHAT>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2)))
k_eval_mma(Prob<float> P, Prm<float> prm, Iter<float> it, Ws<float> ws, float* og, float* oc) {
  constexpr bool KKT = WHAT == EVAL_KKT;
  const int b = blockIdx.y, lane = threadIdx.x, g = lane >> 4, c = lane & 15;
  if (WHAT == EVAL_STOP && skip_instance(ws, b)) return;
  __shared__ float smem[eval_wave_elems<NT>()];
  if (blockIdx.x == gridDim.x - 1) return eval_stage<float, NT, 1, WHAT, true>(P, prm, it, ws, og, oc, b, P.N, smem);
  const int n = P.n, m = P.m, p = P.p, N = P.N, N1 = N + 1;
  const int t = blockIdx.x * 16 + c;
  const bool live = t < N;
  const int tc = live ? t : N - 1;   // a stage with data for the columns past N - 1 (nothing of theirs is kept)
  const float hs = P.h, kap = P.kappa;
  int off[NT][4];
  aop_offsets<NT>(off, n, g, c);

  // f = x + h (A x + B u + kappa tanh(W x)) and the defect
  const rsrc_t rX = make_rsrc(it.X + (size_t)b * N1 * n, N1 * n);
  const rsrc_t rU = make_rsrc(it.U + (size_t)b * N * m, N * m);
  f4 X0[NT], U0, Mt[NT][NT], Wt[NT][NT], Bt[NT], Xn[NT];
#pragma unroll
  for (int k = 0; k < NT; ++k) X0[k] = vload4<WIDE>(rX, tc * n + 16 * k + 4 * g, 16 * k + 4 * g, n);
  U0 = vload4<WIDE>(rU, tc * m + 4 * g, 4 * g, m);
  load_aop_raw<NT, NT, WIDE>(Mt, P.A.at(b, 0), n, n, off);
  {
    const rsrc_t rB = make_rsrc(P.Bm.at(b, 0), n * m);
#pragma unroll
    for (int i = 0; i < NT; ++i) Bt[i] = vload4<WIDE>(rB, (16 * i + c) * m + 4 * g, 4 * g, m);
  }
  load_aop_raw<NT, NT, WIDE>(Wt, P.W.at(b, 0), n, n, off);
#pragma unroll
  for (int i = 0; i < NT; ++i) Xn[i] = vload4<WIDE>(rX, (tc + 1) * n + 16 * i + 4 * g, 16 * i + 4 * g, n);
  __builtin_amdgcn_sched_barrier(0);
  f4 C[NT], SDv[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    f4 a = zero4(), w = zero4();
#pragma unroll
    for (int k = 0; k < NT; ++k)
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        a = mma(Mt[i][k][s], X0[k][s], a);
        w = mma(Wt[i][k][s], X0[k][s], w);
      }
#pragma unroll
    for (int s = 0; s < 4; ++s) a = mma(Bt[i][s], U0[s], a);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const float th = dev_tanh(w[v]);
      SDv[i][v] = 1.f - th * th;
      C[i][v] = 16 * i + 4 * g + v < n ? X0[i][v] + hs * (a[v] + kap * th) - Xn[i][v] : 0.f;
    }
  }

  // the cost 1/2 d'Q d + 1/2 e'R e, with Q d and R e kept for the residual
  load_aop_raw<NT, NT, WIDE>(Mt, P.Q.at(b, 0), n, n, off);
  f4 D0[NT], E0, Rt;
  {
    const rsrc_t rxr = view_rsrc(P.xref, b, N1, n), rur = view_rsrc(P.uref, b, N, m);
#pragma unroll
    for (int k = 0; k < NT; ++k)
      D0[k] = vload4<WIDE>(rxr, (int)(tc * P.xref.st) + 16 * k + 4 * g, 16 * k + 4 * g, n);
    E0 = vload4<WIDE>(rur, (int)(tc * P.uref.st) + 4 * g, 4 * g, m);
    Rt = vload4<WIDE>(make_rsrc(P.R.at(b, 0), m * m), c * m + 4 * g, 4 * g, m);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int k = 0; k < NT; ++k) D0[k] = X0[k] - D0[k];
  E0 = U0 - E0;
  float cost = 0.f, acc = 0.f;
  f4 qa[NT], ra = zero4();
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    f4 q = zero4();
#pragma unroll
    for (int k = 0; k < NT; ++k)
#pragma unroll
      for (int s = 0; s < 4; ++s) q = mma(Mt[i][k][s], D0[k][s], q);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      cost += 0.5f * D0[i][v] * q[v];   // Q's rows past n are 0
      if (WHAT != EVAL_MODEL) acc += C[i][v] * C[i][v];
    }
    qa[i] = q;
  }
#pragma unroll
  for (int s = 0; s < 4; ++s) ra = mma(Rt[s], E0[s], ra);
#pragma unroll
  for (int v = 0; v < 4; ++v) cost += 0.5f * E0[v] * ra[v];   // R's rows past m are 0

  if constexpr (KKT) {
    // grad_x L = Q d + f_x' V_{t+1} - V_t + D'mu, grad_u L = R e + f_u' V_{t+1} + E'mu + nu_hi - nu_lo
    const rsrc_t rV = make_rsrc(it.V + (size_t)b * N1 * n, N1 * n);
    f4 V0[NT], Vn[NT], Bm[1][NT];
    load_aop_t<NT, NT>(Mt, P.A.at(b, 0), n, n, g, c);
    load_aop_t<NT, 1>(Bm, P.Bm.at(b, 0), n, m, g, c);
    load_aop_t<NT, NT>(Wt, P.W.at(b, 0), n, n, g, c);
#pragma unroll
    for (int k = 0; k < NT; ++k) {
      Vn[k] = vload4<WIDE>(rV, (tc + 1) * n + 16 * k + 4 * g, 16 * k + 4 * g, n);
      V0[k] = vload4<WIDE>(rV, tc * n + 16 * k + 4 * g, 16 * k + 4 * g, n);
    }
    __builtin_amdgcn_sched_barrier(0);
    f4 gu = zero4();
#pragma unroll
    for (int k = 0; k < NT; ++k)
#pragma unroll
      for (int s = 0; s < 4; ++s) gu = mma(Bm[0][k][s], Vn[k][s], gu);
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      f4 a = zero4(), w = zero4();
#pragma unroll
      for (int k = 0; k < NT; ++k)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          a = mma(Mt[i][k][s], Vn[k][s], a);
          w = mma(Wt[i][k][s], SDv[k][s] * Vn[k][s], w);
        }
#pragma unroll
      for (int v = 0; v < 4; ++v) qa[i][v] += Vn[i][v] + hs * (a[v] + kap * w[v]) - V0[i][v];
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) ra[v] += hs * gu[v];
    if (p > 0) {
      const rsrc_t rD = view_rsrc(P.D, b, N, p * n), rE = view_rsrc(P.E, b, N, p * m), re = view_rsrc(P.e, b, N, p);
      const rsrc_t rmu = make_rsrc(it.Yeq + (size_t)b * N * p, N * p);
      const int od = (int)(tc * P.D.st) + 4 * g, oe = (int)(tc * P.E.st) + 4 * g;
#pragma unroll 2
      for (int r = 0; r < p; ++r) {
        f4 Dr[NT];
#pragma unroll
        for (int k = 0; k < NT; ++k) Dr[k] = vload4<WIDE>(rD, od + r * n + 16 * k, 16 * k + 4 * g, n);
        const f4 Er = vload4<WIDE>(rE, oe + r * m, 4 * g, m);
        const float ev = rload(re, (int)(tc * P.e.st + r) * 4), mu = rload(rmu, (tc * p + r) * 4);
        float h = 0.f;
#pragma unroll
        for (int k = 0; k < NT; ++k)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            h += Dr[k][v] * X0[k][v];
            qa[k][v] += Dr[k][v] * mu;
          }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          h += Er[v] * U0[v];
          ra[v] += Er[v] * mu;
        }
        h = col_sum4(h) + ev;
        acc += g == 0 ? h * h : 0.f;
      }
    }
    if (P.box) {
      const rsrc_t rYb = make_rsrc(it.Ybox + (size_t)b * N * 2 * m, N * 2 * m);
      const rsrc_t rlo = view_rsrc(P.ulo, b, N, m), rhi = view_rsrc(P.uhi, b, N, m);
      const f4 lo = vload4<WIDE>(rlo, (int)(tc * P.ulo.st) + 4 * g, 4 * g, m);
      const f4 hi = vload4<WIDE>(rhi, (int)(tc * P.uhi.st) + 4 * g, 4 * g, m);
      const f4 nh = vload4<WIDE>(rYb, tc * 2 * m + 4 * g, 4 * g, m);
      const f4 nl = vload4<WIDE>(rYb, tc * 2 * m + m + 4 * g, 4 * g, m);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float c1 = nh[v] * (hi[v] - U0[v]) - prm.mu_b, c2 = nl[v] * (U0[v] - lo[v]) - prm.mu_b;
        ra[v] += nh[v] - nl[v];
        acc += 4 * g + v < m ? c1 * c1 + c2 * c2 : 0.f;
      }
    }
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc += 16 * i + 4 * g + v < n ? qa[i][v] * qa[i][v] : 0.f;
#pragma unroll
    for (int v = 0; v < 4; ++v) acc += 4 * g + v < m ? ra[v] * ra[v] : 0.f;
  }
  if (WHAT == EVAL_MODEL) {
    const rsrc_t rc = make_rsrc(oc + (size_t)b * N1 * n, N1 * n);
#pragma unroll
    for (int i = 0; i < NT; ++i) vstore4<WIDE>(rc, (t + 1) * n + 16 * i + 4 * g, 16 * i + 4 * g, n, live, C[i]);
  }
  cost = col_sum4(cost);
  if (WHAT != EVAL_MODEL) acc = col_sum4(acc);
  if (live && g == 0) {
    const size_t st = (size_t)b * N1 + t;
    if (WHAT == EVAL_MODEL) og[st] = cost;
    if (WHAT == EVAL_STOP) {
      ws.gpart[st * 2] = cost;
      ws.gpart[st * 2 + 1] = acc;
    }
    if (KKT) ws.kpart[st] = acc;
  }
}

}  // namespace mpxk
