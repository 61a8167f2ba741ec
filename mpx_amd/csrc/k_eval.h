// Model evaluation (g, c), the stop test's partials and the KKT residual of an
// iterate for n <= 80: one wave per stage, every matrix read once, by rows.
//
// A group of 16 lanes takes the rows gq, gq + 4, ... of a matrix, lane l of it
// the columns l, l + 16, ... (64 bytes per row and load); a row's product is a
// DPP sum within the group, and the same entries also feed the transposed
// product (columns), which the four groups add once at the end.  A thread per
// row (the general kernels of k_misc.h, for larger n) reads 64 different cache
// lines per load and each matrix once per product.  Bound by the L1's rate of
// loads (about 100 per wave and stage); both evaluations at B = 1024: 76 x 32 x 50, p
// = 12 700 us (a thread per row 5718), stage-varying 19 x 7 x 33, p = 3 119 (215), FP64
// 36 x 12 x 50, p = 8 439 (1475).
#pragma once
#include "k_fwd_block.h"

namespace mpxk {

// v summed over the four lanes l, l + 16, l + 32, l + 48, in each of them
template <typename T>
__device__ __forceinline__ T groups_sum(T v) {
  v += __shfl_xor(v, 16);
  return v + __shfl_xor(v, 32);
}

enum { EVAL_MODEL = 0, EVAL_STOP = 1, EVAL_KKT = 2 };

constexpr int kEvalWaves = 4;

// one wave's LDS: x, x - x_ref, x_{t+1}, V_{t+1}, Q d, A x + B u, W x (16 NC
// each), u, u - u_ref, R e (64 each)
template <int NC>
__host__ __device__ constexpr int eval_wave_elems() { return 7 * 16 * NC + 3 * 64; }

// The rows of one matrix, four at a time (r0, r0 + 4, ... < rows): f(r0, a), a
// the lane's entries of row r0 + gq.  Rows past the matrix lie past the
// descriptor and read 0, columns past it have an offset past every descriptor:
// no masks.  Sixteen rows are requested before the first is used: with few
// stages a wave waits for each request (60 x 20 x 30, B = 1: the two evaluations
// 16.5 and 20.7 us with four rows in flight, 11.7 and 15.9 with sixteen; a
// thread per row 17.2 and 13.8).
template <typename T, int C, typename F>
__device__ __forceinline__ void eval_rows_of(const T* M, int rows, int cols, int gq, int l, F&& f) {
  typedef TileOps<T> O;
  const rsrc_t r = tile_rsrc(M, rows * cols);
  int off[C];
#pragma unroll
  for (int j = 0; j < C; ++j) off[j] = l + 16 * j < cols ? (gq * cols + l + 16 * j) * (int)sizeof(T) : kOOB;
  int r0 = 0;
  for (; r0 + 12 < rows; r0 += 16) {
    T a[4][C];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int j = 0; j < C; ++j) a[k][j] = O::bload(r, off[j], (r0 + 4 * k) * cols * (int)sizeof(T));
#pragma unroll
    for (int k = 0; k < 4; ++k) f(r0 + 4 * k, a[k]);
  }
  for (; r0 < rows; r0 += 4) {
    T a[C];
#pragma unroll
    for (int j = 0; j < C; ++j) a[j] = O::bload(r, off[j], r0 * cols * (int)sizeof(T));
    f(r0, a);
  }
}

// One wave's evaluation of stage t.  WHAT: EVAL_MODEL writes g_t and c_{t+1}
// (c_0 at t = N) to og, oc; EVAL_STOP g_t and |c|^2 to ws.gpart; EVAL_KKT the
// stage's squared residual (k_kkt_stage's terms) to ws.kpart.  n <= 16 NC, m <= 16
// MC; LAST: t = N.  The tanh and the defects are formed once per row, by columns
// of lanes, between the pass over A, B and W and a second one over W (KKT).
template <typename T, int NC, int MC, int WHAT, bool LAST>
__device__ __forceinline__ void eval_stage(const Prob<T>& P, const Prm<T>& prm, const Iter<T>& it, const Ws<T>& ws, T* og,
                                           T* oc, int b, int t, T* sx) {
  constexpr int LX = 16 * NC;
  constexpr bool KKT = WHAT == EVAL_KKT;
  const int n = P.n, m = P.m, p = P.p, N = P.N, N1 = N + 1;
  const int lane = threadIdx.x & 63, gq = lane >> 4, l = lane & 15;
  T *sd = sx + LX, *sxn = sd + LX, *sv = sxn + LX, *sq = sv + LX, *sf = sq + LX, *sw = sf + LX;
  T *su = sw + LX, *se = su + 64, *sr = se + 64;
  const bool caller = P.model == MODEL_CALLER, tanh_model = P.model == MODEL_TANH;
  const bool last = LAST || t == N;
  const T* X = it.X + ((size_t)b * N1 + t) * n;
  const T* xr = caller ? nullptr : P.xref.at(b, t);
  const T* V = KKT ? it.V + ((size_t)b * N1 + t) * n : nullptr;
  const T* U = it.U + ((size_t)b * N + (last ? 0 : t)) * m;
  const T* ur = caller || last ? nullptr : P.uref.at(b, t);
  for (int i = lane; i < LX; i += 64) {
    const bool in = i < n;
    const T x = in ? X[i] : T(0);
    sx[i] = x;
    sd[i] = in && !caller ? x - xr[i] : T(0);
    sxn[i] = in && !last ? X[n + i] : T(0);
    sv[i] = KKT && in && !last ? V[n + i] : T(0);
  }
  {
    const bool in = lane < m && !last;
    const T u = in ? U[lane] : T(0);
    su[lane] = u;
    se[lane] = in && !caller ? u - ur[lane] : T(0);
  }
  wave_lds_sync();
  T cost = T(0), acc = T(0);   // summed over the lanes at the end
  if (!caller) {
    T d[NC];
#pragma unroll
    for (int j = 0; j < NC; ++j) d[j] = sd[l + 16 * j];
    eval_rows_of<T, NC>(last ? P.QN.at(b, 0) : P.Q.at(b, t), n, n, gq, l, [&](int r0, const T (&a)[NC]) {
      T s = T(0);
#pragma unroll
      for (int j = 0; j < NC; ++j) s += a[j] * d[j];
      s = row16_sum(s);
      if (l == 0) sq[r0 + gq] = s;
    });
    if (!last) {
      T e[MC];
#pragma unroll
      for (int j = 0; j < MC; ++j) e[j] = se[l + 16 * j];
      eval_rows_of<T, MC>(P.R.at(b, t), m, m, gq, l, [&](int r0, const T (&a)[MC]) {
        T s = T(0);
#pragma unroll
        for (int j = 0; j < MC; ++j) s += a[j] * e[j];
        s = row16_sum(s);
        if (l == 0) sr[r0 + gq] = s;
      });
    }
  } else if (lane == 0) {
    cost = P.g.at(b, t)[0];
  }
  T x[NC], u[MC], ga[NC], gb[MC];   // ga, gb: the lane's columns of f_x' v (and D'mu), f_u' v
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    x[j] = sx[l + 16 * j];
    ga[j] = T(0);
  }
#pragma unroll
  for (int j = 0; j < MC; ++j) {
    u[j] = su[l + 16 * j];
    gb[j] = T(0);
  }
  if (!last) {
    const int ts = tanh_model ? 0 : t;
    eval_rows_of<T, NC>(P.A.at(b, ts), n, n, gq, l, [&](int r0, const T (&a)[NC]) {
      T s = T(0);
      const T v = sv[r0 + gq];
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        s += a[j] * x[j];
        if (KKT) ga[j] += a[j] * v;
      }
      s = row16_sum(s);
      if (l == 0) sf[r0 + gq] = s;
    });
    if (tanh_model) {
      eval_rows_of<T, NC>(P.W.at(b, 0), n, n, gq, l, [&](int r0, const T (&a)[NC]) {
        T s = T(0);
#pragma unroll
        for (int j = 0; j < NC; ++j) s += a[j] * x[j];
        s = row16_sum(s);
        if (l == 0) sw[r0 + gq] = s;
      });
    }
    eval_rows_of<T, MC>(P.Bm.at(b, ts), n, m, gq, l, [&](int r0, const T (&a)[MC]) {
      T s = T(0);
      const T v = sv[r0 + gq];
#pragma unroll
      for (int j = 0; j < MC; ++j) {
        s += a[j] * u[j];
        if (KKT) gb[j] += a[j] * v;
      }
      s = row16_sum(s);
      if (l == 0) sf[r0 + gq] += s;
    });
  }
  wave_lds_sync();
  // by rows, one per lane: the cost, the dynamics and the defect
  if (!caller) {
    for (int i = lane; i < n; i += 64) cost += T(0.5) * sd[i] * sq[i];
    if (!last && lane < m) cost += T(0.5) * se[lane] * sr[lane];
  }
  if (!last) {
    const T* fb = caller ? P.fbar.at(b, t) : nullptr;
    for (int i = lane; i < LX; i += 64) {
      const bool in = i < n;
      T f;
      if (tanh_model) {
        const T th = dev_tanh(in ? sw[i] : T(0));
        f = sx[i] + P.h * (sf[i] + P.kappa * th);
        if (KKT) sw[i] = in ? P.kappa * (T(1) - th * th) * sv[i] : T(0);
      } else {
        f = caller ? (in ? fb[i] : T(0)) : sf[i];
      }
      if (in) {
        const T c = f - sxn[i];
        if (WHAT == EVAL_MODEL) oc[((size_t)b * N1 + t + 1) * n + i] = c;
        else acc += c * c;
      }
    }
  } else {
    const T* x0 = P.x0.at(b, 0);
    const T* X0 = it.X + (size_t)b * N1 * n;
    for (int i = lane; i < n; i += 64) {
      const T c = x0[i] - X0[i];
      if (WHAT == EVAL_MODEL) oc[(size_t)b * N1 * n + i] = c;
      else acc += c * c;
    }
  }
  if constexpr (KKT) {
    const T* qc = caller ? P.q.at(b, t) : nullptr;
    if (!last) {
      wave_lds_sync();   // sw
      if (tanh_model)
        eval_rows_of<T, NC>(P.W.at(b, 0), n, n, gq, l, [&](int r0, const T (&a)[NC]) {
          const T v = sw[r0 + gq];
#pragma unroll
          for (int j = 0; j < NC; ++j) ga[j] += a[j] * v;
        });
      const T hs = tanh_model ? P.h : T(1);
#pragma unroll
      for (int j = 0; j < NC; ++j) ga[j] *= hs;
#pragma unroll
      for (int j = 0; j < MC; ++j) gb[j] *= hs;
      // equality rows h = D x + E u + e, and D'mu, E'mu by columns
      if (p > 0) {
        const T *e = P.e.at(b, t), *mu = it.Yeq + ((size_t)b * N + t) * p;
        const rsrc_t rD = tile_rsrc(P.D.at(b, t), p * n), rE = tile_rsrc(P.E.at(b, t), p * m);
        for (int r0 = 0; r0 < p; r0 += 4) {
          const int r = r0 + gq;
          const T y = r < p ? mu[r] : T(0);
          T h = T(0);
#pragma unroll
          for (int j = 0; j < NC; ++j) {
            const T d = TileOps<T>::bload(rD, l + 16 * j < n ? (r * n + l + 16 * j) * (int)sizeof(T) : kOOB);
            h += d * x[j];
            ga[j] += d * y;
          }
#pragma unroll
          for (int j = 0; j < MC; ++j) {
            const T d = TileOps<T>::bload(rE, l + 16 * j < m ? (r * m + l + 16 * j) * (int)sizeof(T) : kOOB);
            h += d * u[j];
            gb[j] += d * y;
          }
          h = row16_sum(h);
          if (l == 0 && r < p) acc += (h + e[r]) * (h + e[r]);
        }
      }
      const T* rc = caller ? P.r.at(b, t) : nullptr;
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        const int i = l + 16 * j;
        const T s = groups_sum(ga[j]);
        if (gq == 0 && i < n) {
          const T g = (caller ? qc[i] : sq[i]) + (tanh_model ? sv[i] + s : s) - V[i];
          acc += g * g;
        }
      }
#pragma unroll
      for (int j = 0; j < MC; ++j) {
        const int i = l + 16 * j;
        const T s = groups_sum(gb[j]);
        if (gq == 0 && i < m) {
          T g = (caller ? rc[i] : sr[i]) + s;
          if (P.box) {
            const T* nu = it.Ybox + ((size_t)b * N + t) * 2 * m;
            const T c1 = nu[i] * (P.uhi.at(b, t)[i] - su[i]) - prm.mu_b;
            const T c2 = nu[m + i] * (su[i] - P.ulo.at(b, t)[i]) - prm.mu_b;
            g += nu[i] - nu[m + i];
            acc += c1 * c1 + c2 * c2;
          }
          acc += g * g;
        }
      }
    } else {
      for (int i = lane; i < n; i += 64) {
        const T g = (caller ? qc[i] : sq[i]) - V[i];
        acc += g * g;
      }
    }
  }
  const size_t st = (size_t)b * N1 + t;
  if (!KKT) cost = wave_sum(cost);
  if (WHAT != EVAL_MODEL) acc = wave_sum(acc);
  if (lane == 0) {
    if (WHAT == EVAL_MODEL) og[st] = cost;
    if (WHAT == EVAL_STOP) {
      ws.gpart[st * 2] = cost;
      ws.gpart[st * 2 + 1] = acc;
    }
    if (KKT) ws.kpart[st] = acc;
  }
}

// kEvalWaves stages per block, a wave each.  (Four stages per wave, one after the
// other, past 32768 stages: 19 x 7 x 33, stage-varying, B = 1024 135 us against 124,
// FP64 36 x 12 x 50 558 against 456, 76 x 32 x 50 944 against 725.)
template <typename T, int NC, int MC, int WHAT>
__global__ void __launch_bounds__(64 * kEvalWaves)
k_eval_rows(Prob<T> P, Prm<T> prm, Iter<T> it, Ws<T> ws, T* og, T* oc) {
  __shared__ T smem[kEvalWaves * eval_wave_elems<NC>()];
  const int b = blockIdx.y;
  if (WHAT == EVAL_STOP && skip_instance(ws, b)) return;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int t = blockIdx.x * kEvalWaves + w;
  if (t <= P.N) eval_stage<T, NC, MC, WHAT, false>(P, prm, it, ws, og, oc, b, t, smem + w * eval_wave_elems<NC>());
}

}  // namespace mpxk
