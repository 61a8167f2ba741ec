// The linearisation (K1) and the trials of the line search on the matrix cores
// with the rows of the stage products spread over a block's waves: the tanh
// model with stage-invariant A, W, B, Q, R, for the sizes past k_lin_mma.h and
// k_trials_mma.h (FP32 n <= 80, m <= 32) and, the linearisation, for FP64.
//
// A block takes 16 consecutive stages of one instance, stage t0 + c in lane
// column c; wave i < NT takes rows 16 i .. 16 i + 15 of the state products
// (A x, W x, B u, Q (x - x_ref)), wave NT + i rows 16 i .. of R (u - u_ref)
// and the boxes.  A wave holds the stage vectors as B-operand tiles (lane
// (g, c), register v of tile k: entry 16 k + row(g, v) of stage c) and reads
// its own row tile of each matrix once; a result tile has the rows of the same
// index, so what follows is lane by lane.  The equality rows are dot products
// whose parts (one per wave: its 16 entries) meet in LDS, RQ rows at a time;
// the block after the last takes the terminal stage and the initial row.
//
// Bound by the loads' latency at small batches and by the bytes (f_x, D_t) at
// large ones.  76 x 32 x 50, p = 12, B = 256 (one wave per row of 64 lanes and
// one stage at a time before): linearisation 334 -> 103 us, trials 221 -> 92;
// 76 x 32 x 100, B = 8: 32 -> 16, 25 -> 16; FP64 36 x 12 x 50, p = 8, B = 64:
// linearisation 132 -> 28 (the trials, bound by their FP64 tanh, 36 -> 44: they
// stay on k_trials).
#pragma once
#include "k_lin_mma.h"
#include "k_lqr_tile.h"

namespace mpxk {

__device__ __forceinline__ double col_sum4(double x) {
  x += __shfl_xor(x, 32);
  return x + __shfl_xor(x, 16);
}

// Offset within its 16 of the entry in register v of lane group g (the rows of
// a result tile; the same order serves as the contracted index).
template <typename T>
__device__ __forceinline__ int rows_idx(int g, int v) {
  return sizeof(T) == 4 ? 4 * g + v : 4 * v + g;
}

// Entries 16 k + rows_idx(g, .) < lim of a vector at element offset o, 0 past
// lim.  WIDE (FP32): lim % 4 == 0 and o % 4 == 0, one 128-bit load.
template <typename T, bool WIDE>
__device__ __forceinline__ typename TileOps<T>::V4 rows_load(rsrc_t r, int o, int k, int g, int lim) {
  if constexpr (WIDE && sizeof(T) == 4) {
    return rload4(r, 16 * k + 4 * g < lim ? (o + 16 * k + 4 * g) * 4 : kOOB);
  } else {
    typename TileOps<T>::V4 x;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int e = 16 * k + rows_idx<T>(g, v);
      x[v] = TileOps<T>::bload(r, e < lim ? (o + e) * (int)sizeof(T) : kOOB);
    }
    return x;
  }
}

// The same entries stored (those of lanes with ok).
template <typename T, bool WIDE>
__device__ __forceinline__ void rows_store(rsrc_t r, int o, int k, int g, int lim, bool ok,
                                           const typename TileOps<T>::V4& x) {
  if constexpr (WIDE && sizeof(T) == 4) {
    vstore4<true>(r, o + 16 * k + 4 * g, 16 * k + 4 * g, lim, ok, x);
  } else {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int e = 16 * k + rows_idx<T>(g, v);
      TileOps<T>::bstore(r, ok && e < lim ? (o + e) * (int)sizeof(T) : kOOB, 0, x[v]);
    }
  }
}

// Descriptor over nst stages of a view from stage t on, len elements each; and
// over an array of ours with len elements per stage.
template <typename T>
__device__ __forceinline__ rsrc_t rows_view(const View<T>& v, int b, int t, int nst, int len) {
  return tile_rsrc(v.at(b, t), v.p ? (int)((nst - 1) * v.st + len) : 0);
}
template <typename T>
__device__ __forceinline__ rsrc_t rows_arr(const T* p, size_t stage, int nst, int len) {
  return tile_rsrc(p ? p + stage * len : p, p ? nst * len : 0);
}

// a += M X for one row tile: M row-major (rows x cols) behind r, its rows
// 16 i .., X the stage vectors; KT tiles of the contracted index.
template <typename T, bool WIDE, int KT>
__device__ __forceinline__ void rows_tile(typename TileOps<T>::V4 (&M)[KT], rsrc_t r, int i, int cols, int g, int c) {
#pragma unroll
  for (int k = 0; k < KT; ++k) M[k] = rows_load<T, WIDE>(r, (16 * i + c) * cols, k, g, cols);
}
template <typename T, int KT>
__device__ __forceinline__ typename TileOps<T>::V4 rows_dot(const typename TileOps<T>::V4 (&M)[KT],
                                                            const typename TileOps<T>::V4 (&X)[KT],
                                                            typename TileOps<T>::V4 a) {
#pragma unroll
  for (int k = 0; k < KT; ++k)
#pragma unroll
    for (int s = 0; s < 4; ++s) a = TileOps<T>::mma(M[k][s], X[k][s], a);
  return a;
}

constexpr int kRowsRQ = 8;   // equality rows per pass

// In the block of the terminal stage every lane column holds that stage, column
// 0 counts.
template <typename T, int NT, int MT, bool WIDE>
__global__ void __launch_bounds__(64 * (NT + MT)) __attribute__((amdgpu_waves_per_eu(2)))
k_linearize_rows(Prob<T> P, Prm<T> prm, Iter<T> it, Ws<T> ws) {
  typedef TileOps<T> O;
  typedef typename O::V4 V4;
  constexpr int NW = NT + MT, SD = 16 * NT + 1, RQ = kRowsRQ;
  __shared__ T sdl[16 * SD], part[NW][RQ][16], wl[RQ][16], red[NW][3][16];
  const int b = blockIdx.y, tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int g = lane >> 4, c = lane & 15;
  if (skip_instance(ws, b)) return;
  const int n = P.n, m = P.m, p = P.p, N = P.N, N1 = N + 1;
  const V4 zero = V4{T(0), T(0), T(0), T(0)};
  T cost = 0, vc = 0, cc = 0;
  const int t0 = blockIdx.x * 16;
  const bool term = blockIdx.x == gridDim.x - 1;

  if (term) {
    if (wv < NT) {
      const rsrc_t rX = rows_arr(it.X, (size_t)b * N1 + N, 1, n), rxr = rows_view(P.xref, b, N, 1, n);
      const rsrc_t rX0 = rows_arr(it.X, (size_t)b * N1, 1, n), rx0 = rows_view(P.x0, b, 0, 1, n);
      V4 D0[NT], M[NT];
      rows_tile<T, WIDE, NT>(M, tile_rsrc(P.QN.at(b, 0), n * n), wv, n, g, c);
#pragma unroll
      for (int k = 0; k < NT; ++k) {
        const V4 x = rows_load<T, WIDE>(rX, 0, k, g, n), xr = rows_load<T, WIDE>(rxr, 0, k, g, n);
#pragma unroll
        for (int v = 0; v < 4; ++v) D0[k][v] = x[v] - xr[v];
      }
      const V4 xi = rows_load<T, WIDE>(rX, 0, wv, g, n), xri = rows_load<T, WIDE>(rxr, 0, wv, g, n);
      const V4 x0 = rows_load<T, WIDE>(rx0, 0, wv, g, n), X0 = rows_load<T, WIDE>(rX0, 0, wv, g, n);
      const V4 v0 = rows_load<T, WIDE>(rows_arr(it.V, (size_t)b * N1, 1, n), 0, wv, g, n);
      const V4 q = rows_dot<T, NT>(M, D0, zero);
      V4 ci;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        ci[v] = x0[v] - X0[v];
        cost += T(0.5) * (xi[v] - xri[v]) * q[v];
        vc += v0[v] * ci[v];
        cc += ci[v] * ci[v];
      }
      rows_store<T, WIDE>(rows_arr(ws.qh, (size_t)b * N1 + N, 1, n), 0, wv, g, n, c == 0, q);
      rows_store<T, WIDE>(rows_arr(ws.cdef, (size_t)b * N1, 1, n), 0, wv, g, n, c == 0, ci);
    }
    const T* Bm = P.Bm.at(b, 0);
    for (int e = tid; e < n * m; e += 64 * NW) ws.Blin[(size_t)b * n * m + e] = P.h * Bm[e];
  } else {
    const int ns = min(16, N - t0), tc = min(c, ns - 1);   // columns past the last stage repeat it, nothing of theirs is kept
    const bool live = c < ns;
    const size_t sx = (size_t)b * N1 + t0, su = (size_t)b * N + t0;
    const bool box = P.box != 0;
    const int mb = box ? m : 0;
    const T hs = P.h, kap = P.kappa;
    const rsrc_t rX = rows_arr(it.X, sx, ns + 1, n), rU = rows_arr(it.U, su, ns, m);
    const rsrc_t rlo = rows_view(P.ulo, b, t0, ns, m), rhi = rows_view(P.uhi, b, t0, ns, m);
    const int olo = tc * (int)P.ulo.st, ohi = tc * (int)P.uhi.st;
    // u_t projected into the box interior
    auto inside = [&](V4 u, const V4& lo, const V4& hi, int i) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const T w = T(1e-3) * (hi[v] - lo[v]);
        T y = u[v];
        y = y >= hi[v] ? hi[v] - w : y;
        y = y <= lo[v] ? lo[v] + w : y;
        u[v] = 16 * i + rows_idx<T>(g, v) < mb ? y : u[v];
      }
      return u;
    };
    V4 U0[MT];
#pragma unroll
    for (int k = 0; k < MT; ++k) {
      const V4 u = rows_load<T, WIDE>(rU, tc * m, k, g, m);
      U0[k] = inside(u, rows_load<T, WIDE>(rlo, olo, k, g, mb), rows_load<T, WIDE>(rhi, ohi, k, g, mb), k);
    }
    const int i = wv < NT ? wv : wv - NT;
    V4 out, own;   // q or r of the wave's rows; its entries of x_t or u_t
    V4 lo, hi, C, SDv;
    if (wv < NT) {
      V4 X0[NT], M[NT], Wt[NT], Bt[MT], Q[NT], xr[NT];
#pragma unroll
      for (int k = 0; k < NT; ++k) X0[k] = rows_load<T, WIDE>(rX, tc * n, k, g, n);
      rows_tile<T, WIDE, NT>(M, tile_rsrc(P.A.at(b, 0), n * n), i, n, g, c);
      rows_tile<T, WIDE, NT>(Wt, tile_rsrc(P.W.at(b, 0), n * n), i, n, g, c);
      rows_tile<T, WIDE, MT>(Bt, tile_rsrc(P.Bm.at(b, 0), n * m), i, m, g, c);
      rows_tile<T, WIDE, NT>(Q, tile_rsrc(P.Q.at(b, 0), n * n), i, n, g, c);
      const rsrc_t rxr = rows_view(P.xref, b, t0, ns, n);
      const int oxr = tc * (int)P.xref.st;
#pragma unroll
      for (int k = 0; k < NT; ++k) xr[k] = rows_load<T, WIDE>(rxr, oxr, k, g, n);
      own = rows_load<T, WIDE>(rX, tc * n, i, g, n);
      const V4 xri = rows_load<T, WIDE>(rxr, oxr, i, g, n);
      const V4 xn = rows_load<T, WIDE>(rX, (tc + 1) * n, i, g, n);
      const V4 vn = rows_load<T, WIDE>(rows_arr(it.V, sx, ns + 1, n), (tc + 1) * n, i, g, n);
      // f = x + h (A x + B u + kappa tanh(W x)), c = f - x_{t+1}, sech^2(W x)
      const V4 a = rows_dot<T, MT>(Bt, U0, rows_dot<T, NT>(M, X0, zero));
      const V4 w = rows_dot<T, NT>(Wt, X0, zero);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const T th = dev_tanh(w[v]);
        SDv[v] = T(1) - th * th;
        C[v] = own[v] + hs * (a[v] + kap * th) - xn[v];   // rows past n: 0
        vc += vn[v] * C[v];
        cc += C[v] * C[v];
        sdl[c * SD + 16 * i + rows_idx<T>(g, v)] = SDv[v];
      }
#pragma unroll
      for (int k = 0; k < NT; ++k)
#pragma unroll
        for (int v = 0; v < 4; ++v) X0[k][v] -= xr[k][v];
      out = rows_dot<T, NT>(Q, X0, zero);
#pragma unroll
      for (int v = 0; v < 4; ++v) cost += T(0.5) * (own[v] - xri[v]) * out[v];
    } else {
      V4 R[MT], E0[MT];
      rows_tile<T, WIDE, MT>(R, tile_rsrc(P.R.at(b, 0), m * m), i, m, g, c);
      const rsrc_t rur = rows_view(P.uref, b, t0, ns, m);
      const int our = tc * (int)P.uref.st;
#pragma unroll
      for (int k = 0; k < MT; ++k) E0[k] = U0[k] - rows_load<T, WIDE>(rur, our, k, g, m);
      lo = rows_load<T, WIDE>(rlo, olo, i, g, mb);
      hi = rows_load<T, WIDE>(rhi, ohi, i, g, mb);
      own = inside(rows_load<T, WIDE>(rU, tc * m, i, g, m), lo, hi, i);
      const V4 e = own - rows_load<T, WIDE>(rur, our, i, g, m);
      out = rows_dot<T, MT>(R, E0, zero);
#pragma unroll
      for (int v = 0; v < 4; ++v) cost += T(0.5) * e[v] * out[v];
    }

    // equality rows h = e + D x + E u, w = mu + rho_c h: q += D' w, r += E' w,
    // cost += mu h + rho_c / 2 h^2
    if (p > 0) {
      const bool st = wv < NT;
      const int len = st ? n : m;
      const rsrc_t rD = st ? rows_view(P.D, b, t0, ns, p * n) : rows_view(P.E, b, t0, ns, p * m);
      const rsrc_t re = rows_view(P.e, b, t0, ns, p), rmu = rows_arr(it.Yeq, su, ns, p);
      const int od = tc * (int)(st ? P.D.st : P.E.st);
      for (int r0 = 0; r0 < p; r0 += RQ) {
        V4 Dr[RQ];
#pragma unroll
        for (int q = 0; q < RQ; ++q) Dr[q] = rows_load<T, WIDE>(rD, od + (r0 + q) * len, i, g, r0 + q < p ? len : 0);
        const int hr = tid >> 4;   // tid < 16 RQ: row r0 + hr of stage c
        const bool in = hr < RQ && r0 + hr < p;
        const T ev = O::bload(re, in ? (tc * (int)P.e.st + r0 + hr) * (int)sizeof(T) : kOOB);
        const T mv = O::bload(rmu, in ? (tc * p + r0 + hr) * (int)sizeof(T) : kOOB);
#pragma unroll
        for (int q = 0; q < RQ; ++q) {
          T h = 0;
#pragma unroll
          for (int v = 0; v < 4; ++v) h += Dr[q][v] * own[v];
          h = col_sum4(h);
          if (g == (q & 3)) part[wv][q][c] = h;
        }
        __syncthreads();
        if (hr < RQ) {
          T h = 0;
#pragma unroll
          for (int k = 0; k < NW; ++k) h += part[k][hr][c];
          h += ev;
          wl[hr][c] = in ? mv + prm.rho_c * h : T(0);
          cost += in ? mv * h + T(0.5) * prm.rho_c * h * h : T(0);
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < RQ; ++q) {
          const T w = wl[q][c];
#pragma unroll
          for (int v = 0; v < 4; ++v) out[v] += Dr[q][v] * w;
        }
      }
    } else {
      __syncthreads();
    }

    if (wv < NT) {
      rows_store<T, WIDE>(rows_arr(ws.qh, sx, ns, n), c * n, i, g, n, live, out);
      rows_store<T, WIDE>(rows_arr(ws.cdef, sx, ns + 1, n), (c + 1) * n, i, g, n, live, C);
      rows_store<T, WIDE>(rows_arr(ws.sdh, su, ns, n), c * n, i, g, n, live, SDv);
    } else {
      // the box: barrier cost and gradient, the Hessian diagonal, and the
      // multipliers that are not positive replaced by mu_b / slack
      V4 rd = zero;
      if (box) {
        rows_store<T, WIDE>(rU, c * m, i, g, m, live, own);
        const rsrc_t rYb = rows_arr(it.Ybox, su, ns, 2 * m);
        const V4 nh0 = rows_load<T, WIDE>(rYb, tc * 2 * m, i, g, m), nl0 = rows_load<T, WIDE>(rYb, tc * 2 * m + m, i, g, m);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int e = 16 * i + rows_idx<T>(g, v);
          const bool ok = e < m;
          const T shi = hi[v] - own[v], slo = own[v] - lo[v];
          cost -= ok ? prm.mu_b * (dev_log(shi) + dev_log(slo)) : T(0);
          const bool rh = ok && !(nh0[v] > T(0)), rl = ok && !(nl0[v] > T(0));
          const T nh = rh ? prm.mu_b / shi : nh0[v], nl = rl ? prm.mu_b / slo : nl0[v];
          O::bstore(rYb, live && rh ? (c * 2 * m + e) * (int)sizeof(T) : kOOB, 0, nh);
          O::bstore(rYb, live && rl ? (c * 2 * m + m + e) * (int)sizeof(T) : kOOB, 0, nl);
          out[v] += ok ? prm.mu_b / shi - prm.mu_b / slo : T(0);
          rd[v] = ok ? nh / shi + nl / slo : T(0);
        }
      }
      rows_store<T, WIDE>(rows_arr(ws.rh, su, ns, m), c * m, i, g, m, live, out);
      rows_store<T, WIDE>(rows_arr(ws.rd, su, ns, m), c * m, i, g, m, live, rd);
    }

    // f_x = I + h A + h kappa diag(sech^2(W x)) W by the whole block, stage by
    // stage: a thread keeps its entries of I + h A and h kappa W (the same for
    // every stage), so every store is a run of consecutive entries
    constexpr int KC = (16 * NT * 16 * NT / 4 + 64 * NW - 1) / (64 * NW);
    constexpr int VR = WIDE ? 1 : 4;
    const int nn = n * n;
    const rsrc_t rA = tile_rsrc(P.A.at(b, 0), nn), rW = tile_rsrc(P.W.at(b, 0), nn);
    const rsrc_t rAl = rows_arr(ws.Alin, su, ns, nn);
    V4 hA[KC], hW[KC];
    int row[KC][VR];
#pragma unroll
    for (int k = 0; k < KC; ++k) {
      const int e = 4 * (tid + 64 * NW * k);
#pragma unroll
      for (int v = 0; v < VR; ++v) row[k][v] = min((e + v) / n, n - 1);
      if constexpr (WIDE) {
        hA[k] = O::bload4(rA, e < nn ? e * (int)sizeof(T) : kOOB, 0);
        hW[k] = O::bload4(rW, e < nn ? e * (int)sizeof(T) : kOOB, 0);
      } else {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          hA[k][v] = O::bload(rA, e + v < nn ? (e + v) * (int)sizeof(T) : kOOB);
          hW[k][v] = O::bload(rW, e + v < nn ? (e + v) * (int)sizeof(T) : kOOB);
        }
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int j = row[k][WIDE ? 0 : v];
        hA[k][v] = (e + v - j * n == j ? T(1) : T(0)) + hs * hA[k][v];
        hW[k][v] = hs * kap * hW[k][v];
      }
    }
    for (int tt = 0; tt < ns; ++tt) {
      const T* sd = sdl + tt * SD;
#pragma unroll
      for (int k = 0; k < KC; ++k) {
        const int e = 4 * (tid + 64 * NW * k), o = (tt * nn + e) * (int)sizeof(T);
        V4 y;
#pragma unroll
        for (int v = 0; v < 4; ++v) y[v] = hA[k][v] + sd[row[k][WIDE ? 0 : v]] * hW[k][v];
        if constexpr (WIDE && sizeof(T) == 4) {
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(mpxk_u32x4, y), rAl, e < nn ? o : kOOB, 0, 0);
        } else if constexpr (WIDE) {
#pragma unroll
          for (int v = 0; v < 4; v += 2)
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(mpxk_u32x4, mpxk_f64x2{y[v], y[v + 1]}), rAl,
                                                   e < nn ? o + 8 * v : kOOB, 0, 0);
        } else {
#pragma unroll
          for (int v = 0; v < 4; ++v) O::bstore(rAl, e + v < nn ? o + v * (int)sizeof(T) : kOOB, 0, y[v]);
        }
      }
    }
  }

  // merit parts: the four lanes of a column, then the waves
  cost = col_sum4(cost);
  vc = col_sum4(vc);
  cc = col_sum4(cc);
  if (g == 0) {
    red[wv][MP_COST][c] = cost;
    red[wv][MP_VC][c] = vc;
    red[wv][MP_CC][c] = cc;
  }
  __syncthreads();
  const int t = term ? N : t0 + c;
  if (tid < 48 && (term ? c == 0 : t < N)) {
    T s = 0;
#pragma unroll
    for (int k = 0; k < NW; ++k) s += red[k][tid >> 4][c];
    ws.mpart[((size_t)b * N1 + t) * NMP + (tid >> 4)] = s;
  }
}

// Trials j0 <= j < j1 of the 16 stages of the block (the last block: the
// terminal stage): the merit parts of k_trials.  The quadratic terms are
// polynomials in the step summed once per lane, the model's tanh, the defect
// and the box logarithms run per trial on the rows of each lane; the sums of
// the waves meet in LDS after the last trial.
template <typename T, int NT, int MT, bool WIDE>
__global__ void __launch_bounds__(64 * (NT + MT)) __attribute__((amdgpu_waves_per_eu(2)))
k_trials_rows(Prob<T> P, Prm<T> prm, Iter<T> it, Ws<T> ws, int j0, int j1) {
  typedef TileOps<T> O;
  typedef typename O::V4 V4;
  constexpr int NW = NT + MT, RQ = kRowsRQ;
  __shared__ T part[2][NW][RQ][16], red[MAX_TRIALS][NW][2][16];
  const int b = blockIdx.y, tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int g = lane >> 4, c = lane & 15;
  if (skip_instance(ws, b)) return;
  const int n = P.n, m = P.m, p = P.p, N = P.N, N1 = N + 1;
  if (j0 > 0 && ls_first_accept(prm, ws, b, N1, j0) >= 0) return;   // an earlier pass accepted
  const V4 zero = V4{T(0), T(0), T(0), T(0)};
  const int t0 = blockIdx.x * 16;
  const bool term = blockIdx.x == gridDim.x - 1;
  const int ns = term ? 1 : min(16, N - t0), tc = min(c, ns - 1);
  const size_t sx = (size_t)b * N1 + (term ? N : t0), su = (size_t)b * N + t0;
  const bool box = P.box != 0 && !term;
  const int mb = box ? m : 0;
  const int i = wv < NT ? wv : wv - NT;
  // the lane's rows: defect c0 + a c1 + hk tanh(w0 + a w1), its multiplier
  // v0 + a v1; the quadratic terms p0 + a (p1 + a p2)
  V4 C0 = zero, C1 = zero, W0 = zero, W1 = zero, v0 = zero, v1 = zero, own0, own1, lo, hi;
  T p0 = 0, p1 = 0, p2 = 0;
  if (wv < NT) {
    const int nx = term ? 1 : ns + 1;
    const rsrc_t rX = rows_arr(it.X, sx, nx, n), rdX = rows_arr(ws.dx, sx, nx, n);
    const rsrc_t rxr = rows_view(P.xref, b, term ? N : t0, ns, n);
    const int oxr = tc * (int)P.xref.st;
    V4 X0[NT], X1[NT], Q[NT];
#pragma unroll
    for (int k = 0; k < NT; ++k) {
      X0[k] = rows_load<T, WIDE>(rX, tc * n, k, g, n);
      X1[k] = rows_load<T, WIDE>(rdX, tc * n, k, g, n);
    }
    rows_tile<T, WIDE, NT>(Q, tile_rsrc(term ? P.QN.at(b, 0) : P.Q.at(b, 0), n * n), i, n, g, c);
    own0 = rows_load<T, WIDE>(rX, tc * n, i, g, n);
    own1 = rows_load<T, WIDE>(rdX, tc * n, i, g, n);
    const V4 d0 = own0 - rows_load<T, WIDE>(rxr, oxr, i, g, n);
    if (term) {   // c_init = x0 - X_0 and V_0
      const V4 x0 = rows_load<T, WIDE>(rows_view(P.x0, b, 0, 1, n), 0, i, g, n);
      C0 = x0 - rows_load<T, WIDE>(rows_arr(it.X, (size_t)b * N1, 1, n), 0, i, g, n);
      C1 = zero - rows_load<T, WIDE>(rows_arr(ws.dx, (size_t)b * N1, 1, n), 0, i, g, n);
      v0 = rows_load<T, WIDE>(rows_arr(it.V, (size_t)b * N1, 1, n), 0, i, g, n);
      v1 = rows_load<T, WIDE>(rows_arr(ws.dv, (size_t)b * N1, 1, n), 0, i, g, n);
    } else {
      V4 M[NT], Wt[NT], Bt[MT], U0[MT], U1[MT];
      const rsrc_t rU = rows_arr(it.U, su, ns, m), rdU = rows_arr(ws.du, su, ns, m);
      rows_tile<T, WIDE, NT>(M, tile_rsrc(P.A.at(b, 0), n * n), i, n, g, c);
      rows_tile<T, WIDE, NT>(Wt, tile_rsrc(P.W.at(b, 0), n * n), i, n, g, c);
      rows_tile<T, WIDE, MT>(Bt, tile_rsrc(P.Bm.at(b, 0), n * m), i, m, g, c);
#pragma unroll
      for (int k = 0; k < MT; ++k) {
        U0[k] = rows_load<T, WIDE>(rU, tc * m, k, g, m);
        U1[k] = rows_load<T, WIDE>(rdU, tc * m, k, g, m);
      }
      const V4 xn0 = rows_load<T, WIDE>(rX, (tc + 1) * n, i, g, n), xn1 = rows_load<T, WIDE>(rdX, (tc + 1) * n, i, g, n);
      v0 = rows_load<T, WIDE>(rows_arr(it.V, sx, nx, n), (tc + 1) * n, i, g, n);
      v1 = rows_load<T, WIDE>(rows_arr(ws.dv, sx, nx, n), (tc + 1) * n, i, g, n);
      const V4 a0 = rows_dot<T, MT>(Bt, U0, rows_dot<T, NT>(M, X0, zero));
      const V4 a1 = rows_dot<T, MT>(Bt, U1, rows_dot<T, NT>(M, X1, zero));
      W0 = rows_dot<T, NT>(Wt, X0, zero);
      W1 = rows_dot<T, NT>(Wt, X1, zero);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        C0[v] = own0[v] + P.h * a0[v] - xn0[v];
        C1[v] = own1[v] + P.h * a1[v] - xn1[v];
      }
    }
    // tracking cost 1/2 (d0 + a x1)' Q (d0 + a x1), d0 = x - x_ref
#pragma unroll
    for (int k = 0; k < NT; ++k) X0[k] -= rows_load<T, WIDE>(rxr, oxr, k, g, n);
    const V4 q0 = rows_dot<T, NT>(Q, X0, zero), q1 = rows_dot<T, NT>(Q, X1, zero);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      p0 += d0[v] * q0[v];
      p1 += d0[v] * q1[v] + own1[v] * q0[v];
      p2 += own1[v] * q1[v];
    }
  } else if (!term) {
    V4 R[MT], E0[MT], U1[MT];
    const rsrc_t rU = rows_arr(it.U, su, ns, m), rdU = rows_arr(ws.du, su, ns, m);
    const rsrc_t rur = rows_view(P.uref, b, t0, ns, m);
    const rsrc_t rlo = rows_view(P.ulo, b, t0, ns, m), rhi = rows_view(P.uhi, b, t0, ns, m);
    const int our = tc * (int)P.uref.st;
    rows_tile<T, WIDE, MT>(R, tile_rsrc(P.R.at(b, 0), m * m), i, m, g, c);
#pragma unroll
    for (int k = 0; k < MT; ++k) {
      E0[k] = rows_load<T, WIDE>(rU, tc * m, k, g, m) - rows_load<T, WIDE>(rur, our, k, g, m);
      U1[k] = rows_load<T, WIDE>(rdU, tc * m, k, g, m);
    }
    own0 = rows_load<T, WIDE>(rU, tc * m, i, g, m);
    own1 = rows_load<T, WIDE>(rdU, tc * m, i, g, m);
    lo = rows_load<T, WIDE>(rlo, tc * (int)P.ulo.st, i, g, mb);
    hi = rows_load<T, WIDE>(rhi, tc * (int)P.uhi.st, i, g, mb);
    const V4 e0 = own0 - rows_load<T, WIDE>(rur, our, i, g, m);
    const V4 r0 = rows_dot<T, MT>(R, E0, zero), r1 = rows_dot<T, MT>(R, U1, zero);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      p0 += e0[v] * r0[v];
      p1 += e0[v] * r1[v] + own1[v] * r0[v];
      p2 += own1[v] * r1[v];
    }
  }
  p0 *= T(0.5);
  p1 *= T(0.5);
  p2 *= T(0.5);

  // equality rows at the iterate and along the step, kept in hq for the update
  // of their multipliers, and their part mu h + rho_c / 2 h^2 of the merit
  if (p > 0 && !term) {
    const bool st = wv < NT;
    const int len = st ? n : m;
    const rsrc_t rD = st ? rows_view(P.D, b, t0, ns, p * n) : rows_view(P.E, b, t0, ns, p * m);
    const rsrc_t re = rows_view(P.e, b, t0, ns, p), rmu = rows_arr(it.Yeq, su, ns, p);
    const rsrc_t rhq = rows_arr(ws.hq, su, ns, 2 * p);
    const int od = tc * (int)(st ? P.D.st : P.E.st);
    for (int r0 = 0; r0 < p; r0 += RQ) {
      V4 Dr[RQ];
#pragma unroll
      for (int q = 0; q < RQ; ++q) Dr[q] = rows_load<T, WIDE>(rD, od + (r0 + q) * len, i, g, r0 + q < p ? len : 0);
      const int hr = tid >> 4;
      const bool in = hr < RQ && r0 + hr < p;
      const T ev = O::bload(re, in ? (tc * (int)P.e.st + r0 + hr) * (int)sizeof(T) : kOOB);
      const T mv = O::bload(rmu, in ? (tc * p + r0 + hr) * (int)sizeof(T) : kOOB);
      if (r0 > 0) __syncthreads();   // the parts of the rows before are summed
#pragma unroll
      for (int q = 0; q < RQ; ++q) {
        T h0 = 0, h1 = 0;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          h0 += Dr[q][v] * own0[v];
          h1 += Dr[q][v] * own1[v];
        }
        h0 = col_sum4(h0);
        h1 = col_sum4(h1);
        if (g == (q & 3)) {
          part[0][wv][q][c] = h0;
          part[1][wv][q][c] = h1;
        }
      }
      __syncthreads();
      if (in) {
        T h0 = 0, h1 = 0;
#pragma unroll
        for (int k = 0; k < NW; ++k) {
          h0 += part[0][k][hr][c];
          h1 += part[1][k][hr][c];
        }
        h0 += ev;
        p0 += mv * h0 + T(0.5) * prm.rho_c * h0 * h0;
        p1 += mv * h1 + prm.rho_c * h0 * h1;
        p2 += T(0.5) * prm.rho_c * h1 * h1;
        if (j0 == 0 && c < ns) {
          O::bstore(rhq, (c * 2 * p + r0 + hr) * (int)sizeof(T), 0, h0);
          O::bstore(rhq, (c * 2 * p + p + r0 + hr) * (int)sizeof(T), 0, h1);
        }
      }
    }
  }

  const T hk = P.h * P.kappa;
  T a = ws.lsp[(size_t)b * NLS + LS_AMAX];
  for (int q = 0; q < j0; ++q) a *= prm.beta;
  for (int j = j0; j < j1; ++j, a *= prm.beta) {
    T s1 = p0 + a * (p1 + a * p2), s2 = 0;
    if (wv < NT) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        T cv = C0[v] + a * C1[v];
        if (!term) cv += hk * dev_tanh(W0[v] + a * W1[v]);
        s1 += (v0[v] + a * v1[v]) * cv;
        s2 += cv * cv;
      }
    } else if (box) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const T u = own0[v] + a * own1[v];
        const T y = dev_log(hi[v] - u) + dev_log(u - lo[v]);
        s1 -= 16 * i + rows_idx<T>(g, v) < m ? prm.mu_b * y : T(0);
      }
    }
    s1 = col_sum4(s1);
    s2 = col_sum4(s2);
    if (g == 0) {
      red[j - j0][wv][0][c] = s1;
      red[j - j0][wv][1][c] = s2;
    }
  }
  __syncthreads();
  for (int e = tid; e < 32 * (j1 - j0); e += 64 * NW) {
    const int j = e >> 5, q = (e >> 4) & 1;   // c = e % 16 (64 NW a multiple of 16)
    if (c >= ns) continue;
    T s = 0;
#pragma unroll
    for (int k = 0; k < NW; ++k) s += red[j][k][q][c];
    ws.tpart[(sx + c) * 2 * MAX_TRIALS + 2 * (j0 + j) + q] = s;
  }
}

}  // namespace mpxk
