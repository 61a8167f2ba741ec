// LQR solve (backward recursion and dx chain) of a small caller-linearised
// problem, one wave per instance: FP32 on the matrix cores, n <= 15, m <= 16,
// p <= 16 -- the single-rigid-body quadruped's 13 x 12.  Every matrix is one
// 16 x 16 tile in registers and the wave needs no barrier.
//
// It performs the operations of k_lqr_seq's recursion (riccati_step, chol_lds,
// trsm_lower, trsm_upper_t, fwd_chain) entry by entry in the same order, so
// its results are the same bits: the quadruped's iterations on clipped
// penalties amplify a last-digit change of the step to 1e-4 and more of the
// next iterate, so a recursion of another rounding would return other plans.
//
// A tile X is held "natural": lane (q, r) (q = lane / 16, r = lane % 16),
// register s: X[4 s + q][r] -- matrix instruction s of a product contracts the
// entries 4 s .. 4 s + 3, as mfma_gemm does.  The left operand is loaded with
// its output index permuted, pi(4 a + b) = 4 b + a, so that a result comes out
// natural too (its register v of lane (q, r) is position 4 q + v = entry 4 v +
// q).  H goes through LDS into a row per lane, G into a column per lane; the
// factor's entries pass between the lanes of a row of 16 by DPP.
//
// What bounds it: the instructions of one wave, 2200 a stage, most of them in the
// serial chain of the factorisation and the solves (12 square roots, 36 divisions
// and their sums); the next stage's data is requested
// a stage ahead.  13 x 12 x 25, B = 64: 133 us, k_lqr_seq (block of 256 threads,
// 60 barriers a stage, the factorisation in LDS): 697.
#pragma once
#include <type_traits>
#include "k_lqr_tile.h"

namespace mpxk {

// sum over the four lanes of a column as dot4 adds them: (q0 + q1) + (q2 + q3)
__device__ __forceinline__ float pair_sum4(float x) {
  const unsigned u = __float_as_uint(x);
  const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const float y = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const unsigned w = __float_as_uint(y);
  const auto d = __builtin_amdgcn_permlane32_swap(w, w, false, false);
  return __uint_as_float(d[0]) + __uint_as_float(d[1]);
}

// f(0), ..., with the index as a constant (the lane of a row broadcast is one)
template <int I, int E, typename F>
__device__ __forceinline__ void small_for(F&& f) {
  if constexpr (I < E) {
    f(std::integral_constant<int, I>{});
    small_for<I + 1, E>(f);
  }
}

// x of lane K of the row of 16 (DPP row_newbcast: a modifier of the instruction
// that takes it; through readlane a stage took 17 k cycles)
template <int K>
__device__ __forceinline__ float row_lane(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x150 + K, 0xf, 0xf, false));
}

constexpr int kSmallLD = 17;   // LDS row: 16 entries, rows in different banks

template <int MAXM>
__global__ void __launch_bounds__(64) k_lqr_small(Prob<float> P, Prm<float> prm, Ws<float> ws, LqrIn<float> in) {
  static_assert(MAXM == 12 || MAXM == 16, "control rows of the factorisation");
  constexpr int LD = kSmallLD, MM = MAXM;
  __shared__ float sS[16 * LD], sH[16 * LD], sG[16 * LD], sK[16 * LD], sv[16];
  const int b = blockIdx.x, lane = threadIdx.x, q = lane >> 4, r = lane & 15, pr = 4 * (r & 3) + (r >> 2);
  if (skip_instance(ws, b)) return;
  const int n = P.n, m = P.m, p = P.p, N = P.N, N1 = N + 1;
  const float sr = dev_sqrt(prm.rho_c);
  const bool cross = P.M.p != nullptr;

  // Offsets of a tile X[rows x cols]: entries [4 s + q][j] (nat), [i][4 s + q]
  // (row); opaque, so that they stay in registers rather than as lane masks.
  struct Off {
    int o[4];
  };
  auto nat = [&](int rows, int cols, int j) {
    Off f;
#pragma unroll
    for (int s = 0; s < 4; ++s) f.o[s] = fresh(4 * s + q < rows && j < cols ? ((4 * s + q) * cols + j) * 4 : kOOB);
    return f;
  };
  auto row = [&](int rows, int cols, int i) {
    Off f;
#pragma unroll
    for (int s = 0; s < 4; ++s) f.o[s] = fresh(i < rows && 4 * s + q < cols ? (i * cols + 4 * s + q) * 4 : kOOB);
    return f;
  };
  auto tile = [&](rsrc_t d, const Off& f) {
    f4 x;
#pragma unroll
    for (int s = 0; s < 4; ++s) x[s] = rload(d, f.o[s]);
    return x;
  };
  const Off oA = nat(n, n, r), oAp = nat(n, n, pr), oB = nat(n, m, r), oBp = nat(n, m, pr), oBt = row(n, m, pr),
            oBd = row(n, m, r), oR = nat(m, m, r), oK = nat(m, n, r), oD = nat(p, n, r), oDp = nat(p, n, pr),
            oE = nat(p, m, r), oEp = nat(p, m, pr);
  const int orn = fresh(q == 0 && r < n ? r * 4 : kOOB);
  auto lnat = [&](const float* l, int j) { return f4{l[q * LD + j], l[(4 + q) * LD + j], l[(8 + q) * LD + j], l[(12 + q) * LD + j]}; };
  auto lrow = [&](const float* l, int i) { return f4{l[i * LD + q], l[i * LD + 4 + q], l[i * LD + 8 + q], l[i * LD + 12 + q]}; };
  auto lvec = [&](const float* l) { return f4{l[q], l[4 + q], l[8 + q], l[12 + q]}; };
  auto prod = [&](const f4& x, const f4& y, f4 acc) {
#pragma unroll
    for (int s = 0; s < 4; ++s) acc = mma(x[s], y[s], acc);
    return acc;
  };

  struct Stage {
    f4 A, Ap, B, Bp, Bt, Bd, Q, R, M, D, Dp, E, Ep, c;
    float cr, qr, rr, rdr;
  };
  // the next stage to load, t = N - 1 first
  struct Ptr {
    const float *A, *B, *Q, *R, *M, *D, *E, *c, *q, *r, *rd;
  } at = {in.A.at(b, N - 1), in.Bm.at(b, N - 1), P.Q.at(b, N - 1), P.R.at(b, N - 1), P.M.at(b, N - 1),
          P.D.at(b, N - 1),  P.E.at(b, N - 1),   ws.cdef + ((size_t)b * N1 + N) * n, ws.qh + ((size_t)b * N1 + N - 1) * n,
          ws.rh + ((size_t)b * N + N - 1) * m, ws.rd + ((size_t)b * N + N - 1) * m};
  auto load = [&](Stage& d) {
    const rsrc_t rA = make_rsrc(at.A, n * n), rB = make_rsrc(at.B, n * m);
    d.A = tile(rA, oA);
    d.Ap = tile(rA, oAp);
    d.B = tile(rB, oB);
    d.Bp = tile(rB, oBp);
    d.Bt = tile(rB, oBt);
    d.Bd = tile(rB, oBd);
    d.Q = tile(make_rsrc(at.Q, n * n), oA);
    d.R = tile(make_rsrc(at.R, m * m), oR);
    d.M = tile(make_rsrc(at.M, cross ? n * m : 0), oBd);   // M'[4 s + q][r]; 0 without one
    if (p > 0) {
      const rsrc_t rD = make_rsrc(at.D, p * n), rE = make_rsrc(at.E, p * m);
      d.D = tile(rD, oD);
      d.Dp = tile(rD, oDp);
      d.E = tile(rE, oE);
      d.Ep = tile(rE, oEp);
    }
    const rsrc_t rc = make_rsrc(at.c, n);
#pragma unroll
    for (int s = 0; s < 4; ++s) d.c[s] = rload(rc, (4 * s + q) * 4);
    d.cr = rload(rc, r * 4);
    d.qr = rload(make_rsrc(at.q, n), r * 4);
    d.rr = rload(make_rsrc(at.r, m), r * 4);
    d.rdr = rload(make_rsrc(at.rd, m), r * 4);
  };
  // where the stage being solved goes, t = N (S, s) and N - 1 first
  struct Out {
    float *S, *s, *F, *f, *K, *k;
  } to = {ws.S + ((size_t)b * N1 + N) * n * n, ws.s + ((size_t)b * N1 + N) * n, ws.F + ((size_t)b * N + N) * n * n,
          ws.f + ((size_t)b * N + N) * n,      ws.K + ((size_t)b * N + N) * m * n, ws.k + ((size_t)b * N + N) * m};
  auto back = [&] {
    at = {at.A - in.A.st, at.B - in.Bm.st, at.Q - P.Q.st, at.R - P.R.st, at.M - P.M.st, at.D - P.D.st,
          at.E - P.E.st,  at.c - n,        at.q - n,      at.r - m,      at.rd - m};
  };
  // S (row-major n x n) and s to the workspace
  auto store_value = [&](float sval) {
    const rsrc_t rS = make_rsrc(to.S, n * n), rs = make_rsrc(to.s, n);
    const f4 S = lnat(sS, r);
#pragma unroll
    for (int s = 0; s < 4; ++s) rstore(rS, oA.o[s], S[s]);
    rstore(rs, orn, sval);
  };

  for (int e = lane; e < 16 * LD; e += 64) sS[e] = sH[e] = sG[e] = sK[e] = 0.f;
  wave_lds_sync();
  float sval = rload(make_rsrc(ws.qh + ((size_t)b * N1 + N) * n, n), r * 4);
  {
    const f4 S = tile(make_rsrc(P.QN.at(b, 0), n * n), oA);
#pragma unroll
    for (int s = 0; s < 4; ++s) sS[(4 * s + q) * LD + r] = S[s];
  }
  wave_lds_sync();
  store_value(sval);

  Stage nx;
  load(nx);
  for (int t = N - 1; t >= 0; --t) {
    Stage d = nx;
    const int ro = fresh(r);   // (comparisons with it are made here, not kept as lane masks)
    if (p > 0) {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        d.D[s] *= sr;
        d.Dp[s] *= sr;
        d.E[s] *= sr;
        d.Ep[s] *= sr;
      }
    }
    if (t > 0) back();   // (the last stage's data is requested once more)
    load(nx);
    __builtin_amdgcn_sched_barrier(0);

    // T = S A, SB = S B, Sc = S c + s
    const f4 Sp = lrow(sS, pr), Sd = lrow(sS, r);
    const f4 T1 = prod(Sp, d.A, zero4()), SB = prod(Sp, d.B, zero4());
    float v = 0.f;
#pragma unroll
    for (int s = 0; s < 4; ++s) v += Sd[s] * d.c[s];
    const float Scr = sval + pair_sum4(v);
    if (q == 0) sv[r] = Scr;
    // H = B'SB + rho_c E'E + (R + diag(rd)), [G | g] = [B'T + rho_c E'D + M' | r + B'Sc]
    f4 H = prod(d.Bp, SB, zero4()), G = prod(d.Bp, T1, zero4());
    if (p > 0) {
      H = prod(d.Ep, d.E, H);
      G = prod(d.Ep, d.D, G);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      float add = d.R[s];
      add += 4 * s + q == ro ? d.rdr : 0.f;
      const float hv = H[s] + add;
      sH[(4 * s + q) * LD + r] = 4 * s + q < m && ro < m ? hv : (4 * s + q == ro ? 1.f : 0.f);
      const float gv = G[s] + d.M[s];
      if (ro < n && 4 * s + q < m) sG[(4 * s + q) * LD + r] = gv;
    }
    wave_lds_sync();
    const f4 Sc = lvec(sv);
    v = 0.f;
#pragma unroll
    for (int s = 0; s < 4; ++s) v += d.B[s] * Sc[s];
    v = pair_sum4(v);
    if (q == 0 && r < m) sG[r * LD + n] = d.rr + v;
    wave_lds_sync();

    // H = L L' (chol_lds), row r of L in lane r; the rows past m are the
    // identity's, which changes no other row
    float h[MM], x[MM];
#pragma unroll
    for (int k = 0; k < MM; ++k) {
      h[k] = sH[r * LD + k];
      x[k] = sG[k * LD + r];   // column r of [G | g]; 0 past row m
    }
    small_for<0, MM>([&](auto J) {
      constexpr int j = decltype(J)::value;
      float h0 = h[j];
#pragma unroll
      for (int k = 0; k < j; ++k) h0 += h[k] * h[k];
      const float dj = row_lane<j>(dev_sqrt(floored_pivot(h[j], h0, prm.hfloor)));
      h[j] = ro == j ? dj : (ro < m ? h[j] / dj : 0.f);
      small_for<j + 1, MM>([&](auto K) { h[K] -= h[j] * row_lane<K>(h[j]); });
    });
    // W = L^{-1} [G | g], [K | k] = L^{-T} W
    small_for<0, MM>([&](auto I) {
      constexpr int i = decltype(I)::value;
      float y = x[i];
      small_for<0, i>([&](auto K) { y -= row_lane<i>(h[K]) * x[K]; });
      x[i] = y / row_lane<i>(h[i]);
    });
    wave_lds_sync();   // every column of G has been read
#pragma unroll
    for (int i = 0; i < MM; ++i) sG[i * LD + r] = x[i];
    small_for<0, MM>([&](auto I) {
      constexpr int i = MM - 1 - decltype(I)::value;
      float y = x[i];
      small_for<i + 1, MM>([&](auto K) { y -= row_lane<K>(h[i]) * x[K]; });
      x[i] = y / row_lane<i>(h[i]);
    });
#pragma unroll
    for (int i = 0; i < MM; ++i) sK[i * LD + r] = x[i];
    wave_lds_sync();

    // S = A'T - W'W + rho_c D'D + Q (the upper triangle, mirrored), s = q + A'Sc - W'w
    const f4 W = lnat(sG, r), Wp = -lnat(sG, pr), wv = lnat(sG, n), kv = lnat(sK, n), K = lnat(sK, r);
    f4 S = prod(Wp, W, prod(d.Ap, T1, zero4()));
    if (p > 0) S = prod(d.Dp, d.D, S);
    const f4 F = prod(-d.Bt, K, zero4());
    v = 0.f;
#pragma unroll
    for (int s = 0; s < 4; ++s) v += d.A[s] * Sc[s];
    // the rows past m of W, w and k are 0
#pragma unroll
    for (int s = 0; s < 4; ++s) v -= W[s] * wv[s];
    sval = r < n ? d.qr + pair_sum4(v) : 0.f;
    float f = 0.f;
#pragma unroll
    for (int s = 0; s < 4; ++s) f -= d.Bd[s] * kv[s];
    f = d.cr + pair_sum4(f);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int i = 4 * s + q;
      if (i <= ro && ro < n) {
        const float y = S[s] + d.Q[s];
        sS[i * LD + r] = y;
        sS[r * LD + i] = y;
      }
    }
    wave_lds_sync();
    to = {to.S - n * n, to.s - n, to.F - n * n, to.f - n, to.K - m * n, to.k - m};
    store_value(sval);
    const rsrc_t rF = make_rsrc(to.F, n * n), rf = make_rsrc(to.f, n);
    const rsrc_t rK = make_rsrc(to.K, m * n), rk = make_rsrc(to.k, m);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      rstore(rF, oA.o[s], F[s] + d.A[s]);
      rstore(rK, oK.o[s], K[s]);
      rstore(rk, r == 0 ? (4 * s + q) * 4 : kOOB, kv[s]);
    }
    rstore(rf, orn, f);
  }

  // dx_{t+1} = F_t dx_t + f_t, row r in lane r (fwd_chain)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // F, f are in memory
  struct Fwd {
    float F[15], f;
  };
  const int ofr = fresh(r < n ? r * n * 4 : kOOB);
  auto loadf = [&](Fwd& d, int t) {
    const rsrc_t rF = make_rsrc(ws.F + ((size_t)b * N + t) * n * n, n * n);
#pragma unroll
    for (int j = 0; j < 15; ++j) d.F[j] = rload(rF, j < n ? ofr + 4 * j : kOOB);
    d.f = rload(make_rsrc(ws.f + ((size_t)b * N + t) * n, n), r * 4);
  };
  float y = rload(make_rsrc(ws.cdef + (size_t)b * N1 * n, n), r * 4);
  Fwd f0, f1;
  loadf(f0, 0);
  loadf(f1, min(1, N - 1));
  for (int t = 0; t < N; ++t) {
    const Fwd d = f0;
    f0 = f1;
    loadf(f1, min(t + 2, N - 1));
    __builtin_amdgcn_sched_barrier(0);
    rstore(make_rsrc(ws.dx + ((size_t)b * N1 + t) * n, n), orn, y);
    float z = d.f;
    small_for<0, 15>([&](auto J) { z += d.F[J] * row_lane<J>(y); });   // entries past n add 0
    y = z;
  }
  rstore(make_rsrc(ws.dx + ((size_t)b * N1 + N) * n, n), orn, y);
}

}  // namespace mpxk
