// The recursion of k_lqr_wave on NT + 1 waves per instance, for batches that
// leave most of the chip's SIMDs without a wave: wave J < NT takes column tile
// J of S~ A~, G~, Pm, W~, K~ and S~ (and row tile J of S~ B~), wave NT the
// factorisation beside them.  The products and their order are those of
// k_lqr_wave, tile by tile, so the results are the same bits whichever of the
// two kernels the batch size selects.
//
// One stage, a barrier after each part:
//   1  SB tiles (waves J)                    -> LDS
//   2  wave NT: H, Z, Z' -> LDS; waves J: S~ A~, G~, Pm of their column
//   3  W~ = Z G~ (waves J)                   -> LDS
//   4  K~, S~ = Pm - W~'W~ of the column, mirrored -> LDS; every wave reads S~
// (a lane's f4 of a tile is one 16-byte entry: every read is the lane's own
// slot, free of conflicts).  Bound by the chain 1 - H - factorisation - 3 - 4.
// 36 x 12 x 50, p = 8, B = 1: 151 us (k_lqr_wave 304); 19 x 7 x 33, stage-varying,
// p = 3, B = 333: 116 (142); 12 x 12 x 25, B = 1: 50 (55).
#pragma once
#include "k_lqr_wave.h"

namespace mpxk {

template <int NT>
struct WavesLds {
  f4 S[NT * NT][64], SB[NT][64], W[NT][64], Z[64], Zt[64];
  float tbuf[NT + 1][16 * 17];
};

// Wave J's data of stage t beyond E and r: columns <= J of A~ (FA: sech^2
// instead, and column n's c), D, q or Q~'s tiles (., J), B~.
template <int NT, int J, bool CQ, bool FA>
__device__ __forceinline__ void waves_load_mats(IlStage<NT>& d, const Prob<float>& P, const Ws<float>& ws,
                                                const LqrIn<float>& in, int b, int t, int g, bool homlane,
                                                const IlOff<NT>& L) {
  const int n = P.n, m = P.m, p = P.p, N = P.N, N1 = N + 1, cn = n & 15;
  const rsrc_t rc = make_rsrc(ws.cdef + ((size_t)b * N1 + t + 1) * n, n);
  if constexpr (FA) {
    const rsrc_t rs = make_rsrc(ws.sdh + ((size_t)b * N + t) * n, n);
#pragma unroll
    for (int i = 0; i < NT; ++i) d.sdr[i] = il_rows(rs, L.g4, i);
    if constexpr (J == NT - 1) {
      if (homlane) {
#pragma unroll
        for (int i = 0; i < NT; ++i) d.A[i][NT - 1] = il_rows(rc, L.g4, i);
      }
    }
  } else {
    const rsrc_t rA = make_rsrc(in.A.at(b, t), n * n);
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int j = 0; j <= J; ++j) {
        f4 x = il_tile_n<NT>(rA, n, i, j, L);
        if (j == NT - 1 && homlane) x = il_rows(rc, L.g4, i);
        d.A[i][j] = x;
      }
  }
  const rsrc_t rD = make_rsrc(P.D.at(b, t), p * n);
#pragma unroll
  for (int j = 0; j <= J; ++j)
#pragma unroll
    for (int v = 0; v < 4; ++v) d.D[j][v] = rload(rD, L.nn[j] + 4 * v * n * 4);
  const rsrc_t rq = make_rsrc(ws.qh + ((size_t)b * N1 + t) * n, n);
  if constexpr (CQ) {
    if constexpr (J == NT - 1) {
#pragma unroll
      for (int i = 0; i < NT; ++i) d.qrow[i] = il_rows(rq, L.hom, i);
      d.qcol[J] = rload(rq, L.pc4 + 64 * J);
    }
  } else {
    const rsrc_t rQ = make_rsrc(P.Q.at(b, t), n * n);
#pragma unroll
    for (int i = 0; i <= J; ++i) {
      f4 x = il_tile_n<NT>(rQ, n, i, J, L);
      if (J == NT - 1 && homlane) x = il_rows(rq, L.g4, i);
      if (i == NT - 1) {
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (4 * v + g == cn) x[v] = rload(rq, L.pc4 + 64 * J);
      }
      d.Q[i][J] = x;
    }
    const rsrc_t rB = make_rsrc(in.Bm.at(b, t), n * m);
#pragma unroll
    for (int i = 0; i < NT; ++i) d.B[i] = il_tile_m<NT>(rB, m, i, L);
  }
}

// E (and r on the wave of column n)
template <int NT, int J>
__device__ __forceinline__ void waves_load_vecs(IlStage<NT>& d, const Prob<float>& P, const Ws<float>& ws, int b,
                                                int t, const IlOff<NT>& L) {
  const int m = P.m, p = P.p, N = P.N;
  const rsrc_t rE = make_rsrc(P.E.at(b, t), p * m);
#pragma unroll
  for (int v = 0; v < 4; ++v) d.E[v] = rload(rE, L.mm + 4 * v * m * 4);
  if constexpr (J == NT - 1) d.rh = il_rows(make_rsrc(ws.rh + ((size_t)b * N + t) * m, m), L.hom, 0);
}

// Wave J < NT: column tile J, every stage.
template <int NT, int J, bool CQ, int KSN, bool FA, bool AS>
__device__ __forceinline__ void waves_column(const Prob<float>& P, const Prm<float>& prm, const Ws<float>& ws,
                                             const LqrIn<float>& in, WavesLds<NT>& lds, const f4* fab, int b) {
  constexpr int KSS = AS ? KSN - 1 : KSN;
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const int n = P.n, m = P.m, p = P.p, N = P.N, N1 = N + 1;
  const float sr = sqrtf(prm.rho_c);
  const int ksm = (m + 3) >> 2, ksp = (p + 3) >> 2;
  const int cn = n & 15, pc = 4 * (c & 3) + (c >> 2);
  const IlOff<NT> L = il_offsets<NT>(n, m, g, c);
  float* tbuf = lds.tbuf[J];

  f4 S[NT][NT];
  il_load_qbar<NT>(S, P.QN.at(b, 0), ws.qh + ((size_t)b * N1 + N) * n, n, false, g, pc == cn, L);
  f4 Qc[J + 1], Bc[NT];
  if constexpr (CQ) {
    const rsrc_t rQ = make_rsrc(P.Q.at(b, 0), n * n), rB = make_rsrc(in.Bm.at(b, 0), n * m);
#pragma unroll
    for (int i = 0; i <= J; ++i) Qc[i] = il_tile_n<NT>(rQ, n, i, J, L);
#pragma unroll
    for (int i = 0; i < NT; ++i) Bc[i] = il_tile_m<NT>(rB, m, i, L);
  }
  IlStage<NT> cur;
  waves_load_vecs<NT, J>(cur, P, ws, b, N - 1, L);
  waves_load_mats<NT, J, CQ, FA>(cur, P, ws, in, b, N - 1, g, pc == cn, L);
  auto store_value = [&](int t, const IlOff<NT>& Lo) {
    const rsrc_t rS = make_rsrc(ws.S + ((size_t)b * N1 + t) * n * n, n * n);
    const rsrc_t rs = make_rsrc(ws.s + ((size_t)b * N1 + t) * n, n);
#pragma unroll
    for (int i = 0; i <= J; ++i) il_store_hom<NT>(S[i][J], rS, rs, n, i, J, Lo);
  };
  if constexpr (!FA) store_value(N, L);
  for (int t = N - 1; t >= 0; --t) {
    const int gf = fresh(g), cf = fresh(c);
    const IlOff<NT> Ls = il_offsets<NT>(n, m, gf, cf);
    const bool homlane = 4 * (cf & 3) + (cf >> 2) == cn;
    f4 rown;
#pragma unroll
    for (int v = 0; v < 4; ++v) rown[v] = 4 * v + gf == cn ? 1.f : 0.f;
    const int tp = __builtin_amdgcn_readfirstlane(t > 0 ? t - 1 : 0);
    f4 Bt[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) Bt[i] = CQ ? Bc[i] : cur.B[i];
    {   // 1: SB tile J
      f4 acc = zero4();
#pragma unroll
      for (int k = 0; k < NT - 1; ++k) acc = mma_k<4>(S[k][J], Bt[k], acc);
      lds.SB[J][lane] = mma_k<KSS>(S[NT - 1][J], Bt[NT - 1], acc);
    }
    lds_sync();
    // 2: G~ and Pm of the column
    f4 G = J == NT - 1 ? cur.rh : zero4();
    if (p > 0) {
#pragma unroll
      for (int v = 0; v < 4; ++v) cur.E[v] *= sr;
#pragma unroll
      for (int j = 0; j <= J; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) cur.D[j][v] *= sr;
      with_steps<1, 4>(ksp, [&](auto KP) { G = mma_k<decltype(KP)::value>(cur.E, cur.D[J], G); });
    }
    waves_load_vecs<NT, J>(cur, P, ws, b, tp, Ls);
    if constexpr (FA) {   // A~ = I + h A + diag(sd) h kappa W, column n = c on its lanes
#pragma unroll
      for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j <= J; ++j) {
          const f4 a = fab[(i * NT + j) * 64 + lane], w = fab[(NT * NT + i * NT + j) * 64 + lane];
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const float x = fmaf(cur.sdr[i][v], w[v], a[v]);
            cur.A[i][j][v] = (j == NT - 1 && homlane) ? cur.A[i][j][v] : x;
          }
        }
    }
    if constexpr (!AS && J == NT - 1) {
#pragma unroll
      for (int v = 0; v < 4; ++v) cur.A[NT - 1][NT - 1][v] += homlane ? rown[v] : 0.f;
    }
    f4 Pm[J + 1];
    {
      f4 SAc[NT];
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        f4 acc = zero4();
#pragma unroll
        for (int k = 0; k < NT - 1; ++k) acc = mma_k<4>(S[k][i], cur.A[k][J], acc);
        SAc[i] = mma_k<KSS>(S[NT - 1][i], cur.A[NT - 1][J], acc);
        if constexpr (AS && J == NT - 1) {
          const float hm = homlane ? 1.f : 0.f;
#pragma unroll
          for (int v = 0; v < 4; ++v) SAc[i][v] = fmaf(hm, S[i][NT - 1][v], SAc[i][v]);
        }
      }
#pragma unroll
      for (int k = 0; k < NT - 1; ++k) G = mma_k<4>(Bt[k], SAc[k], G);
      G = mma_k<KSS>(Bt[NT - 1], SAc[NT - 1], G);
#pragma unroll
      for (int i = 0; i <= J; ++i) {
        f4 acc;
        if constexpr (CQ) {
          acc = Qc[i];
          if (J == NT - 1) {
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[v] += cur.qrow[i][v];
          }
          if (i == NT - 1) {
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[v] = fmaf(rown[v], cur.qcol[J], acc[v]);
          }
        } else {
          acc = cur.Q[i][J];
        }
        if (p > 0) acc = mma_ks(cur.D[i], cur.D[J], acc, ksp);
#pragma unroll
        for (int k = 0; k < NT - 1; ++k) acc = mma_k<4>(cur.A[k][i], SAc[k], acc);
        acc = mma_k<KSS>(cur.A[NT - 1][i], SAc[NT - 1], acc);
        if constexpr (AS) {
          if (i == NT - 1) {
            constexpr int v = KSN - 1;
            acc[v] = fmaf(rown[v], SAc[NT - 1][v], acc[v]);
          }
        }
        Pm[i] = acc;
      }
    }
    waves_load_mats<NT, J, CQ, FA>(cur, P, ws, in, b, tp, gf, homlane, Ls);
    lds_sync();
    // 3, 4: W~, K~ and S~
    const f4 Zt = lds.Zt[lane], Z = lds.Z[lane];
    f4 K;
    with_steps<1, 4>(ksm, [&](auto KM) {
      constexpr int km = decltype(KM)::value;
      const f4 w = mma_k<km>(Zt, G, zero4());
      lds.W[J][lane] = w;
      K = mma_k<km>(Z, w, zero4());
      lds_sync();
#pragma unroll
      for (int i = 0; i <= J; ++i) {
        f4 Wn = i == J ? w : lds.W[i][lane];
#pragma unroll
        for (int v = 0; v < 4; ++v) Wn[v] = -Wn[v];
        S[i][J] = mma_k<km>(Wn, w, Pm[i]);
      }
    });
    {
      const f4 d = tile_transpose(S[J][J], tbuf, g, c);
#pragma unroll
      for (int v = 0; v < 4; ++v) S[J][J][v] = 0.5f * (S[J][J][v] + d[v]);
    }
#pragma unroll
    for (int i = 0; i < J; ++i) {
      S[J][i] = tile_transpose(S[i][J], tbuf, g, c);
      lds.S[J * NT + i][lane] = S[J][i];
      lds.S[i * NT + J][lane] = S[i][J];
    }
    if constexpr (J == NT - 1) {
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (homlane && 4 * v + gf == cn) S[NT - 1][NT - 1][v] = 0.f;
    }
    lds.S[J * NT + J][lane] = S[J][J];
    lds_sync();
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
        if ((i > J || j > J) || (i < J && j < J)) S[i][j] = lds.S[i * NT + j][lane];
    if constexpr (!FA) store_value(t, Ls);
    {
      const rsrc_t rK = make_rsrc(ws.K + ((size_t)b * N + t) * m * n, m * n);
      const rsrc_t rk = make_rsrc(ws.k + ((size_t)b * N + t) * m, m);
      il_store_hom<NT>(K, rK, rk, n, 0, J, Ls);
    }
  }
}

// Wave NT: H and its factorisation, every stage.
template <int NT, bool CQ, int KSS>
__device__ __forceinline__ void waves_factor(const Prob<float>& P, const Prm<float>& prm, const Ws<float>& ws,
                                             const LqrIn<float>& in, WavesLds<NT>& lds, int b) {
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const int n = P.n, m = P.m, p = P.p, N = P.N;
  const float sr = sqrtf(prm.rho_c);
  const int ksm = (m + 3) >> 2, ksp = (p + 3) >> 2;
  const IlOff<NT> L = il_offsets<NT>(n, m, g, c);
  f4 dmask, Rc, Bt[NT], E, rdv;
#pragma unroll
  for (int v = 0; v < 4; ++v) dmask[v] = 4 * g + v == c ? 1.f : 0.f;
  auto load = [&](int t) {
    const rsrc_t rE = make_rsrc(P.E.at(b, t), p * m);
#pragma unroll
    for (int v = 0; v < 4; ++v) E[v] = rload(rE, L.mm + 4 * v * m * 4);
    rdv = il_rows(make_rsrc(ws.rd + ((size_t)b * N + t) * m, m), L.g4, 0);
    if constexpr (!CQ) {
      Rc = il_tile_m<NT>(make_rsrc(P.R.at(b, t), m * m), m, 0, L);
      const rsrc_t rB = make_rsrc(in.Bm.at(b, t), n * m);
#pragma unroll
      for (int i = 0; i < NT; ++i) Bt[i] = il_tile_m<NT>(rB, m, i, L);
    }
  };
  if constexpr (CQ) {
    const rsrc_t rB = make_rsrc(in.Bm.at(b, 0), n * m);
#pragma unroll
    for (int i = 0; i < NT; ++i) Bt[i] = il_tile_m<NT>(rB, m, i, L);
    Rc = il_tile_m<NT>(make_rsrc(P.R.at(b, 0), m * m), m, 0, L);
#pragma unroll
    for (int v = 0; v < 4; ++v) Rc[v] += (4 * g + v == c && 4 * v + g >= m) ? 1.f : 0.f;
  }
  load(N - 1);
  for (int t = N - 1; t >= 0; --t) {
    const int tp = __builtin_amdgcn_readfirstlane(t > 0 ? t - 1 : 0);
    lds_sync();
    f4 H;
#pragma unroll
    for (int v = 0; v < 4; ++v)
      H[v] = fmaf(dmask[v], rdv[v], CQ ? Rc[v] : Rc[v] + (dmask[v] != 0.f && 4 * v + g >= m ? 1.f : 0.f));
#pragma unroll
    for (int k = 0; k < NT - 1; ++k) H = mma_k<4>(Bt[k], lds.SB[k][lane], H);
    H = mma_k<KSS>(Bt[NT - 1], lds.SB[NT - 1][lane], H);
    if (p > 0) {
#pragma unroll
      for (int v = 0; v < 4; ++v) E[v] *= sr;
      with_steps<1, 4>(ksp, [&](auto KP) { H = mma_k<decltype(KP)::value>(E, E, H); });
    }
    load(tp);
    f4 Z;
#pragma unroll
    for (int v = 0; v < 4; ++v) Z[v] = dmask[v];
    with_steps<1, 4>(ksm, [&](auto KM) { chol_lower_inv<decltype(KM)::value>(H, Z, prm.hfloor); });
    lds.Z[lane] = Z;
    lds.Zt[lane] = tile_transpose(Z, lds.tbuf[NT], g, c);
    lds_sync();
    lds_sync();
    lds_sync();
  }
}

// Parameters and limits as for k_lqr_wave.
template <int NT, bool CQ, int KSN, bool FA, bool AS>
__global__ void __launch_bounds__(64 * (NT + 1)) k_lqr_waves(Prob<float> P, Prm<float> prm, Ws<float> ws,
                                                            LqrIn<float> in) {
  static_assert(!FA || CQ, "A~ is formed from stage-invariant A, W only with stage-invariant Q, B, R");
  static_assert(!AS || CQ, "the homogeneous step is split off only with the step count of n");
  __shared__ WavesLds<NT> lds;
  __shared__ f4 fab[FA ? 2 * NT * NT * 64 : 1];   // as in k_lqr_wave, read by every column wave
  const int b = blockIdx.x, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (skip_instance(ws, b)) return;
  if constexpr (FA) {
    const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15, pc = 4 * (c & 3) + (c >> 2), n = P.n;
    const IlOff<NT> L = il_offsets<NT>(n, P.m, g, c);
    const rsrc_t rA = make_rsrc(P.A.at(b, 0), n * n), rW = make_rsrc(P.W.at(b, 0), n * n);
    const float hs = P.h, hk = P.h * P.kappa;
    if (wv < NT) {
#pragma unroll
      for (int j = 0; j < NT; ++j) {   // row tile wv
        f4 a, w;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          a[v] = rload(rA, L.nn[j] + (16 * wv + 4 * v) * n * 4);
          w[v] = rload(rW, L.nn[j] + (16 * wv + 4 * v) * n * 4);
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = 16 * wv + 4 * v + g, col = 16 * j + pc;
          a[v] = (row == col && row < n ? 1.f : 0.f) + hs * a[v];
          w[v] = hk * w[v];
        }
        fab[(wv * NT + j) * 64 + lane] = a;
        fab[(NT * NT + wv * NT + j) * 64 + lane] = w;
      }
    }
  }
  lds_sync();
  constexpr int KSS = AS ? KSN - 1 : KSN;
  if (wv == NT) return waves_factor<NT, CQ, KSS>(P, prm, ws, in, lds, b);
  if (wv == 0) return waves_column<NT, 0, CQ, KSN, FA, AS>(P, prm, ws, in, lds, fab, b);
  if constexpr (NT >= 2) {
    if (wv == 1) return waves_column<NT, 1, CQ, KSN, FA, AS>(P, prm, ws, in, lds, fab, b);
  }
  if constexpr (NT == 3) waves_column<NT, 2, CQ, KSN, FA, AS>(P, prm, ws, in, lds, fab, b);
}

}  // namespace mpxk
