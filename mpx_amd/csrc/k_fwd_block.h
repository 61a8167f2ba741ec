// Forward pass of the LQR solve, one block of 512 threads per instance:
//   du_t = -(K_t dx_t + k_t),  dx_{t+1} = A_t dx_t + B_t du_t + c_{t+1},
// on the vector ALU.  A group of 16 lanes takes the rows q, q + 32, ... of A
// and B and row q of K (m <= 32), lane l of it the columns l, l + 16, ...; row
// sums are DPP rotations within the group.  dx and du pass between the groups
// through LDS, two barriers per stage; the next stage's matrices are requested
// a stage ahead.  A dx needs no du and is formed before the barrier.
#pragma once
#include "k_lqr_tile.h"

namespace mpxk {

// sum over the 16 lanes of a row, in every lane
template <typename T>
__device__ __forceinline__ T row16_sum(T v) {
  v += dpp_ror<0x128>(v);
  v += dpp_ror<0x124>(v);
  v += dpp_ror<0x122>(v);
  v += dpp_ror<0x121>(v);
  return v;
}

// n <= 16 NC, m <= 16 MC (MC <= 2)
template <typename T, int NC, int MC>
__global__ void __launch_bounds__(512) k_fwd_block(Prob<T> P, Ws<T> ws, LqrIn<T> in) {
  typedef TileOps<T> O;
  constexpr int RR = (NC + 1) / 2, ES = sizeof(T);
  const int b = blockIdx.x;
  if (skip_instance(ws, b)) return;
  const int tid = threadIdx.x, q = tid >> 4, l = tid & 15;
  const int n = P.n, m = P.m, N = P.N, N1 = N + 1;
  __shared__ T sx[2][16 * NC], su[16 * MC];
  struct Stage {
    T A[RR][NC], B[RR][MC], K[NC], c[RR], k;
  };
  const bool bconst = in.Bm.st == 0;
  auto load_b = [&](T (&B)[RR][MC], int t) {
    const rsrc_t rB = tile_rsrc(in.Bm.at(b, t), n * m);
#pragma unroll
    for (int i = 0; i < RR; ++i)
#pragma unroll
      for (int j = 0; j < MC; ++j) B[i][j] = O::bload(rB, l + 16 * j < m ? ((q + 32 * i) * m + l + 16 * j) * ES : kOOB);
  };
  auto load = [&](Stage& s, int t) {
    const rsrc_t rA = tile_rsrc(in.A.at(b, t), n * n);
    const rsrc_t rK = tile_rsrc(ws.K + ((size_t)b * N + t) * m * n, m * n);
    const rsrc_t rc = tile_rsrc(ws.cdef + ((size_t)b * N1 + t + 1) * n, n);
    const rsrc_t rk = tile_rsrc(ws.k + ((size_t)b * N + t) * m, m);
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const bool in_row = l + 16 * j < n;
      s.K[j] = O::bload(rK, in_row ? (q * n + l + 16 * j) * ES : kOOB);
#pragma unroll
      for (int i = 0; i < RR; ++i) s.A[i][j] = O::bload(rA, in_row ? ((q + 32 * i) * n + l + 16 * j) * ES : kOOB);
    }
#pragma unroll
    for (int i = 0; i < RR; ++i) s.c[i] = O::bload(rc, (q + 32 * i) * ES);
    s.k = O::bload(rk, q * ES);
    if (!bconst) load_b(s.B, t);
  };
  Stage s0, s1;
  for (int i = tid; i < 16 * NC; i += 512) {
    sx[0][i] = i < n ? ws.cdef[(size_t)b * N1 * n + i] : T(0);
    sx[1][i] = T(0);
  }
  if (tid < 16 * MC) su[tid] = T(0);
  if (tid < n) ws.dx[(size_t)b * N1 * n + tid] = ws.cdef[(size_t)b * N1 * n + tid];
  load(s0, 0);
  if (bconst) {
    load_b(s0.B, 0);
#pragma unroll
    for (int i = 0; i < RR; ++i)
#pragma unroll
      for (int j = 0; j < MC; ++j) s1.B[i][j] = s0.B[i][j];
  }
  __syncthreads();
  auto step = [&](Stage& cur, Stage& nxt, int t, int buf) {
    load(nxt, t + 1 < N ? t + 1 : t);
    T x[NC];
#pragma unroll
    for (int j = 0; j < NC; ++j) x[j] = sx[buf][l + 16 * j];
    T kx = T(0);
#pragma unroll
    for (int j = 0; j < NC; ++j) kx += cur.K[j] * x[j];
    kx = row16_sum(kx);
    const T u = -(kx + cur.k);
    if (l == 0 && q < m) {
      su[q] = u;
      ws.du[((size_t)b * N + t) * m + q] = u;
    }
    T acc[RR];
#pragma unroll
    for (int i = 0; i < RR; ++i) {
      acc[i] = T(0);
#pragma unroll
      for (int j = 0; j < NC; ++j) acc[i] += cur.A[i][j] * x[j];
    }
    lds_sync();
#pragma unroll
    for (int j = 0; j < MC; ++j) {
      const T uj = su[l + 16 * j];
#pragma unroll
      for (int i = 0; i < RR; ++i) acc[i] += cur.B[i][j] * uj;
    }
#pragma unroll
    for (int i = 0; i < RR; ++i) {
      const T y = row16_sum(acc[i]) + cur.c[i];
      const int r = q + 32 * i;
      if (l == 0 && r < n) {
        sx[buf ^ 1][r] = y;
        ws.dx[((size_t)b * N1 + t + 1) * n + r] = y;
      }
    }
    lds_sync();
  };
  int t = 0;
  for (; t + 1 < N; t += 2) {
    step(s0, s1, t, 0);
    step(s1, s0, t + 1, 1);
  }
  if (t < N) step(s0, s1, t, 0);
}

}  // namespace mpxk
