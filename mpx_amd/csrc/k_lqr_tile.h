// Backward Riccati recursion of one instance per block, every product on the
// matrix cores from operand tiles in LDS (FP32 v_mfma_f32_16x16x4f32, FP64
// v_mfma_f64_16x16x4f64).
//
// Same recursion, in the homogeneous form of k_lqr_wave.h (x~ = [x; 1]):
//   T = S~ A~, SB = S~ B~,  H = R + diag(rd) + rho_c E'E + B~' SB,
//   G~ = [M' | r] + rho_c E'[D | 0] + B~' T,  W~ = Z G~, K~ = Z' W~ (Z = L^{-1}),
//   S~ <- Q~ + rho_c [D|0]'[D|0] + A~' T - W~' W~.
//
// Layout.  LDS holds every matrix as the rows a matrix instruction's operand
// reads along: S, A~', B~', T', SB', G', W', Z, Z', D', E', one row per
// non-contracted index, the contracted index contiguous.  Lane (g, c) (g =
// lane / 16, c = lane % 16) reads positions 4 g .. 4 g + 3 of a 16-wide k tile
// of row c as one 128-bit load (FP64: two), which feeds the four matrix
// instructions of that k tile, and a result tile (lane (g, c): four rows of
// column c) is stored the same way.  Rows are padded by 16 bytes so that the
// 16 rows a load touches start in different banks.
// Positions.  Entry x of a dimension sits at position 16 (x / 16) + pi(x % 16),
// pi(4 a + b) = 4 b + a (the order of k_lqr_wave's tiles, which the
// factorisation's steps take): the four positions of lane group g are the
// entries g, 4 + g, 8 + g, 12 + g.
//
// Rounding.  The products with A~ are formed with Delta = A~ - diag(e), e_j = 1
// where A_jj lies in [1/2, 2] (the difference is then exact) and for the
// homogeneous index, else 0: T = S~ diag(e) + S~ Delta, A~'T = diag(e) T +
// Delta' T.  A discretised model's Delta is small, so the sums' roundings are
// too (at n = 76, m = 32, p = 12 the error of dX falls to 0.4 of the direct
// products', that of dU to 0.7), and row n of Delta is 0: the sums over the
// state have n terms.  Sums start from zero and take their addend (Q~, R, [M' | r], P) last: started
// from the addend, every matrix instruction rounds at its size, which doubled
// the error of U and V at n = 76, m = 32.
//
// One stage, a barrier after each phase (global stores are not waited for):
//   A  SB, and as many tiles of T as fill the round
//   B  (m > 16) the tiles of H by three waves, tiles of T by the others
//   C  the first wave: (m <= 16: H,) the first half of the factorisation in its
//      registers; the others: the rest of T
//   D  the first wave: the second half, Z; the others: G~ and
//      Q~ + rho_c D'D + A~'T, the latter kept in the registers of their owners
//   E  W~; the next stage's data from registers to LDS
//   F  S~ and K~
// so that the factorisation's serial steps run beside the large products.  In
// each phase a wave forms all its tiles before it stores the first: a store to
// LDS would hold back the loads of the next tile.  The next stage's data is
// requested at the start of a stage, a 4 x 4 block per thread as four 128-bit
// loads of rows (dword aligned) that land as four columns.
//
// What bounds it (76 x 32, one block per CU, clocks of one stage): 1450 matrix
// instructions of 32 cycles on four SIMDs are 11.6 k cycles, the other vector
// instructions beside them 4 to 5 k (they do not overlap), and a stage takes
// 27.5 k: the rest is the start of each phase (LDS latency, addresses) and
// uneven tile counts.  k_lqr_seq takes 161 k on the same stage.  Fewer
// instructions per access (scalar row steps, addresses formed once) brought 32 k
// to 27.5 k; 16 waves per block spill (34 k and more); T and SB in one phase and
// the whole factorisation beside G~ and P took 34 k.
#pragma once
#include "k_lqr_wave.h"

namespace mpxk {

typedef double mpxk_f64x4 __attribute__((ext_vector_type(4)));
typedef double mpxk_f64x2 __attribute__((ext_vector_type(2)));

template <typename T>
struct TileOps;
template <>
struct TileOps<float> {
  typedef f4 V4;
  static constexpr int PAD = 4;
  // entry offset, within its 16, of the row in register v of a result tile,
  // and (pos) the position it sits at
  static constexpr int RG = 1, RV = 4;   // row(g, v) = RG g + RV v
  static __device__ __forceinline__ V4 mma(float a, float b, V4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ V4 load(const float* p) { return *reinterpret_cast<const f4*>(p); }
  static __device__ __forceinline__ void store4(float* p, const V4& x) { *reinterpret_cast<f4*>(p) = x; }
  // a result tile's column c: the rows of lane group g
  static __device__ __forceinline__ void store_col(float* p, int g, const V4& x) {
    *reinterpret_cast<f4*>(p + 4 * g) = x;
  }
  static __device__ __forceinline__ V4 load_col(const float* p, int g) { return *reinterpret_cast<const f4*>(p + 4 * g); }
  static __device__ __forceinline__ int pos(int g, int v) { return 4 * g + v; }
  // entry at byte off + soff (soff uniform: the scalar offset of the access)
  static __device__ __forceinline__ float bload(rsrc_t r, int off, int soff = 0) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, soff, 0));
  }
  // four consecutive entries (dword aligned)
  static __device__ __forceinline__ V4 bload4(rsrc_t r, int off, int soff) {
    return __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(r, off, soff, 0));
  }
  static __device__ __forceinline__ void bstore(rsrc_t r, int off, int soff, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned int, v), r, off, soff, 0);
  }
};

// (FP64: a result tile's register v of lane group g is row 4 v + g, not 4 g + v)
template <>
struct TileOps<double> {
  typedef mpxk_f64x4 V4;
  typedef unsigned int u2 __attribute__((ext_vector_type(2)));
  static constexpr int PAD = 2;
  static constexpr int RG = 4, RV = 1;
  static __device__ __forceinline__ V4 mma(double a, double b, V4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ V4 load(const double* p) {
    const mpxk_f64x2 a = reinterpret_cast<const mpxk_f64x2*>(p)[0], b = reinterpret_cast<const mpxk_f64x2*>(p)[1];
    return V4{a[0], a[1], b[0], b[1]};
  }
  static __device__ __forceinline__ void store4(double* p, const V4& x) {
    reinterpret_cast<mpxk_f64x2*>(p)[0] = mpxk_f64x2{x[0], x[1]};
    reinterpret_cast<mpxk_f64x2*>(p)[1] = mpxk_f64x2{x[2], x[3]};
  }
  static __device__ __forceinline__ void store_col(double* p, int g, const V4& x) {
#pragma unroll
    for (int v = 0; v < 4; ++v) p[4 * v + g] = x[v];
  }
  static __device__ __forceinline__ V4 load_col(const double* p, int g) {
    return V4{p[g], p[4 + g], p[8 + g], p[12 + g]};
  }
  static __device__ __forceinline__ int pos(int g, int v) { return 4 * v + g; }
  static __device__ __forceinline__ double bload(rsrc_t r, int off, int soff = 0) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off, soff, 0));
  }
  static __device__ __forceinline__ V4 bload4(rsrc_t r, int off, int soff) {
    const mpxk_f64x2 a = __builtin_bit_cast(mpxk_f64x2, __builtin_amdgcn_raw_buffer_load_b128(r, off, soff, 0));
    const mpxk_f64x2 b = __builtin_bit_cast(mpxk_f64x2, __builtin_amdgcn_raw_buffer_load_b128(r, off + 16, soff, 0));
    return V4{a[0], a[1], b[0], b[1]};
  }
  static __device__ __forceinline__ void bstore(rsrc_t r, int off, int soff, double v) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, v), r, off, soff, 0);
  }
};

template <typename T>
__device__ __forceinline__ rsrc_t tile_rsrc(const T* p, int nelem) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(p), (short)0, nelem * (int)sizeof(T), 0x00020000);
}

// position of entry x, and entry at position x (its own inverse)
__device__ __host__ __forceinline__ int tile_pos(int x) { return (x & ~15) | (4 * (x & 3) + ((x >> 2) & 3)); }

// LDS plan in elements.
template <typename T, int NT, int MT>
struct TileLds {
  static constexpr int LD = 16 * NT + TileOps<T>::PAD, LM = 16 * MT + TileOps<T>::PAD, LP = 16 + TileOps<T>::PAD;
  static constexpr int S = 0;
  static constexpr int AT = S + 16 * NT * LD;
  static constexpr int TT = AT + 16 * NT * LD;
  static constexpr int BT = TT + 16 * NT * LD;
  static constexpr int SBT = BT + 16 * MT * LD;
  static constexpr int GT = SBT + 16 * MT * LD;
  static constexpr int WT = GT + 16 * NT * LM;
  static constexpr int Z = WT + 16 * NT * LM;
  static constexpr int ZT = Z + 16 * MT * LM;
  static constexpr int DT = ZT + 16 * MT * LM;
  static constexpr int ET = DT + 16 * NT * LP;
  static constexpr int RV = ET + 16 * MT * LP;   // r and rd by position
  static constexpr int RD = RV + 16 * MT;
  static constexpr int QV = RD + 16 * MT;        // q by position
  static constexpr int EV = QV + 16 * NT;        // the unit diagonal taken out of A~ (0 or 1) by position
  static constexpr int NONE = EV + 16 * NT;      // what a block has past its matrix lands here, never read
  static constexpr int SKEW = NONE + 64;         // whether Q_N is not symmetric
  static constexpr int TOTAL = SKEW + 4;
};

// a b over KT k tiles; the even and the odd ones in two chains (half the
// roundings at the sum's size, and two chains in flight).  Padding entries are
// 0, so every tile takes all its steps (no branches).
template <typename T, int KT>
__device__ __forceinline__ typename TileOps<T>::V4 tile_dot(const T* a, const T* b) {
  typedef TileOps<T> O;
  constexpr int GR = sizeof(T) == 8 ? 2 : KT;   // k tiles whose operands are in registers at once
  typename O::V4 x[KT], y[KT], acc[2];
#pragma unroll
  for (int v = 0; v < 4; ++v) acc[0][v] = acc[1][v] = T(0);
#pragma unroll
  for (int k0 = 0; k0 < KT; k0 += GR) {
#pragma unroll
    for (int k = k0; k < KT && k < k0 + GR; ++k) {
      x[k] = O::load(a + 16 * k);
      y[k] = O::load(b + 16 * k);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
#pragma unroll
      for (int k = k0; k < KT && k < k0 + GR; ++k) acc[k & 1] = O::mma(x[k][s], y[k][s], acc[k & 1]);
    }
    if (GR < KT) __builtin_amdgcn_sched_barrier(0);
  }
  return KT > 1 ? acc[0] + acc[1] : acc[0];
}

// tile (i, j), i <= j, number u < 21 of the upper triangle, column by column, as
// i + 16 j
__device__ __forceinline__ int tile_upper(int u) {
  const int j = (u >= 1) + (u >= 3) + (u >= 6) + (u >= 10) + (u >= 15);
  return u - j * (j + 1) / 2 + 16 * j;
}

enum { TILE_A = 0, TILE_CALLER = 1 };

// FP32: Z = L^{-1} of the floored Cholesky factor of H (16 MT square, identity
// past m), in two halves, from its upper tiles in the registers of one wave, to
// LDS as rows of Z and of Z'.  MT = 1: eight pivots each.  MT = 2 by blocks:
// H00 = L00 L00', V = Z00 H01 (= L10'), then L11 L11' = H11 - V'V and
// Z10 = -Z11 (V' Z00).  The pivot floors are those of H's own diagonal.
template <typename T, int MT>
struct TileFactor;

template <int MT>
struct TileFactor<float, MT> {
  static constexpr int LM = 16 * MT + 4;
  f4 h, z, d, u;   // the block under factorisation, its Z, its own H, -V' Z00
  template <int J0, int J1, int KM>
  __device__ __forceinline__ void steps(float floor) {
    static_for<J0, J1>([&](auto JJ) {
      constexpr int J = decltype(JJ)::value;
      chol_step<J, KM>(h, z, floor * fabsf(rlane(d[J >> 2], 16 * (J & 3) + 4 * (J & 3) + (J >> 2))));
    });
  }
  __device__ __forceinline__ void start(const f4& block, int g, int c) {
    h = block;
#pragma unroll
    for (int v = 0; v < 4; ++v) z[v] = 4 * g + v == c ? 1.f : 0.f;
  }
  // Z's tile (i, j): rows 16 i + 4 g + v, column 16 j + c, and its transpose
  static __device__ __forceinline__ void put(const f4& x, int i, int j, float* zr, float* zt, int g, int c) {
#pragma unroll
    for (int v = 0; v < 4; ++v) zr[(16 * i + 4 * g + v) * LM + 16 * j + c] = x[v];
    *reinterpret_cast<f4*>(zt + (16 * j + c) * LM + 16 * i + 4 * g) = x;
  }
  // an A operand: the transpose of diagonal tile i of Z, by rows of Z'
  static __device__ __forceinline__ f4 transposed(int i, const float* zt, int g, int c) {
    wave_lds_sync();
    f4 x;
#pragma unroll
    for (int v = 0; v < 4; ++v) x[v] = zt[(16 * i + 4 * g + v) * LM + 16 * i + c];
    return x;
  }
  __device__ __forceinline__ void first(const f4 (&H)[MT][MT], float* zr, float* zt, int ksm, float floor, int g, int c) {
    d = H[0][0];
    start(H[0][0], g, c);
    if constexpr (MT == 1) {
      with_steps<1, 4>(ksm, [&](auto KM) {
        constexpr int km = decltype(KM)::value;
        steps<0, (km < 2 ? 4 * km : 8), km>(floor);
      });
    } else {
      steps<0, 16, 4>(floor);
      put(z, 0, 0, zr, zt, g, c);
      const f4 v01 = mma_k<4>(transposed(0, zt, g, c), H[0][1], zero4());
      f4 nv;
#pragma unroll
      for (int v = 0; v < 4; ++v) nv[v] = -v01[v];
      u = mma_k<4>(nv, z, zero4());
      d = H[1][1];
      const f4 s = mma_k<4>(nv, v01, zero4());
      start(d + s, g, c);
    }
  }
  __device__ __forceinline__ void second(float* zr, float* zt, int ksm, float floor, int g, int c) {
    with_steps<1, 4>(ksm, [&](auto KM) {
      constexpr int km = decltype(KM)::value;
      if constexpr (MT == 2) steps<0, 4 * km, km>(floor);
      else if constexpr (km > 2) steps<8, 4 * km, km>(floor);
    });
    put(z, MT - 1, MT - 1, zr, zt, g, c);
    if constexpr (MT == 2) put(mma_k<4>(transposed(1, zt, g, c), u, zero4()), 1, 0, zr, zt, g, c);
  }
};

// FP64, m <= 16: lane k holds column k of H (identity past m) and of Z; pivot j
// forms row j of L', divides by it and takes L[i][j] from lane i by readlane for
// the trailing column and the forward substitution.
template <>
struct TileFactor<double, 1> {
  static constexpr int LM = 18;
  double h[16], z[16], hkk;
  template <int J0, int J1>
  __device__ __forceinline__ void steps(double floor, int k) {
    static_for<J0, J1>([&](auto JJ) {
      constexpr int J = decltype(JJ)::value;
      const double d = dev_sqrt(floored_pivot(rlane(h[J], J), rlane(hkk, J), floor)), id = 1.0 / d;
      const double lk = k > J ? h[J] * id : 0.0, zj = z[J] * id;
      z[J] = zj;
      static_for<J + 1, 16>([&](auto II) {
        constexpr int i = decltype(II)::value;
        const double lij = rlane(lk, i);
        h[i] -= lij * lk;
        z[i] -= lij * zj;
      });
    });
  }
  __device__ __forceinline__ void first(const mpxk_f64x4 (&H)[1][1], double* zr, double* zt, int ksm, double floor, int g,
                                        int c) {
    // through Z's place: rows and columns by position, column k = entry k
#pragma unroll
    for (int v = 0; v < 4; ++v) zr[(4 * v + g) * LM + c] = H[0][0][v];
    wave_lds_sync();
    const int k = 16 * g + c, kp = tile_pos(c);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      h[i] = zr[tile_pos(i) * LM + kp];
      z[i] = k == i ? 1.0 : 0.0;
      hkk = c == i ? h[i] : hkk;
    }
    wave_lds_sync();
    steps<0, 8>(floor, k);
  }
  __device__ __forceinline__ void second(double* zr, double* zt, int ksm, double floor, int g, int c) {
    const int k = 16 * g + c, kp = tile_pos(c);
    if (ksm > 2) steps<8, 16>(floor, k);
    if (g == 0) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        zr[tile_pos(i) * LM + kp] = z[i];
        zt[kp * LM + tile_pos(i)] = z[i];
      }
    }
  }
};

// n + 1 <= 16 NT (NT minimal), 16 (MT - 1) < m <= 16 MT, p <= 16.  Stores K~_t,
// the upper tiles of S_t (Q_N whole) and s_t (k_costate_one).  MODE TILE_CALLER
// adds the caller's cross Hessian M_t (may be null).
// FP64: m <= 16, n + 1 <= 64, both triangles of S_t.
//
// A Q_N that is not symmetric to the bit (a caller's J'WJ) is read by its rows, as
// k_lqr_seq reads it, which makes stage N - 1 a special one: the columns of S~
// diag(e) cannot be taken from its rows, so e_j = 0 where column and row j of Q_N
// differ, and one triangle counts, as there: of H the lower (m <= 16) or the
// upper one, of P the upper (corrections formed before the loop).
template <typename T, int NT, int MT, int NW, int MODE>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2)))
k_lqr_tile(Prob<T> P, Prm<T> prm, Ws<T> ws, LqrIn<T> in) {
  typedef TileOps<T> O;
  typedef typename O::V4 V4;
  typedef TileLds<T, NT, MT> X;
  constexpr int LD = X::LD, LM = X::LM, LP = X::LP, NTH = 64 * NW, ES = sizeof(T);
  constexpr int NPM = NT * (NT + 1) / 2, NG = MT * NT, NWK = NW - 1;   // waves 1.. own Pm and G tiles
  constexpr int PSL = (NPM + NWK - 1) / NWK, GSL = (NG + NWK - 1) / NWK;
  constexpr int NB = NT * MT, NTT = NT * NT;                    // tiles of SB and of T
  constexpr int RA = (NB + NW - 1) / NW, T_B = RA * NW - NB;    // rounds of phase A; T's tiles from T_B on come later
  constexpr int T_C = MT == 2 ? T_B + NW - 3 : T_B;             // ... from T_C on in phase C
  constexpr int RC = T_C < NTT ? (NTT - T_C + NWK - 1) / NWK : 0;
  constexpr int RG = (NG + NW - 1) / NW;
  static_assert(16 * NT * NT <= NTH, "a 4 x 4 block per thread");
  const int b = blockIdx.x;
  if (skip_instance(ws, b)) return;
  const int tid = threadIdx.x;
  int g = (tid & 63) >> 4, c = tid & 15;
  int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = P.n, m = P.m, p = P.p, N = P.N, N1 = N + 1;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T* sm = reinterpret_cast<T*>(smem_raw);
  const int ksm = (m - 16 * (MT - 1) + 3) >> 2;   // fours of pivots in the last control tile
  int pc = 4 * (c & 3) + (c >> 2);   // the entry at position c
  const int pn = tile_pos(n);        // the position of the homogeneous index
  const T sr = dev_sqrt(prm.rho_c), hfloor = prm.hfloor;
  const T T0 = T(0);
  // this instance's arrays (stage strides in elements): held in scalar
  // registers for the whole recursion instead of the problem's views
  const T *pA = in.A.at(b, 0), *pB = in.Bm.at(b, 0), *pQ = P.Q.at(b, 0), *pR = P.R.at(b, 0);
  const T *pD = P.D.at(b, 0), *pE = P.E.at(b, 0), *pM = MODE == TILE_CALLER ? P.M.at(b, 0) : nullptr;
  const bool has_m = MODE == TILE_CALLER && P.M.p != nullptr;
  const long long sA = in.A.st, sB = in.Bm.st, sQ = P.Q.st, sR = P.R.st, sD = P.D.st, sE = P.E.st, sM = P.M.st;
  const T *pc_ = ws.cdef + ((size_t)b * N1 + 1) * n, *pq = ws.qh + (size_t)b * N1 * n;
  const T *pr = ws.rh + (size_t)b * N * m, *prd = ws.rd + (size_t)b * N * m;
  T *pK = ws.K + (size_t)b * N * m * n, *pk = ws.k + (size_t)b * N * m;
  T *pS = ws.S + (size_t)b * N1 * n * n, *ps = ws.s + (size_t)b * N1 * n;

  // ---- this thread's share of a stage's data: 4 x 4 blocks (rows g, 4 + g,
  // 8 + g, 12 + g of a k tile, four columns), a 128-bit LDS store per column.
  // The lanes of a 16 take the 4 x 4 blocks of a tile (64 bytes of each row;
  // the columns' stores mostly in different banks).  B~, D and E (in one k tile
  // each) are the last waves' besides, each wave has one of them at most.
  const bool bconst = in.Bm.st == 0;
  const int na = (n + 15) >> 4, mb = (m + 15) >> 4;   // column tiles
  constexpr int WB = (NT * MT + 3) / 4, WD = (NT + 3) / 4;
  static_assert(WB + WD + 1 <= NW, "a wave for each small array");
  const int role = w >= NW - WB ? 0 : w >= NW - WB - WD ? 1 : w == NW - WB - WD - 1 ? 2 : 3;   // B~, D, E, none
  struct Block {
    int off, lds[4];   // byte offset (kOOB: none), its columns' quads
  };
  auto block_of = [&](int e, int rows, int cols, int ld, int base, int stride) {
    Block k;
    const int kt = (e >> 4) / cols, ct = (e >> 4) - kt * cols, cb = e & 3, kq = (e >> 2) & 3, col = 16 * ct + 4 * cb;
    k.off = e >= 0 && kt < rows && col < ld ? ((16 * kt + kq) * ld + col) * ES : kOOB;
#pragma unroll
    for (int j = 0; j < 4; ++j)   // column 4 cb + j: position + 4 j
      k.lds[j] = k.off != kOOB && col + j < ld ? base + (16 * ct + cb + 4 * j) * stride + 16 * kt + 4 * kq
                                               : X::NONE + 4 * (tid & 15);
    return k;
  };
  const Block ka = block_of(tid, NT, na, n, X::AT, LD);
  const int ts = tid - 64 * (role == 0 ? NW - WB : role == 1 ? NW - WB - WD : NW - WB - WD - 1);
  const Block kb = role == 0 ? block_of(ts, NT, mb, m, X::BT, LD)
                 : role == 1 ? block_of(ts, 1, na, n, X::DT, LP)
                             : block_of(role == 2 ? ts : -1, 1, mb, m, X::ET, LP);
  V4 ra[4], rb[4], rcv;
  T rvr, rvd, rvq, rdg;
  // (absent entries past the descriptor: branches around loads would make the
  // later waits, which count requests, wait for more than they need)
  const int cvo = tid < 4 * NT ? (16 * (tid >> 2) + (tid & 3)) * ES : kOOB;
  const int rvo = tid < 16 * MT ? tile_pos(tid) * ES : kOOB, qvo = tid < 16 * NT ? tile_pos(tid) * ES : kOOB;
  const int dgo = tid < n ? tid * (n + 1) * ES : kOOB;
  auto block_load = [&](V4 (&x)[4], rsrc_t r, int off, int ld) {
#pragma unroll
    for (int s = 0; s < 4; ++s) x[s] = O::bload4(r, off, 4 * s * ld * ES);
  };
  auto block_store = [&](const V4 (&x)[4], const Block& k) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const V4 y = {x[0][j], x[1][j], x[2][j], x[3][j]};
      O::store4(sm + k.lds[j], y);
    }
  };
  auto load_data = [&](int t) {
    // first what not every call has: the waits count the requests after it
    if (role == 0 ? !bconst : role < 3 && p > 0) {
      const T* q = role == 0 ? pB + t * sB : role == 1 ? pD + t * sD : pE + t * sE;
      const int cols = role == 1 ? n : m, rows = role == 0 ? n : p;
      block_load(rb, tile_rsrc(q, rows * cols), kb.off, cols);
    }
    const rsrc_t rA = tile_rsrc(pA + t * sA, n * n);
    block_load(ra, rA, ka.off, n);
    rdg = O::bload(rA, dgo);
    const rsrc_t rc = tile_rsrc(pc_ + (size_t)t * n, n);
#pragma unroll
    for (int s = 0; s < 4; ++s) rcv[s] = O::bload(rc, cvo, 4 * s * ES);
    rvr = O::bload(tile_rsrc(pr + (size_t)t * m, m), rvo);
    rvd = O::bload(tile_rsrc(prd + (size_t)t * m, m), rvo);
    rvq = O::bload(tile_rsrc(pq + (size_t)t * n, n), qvo);
  };
  auto store_data = [&]() {
    block_store(ra, ka);
    if (role == 0 ? !bconst : role < 3 && p > 0) {
      if (role > 0) {
#pragma unroll
        for (int s = 0; s < 4; ++s) rb[s] *= sr;
      }
      block_store(rb, kb);
    }
    if (tid < 4 * NT) O::store4(sm + X::AT + pn * LD + 4 * tid, rcv);   // column n: c
    if (tid < 16 * MT) {
      sm[X::RV + tid] = rvr;
      sm[X::RD + tid] = rvd;
    }
    if (tid < 16 * NT) sm[X::QV + tid] = rvq;
  };
  // after store_data and a barrier: the unit diagonal taken out of A~ (for the
  // first stage from the columns not marked in its place)
  auto store_diag = [&](bool first) {
    if (tid < n) {
      const int d = tile_pos(tid);
      const bool keep = first && sm[X::EV + d] != T0;
      const T e = !keep && rdg >= T(0.5) && rdg <= T(2) ? T(1) : T0;
      sm[X::AT + d * LD + d] = rdg - e;
      sm[X::EV + d] = e;
    }
  };

  // ---- addends in the registers of the waves that use them: Q (upper
  // tiles) and M' of the owners, R of the first wave
  // Their tiles: P's number w - 1 + NWK s (w > 0); G's gw + NWK s, the wave with
  // the most tiles of P taking the fewest of G; K's NW - 1 - w + NW r.
  const int gw = w == 0 ? NG : w == 1 ? NWK - 1 : w - 2;
  int pij[PSL], qo[PSL];
#pragma unroll
  for (int s = 0; s < PSL; ++s) {
    const int u = w - 1 + s * NWK, col0 = 16 * (tile_upper(u) >> 4) + pc;
    pij[s] = tile_upper(u);
    qo[s] = w > 0 && u < NPM && col0 < n ? ((16 * (pij[s] & 15) + O::RG * g) * n + col0) * ES : kOOB;
  }
  const int svo = c == (pn & 15) ? O::RG * g * ES : kOOB;   // column n of a tile's rows
  const int srow = O::RV * n * ES;                          // the step between a lane's rows
  int ko[RG];
#pragma unroll
  for (int r = 0; r < RG; ++r) {
    const int u = NW - 1 - w + r * NW, col = 16 * (u % NT) + pc;
    ko[r] = col < n ? ((16 * (u / NT) + O::RG * g) * n + col) * ES : kOOB;
  }
  const int ro = w < (MT == 2 ? 3 : 1) && 16 * ((w + 1) >> 1) + pc < m
                     ? ((16 * (w >> 1) + O::RG * g) * m + 16 * ((w + 1) >> 1) + pc) * ES : kOOB;
  V4 qv[PSL], mv[MODE == TILE_CALLER ? GSL : 1], rv;
  auto load_addends = [&](int t) {
    const rsrc_t rQ = tile_rsrc(pQ + t * sQ, n * n);
#pragma unroll
    for (int s = 0; s < PSL; ++s)
#pragma unroll
      for (int v = 0; v < 4; ++v) qv[s][v] = O::bload(rQ, qo[s], v * srow);
    if constexpr (MODE == TILE_CALLER) {
      const rsrc_t rM = tile_rsrc(pM + t * sM, has_m ? n * m : 0);
#pragma unroll
      for (int s = 0; s < GSL; ++s) {
        const int u = gw + s * NWK;
        const int i = u / NT, j = u - i * NT, col = 16 * j + pc;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = 16 * i + O::RG * g + O::RV * v;
          mv[s][v] = O::bload(rM, row < m ? (col * m + row) * ES : kOOB);
        }
      }
    }
    const rsrc_t rR = tile_rsrc(pR + t * sR, m * m);
#pragma unroll
    for (int v = 0; v < 4; ++v) rv[v] = O::bload(rR, ro, v * O::RV * m * ES);
  };

  // ---- start: LDS cleared (padding rows and columns stay 0), S~_N, stage N - 1
  for (int e = tid; e < X::TOTAL; e += NTH) sm[e] = T0;
  __syncthreads();
  if (tid < 16 * NT && tid == pn) sm[X::EV + tid] = T(1);
  {
    const T* QN = P.QN.at(b, 0);
    const T* qN = pq + (size_t)N * n;
    for (int e = tid; e < n * n; e += NTH) {
      const int i = e / n, j = e - i * n;
      sm[X::S + tile_pos(i) * LD + tile_pos(j)] = QN[e];
      pS[(size_t)N * n * n + e] = QN[e];
    }
    for (int i = tid; i < n; i += NTH) {
      const T q = qN[i];
      sm[X::S + tile_pos(i) * LD + pn] = q;
      sm[X::S + pn * LD + tile_pos(i)] = q;
      ps[(size_t)N * n + i] = q;
    }
  }
  if (bconst && role == 0) {
    block_load(rb, tile_rsrc(pB, n * m), kb.off, m);
    block_store(rb, kb);
  }
  load_data(N - 1);
  load_addends(N - 1);
  store_data();
  lds_sync();
  // where column j of Q_N differs from row j, j is marked in e's place
#pragma unroll
  for (int k = 0; k < (256 * NT * NT + NTH - 1) / NTH; ++k) {
    const int f = tid + k * NTH, i = f / (16 * NT), j = f - i * 16 * NT;
    if (f < 256 * NT * NT && !(sm[X::S + i * LD + j] == sm[X::S + j * LD + i])) sm[X::EV + j] = sm[X::SKEW] = T(1);
  }
  lds_sync();
  store_diag(true);
  lds_sync();

  auto sb_tile = [&](int u) {   // SB tile u = j NT + i
    const int j = u / NT, i = u - j * NT;
    return tile_dot<T, NT>(sm + X::S + 16 * i * LD + (c * LD + 4 * g), sm + X::BT + 16 * j * LD + (c * LD + 4 * g));
  };
  auto t_tile = [&](int u) {
    const int j = u / NT, i = u - j * NT;
    V4 acc = tile_dot<T, NT>(sm + X::S + 16 * i * LD + (c * LD + 4 * g), sm + X::AT + 16 * j * LD + (c * LD + 4 * g));
    // + S~ diag(e) (S~ symmetric: its column as a row)
    const V4 x = O::load_col(sm + X::S + (16 * j + c) * LD + 16 * i, g);
    const T e = sm[X::EV + 16 * j + c];
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[v] += e * x[v];
    return acc;
  };
  auto put_t = [&](int u, const V4& x) {
    const int j = u / NT, i = u - j * NT;
    O::store_col(sm + X::TT + (16 * j + c) * LD + 16 * i, g, x);
  };
  auto put_sb = [&](int u, const V4& x) {
    const int j = u / NT, i = u - j * NT;
    O::store_col(sm + X::SBT + (16 * j + c) * LD + 16 * i, g, x);
  };
  auto h_tile = [&](int i, int j) {
    V4 acc = tile_dot<T, NT>(sm + X::BT + 16 * i * LD + (c * LD + 4 * g), sm + X::SBT + 16 * j * LD + (c * LD + 4 * g));
    if (p > 0) acc += tile_dot<T, 1>(sm + X::ET + 16 * i * LP + (c * LP + 4 * g), sm + X::ET + 16 * j * LP + (c * LP + 4 * g));
    acc += rv;
#pragma unroll
    for (int v = 0; v < 4; ++v)
      if (i == j && O::pos(g, v) == c) acc[v] = 16 * i + pc < m ? acc[v] + sm[X::RD + 16 * i + c] : T(1);
    return acc;
  };
  auto at_tile = [&](int i, int j) {   // A~' T
    V4 acc = tile_dot<T, NT>(sm + X::AT + 16 * i * LD + (c * LD + 4 * g), sm + X::TT + 16 * j * LD + (c * LD + 4 * g));
    const V4 x = O::load_col(sm + X::TT + (16 * j + c) * LD + 16 * i, g), e = O::load_col(sm + X::EV + 16 * i, g);
    return acc + e * x;
  };
  // what makes a diagonal tile symmetric from one of its triangles, through buf
  // (rows of LM)
  auto one_triangle = [&](const V4& x, T* buf, bool lower) {
    V4 d;
#pragma unroll
    for (int v = 0; v < 4; ++v) buf[O::pos(g, v) * LM + c] = x[v];
    wave_lds_sync();
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = O::RG * g + O::RV * v;
      d[v] = (lower ? row < pc : row > pc) ? buf[c * LM + O::pos(g, v)] - x[v] : T0;
    }
    return d;
  };
  // Q_N not symmetric: the corrections to stage N - 1's H and P join R and Q (no
  // branch in the loop: one between H and its factorisation, or beside P, cost 2 %
  // of a stage)
  if (__any(sm[X::SKEW] != T0)) {
    for (int u = w; u < NB; u += NW) put_sb(u, sb_tile(u));
    for (int u = w; u < NTT; u += NW) put_t(u, t_tile(u));
    lds_sync();
    if (w == 0 || (MT == 2 && w == 2)) {
      const int i = w >> 1;
      rv += one_triangle(h_tile(i, i), sm + X::Z + 16 * i * LM, MT == 1);
    }
    if (w > 0) {
#pragma unroll
      for (int s = 0; s < PSL; ++s) {
        const int i = pij[s] & 15;
        if (((s + 1) * NWK <= NPM || w - 1 + s * NWK < NPM) && i == pij[s] >> 4)
          qv[s] += one_triangle(at_tile(i, i), sm + X::WT + 16 * i * LM, false);
      }
    }
    lds_sync();
  }

  for (int t = N - 1; t >= 0; --t) {
    // (pinned to a scalar register: a select into a vector register would make
    // every descriptor built from it look divergent)
    const int tp = __builtin_amdgcn_readfirstlane(t > 0 ? t - 1 : 0);
    // opaque copies: the tiles' addresses are formed anew in every phase (hoisted
    // out of the loop, or kept from phase to phase, they fill the registers and
    // spill)
    auto phase = [&]() {
      asm volatile("" : "+s"(w), "+v"(g), "+v"(c));
      pc = 4 * (c & 3) + (c >> 2);
    };
    phase();
    load_data(tp);
    // A
    {
      V4 acc[RA];
#pragma unroll
      for (int r = 0; r < RA; ++r) {
        const int u = w + r * NW;
        if ((r + 1) * NW <= NB || u < NB) acc[r] = sb_tile(u);
        else if (u - NB < NTT) acc[r] = t_tile(u - NB);
      }
#pragma unroll
      for (int r = 0; r < RA; ++r) {
        const int u = w + r * NW;
        if ((r + 1) * NW <= NB || u < NB) put_sb(u, acc[r]);
        else if (u - NB < NTT) put_t(u - NB, acc[r]);
      }
    }
    lds_sync();
    phase();
    V4 H[MT][MT];
    // B: H's tiles, the first in the first wave's registers, the others through
    // Z's place (lane by lane)
    if constexpr (MT == 2) {
      if (w < 3) {
        const V4 x = h_tile(w >> 1, (w + 1) >> 1);
        if (w == 0) {
          H[0][0] = x;
        } else {
#pragma unroll
          for (int v = 0; v < 4; ++v) sm[X::Z + (w - 1) * 256 + 64 * v + 16 * g + c] = x[v];
        }
      } else if (T_B + w - 3 < NTT) {
        put_t(T_B + w - 3, t_tile(T_B + w - 3));
      }
      lds_sync();
    }
    TileFactor<T, MT> fac;
    // C
    if (w == 0) {
      __builtin_amdgcn_s_setprio(3);
      if constexpr (MT == 1) {
        H[0][0] = h_tile(0, 0);
      } else {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          H[0][1][v] = sm[X::Z + 64 * v + 16 * g + c];
          H[1][1][v] = sm[X::Z + 256 + 64 * v + 16 * g + c];
        }
        wave_lds_sync();
      }
      fac.first(H, sm + X::Z, sm + X::ZT, ksm, hfloor, g, c);
      __builtin_amdgcn_s_setprio(0);
    } else if constexpr (RC > 0) {
      V4 acc[RC];
#pragma unroll
      for (int r = 0; r < RC; ++r) {
        const int u = T_C + w - 1 + r * NWK;
        if (T_C + (r + 1) * NWK <= NTT || u < NTT) acc[r] = t_tile(u);
      }
#pragma unroll
      for (int r = 0; r < RC; ++r) {
        const int u = T_C + w - 1 + r * NWK;
        if (T_C + (r + 1) * NWK <= NTT || u < NTT) put_t(u, acc[r]);
      }
    }
    lds_sync();
    phase();
    // D
    V4 pm[PSL];
    if (w == 0) {
      __builtin_amdgcn_s_setprio(3);
      fac.second(sm + X::Z, sm + X::ZT, ksm, hfloor, g, c);
      __builtin_amdgcn_s_setprio(0);
    } else {
      V4 ga[GSL];
#pragma unroll
      for (int s = 0; s < GSL; ++s) {
        const int u = gw + s * NWK;
        if ((s + 1) * NWK <= NG || u < NG) {
          const int i = u / NT, j = u - i * NT;
          V4 acc = tile_dot<T, NT>(sm + X::BT + 16 * i * LD + (c * LD + 4 * g), sm + X::TT + 16 * j * LD + (c * LD + 4 * g));
          if (p > 0) acc += tile_dot<T, 1>(sm + X::ET + 16 * i * LP + (c * LP + 4 * g), sm + X::DT + 16 * j * LP + (c * LP + 4 * g));
          if constexpr (MODE == TILE_CALLER) acc += mv[s];
          if (j == NT - 1 && c == (pn & 15)) acc += O::load_col(sm + X::RV + 16 * i, g);
          ga[s] = acc;
        }
      }
#pragma unroll
      for (int s = 0; s < PSL; ++s) {
        const int u = w - 1 + s * NWK;
        if ((s + 1) * NWK <= NPM || u < NPM) {
          const int i = pij[s] & 15, j = pij[s] >> 4;
          V4 acc = tile_dot<T, NT>(sm + X::AT + 16 * i * LD + (c * LD + 4 * g), sm + X::TT + 16 * j * LD + (c * LD + 4 * g));
          if (p > 0) acc += tile_dot<T, 1>(sm + X::DT + 16 * i * LP + (c * LP + 4 * g), sm + X::DT + 16 * j * LP + (c * LP + 4 * g));
          const V4 x = O::load_col(sm + X::TT + (16 * j + c) * LD + 16 * i, g), e = O::load_col(sm + X::EV + 16 * i, g);
          acc += e * x;
          acc += qv[s];
          if (j == NT - 1) {   // column and row n: q
            if (c == (pn & 15)) acc += O::load_col(sm + X::QV + 16 * i, g);
            if (i == j) {
              const T q = sm[X::QV + 16 * j + c];
#pragma unroll
              for (int v = 0; v < 4; ++v) acc[v] += 16 * i + O::pos(g, v) == pn ? q : T0;
            }
          }
          pm[s] = acc;
        }
      }
#pragma unroll
      for (int s = 0; s < GSL; ++s) {
        const int u = gw + s * NWK;
        const int i = u / NT, j = u - i * NT;
        if ((s + 1) * NWK <= NG || u < NG) O::store_col(sm + X::GT + (16 * j + c) * LM + 16 * i, g, ga[s]);
      }
    }
    load_addends(tp);
    lds_sync();
    phase();
    // E: W~ = Z G~ (Z lower triangular), stored W~'
    {
      V4 acc[RG];
#pragma unroll
      for (int r = 0; r < RG; ++r) {
        const int u = w + r * NW;
        if ((r + 1) * NW <= NG || u < NG) {
          const int i = u / NT, j = u - i * NT;
          const T* z = sm + X::Z + 16 * i * LM + c * LM + 4 * g;
          const T* gt = sm + X::GT + 16 * j * LM + c * LM + 4 * g;
          if (MT == 1 || i == 0) acc[r] = tile_dot<T, 1>(z, gt);
          else acc[r] = tile_dot<T, MT>(z, gt);
        }
      }
#pragma unroll
      for (int r = 0; r < RG; ++r) {
        const int u = w + r * NW;
        const int i = u / NT, j = u - i * NT;
        if ((r + 1) * NW <= NG || u < NG) O::store_col(sm + X::WT + (16 * j + c) * LM + 16 * i, g, acc[r]);
      }
    }
    if (t > 0) store_data();   // A~', B~', D', E', e, r, rd of this stage are no longer read
    lds_sync();
    phase();
    // F: S~ <- P - W~'W~ (both triangles), K~ = Z' W~
    {
      V4 sa[PSL], kc[RG];
      if (w > 0) {
#pragma unroll
        for (int s = 0; s < PSL; ++s) {
          const int u = w - 1 + s * NWK;
          if ((s + 1) * NWK <= NPM || u < NPM) {
            const int i = pij[s] & 15, j = pij[s] >> 4;
            sa[s] = pm[s] - tile_dot<T, MT>(sm + X::WT + 16 * i * LM + (c * LM + 4 * g), sm + X::WT + 16 * j * LM + (c * LM + 4 * g));
          }
        }
      }
#pragma unroll
      for (int r = 0; r < RG; ++r) {
        const int u = NW - 1 - w + r * NW;
        if ((r + 1) * NW <= NG || u < NG) {
          const int i = u / NT, j = u - i * NT;
          const T* z = sm + X::ZT + 16 * i * LM + c * LM + 4 * g;
          const T* wt = sm + X::WT + 16 * j * LM + c * LM + 4 * g;
          if (MT > 1 && i == MT - 1) kc[r] = tile_dot<T, 1>(z + 16 * i, wt + 16 * i);
          else kc[r] = tile_dot<T, MT>(z, wt);
        }
      }
      if (w > 0) {
        const rsrc_t rS = tile_rsrc(pS + (size_t)t * n * n, n * n);
        const rsrc_t rs = tile_rsrc(ps + (size_t)t * n, n);
#pragma unroll
        for (int s = 0; s < PSL; ++s) {
          const int u = w - 1 + s * NWK;
          if ((s + 1) * NWK <= NPM || u < NPM) {
            const int i = pij[s] & 15, j = pij[s] >> 4;
            V4 acc = sa[s];
            if (i == j) {
              // the upper triangle to both sides; the corner (n, n) is not carried
#pragma unroll
              for (int v = 0; v < 4; ++v) {
                const int r = 16 * i + O::pos(g, v), q = 16 * i + c;
                if (O::pos(g, v) <= c) {
                  const T x = r == pn && q == pn ? T0 : acc[v];
                  sm[X::S + r * LD + q] = x;
                  sm[X::S + q * LD + r] = x;
                }
              }
            } else {
#pragma unroll
              for (int v = 0; v < 4; ++v) sm[X::S + (16 * i + O::pos(g, v)) * LD + 16 * j + c] = acc[v];
              O::store_col(sm + X::S + (16 * j + c) * LD + 16 * i, g, acc);
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) O::bstore(rS, qo[s], v * srow, acc[v]);
            if (sizeof(T) == 8 && i != j) {   // both triangles (k_fwd_stage)
              const int qt = 16 * j + pc < n ? ((16 * j + pc) * n + 16 * i + O::RG * g) * ES : kOOB;
#pragma unroll
              for (int v = 0; v < 4; ++v) O::bstore(rS, qt, v * O::RV * ES, acc[v]);
            }
            if (j == NT - 1) {
#pragma unroll
              for (int v = 0; v < 4; ++v) O::bstore(rs, svo, (16 * i + O::RV * v) * ES, acc[v]);
            }
          }
        }
      }
      const rsrc_t rK = tile_rsrc(pK + (size_t)t * m * n, m * n);
      const rsrc_t rk = tile_rsrc(pk + (size_t)t * m, m);
#pragma unroll
      for (int r = 0; r < RG; ++r) {
        const int u = NW - 1 - w + r * NW;
        if ((r + 1) * NW <= NG || u < NG) {
          const int i = u / NT, j = u - i * NT;
#pragma unroll
          for (int v = 0; v < 4; ++v) O::bstore(rK, ko[r], v * srow, kc[r][v]);
          if (j == NT - 1) {
#pragma unroll
            for (int v = 0; v < 4; ++v) O::bstore(rk, svo, (16 * i + O::RV * v) * ES, kc[r][v]);
          }
        }
      }
    }
    if (t > 0) store_diag(false);
    lds_sync();
  }
}

}  // namespace mpxk
