// The partition sweep and the interface recursion of pyro_spike.hpp for
// 16 < NV <= 63 with their block algebra on the FP64 matrix cores
// (v_mfma_f64_16x16x4f64), four waves per workgroup.
//
// A 64 x 64 block (NV used, the rest zero; column NV carries a right-hand
// side where there is one) is spread by columns: wave w holds the column
// tile 16 w .. 16 w + 15 as four row tiles in the MFMA accumulator layout:
// in row tile rt, lane l and register r hold row (l / 16) + 4 r + 16 rt of
// column 16 w + l % 16.  The layout of the B operand (B[k][j] from lane
// j + 16 k) is that of one register of it: rows 4 r .. 4 r + 3 of a row
// tile are acc[rt][r].  So a product A B with B in accumulators needs only
// its A operand (A[i][k] from lane i + 16 k) from LDS, and the pivot rows of
// a panel, which are the panel's own rows, are registers of each tile.
//
// gj_tiles reduces [A | ...] to [I | X]: rows are scaled by powers of two,
// then the A columns are eliminated in panels of eight.  The wave that
// holds a panel copies it to one row per lane and reduces it alone; pivot k
// is row k unless an unused row's entry is more than kPivotRatio times
// larger, in which case the two rows are exchanged (in the panel at once, in
// every tile before the panel is applied).  The eight elementary transforms
// I - g_k e_k^T compose to T = I - W E_P^T, accumulated as the panel is
// reduced (W[:, k] = g_k, W[:, c<k] -= g_k W[k, c]), and every wave applies
// it to its tiles with two MFMAs per 16 x 16 tile.  The wave that holds the
// next panel updates that tile first and reduces the next panel before its
// other tiles: one workgroup barrier per panel.
//
// The chain of 54 pivots per block row (recip, broadcast, 7 columns each)
// bounds it.  With pivot rows left in place (a search over all rows per
// pivot, and the panel's rows gathered through LDS for every tile) a block
// row of the sweep took about 107k cycles at nv = 54.
#pragma once

#include "pyro_spike.hpp"

namespace pyro_spike {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int kMfmaWaves = 4;

__device__ __forceinline__ d4 mfma_f64(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Workgroup barrier for LDS data only: waits for this wave's LDS accesses,
// not for its global loads, so the next block's prefetch stays in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

struct alignas(16) TileShared {
  double W[2][64 * 9];         // -W of the panel, [row][k], by panel parity
  double pnl[64 * 9];          // a panel as one row per lane, [row][c]
  double swap[kMfmaWaves][2][48];  // per wave: the two rows of an exchange
  int smax[64][kMfmaWaves];    // high words of the rows' largest |A|, per wave
  unsigned long long with[2];  // byte k: row exchanged with pivot row k
  int any[2];                  // whether the panel exchanges rows at all
  int singular;
};

// Max over each 16-lane row of a non-negative 32-bit value.
__device__ __forceinline__ int row16_max(int v) {
#define PYRO_ROR_MAX(N)                                                      \
  {                                                                          \
    const int o = __builtin_amdgcn_update_dpp(0, v, 0x120 + N, 0xF, 0xF,     \
                                              true);                         \
    v = v > o ? v : o;                                                       \
  }
  PYRO_ROR_MAX(8)
  PYRO_ROR_MAX(4)
  PYRO_ROR_MAX(2)
  PYRO_ROR_MAX(1)
#undef PYRO_ROR_MAX
  return v;
}

// Reduce panel P (columns 8 P .. of the A tile acc of the wave that calls
// it) and publish its transform and row exchanges.
template <int NV, int P>
__device__ __forceinline__ void tile_panel(const d4 (&acc)[4], int lane,
                                           TileShared& sh, bool& singular) {
  constexpr int kBuf = P & 1;
  constexpr int kCol = 8 * (P & 1);  // the panel's first column in the tile
  constexpr int kNum = NV - 8 * P < 8 ? NV - 8 * P : 8;
  const int g = lane >> 4, cl = lane & 15;
  if (cl >= kCol && cl < kCol + 8) {
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        sh.pnl[(16 * rt + g + 4 * r) * 9 + (cl - kCol)] = acc[rt][r];
  }
  wave_lds_fence();
  double pn[8], wr[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    pn[k] = sh.pnl[lane * 9 + k];
    wr[k] = 0.0;
  }
  // (lane through an empty asm: the pivots' lane masks are formed where
  // they are used instead of kept, and spilled, across block rows)
  int ln = lane;
  asm volatile("" : "+v"(ln));
  unsigned long long with = 0ull;  // one byte per pivot
  bool any = false;
#pragma unroll
  for (int k = 0; k < kNum; ++k) {
    const int q = 8 * P + k;
    // the unused rows after row q
    const unsigned long long later =
        ((1ull << NV) - 1ull) & ~((2ull << q) - 1ull);
    int row = q;
    double piv = bcast(pn[k], q);
    double inv = pyro::recip(piv);
    if (__builtin_amdgcn_ballot_w64(fabs(pn[k]) > kPivotRatio * fabs(piv)) &
        later) {
      // the largest candidate
      row = pyro_bt::pivot_lane<NV>(
          pyro_bt::pivot_key(pn[k], ln >= q && ln < NV, ln), 0ull, 1ull << q);
      const int src = ln == q ? row : ln == row ? q : ln;
#pragma unroll
      for (int x = 0; x < 8; ++x) {
        if (x >= k) pn[x] = __shfl(pn[x], src);
        if (x < k) wr[x] = __shfl(wr[x], src);
      }
      any = true;
      piv = bcast(pn[k], q);
      inv = pyro::recip(piv);
    }
    with |= static_cast<unsigned long long>(row) << (8 * k);
    singular = singular || !(fabs(piv) > 0.0);
    // wr holds -W
    const double h = (ln == q) ? inv - 1.0 : -(pn[k] * inv);
#pragma unroll
    for (int x = k + 1; x < kNum; ++x) pn[x] = fma(h, bcast(pn[x], q), pn[x]);
#pragma unroll
    for (int x = 0; x < k; ++x) wr[x] = fma(h, bcast(wr[x], q), wr[x]);
    wr[k] = h;
  }
#pragma unroll
  for (int k = 0; k < 8; ++k) sh.W[kBuf][lane * 9 + k] = wr[k];
  if (lane == 0) {
    sh.with[kBuf] = with;
    sh.any[kBuf] = any;
  }
}

// The row exchanges of panel P in this wave's tiles, in the order they were
// made.
template <int NV, int NB, int P>
__device__ __forceinline__ void tile_swaps(d4 (&acc)[NB][4], int wv, int lane,
                                           TileShared& sh) {
  constexpr int kBuf = P & 1;
  constexpr int kNum = NV - 8 * P < 8 ? NV - 8 * P : 8;
  const int g = lane >> 4, cl = lane & 15;
  const unsigned lo = __builtin_amdgcn_readfirstlane(
      static_cast<unsigned>(sh.with[kBuf]));
  const unsigned hi = __builtin_amdgcn_readfirstlane(
      static_cast<unsigned>(sh.with[kBuf] >> 32));
#pragma unroll 1
  for (int k = 0; k < kNum; ++k) {
    const int q = 8 * P + k;
    const int w = ((k < 4 ? lo >> (8 * k) : hi >> (8 * (k - 4))) & 255u);
    if (w == q) continue;
    // register 4 rt + r and lane group of each of the two rows
    const int qi = (q >> 4) * 4 + ((q >> 2) & 3), wi = (w >> 4) * 4 + ((w >> 2) & 3);
    const bool mq = g == (q & 3), mw = g == (w & 3);
    double* sq = sh.swap[wv][0] + cl;
    double* sw = sh.swap[wv][1] + cl;
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      if (u == qi && mq)
#pragma unroll
        for (int j = 0; j < NB; ++j) sq[16 * j] = acc[j][u / 4][u % 4];
      if (u == wi && mw)
#pragma unroll
        for (int j = 0; j < NB; ++j) sw[16 * j] = acc[j][u / 4][u % 4];
    }
    wave_lds_fence();
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      if (u == qi && mq)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[j][u / 4][u % 4] = sw[16 * j];
      if (u == wi && mw)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[j][u / 4][u % 4] = sq[16 * j];
    }
    wave_lds_fence();
  }
}

template <int NV, int NB, int P>
__device__ __forceinline__ void gj_tiles_from(d4 (&acc)[NB][4], int wv,
                                              int lane, TileShared& sh,
                                              bool& singular) {
  constexpr int kBuf = P & 1;
  constexpr int kPanels = (NV + 7) / 8;
  const int g = lane >> 4, cl = lane & 15;
  if (__builtin_amdgcn_readfirstlane(sh.any[kBuf]))
    tile_swaps<NV, NB, P>(acc, wv, lane, sh);
  double aw[4][2];
#pragma unroll
  for (int rt = 0; rt < 4; ++rt)
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
      aw[rt][ks] = sh.W[kBuf][(16 * rt + cl) * 9 + 4 * ks + g];
  auto apply = [&](int j) {
    const double b0 = acc[j][P / 2][2 * (P & 1)];
    const double b1 = acc[j][P / 2][2 * (P & 1) + 1];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
      acc[j][rt] = mfma_f64(aw[rt][0], b0, acc[j][rt]);
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
      acc[j][rt] = mfma_f64(aw[rt][1], b1, acc[j][rt]);
  };
  // the A tile: live while it holds a column >= 8 (P + 1)
  if (16 * wv + 16 > 8 * (P + 1)) apply(0);
  if constexpr (P + 1 < kPanels) {
    if (wv == (P + 1) / 2) tile_panel<NV, P + 1>(acc[0], lane, sh, singular);
  }
#pragma unroll
  for (int j = 1; j < NB; ++j) apply(j);
  lds_barrier();
  if constexpr (P + 1 < kPanels)
    gj_tiles_from<NV, NB, P + 1>(acc, wv, lane, sh, singular);
}

// [A | ...] -> [I | X] as described above; row q of X in row q.  Every wave
// of the workgroup calls it together; its LDS may be reused after it.
template <int NV, int NB>
__device__ __forceinline__ void gj_tiles(d4 (&acc)[NB][4], int wv, int lane,
                                         TileShared& sh, bool& singular) {
  static_assert(NB <= 3, "three tiles per wave pass the exchange buffer");
  const int g = lane >> 4, cl = lane & 15;
  // rows scaled by 2^-e of their largest |A| entry
#pragma unroll
  for (int rt = 0; rt < 4; ++rt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int hi = static_cast<int>(__double_as_longlong(acc[0][rt][r]) >> 32)
                     & 0x7fffffff;
      const int mx = row16_max(hi);
      if (cl == 0) sh.smax[16 * rt + g + 4 * r][wv] = mx;
    }
  lds_barrier();
#pragma unroll
  for (int rt = 0; rt < 4; ++rt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int4 m = *reinterpret_cast<const int4*>(
          &sh.smax[16 * rt + g + 4 * r][0]);
      const int mx = max(max(m.x, m.y), max(m.z, m.w)) >> 20;
      // 2^(1023 - mx); rows of zeros, infinities or NaN stay as they are
      const int e = (mx > 0 && mx < 2046) ? 2046 - mx : 1023;
      const double sc =
          __longlong_as_double(static_cast<long long>(e) << 52);
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[j][rt][r] *= sc;
    }
  if (wv == 0) tile_panel<NV, 0>(acc[0], lane, sh, singular);
  lds_barrier();
  gj_tiles_from<NV, NB, 0>(acc, wv, lane, sh, singular);
}

// One sweep over a partition, one workgroup per sweep task (blockIdx = 2
// partition + (0 down, 1 up)), as k_spike_sweep_waves: acc[0] C', acc[1]
// slot (the coupling to the next row), acc[2] E (the outside unknown met
// first) with the right-hand side in column NV.
template <int NV>
__global__ void __launch_bounds__(64 * kMfmaWaves, 2)
k_spike_sweep_mfma(const double* __restrict__ L, const double* __restrict__ C,
                   const double* __restrict__ U, const double* __restrict__ R,
                   const int64_t* __restrict__ off,
                   const int64_t* __restrict__ pstart,
                   const int64_t* __restrict__ pend,
                   const int* __restrict__ psys, double* __restrict__ fact,
                   double* __restrict__ maps, int* __restrict__ n_singular) {
  static_assert(NV > 16 && NV <= 63, "column NV carries the right-hand side");
  constexpr int MW = 2 * NV + 1;
  __shared__ TileShared sh;
  const int64_t part = blockIdx.x >> 1;
  const bool down = (blockIdx.x & 1) == 0;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, cl = lane & 15;
  const int64_t s = pstart[part], e = pend[part];
  const int sy = psys[part];
  const int64_t s0 = off[sy], s1 = off[sy + 1];
  const int64_t m = e - s;
  if (!down && s == s0) return;  // never used; the whole workgroup leaves
  if (threadIdx.x == 0) sh.singular = 0;
  auto row = [&](int64_t t) { return down ? s + t : e - 1 - t; };
  auto slot_coef = [&](int64_t i) -> double {
    if (down) return i < s1 - 1 ? U[i] : 0.0;
    return i > s0 ? L[i - 1] : 0.0;
  };
  auto back_coef = [&](int64_t i) -> double {
    return down ? L[i] : U[i - 1];
  };
  const int c = 16 * wv + cl;  // this lane's column in each block
  auto rowq = [&](int rt, int r) { return 16 * rt + g + 4 * r; };

  d4 acc[3][4];
  {
    const int64_t i = row(0);
    const double sc = slot_coef(i);
    double ec = 0.0;
    if (down && s > s0) ec = -L[s - 1];
    if (!down && e < s1) ec = -U[e - 1];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int q = rowq(rt, r);
        const bool live = q < NV;
        acc[0][rt][r] = (live && c < NV) ? C[(i * NV + q) * NV + c] : 0.0;
        acc[1][rt][r] = (live && c == q) ? sc : 0.0;
        acc[2][rt][r] = !live ? 0.0
                        : c == q ? ec : (c == NV ? R[i * NV + q] : 0.0);
      }
  }
  // the loop below reads acc with no wait for these loads
  __builtin_amdgcn_s_waitcnt(0);
  bool singular = false;
  for (int64_t t = 0; t < m; ++t) {
    const int64_t i = row(t);
    // the next block's rows, in flight during this one (from clamped, valid
    // addresses; entries outside the block are masked where they are used)
    // column NV's lanes fetch the right-hand side
    d4 cpre[4] = {};
    double bpre = 0.0, spre = 0.0;
    const bool more = t + 1 < m;
    if (more) {
      const int64_t i1 = row(t + 1);
      const double* base = c < NV ? C + i1 * NV * NV + c : R + i1 * NV;
      const int ld = c < NV ? NV : 1;
#pragma unroll
      for (int rt = 0; rt < 4; ++rt)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          cpre[rt][r] = base[(rowq(rt, r) < NV ? rowq(rt, r) : NV - 1) * ld];
      bpre = back_coef(i);
      spre = slot_coef(i1);
    }
    gj_tiles<NV, 3>(acc, wv, lane, sh, singular);
    if (down) {
      // [X_U | X_r | X_W]: slot -> columns 0..NV-1, x -> NV, E -> NV+1..2NV
#pragma unroll
      for (int rt = 0; rt < 4; ++rt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (rowq(rt, r) >= NV) continue;
          double* f = fact + (i * NV + rowq(rt, r)) * MW;
          if (c < NV) {
            f[c] = acc[1][rt][r];
            f[NV + 1 + c] = acc[2][rt][r];
          } else if (c == NV) {
            f[NV] = acc[2][rt][r];
          }
        }
    }
    if (!more) break;
    // next block row: C_next - l X_slot | diag(spre) | -l E with r - l x
    const double l = bpre;
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int q = rowq(rt, r);
        const bool live = q < NV;
        acc[0][rt][r] =
            (live && c < NV) ? fma(-l, acc[1][rt][r], cpre[rt][r]) : 0.0;
        acc[1][rt][r] = (live && c == q) ? spre : 0.0;
        acc[2][rt][r] = fma(-l, acc[2][rt][r],
                            (live && c == NV) ? cpre[rt][r] : 0.0);
      }
  }
  // the partition's map from its last block row:
  //   down: x_{e-1} = X_r + X_W x_{s-1} - X_U x_e
  //   up:   x_s     = X_r + X_V x_e     - X_L x_{s-1}
#pragma unroll
  for (int rt = 0; rt < 4; ++rt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int q = rowq(rt, r);
      if (q >= NV || c > NV) continue;
      double* mp = maps + ((part * 2 + (down ? 0 : 1)) * NV + q) * MW;
      if (c == NV) {
        mp[0] = acc[2][rt][r];
      } else {
        // E: coefficient of the outside unknown; slot: minus the next's
        mp[(down ? 1 : 1 + NV) + c] = acc[2][rt][r];
        mp[(down ? 1 + NV : 1) + c] = -acc[1][rt][r];
      }
    }
  if (singular && lane == 0) sh.singular = 1;
  __syncthreads();
  if (threadIdx.x == 0 && sh.singular && n_singular) atomicAdd(n_singular, 1);
}

// k_spike_reduced_waves in the tile layout, one workgroup of four waves per
// system.  [G | beta] of the partition before stays in accumulators (column
// NV: beta), so per partition q:
//   [Q | .] = B'_q [G | beta], [P | .] = B_q [G | beta]  (B', B from LDS),
//   gj_tiles on [I - Q | D'_q with a' + B' beta] -> [H | tau],
//   [G | beta] = [D_q | a_q + B beta] + P [H | tau]      (P from LDS).
template <int NV>
__global__ void __launch_bounds__(64 * kMfmaWaves)
k_spike_reduced_mfma(const double* __restrict__ maps,
                     const int64_t* __restrict__ roff,
                     double* __restrict__ red, double* __restrict__ Z,
                     int* __restrict__ n_singular) {
  static_assert(NV > 16 && NV <= 63, "column NV carries the right-hand side");
  constexpr int MW = 2 * NV + 1;
  constexpr int N2 = 2 * NV;
  constexpr int RW = 2 * NV + 2;
  constexpr int KS = (NV + 3) / 4;  // k-steps of 4
  constexpr int LD = 65;            // LDS row stride of the A operands (odd)
  __shared__ TileShared sh;
  // A operands, zero outside the NV x NV block
  __shared__ double Bp[64 * LD], Bm[64 * LD];
  const int sy = blockIdx.x;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, cl = lane & 15;
  const int c = 16 * wv + cl;
  const int64_t j0 = roff[sy], j1 = roff[sy + 1];
  const int64_t nq = j1 - j0 + 1;
  if (nq < 2) return;  // the whole workgroup leaves
  const int64_t q0 = j0 + sy;
  auto mrow = [&](int64_t q, int dir, int row) {
    return maps + ((q * 2 + dir) * NV + row) * MW;
  };
  auto rrow = [&](int64_t q, int row) { return red + (q * NV + row) * RW; };
  auto rowq = [&](int rt, int r) { return 16 * rt + g + 4 * r; };
  // column c of [D | a] of a map row
  auto dcol = [&](const double* mr) { return c < NV ? mr[1 + NV + c] : mr[0]; };
  for (int idx = threadIdx.x; idx < 64 * LD; idx += 64 * kMfmaWaves)
    Bp[idx] = Bm[idx] = 0.0;
  if (threadIdx.x == 0) sh.singular = 0;
  bool singular = false;
  d4 G[4];
  auto store_G = [&](int64_t q) {
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (rowq(rt, r) < NV && c <= NV)
          rrow(q, rowq(rt, r))[c < NV ? 1 + c : 0] = G[rt][r];
  };
#pragma unroll
  for (int rt = 0; rt < 4; ++rt)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      G[rt][r] = (rowq(rt, r) < NV && c <= NV)
                     ? dcol(mrow(q0, 0, rowq(rt, r))) : 0.0;
  store_G(q0);
  // acc += A B over KS k-steps, A in LDS, B a column tile in accumulators
  auto product = [&](const double* A, const d4 (&B)[4], d4 (&acc)[4]) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int rt = 0; rt < 4; ++rt)
        acc[rt] = mfma_f64(A[(16 * rt + cl) * LD + 4 * ks + g],
                           B[ks / 4][ks % 4], acc[rt]);
  };
  __syncthreads();
  for (int64_t q = q0 + 1; q < q0 + nq; ++q) {
    // B'_q and B_q (rows of the up and down maps) to LDS; D' and D to
    // registers
    for (int idx = threadIdx.x; idx < NV * NV; idx += 64 * kMfmaWaves) {
      const int row = idx / NV, k = idx - row * NV;
      Bp[row * LD + k] = mrow(q, 1, row)[1 + k];
      Bm[row * LD + k] = mrow(q, 0, row)[1 + k];
    }
    d4 acc[2][4], D[4];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool ok = rowq(rt, r) < NV && c <= NV;
        const int row = ok ? rowq(rt, r) : 0;
        const double d1 = dcol(mrow(q, 1, row)), d0 = dcol(mrow(q, 0, row));
        acc[1][rt][r] = ok ? d1 : 0.0;
        D[rt][r] = ok ? d0 : 0.0;
      }
    __syncthreads();
    d4 Q[4] = {}, P[4] = {};
    product(Bp, G, Q);
    product(Bm, G, P);
    // [I - Q | D' with a' + B' beta], and D with a + B beta
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = rowq(rt, r);
        acc[0][rt][r] = (row < NV && c < NV)
                            ? ((row == c) ? 1.0 : 0.0) - Q[rt][r] : 0.0;
        if (c == NV) {
          acc[1][rt][r] += Q[rt][r];
          D[rt][r] += P[rt][r];
        }
      }
    __syncthreads();  // every wave has read B
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (c < NV) Bm[rowq(rt, r) * LD + c] = P[rt][r];
    gj_tiles<NV, 2>(acc, wv, lane, sh, singular);
    // (its barriers also order P's stores before the reads below)
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (rowq(rt, r) < NV && c <= NV)
          rrow(q, rowq(rt, r))[1 + NV + (c < NV ? 1 + c : 0)] = acc[1][rt][r];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) G[rt] = D[rt];
    product(Bm, acc[1], G);
    store_G(q);
    __syncthreads();  // every wave has read P before the next B is staged
  }
  if (singular && lane == 0) sh.singular = 1;
  __syncthreads();
  if (threadIdx.x == 0 && sh.singular && n_singular) atomicAdd(n_singular, 1);
  if (wv != 0) return;
  // back substitution on wave 0 (the rows of red were written by all the
  // waves before the last barrier); t in natural row order, lane r
  const bool active = lane < NV;
  const int r = active ? lane : 0;
  const int64_t ql = q0 + nq - 1;
  double t = rrow(ql, r)[1 + NV];
  for (int64_t q = ql - 1; q >= q0; --q) {
    const double* o = rrow(q, r);
    double b = o[0], tn = o[1 + NV];
#pragma unroll
    for (int mm = 0; mm < NV; ++mm) {
      const double tm = bcast(t, mm);
      b = fma(o[1 + mm], tm, b);
      tn = fma(o[2 + NV + mm], tm, tn);
    }
    const int64_t j = j0 + (q - q0);
    if (active) {
      Z[j * N2 + r] = b;
      Z[j * N2 + NV + r] = t;
    }
    t = tn;  // of q0: never used
  }
}

// Form for 16 < NV <= 63: 1 the blocked MFMA sweep and the MFMA recursion
// above (default), 0 k_spike_sweep_waves and k_spike_reduced_waves.
inline int& sweep_form() {
  static int form = 1;
  return form;
}

// Host side: the three launches.  All arrays are device arrays prepared by
// the caller (see pyro_flamelet_thomas_partitioned).
template <int NV>
int solve(const double* L, const double* C, const double* U, const double* R,
          double* X, const int64_t* off, const int64_t* pstart,
          const int64_t* pend, const int* psys, int64_t nparts,
          const int64_t* jbefore, const int64_t* jafter, const int64_t* roff,
          int64_t nsys, int64_t nj, double* fact, double* maps, double* red,
          double* Z, int* n_singular, hipStream_t stream) {
  if constexpr (NV <= 16) {
    k_spike_sweep_grp<NV>
        <<<static_cast<unsigned>((2 * nparts + 3) / 4), 64, 0, stream>>>(
            L, C, U, R, off, pstart, pend, psys, nparts, fact, maps,
            n_singular);
  } else {
    bool blocked = false;
    if constexpr (NV <= 63) {
      if (sweep_form() == 1) {
        blocked = true;
        k_spike_sweep_mfma<NV>
            <<<static_cast<unsigned>(2 * nparts), 64 * kMfmaWaves, 0,
               stream>>>(
                L, C, U, R, off, pstart, pend, psys, fact, maps, n_singular);
      }
    }
    if (!blocked)
      k_spike_sweep_waves<NV>
          <<<static_cast<unsigned>(2 * nparts), 64 * kWaves, 0, stream>>>(
              L, C, U, R, off, pstart, pend, psys, fact, maps, n_singular);
  }
  if (nj > 0) {
    if constexpr (NV <= 16)
      k_spike_reduced<NV><<<static_cast<unsigned>(nsys), 64, 0, stream>>>(
          maps, roff, red, Z, n_singular);
    else {
      bool mfma = false;
      if constexpr (NV <= 63) {
        if (sweep_form() == 1) {
          mfma = true;
          k_spike_reduced_mfma<NV>
              <<<static_cast<unsigned>(nsys), 64 * kMfmaWaves, 0, stream>>>(
                  maps, roff, red, Z, n_singular);
        }
      }
      if (!mfma)
        k_spike_reduced_waves<NV>
            <<<static_cast<unsigned>(nsys), 64 * kWaves, 0, stream>>>(
                maps, roff, red, Z, n_singular);
    }
  }
  if constexpr (NV <= 16)
    k_spike_recover_grp<NV><<<static_cast<unsigned>((nparts + 3) / 4), 64, 0,
                              stream>>>(fact, pstart, pend, nparts, jbefore,
                                        jafter, Z, X);
  else
    k_spike_recover<NV><<<static_cast<unsigned>(nparts), 256, 0, stream>>>(
        fact, pstart, pend, jbefore, jafter, Z, X);
  return pyro::launch_status();
}

}  // namespace pyro_spike
