// Flamelet source kernel of a generated mechanism with NS <= 16: T(h, Y),
// S and the NV x NV source Jacobian per point in one pass, with the NS x NS
// kinetics Jacobian held in registers (mech::net_production_rates_jac).
//
// Included after pyro_flamelet_kernels.hpp.  Larger mechanisms form the
// source Jacobian with pyro_source_jacobian instead.
#pragma once

#include "pyro_flamelet_kernels.hpp"

namespace pyro_fl {

// Source term S = [vd/rho ; W_k w_k / rho] of one point
// (flamelets/equations.py:313-389) and, if jout != nullptr, its Jacobian
// dS/dphi (NV x NV, row-major) by the chain rule through T(h, Y) and
// rho(T, Y) = p W/(R T):
//   dT/dh = 1/cp, dT/dY_m = -h_m/cp, drho/dh = -rho/T dT/dh,
//   drho/dY_m = -rho W/W_m - rho/T dT/dY_m, dC_k = (Y_k/W_k) drho + rho/W_k dY_k.
// kRef: T and dT/dphi from the reference's loop (temperature_from_h_tangent)
// instead of the converged Newton and the exact derivative of T(h, Y).
// The Jacobian's rows go to put(r, row) in order, if jac.
template <bool kRef, class Put>
__device__ __forceinline__ bool point_source(const double h,
                                             const double (&Y)[NS],
                                             const double vd,
                                             const double tguess,
                                             const double p, const double tol,
                                             const int maxit, double& T,
                                             double (&S)[NV], const bool jac,
                                             Put put) {
  double th_ref = 0.0, tY_ref[NS];
  bool ok;
  if constexpr (kRef)
    ok = temperature_from_h_tangent(h, Y, tguess, tol, maxit, T, th_ref,
                                    tY_ref);
  else
    ok = temperature_from_h(h, Y, tguess, tol, maxit, T);
  double s = 0.0;
#pragma unroll
  for (int k = 0; k < NS; ++k) s = fma(mech::kInvW[k], Y[k], s);
  const double mmw = 1.0 / s;
  const double rho = p * mmw / (kGasConstant * T);
  double C[NS], w[NS];
#pragma unroll
  for (int k = 0; k < NS; ++k) C[k] = mech::kInvW[k] * rho * Y[k];
  const double irho = 1.0 / rho;
  if (!jac) {
    mech::net_production_rates(T, C, w);
  } else {
    double J[NS][NS], JT[NS];
    mech::net_production_rates_jac(T, C, w, J, JT);
    double hrt[NS], cpr[NS];
    mech::species_h_rt(T, 1.0 / T, hrt);
    mech::species_cp_r(T, cpr);
    double sc = 0.0;
#pragma unroll
    for (int k = 0; k < NS; ++k) sc = fma(Y[k] * mech::kInvW[k], cpr[k], sc);
    const double cp = kGasConstant * sc;
    const double dTdh = kRef ? th_ref : 1.0 / cp;
    const double rT = rho / T;
    const double drdh = -rT * dTdh;
    double dTdY[NS], drdY[NS];
#pragma unroll
    for (int m = 0; m < NS; ++m) {
      dTdY[m] = kRef ? tY_ref[m]
                     : -(kGasConstant * T * hrt[m] * mech::kInvW[m]) * dTdh;
      drdY[m] = fma(-rT, dTdY[m], -rho * mmw * mech::kInvW[m]);
    }
    // row 0: d(vd/rho)
    const double c0 = -vd * irho * irho;
    double row[NV];
    row[0] = c0 * drdh;
#pragma unroll
    for (int m = 0; m < NS; ++m) row[1 + m] = c0 * drdY[m];
    put(0, row);
#pragma unroll
    for (int k = 0; k < NS; ++k) {
      double a = 0.0;
#pragma unroll
      for (int j = 0; j < NS; ++j) a = fma(J[k][j], Y[j] * mech::kInvW[j], a);
      const double f = mech::kW[k] * irho;
      const double wr = w[k] * irho;
      const double dwh = fma(a, drdh, JT[k] * dTdh);
      row[0] = f * fma(-wr, drdh, dwh);
#pragma unroll
      for (int m = 0; m < NS; ++m) {
        const double dwm = fma(J[k][m], rho * mech::kInvW[m],
                               fma(a, drdY[m], JT[k] * dTdY[m]));
        row[1 + m] = f * fma(-wr, drdY[m], dwm);
      }
      put(1 + k, row);
    }
  }
  S[0] = vd * irho;
#pragma unroll
  for (int k = 0; k < NS; ++k) S[1 + k] = mech::kW[k] * w[k] * irho;
  return ok;
}

// What turns the source Jacobian's blocks into the central blocks of the
// system (k_flamelet_blocks) while they are written; chi null: they are
// written as they are.
struct BlockArgs {
  const double* chi;
  const double* chi0;
  const double* lb;
  const int* sys;
  const int64_t* off;
  const int* modes;
  const double* dt;
};

// Each wave passes a Jacobian row of its 64 points through LDS, so that a
// store instruction writes whole rows of a few points instead of one entry
// of 64.  143k sandiego points: 129 us with J written entry by entry, 146 us
// with the finished blocks, which take the place of a 65 us pass that read
// and wrote all of J again; bound by the FP64 chain of one point per lane
// (one wave per SIMD for the NS x NS Jacobian in registers).
template <bool kRef>
__global__ void __launch_bounds__(256)
k_flamelet_source(const double* __restrict__ phi, int64_t ldp,
                  const double* __restrict__ vd,
                  const double* __restrict__ tguess, int64_t tg_stride,
                  const double* __restrict__ p, int64_t p_stride,
                  double* __restrict__ S, int64_t lds,
                  double* __restrict__ T_out, double* __restrict__ J,
                  int64_t n, double tol, int maxit, int* __restrict__ n_fail,
                  BlockArgs blk) {
  constexpr int kLd = NV | 1;
  __shared__ double stage[4][64 * kLd];
  const int lane = threadIdx.x & 63;
  const int64_t i1 = cell_index();
  const int64_t i0 = i1 - lane;  // the wave's first point
  if (i0 >= n) return;           // whole waves leave
  const bool live = i1 < n;
  const int64_t i = live ? i1 : n - 1;  // lanes past the end store nothing
  double Y[NS], s[NV], T;
  const double h = phi[i];
#pragma unroll
  for (int k = 0; k < NS; ++k) Y[k] = phi[(1 + k) * ldp + i];
  double hc = 0.0, diag = 0.0, mask = 1.0, hdt = 0.0;
  bool cn = false;
  if (J && blk.chi) {
    const int sy = blk.sys[i];
    const bool end = i == blk.off[sy] || i == blk.off[sy + 1] - 1;
    const int mode = blk.modes ? blk.modes[sy] : 0;
    hc = 0.5 * (((mode & 2) && blk.chi0) ? blk.chi0[i] : blk.chi[i]);
    diag = blk.lb[i];
    mask = end ? 0.0 : 1.0;
    cn = mode & 1;
    hdt = cn ? 0.5 * blk.dt[sy] : 0.0;
  }
  double* st = stage[threadIdx.x >> 6];
  double* Jw = J + i0 * NV * NV;
  const int pts = n - i0 < 64 ? static_cast<int>(n - i0) : 64;
  const bool blocks = blk.chi != nullptr;
  auto put = [&](int r, double (&row)[NV]) {
#pragma unroll
    for (int c = 0; c < NV; ++c) {
      double v = row[c];
      if (blocks) {
        v *= mask;
        if (c == r) v = fma(hc, diag, v);
        if (cn) v = (c == r ? 1.0 : 0.0) - hdt * v;
      }
      st[lane * kLd + c] = v;
    }
    pyro_spike::wave_lds_fence();
#pragma unroll
    for (int u = 0; u < NV; ++u) {
      const unsigned f = u * 64u + lane;
      const unsigned pt = f / NV, c = f - pt * NV;
      if (static_cast<int>(pt) < pts)
        Jw[pt * (NV * NV) + r * NV + c] = st[pt * kLd + c];
    }
    pyro_spike::wave_lds_fence();
  };
  const bool ok = point_source<kRef>(h, Y, vd ? vd[i] : 0.0,
                                     tguess[i * tg_stride], p[i * p_stride],
                                     tol, maxit, T, s, J != nullptr, put);
  if (!live) return;
  // a point whose temperature did not converge poisons its flamelet's
  // update (NaN S), which the caller sees in the update norm
  const double bad = __builtin_nan("");
#pragma unroll
  for (int v = 0; v < NV; ++v) S[v * lds + i] = ok ? s[v] : bad;
  if (T_out) T_out[i] = ok ? T : bad;
  if (!ok && n_fail) atomicAdd(n_fail, 1);
}

inline int launch_source(const double* phi, int64_t ldp, const double* vd,
                         const double* tguess, int64_t tg_stride,
                         const double* p, int64_t p_stride, double* S,
                         int64_t lds, double* T_out, double* J, int64_t n,
                         double tol, int maxit, int* n_fail, int semantics,
                         const BlockArgs& blk, hipStream_t stream) {
  if (n < 0 || ldp < n || lds < n || !phi || !tguess || !p || !S ||
      (semantics != 0 && semantics != 1))
    return kInvalidArgument;
  if (semantics == 1)
    k_flamelet_source<true><<<grid_for(n, 256), 256, 0, stream>>>(
        phi, ldp, vd, tguess, tg_stride, p, p_stride, S, lds, T_out, J, n,
        tol, maxit, n_fail, blk);
  else
    k_flamelet_source<false><<<grid_for(n, 256), 256, 0, stream>>>(
        phi, ldp, vd, tguess, tg_stride, p, p_stride, S, lds, T_out, J, n,
        tol, maxit, n_fail, blk);
  return launch_status();
}

}  // namespace pyro_fl

PYRO_API int pyro_flamelet_source(const double* phi, int64_t ldp,
                                  const double* vd, const double* tguess,
                                  int64_t tg_stride, const double* p,
                                  int64_t p_stride, double* S, int64_t lds,
                                  double* T_out, double* J, int64_t n,
                                  double tol, int maxit, int* n_fail,
                                  int semantics, hipStream_t stream) {
  if (n == 0) return pyro::kOk;
  return pyro_fl::launch_source(phi, ldp, vd, tguess, tg_stride, p, p_stride,
                                S, lds, T_out, J, n, tol, maxit, n_fail,
                                semantics, pyro_fl::BlockArgs{}, stream);
}

// pyro_flamelet_source followed by the part of pyro_flamelet_assemble that
// turns J into the system's central blocks, in one pass over the blocks;
// pyro_flamelet_residual does the rest of it.
PYRO_API int pyro_flamelet_source_blocks(
    const double* phi, int64_t ldp, const double* vd, const double* tguess,
    int64_t tg_stride, const double* p, int64_t p_stride, double* S,
    int64_t lds, double* T_out, double* J, const double* chi,
    const double* chi0, const double* lb, const int* sys, const int64_t* off,
    const int* modes, const double* dt, int64_t n, double tol, int maxit,
    int* n_fail, int semantics, hipStream_t stream) {
  if (n == 0) return pyro::kOk;
  if (!J || !chi || !lb || !sys || !off || (modes && !dt))
    return pyro::kInvalidArgument;
  return pyro_fl::launch_source(
      phi, ldp, vd, tguess, tg_stride, p, p_stride, S, lds, T_out, J, n, tol,
      maxit, n_fail, semantics,
      pyro_fl::BlockArgs{chi, chi0, lb, sys, off, modes, dt}, stream);
}
