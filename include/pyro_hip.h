/*
 * pyro_hip.h -- C ABI of the MI355X thermochemistry / flamelet libraries.
 *
 * Two kinds of shared library export these symbols:
 *   libpyro_<mech>_<digest>.so   one per mechanism, generated by the "hip"
 *                                code-generation target (pointwise chemistry)
 *   libpyro_core.so              mechanism-independent (block-Thomas)
 *
 * Conventions (every function):
 *   - all array pointers are DEVICE pointers owned by the caller;
 *   - arrays are float64 struct-of-arrays: a per-species array is (ns, ld)
 *     with cell i of species k at [k*ld + i]; a per-reaction array likewise
 *     (nr, ld);
 *   - a per-cell scalar input comes with a stride: 0 broadcasts element 0,
 *     1 reads one value per cell;
 *   - work is enqueued on `stream` (a hipStream_t; NULL = default stream)
 *     and the call returns without synchronising;
 *   - return value: 0 = ok, < 0 = invalid argument (-1) or launch error
 *     (-2); no C++ exception crosses the boundary.
 *   - n == 0 is valid and does nothing.
 *
 * The reference (pyrometheus 1.1.1) has no C ABI: its hot path is the
 * generated Python class.  Each entry point below names the generated method
 * (pyrometheus/codegen/python.py) or flamelet function it replaces.
 */
#ifndef PYRO_HIP_H
#define PYRO_HIP_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef struct ihipStream_t* pyro_stream_t; /* == hipStream_t */

/* ---- per-mechanism library ------------------------------------------- */

/* out[0..3] = {num_species, num_reactions, num_falloff, abi_version}.
 * Replaces the generated attributes num_species/num_reactions/num_falloff
 * (codegen/python.py:180-186). */
int pyro_mech_info(int64_t* out, int n);

/* which: 0 cp/R, 1 h/RT, 2 s/R, 3 g/RT, 4 d(cp/R)/dT, 5 d(h/RT)/dT,
 *        6 d(s/R)/dT;  out is (ns, ld).
 * Replaces get_species_specific_heats_r / _enthalpies_rt / _entropies_r /
 * _gibbs_rt and the *_derivative methods (codegen/python.py:313-358). */
int pyro_species_thermo(int which, const double* T, int64_t t_stride,
                        double* out, int64_t ld, int64_t n,
                        pyro_stream_t stream);

/* which: 0 cp, 1 cv, 2 h, 3 e (mass-specific mixture values).
 * Replaces get_mixture_specific_heat_cp_mass / _cv_mass,
 * get_mixture_enthalpy_mass, get_mixture_internal_energy_mass
 * (codegen/python.py:293-311). */
int pyro_mixture_thermo(int which, const double* T, int64_t t_stride,
                        const double* Y, int64_t ldY, double* out, int64_t n,
                        pyro_stream_t stream);

/* which: 0 mixture molecular weight(Y), 1 specific gas constant(Y),
 *        2 density(a = p, T, Y), 3 pressure(a = rho, T, Y).
 * Replaces get_mixture_molecular_weight, get_specific_gas_constant,
 * get_density, get_pressure (codegen/python.py:248-270). */
int pyro_mixture_state(int which, const double* a, int64_t a_stride,
                       const double* T, int64_t t_stride, const double* Y,
                       int64_t ldY, double* out, int64_t n,
                       pyro_stream_t stream);

/* which: 0 concentrations(a = rho), 1 mole fractions(a = mmw); out (ns, ld).
 * Replaces get_concentrations, get_mole_fractions
 * (codegen/python.py:272-285). */
int pyro_species_state(int which, const double* a, int64_t a_stride,
                       const double* Y, int64_t ldY, double* out, int64_t ld,
                       int64_t n, pyro_stream_t stream);

/* Per-reaction quantities from (T, concentrations C (ns, ldC)); any output
 * may be NULL.  kf: forward rate coefficients incl. falloff and three-body
 * factors; nlk: -ln K_c (irreversible: -0.17364695002734*T); rf, rr, rnet:
 * forward, reverse, net rates of progress.  Outputs are (nr, ldR).
 * Replaces get_fwd_rate_coefficients (codegen/python.py:453-473),
 * get_equilibrium_constants (:360-373), get_fwd_rates_of_progress (:497),
 * get_rev_rates_of_progress (:506), get_net_rates_of_progress (:475). */
int pyro_reaction_quantities(const double* T, const double* C, int64_t ldC,
                             double* kf, double* nlk, double* rf, double* rr,
                             double* rnet, int64_t ldR, int64_t n,
                             pyro_stream_t stream);

/* Net molar production rates (ns, ldW) from rho, T, Y: one fused kernel.
 * Replaces get_net_production_rates (codegen/python.py:486-495). */
int pyro_wdot(const double* rho, const double* T, const double* Y,
              int64_t ldY, double* wdot, int64_t ldW, int64_t n,
              pyro_stream_t stream);

/* Creation and destruction rates (ns, ldW).
 * Replaces get_creation_destruction_rates (codegen/python.py:543-562). */
int pyro_creation_destruction(const double* rho, const double* T,
                              const double* Y, int64_t ldY, double* cdot,
                              double* ddot, int64_t ldW, int64_t n,
                              pyro_stream_t stream);

/* Per-lane Newton for T from e (do_energy != 0) or h.
 * mode 0: take the step, stop when |step| < tol (get_temperature,
 *         codegen/python.py:375-396);
 * mode 1: stop when |step| <= tol without taking it
 *         (get_temperature_from_enthalpy, flamelets/make_pyro.py:255-299).
 * *n_fail (device int, may be NULL) is incremented once per lane that did
 * not converge in maxit steps; iters (device int array, may be NULL) gets
 * the per-lane iteration count, -1 for a lane that did not converge. */
int pyro_temperature(const double* target, int64_t target_stride,
                     const double* t_guess, int64_t guess_stride,
                     const double* Y, int64_t ldY, double* T_out, int64_t n,
                     int do_energy, int mode, double tol, int maxit,
                     int* n_fail, int* iters, pyro_stream_t stream);

/* ---- derivatives of the net production rates -------------------------
 * Exported by every mechanism library.  Tangents and cotangents follow the
 * layout of the primal: v_rho, v_T, g_rho, g_T are (n,), v_Y, g_Y, wbar,
 * jvp are (ns, ld).  A NULL tangent counts as zero; a NULL gradient output
 * is skipped.  The reference differentiates the generated class with JAX
 * (flamelets/equations.py:124-129, vmap(jacfwd(local_source_terms))); these
 * are the hand-written forward and reverse products of
 * get_net_production_rates (codegen/python.py:486-495). */

/* jvp = dw/drho v_rho + dw/dT v_T + dw/dY v_Y; wdot (may be NULL) gets w. */
int pyro_wdot_jvp(const double* rho, const double* T, const double* Y,
                  int64_t ldY, const double* v_rho, const double* v_T,
                  const double* v_Y, int64_t ldV, double* wdot, double* jvp,
                  int64_t ldO, int64_t n, pyro_stream_t stream);

/* g_rho = wbar . dw/drho, g_T = wbar . dw/dT, g_Y = wbar . dw/dY. */
int pyro_wdot_vjp(const double* rho, const double* T, const double* Y,
                  int64_t ldY, const double* wbar, int64_t ldB, double* g_rho,
                  double* g_T, double* g_Y, int64_t ldG, int64_t n,
                  pyro_stream_t stream);

/* Doubles of workspace pyro_source_jacobian needs in its current form: 0
 * for the one-pass form (the default), else the per-reaction cache (k_f,
 * k_r, q, dq/dT, dq/d[M]) of one fixed-size chunk of cells. */
int64_t pyro_source_jacobian_work_doubles(void);

/* Form of pyro_source_jacobian for this process: 1 one pass (each row
 * evaluates the rate coefficients of its species' reactions; no workspace;
 * the default), 0 two passes through the per-reaction cache.  waves: the
 * waves that share each 64 cells in the one-pass form (1, 2, 4 or 8; 0
 * the default, one wave per row group); the values do not depend on it.  A
 * negative form only queries.  Returns the previous form, or -1 (invalid
 * argument).  No counterpart in the reference, whose Jacobian is jacfwd. */
int pyro_source_jacobian_form(int form, int waves);

/* Full (ns+1) x (ns+1) Jacobian of the flamelet source S = [vd/rho;
 * W_k w_k/rho] with respect to phi = [h; Y] per cell, at a temperature T
 * consistent with h and rho = p W/(R T) (p with stride p_stride; vd may be
 * NULL = 0).  Entry (r, c) of cell i is written to out[(r*nv + c)*s_rc +
 * i*s_i]: s_rc = 1, s_i = nv*nv gives the reference's (n, nv, nv) layout,
 * s_rc = ld, s_i = 1 an entry-major (nv, nv, ld) one.  The one-pass form
 * writes the entry-major layout with streaming stores; with s_rc = 1 (any
 * s_i, so padded blocks too) it stages each row through LDS and writes 64
 * contiguous bytes per cell and store.  S (nv, ldS), if not
 * NULL, receives S.  work holds pyro_source_jacobian_work_doubles()
 * doubles (the two-pass form processes the cells chunk by chunk through
 * it; the one-pass form ignores it and accepts NULL).  Replaces
 * vmap(jacfwd(local_source_terms)) (flamelets/equations.py:124-129,
 * :361-389). */
int pyro_source_jacobian(const double* T, const double* p, int64_t p_stride,
                         const double* Y, int64_t ldY, const double* vd,
                         double* out, int64_t s_rc, int64_t s_i, double* S,
                         int64_t ldS, double* work, int64_t n,
                         pyro_stream_t stream);

/* ---- flamelet kernels ------------------------------------------------
 * Exported by libraries of mechanisms with ns <= 16 (nv = ns + 1 <= 17).
 * A batch of B flamelets is stored with its grid points concatenated:
 * P = sum_s N_s points, point i of system s = sys[i] lies in
 * [off[s], off[s+1]).  phi is (nv, ldp): row 0 the mass enthalpy, rows
 * 1..ns the mass fractions (flamelets/state.py:297-316).  Blocks are
 * (P, nv, nv) row-major per point. */

/* Per point: T(h, Y) by Newton from tguess (take the step, stop when
 * |step| < tol; equations.py:284-311 with make_pyro.py:255-299), the source
 * S = [vd/rho; W_k w_k/rho] (equations.py:361-389) into S (nv, lds) and, if
 * J != NULL, dS/dphi (nv x nv) by the chain rule through T(h, Y) and
 * rho = p W/(R T) (replaces equations.py:124-129).  vd may be NULL (zero).
 * T_out may be NULL; *n_fail counts points whose Newton did not converge,
 * and such a point gets T = NaN and S = NaN (so the update of its flamelet
 * is not finite and the caller can stop it at once).
 * semantics 0: the Newton takes the step and stops once |step| < tol, and J
 * uses the exact derivative of T(h, Y) (dT/dh = 1/cp, dT/dY_m = -h_m/cp);
 * semantics 1: the reference's loop (make_pyro.py:255-299 as a
 * lax.while_loop: stop before the step once |step| <= tol) with dT/dphi the
 * forward-mode tangent carried through the iterations taken, which is what
 * jax.jacfwd gives there (0 when the guess already meets the test). */
int pyro_flamelet_source(const double* phi, int64_t ldp, const double* vd,
                         const double* tguess, int64_t tg_stride,
                         const double* p, int64_t p_stride, double* S,
                         int64_t lds, double* T_out, double* J, int64_t n,
                         double tol, int maxit, int* n_fail, int semantics,
                         pyro_stream_t stream);

/* Residual and block-tridiagonal Jacobian, steady (bit 0 of modes[s]
 * clear, or modes == NULL) or Crank-Nicolson (bit 0 set, with phi_prev,
 * r_prev and dt[s]); bit 1 of modes[s] selects the dissipation rate chi0
 * instead of chi (the equilibration phase; chi0 may be NULL otherwise);
 * bits 0 and 2 together start a time step: phi_prev = phi and r_prev =
 * R(phi) are written first (the step's first Newton iteration).
 * R_i = chi_i/2 (a_i phi_{i-1} + b_i phi_i + c_i phi_{i+1}) + m_i S_i
 * - BC_i with m_i = 0 on the end points and bc (B, 2, nv) the
 * oxidiser/fuel states (equations.py:167-282; onedim_laplacian.py:144-212;
 * CN form solver.py:253-306).  Writes rhs = -R as (P, nv), the central
 * blocks in place of J, the scalar coupling coefficients L, U (P,), and R
 * itself into r_out (nv, ldp) when r_out != NULL. */
int pyro_flamelet_assemble(const double* phi, int64_t ldp, const double* S,
                           int64_t lds, double* J, const double* chi,
                           const double* chi0, const double* la,
                           const double* lb, const double* lc, const int* sys,
                           const int64_t* off, const double* bc,
                           const int* modes, double* phi_prev,
                           double* r_prev, const double* dt,
                           double* rhs, double* L, double* U, double* r_out,
                           int64_t n, pyro_stream_t stream);

/* pyro_flamelet_assemble without the central blocks. */
int pyro_flamelet_residual(const double* phi, int64_t ldp, const double* S,
                           int64_t lds, const double* chi,
                           const double* chi0, const double* la,
                           const double* lb, const double* lc, const int* sys,
                           const int64_t* off, const double* bc,
                           const int* modes, double* phi_prev,
                           double* r_prev, const double* dt,
                           double* rhs, double* L, double* U, double* r_out,
                           int64_t n, pyro_stream_t stream);

/* pyro_flamelet_source with J written as the central blocks that
 * pyro_flamelet_assemble would make of it (mechanisms of at most 16
 * species), so that the blocks are written once. */
int pyro_flamelet_source_blocks(const double* phi, int64_t ldp,
                                const double* vd, const double* tguess,
                                int64_t tg_stride, const double* p,
                                int64_t p_stride, double* S, int64_t lds,
                                double* T_out, double* J, const double* chi,
                                const double* chi0, const double* lb,
                                const int* sys, const int64_t* off,
                                const int* modes, const double* dt,
                                int64_t n, double tol, int maxit,
                                int* n_fail, int semantics,
                                pyro_stream_t stream);

/* Block Thomas over B systems whose off-diagonal blocks are L[i] I and
 * U[i] I (the Laplacian coupling), one wavefront per system; X (P, nv).
 * work holds P nv (nv + 1) doubles.  Replaces block_thomas
 * (flamelets/linear_solver.py:6-103) for the flamelet Jacobian. */
int pyro_flamelet_thomas(const double* L, const double* C, const double* U,
                         const double* R, double* X, const int64_t* off,
                         int64_t nsys, double* work, int* n_singular,
                         pyro_stream_t stream);

/* phi += X for points of systems with active[s] != 0 (active NULL = all),
 * for the same points tg = T_new when tg != NULL (the next temperature
 * guess), and, if norm2 != NULL, norm2[2s] = sum of X_s^2 over the
 * enthalpy row and norm2[2s+1] over the species rows, each with a fixed-order reduction (the
 * Newton update and its norm, solver.py:63-147). */
int pyro_flamelet_update(double* phi, int64_t ldp, const double* x,
                         const int* sys, const int* active,
                         const double* T_new, double* tg, const int64_t* off,
                         int64_t nsys, double* norm2, int64_t n,
                         pyro_stream_t stream);

/* Block Thomas as pyro_flamelet_thomas, with every system cut into
 * partitions [pstart[p], pend[p]) of system psys[p] (consecutive within a
 * system; those of system s are roff[s] + s .. roff[s+1] + s), each swept
 * from both ends by two sweeps (four sweeps per wavefront for nv <= 16;
 * above, by default for nv <= 63 a blocked Gauss-Jordan with FP64 MFMA
 * trailing updates on four wavefronts per sweep, else eight wavefronts
 * with one row per lane; eight wavefronts per system's recursion, its
 * products on MFMA by default),
 * and the unknowns at the partition interfaces found by an nv-sized block
 * recursion over each system's partitions (roff: interface offsets per
 * system, jbefore/jafter[p]: interface on either side of partition p or
 * -1).  Work arrays: fact P*nv*(2nv+1), maps nparts*2*nv*(2nv+1), red
 * nparts*nv*(2nv+2), Z nj*2nv doubles.  nv <= 64; returns -3 otherwise.
 * Same solution as block_thomas (flamelets/linear_solver.py:6-103) in a
 * different order of elimination. */
int pyro_flamelet_thomas_partitioned(
    const double* L, const double* C, const double* U, const double* R,
    double* X, const int64_t* off, int64_t nsys, const int64_t* pstart,
    const int64_t* pend, const int* psys, int64_t nparts,
    const int64_t* jbefore, const int64_t* jafter, const int64_t* roff,
    int64_t nj, double* fact, double* maps, double* red, double* Z,
    int* n_singular, pyro_stream_t stream);

/* Form of pyro_flamelet_thomas_partitioned for 16 < nv <= 63: 1 (default)
 * the blocked Gauss-Jordan sweep with FP64 MFMA trailing updates and the
 * interface recursion with its nv x nv products on MFMA, 0 the row-per-lane
 * eight-wavefront sweep and recursion; a negative form only queries.
 * Returns the previous form, or -3 where nv has a single form.  No
 * counterpart in the reference (a tuning switch of this solver). */
int pyro_flamelet_thomas_sweep_form(int form);

/* ---- transport -------------------------------------------------------
 * Exported by libraries of mechanisms whose species all carry transport
 * data.  The fits are polynomials in ln T (pyrometheus_amd.transport):
 * mu_k = sqrt(T) (sum a (ln T)^n)^2, lambda_k = sqrt(T) sum b (ln T)^n,
 * D_ij p = T^1.5 sum d (ln T)^n (chem_expr.py:190-243). */

/* which: 0 species viscosities, 1 species thermal conductivities (out
 * (ns, ld)), 2 binary mass diffusivities times p (out (ns, ns, ld)).
 * Replace get_species_viscosities, get_species_thermal_conductivities,
 * get_species_binary_mass_diffusivities (codegen/python.py:564-591). */
int pyro_species_transport(int which, const double* T, int64_t t_stride,
                           double* out, int64_t ld, int64_t n,
                           pyro_stream_t stream);

/* which: 0 mixture viscosity by Wilke's rule, 1 mixture conductivity
 * (out (n,)); 2 mixture-averaged species mass diffusivities at pressure p
 * (out (ns, ld)).  Replace get_mixture_viscosity_mixavg,
 * get_mixture_thermal_conductivity_mixavg and
 * get_species_mass_diffusivities_mixavg (codegen/python.py:593-641). */
int pyro_mixture_transport(int which, const double* p, int64_t p_stride,
                           const double* T, int64_t t_stride,
                           const double* Y, int64_t ldY, double* out,
                           int64_t ld, int64_t n, pyro_stream_t stream);

/* The fit coefficients compiled in, into HOST memory: which 0 viscosity
 * (ns, 5), 1 conductivity (ns, 5), 2 binary diffusivity (ns, ns, 5), in
 * ascending powers of ln T (Cantera's get_*_polynomial counterparts). */
int pyro_transport_fits(int which, double* out, int64_t n);

/* ---- compressible-EOS adjoint solves ---------------------------------
 * Exported by every mechanism library; batches as for the flamelet kernels.
 * Replace the pieces CompressibleEOS (flamelets/thermodynamic_consistency.py
 * :106-308) takes from FlameletEquations. */

/* rt[i] = R T of point i (R = R_u / W; local_compressible_eos_rt,
 * flamelets/equations.py:518-535) with T(h, Y) by Newton from tguess, and,
 * if rtj != NULL, its gradient d(RT)/dphi into rtj (nv, ldj) (the jacfwd of
 * it, equations.py:140-149).  semantics as for pyro_flamelet_source; a
 * point whose Newton did not converge gets NaN and counts in *n_fail. */
int pyro_flamelet_eos_rt(const double* phi, int64_t ldp, const double* tguess,
                         int64_t tg_stride, double* rt, double* rtj,
                         int64_t ldj, int64_t n, double tol, int maxit,
                         int* n_fail, int semantics, pyro_stream_t stream);

/* The adjoint operator (FlameletEquations.adjoint_operator, equations.py:
 * 451-516) in place of the source-Jacobian blocks J (P, nv, nv): interior
 * central blocks b_i I + 2 J_i^T / chi_i, identity rows at both ends of each
 * system, and the Laplacian's couplings as scalars L (row i+1 to x_i) and
 * U (row i to x_{i+1}), ready for pyro_flamelet_thomas[_partitioned]. */
int pyro_flamelet_adjoint_blocks(double* J, const double* chi,
                                 const double* la, const double* lb,
                                 const double* lc, const int* sys,
                                 const int64_t* off, double* L, double* U,
                                 int64_t n, pyro_stream_t stream);

#ifdef __cplusplus
}
#endif

#endif /* PYRO_HIP_H */
