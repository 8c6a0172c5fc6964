"""The work this framework is used for, as measurable cases.

Each case is one call (or one forward and backward pass) through a public
entry point, on float64 state resident in HBM, the only type the framework
takes.  The mechanisms are the two that the benchmark and the server use:
sandiego (9 species, 24 reactions) and GRI-3.0 (53 species, 325 reactions).
Cell states are drawn like the benchmark's: T uniform in [300, 2500] K, p
log-uniform in [0.5, 20] atm, Y half Dirichlet(0.5) and half N2.  Flamelets
are the benchmark's H2:N2 / air flames: grids clustered about the
stoichiometric mixture fraction, dissipation rate log-uniform in [1, 1000]
1/s.

``exact`` evaluates the same formulas with plain torch operations in 64 bits
(and torch's autograd for the derivatives), from the mechanism's numbers
alone.
"""

import math

import numpy as np
import torch

from pyrometheus_amd import bundled, get_thermochem_class
from pyrometheus_amd.adjoint import (net_production_rates, source_jacobian,
                                     wdot_jvp)
from pyrometheus_amd.flamelets.engine import FlameletBatch
from pyrometheus_amd.flamelets.solver import solve_batch
from pyrometheus_amd.flamelets.workload import make_problem, streams
from pyrometheus_amd.flops import wdot_flops
from pyrometheus_amd.mechanism import GAS_CONSTANT, ONE_ATM

_F64 = torch.float64
_DEV = "cuda"


def listed():
    return [
        # a served production-rate request of the smallest kind: latency
        {"name": "wdot_sandiego_small", "op": "wdot", "mech": "sandiego",
         "cells": 4096},
        # one CFD block of ordinary, ragged size
        {"name": "wdot_gri30_mid", "op": "wdot", "mech": "gri30",
         "cells": 100003},
        # the headline benchmark: a whole domain on one GPU
        {"name": "wdot_gri30_large", "op": "wdot", "mech": "gri30",
         "cells": 1 << 24},
        # T recovery from the conserved energy, once per time step
        {"name": "temperature_gri30", "op": "temperature", "mech": "gri30",
         "cells": 1000003, "energy": True},
        # omega-dot and its reverse pass under torch autograd
        {"name": "backward_gri30", "op": "backward", "mech": "gri30",
         "cells": 262144},
        # omega-dot and its forward-mode product (matrix-free implicit step)
        {"name": "jvp_gri30", "op": "jvp", "mech": "gri30", "cells": 200001},
        # the full source Jacobian, one block per cell (implicit chemistry)
        {"name": "jacobian_gri30", "op": "jacobian", "mech": "gri30",
         "cells": 65536, "layout": "cell"},
        # per-reaction net rates (reaction-path analysis)
        {"name": "progress_gri30", "op": "progress", "mech": "gri30",
         "cells": 262144, "what": "net"},
        # the mixture-averaged transport properties of one CFD step
        {"name": "transport_gri30", "op": "transport", "mech": "gri30",
         "cells": 262144},
        # one implicit update of the benchmark's batch of 256 flamelets
        {"name": "newton_sandiego_batch", "op": "newton", "mech": "sandiego",
         "flamelets": 256, "n_min": 64, "n_max": 1024},
        # one implicit update of a served batch of 53-species flamelets
        {"name": "newton_gri30_batch", "op": "newton", "mech": "gri30",
         "flamelets": 16, "n_min": 64, "n_max": 512},
        # a whole batched solve: equilibration, time march, Newton
        {"name": "solve_sandiego", "op": "solve", "mech": "sandiego",
         "flamelets": 48, "n_min": 64, "n_max": 512},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["wdot", "wdot", "temperature", "backward", "jvp",
                     "jacobian", "progress", "transport", "newton", "newton",
                     "solve"])
    mech = rng.choice(["sandiego", "gri30"])
    big = mech == "gri30"
    case = {"op": op, "mech": mech}
    if op == "wdot":
        case["cells"] = _log_int(rng, 1000, 1 << 24)
    elif op == "temperature":
        case["cells"] = _log_int(rng, 1000, 1 << 22)
        case["energy"] = rng.random() < 0.5
    elif op in ("backward", "jvp", "transport"):
        case["cells"] = _log_int(rng, 1000, 1 << 20)
    elif op == "jacobian":
        case["cells"] = _log_int(rng, 1000, 1 << (18 if big else 20))
        case["layout"] = rng.choice(["cell", "entry"])
    elif op == "progress":
        case["cells"] = _log_int(rng, 1000, 1 << (19 if big else 20))
        case["what"] = rng.choice(["kf", "net"])
    elif op == "newton":
        case["flamelets"] = _log_int(rng, 1, 16 if big else 256)
        case["n_min"] = rng.randint(64, 256)
        case["n_max"] = rng.randint(256, 512 if big else 1024)
    else:
        case["mech"] = "sandiego"
        case["flamelets"] = _log_int(rng, 8, 64)
        case["n_min"] = rng.randint(64, 256)
        case["n_max"] = rng.randint(256, 512)
    return case


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
_GAS = {}


def _gas(name):
    if name not in _GAS:
        _GAS[name] = get_thermochem_class(bundled(name))(device=_DEV)
    return _GAS[name]


def _rand(g, *shape):
    return torch.rand(shape, generator=g, dtype=_F64, device=_DEV)


def _cells(mech, n, g):
    """T, p, Y of n cells, and rho = p W / (R T)."""
    T = 300.0 + 2200.0 * _rand(g, n)
    p = ONE_ATM * torch.exp(math.log(0.5) + math.log(40.0) * _rand(g, n))
    ns = mech.n_species
    Y = torch._standard_gamma(torch.full((ns, n), 0.5, dtype=_F64,
                                         device=_DEV), generator=g)
    Y /= Y.sum(0, keepdim=True)
    Y *= 0.5
    Y[mech.species_index("N2")] += 0.5
    inv_w = torch.tensor(1.0 / mech.molecular_weights, dtype=_F64,
                         device=_DEV)
    return T, p, Y, p / (GAS_CONSTANT * T * (inv_w @ Y))


def _sizes(case):
    return [int(round(x)) for x in np.linspace(case["n_min"], case["n_max"],
                                               case["flamelets"])]


def _problems(case, gas, seed):
    rng = np.random.default_rng(seed)
    st = streams(gas, t_ox=800.0, t_fu=300.0)
    chis = np.exp(rng.uniform(0.0, math.log(1000.0), case["flamelets"]))
    return [make_problem(gas, st, n, float(c))[1]
            for n, c in zip(_sizes(case), chis)], rng


def _flamelets(case, gas, seed):
    """A batch in the middle of its time march: burnt profiles disturbed by
    a smooth per-flamelet composition, a Crank-Nicolson step of 1e-5 s."""
    probs, rng = _problems(case, gas, seed)
    ns = gas.num_species
    for q in probs:
        d = rng.dirichlet(0.5 * np.ones(ns))[:, None]
        q.phi[1:] += 0.08 * q.x * (1.0 - q.x) * (d - q.phi[1:])
    cat = lambda rows: torch.tensor(np.concatenate(rows, axis=-1), dtype=_F64,
                                    device=_DEV)
    b = FlameletBatch(gas, [q.x for q in probs],
                      np.stack([q.y_ox for q in probs]),
                      np.stack([q.y_fu for q in probs]), device=_DEV)
    b.set_boundary_enthalpy([q.h_ox for q in probs], [q.h_fu for q in probs])
    s = {"batch": b, "phi": cat([q.phi for q in probs]),
         "chi": cat([q.chi for q in probs]),
         "tg": cat([q.t_guess for q in probs]),
         "p": cat([np.full(len(q.x), q.pressure) for q in probs])}
    s["vd"] = torch.zeros_like(s["chi"])
    b.modes.fill_(1)
    b.dt.fill_(1e-5)
    s["phi_prev"] = s["phi"].clone()
    s["r_prev"] = b.residual(s["phi"], s["chi"], s["vd"], s["tg"], s["p"],
                             torch.empty_like(s["phi"]))
    return s


def prepare(case, seed):
    gas = _gas(case["mech"])
    mech, op = gas._mech, case["op"]
    state = {"op": op, "gas": gas}
    if op == "newton":
        return dict(state, **_flamelets(case, gas, seed))
    if op == "solve":
        return dict(state, problems=_problems(case, gas, seed)[0])
    n, ns = case["cells"], mech.n_species
    g = torch.Generator(device=_DEV).manual_seed(seed)
    T, p, Y, rho = _cells(mech, n, g)
    state.update(T=T, p=p, Y=Y, rho=rho)
    if op == "temperature":
        state["energy"] = case["energy"]
        state["target"] = (gas.get_mixture_internal_energy_mass(T, Y)
                           if case["energy"] else
                           gas.get_mixture_enthalpy_mass(T, Y))
        state["guess"] = (T + 600.0 * (_rand(g, n) - 0.5)).clamp(200.0,
                                                                 3500.0)
    elif op == "backward":
        for k in ("rho", "T", "Y"):
            state[k] = state[k].requires_grad_()
        state["wbar"] = torch.randn((ns, n), generator=g, dtype=_F64,
                                    device=_DEV)
    elif op == "jvp":
        state["v"] = (rho * (_rand(g, n) - 0.5), 200.0 * (_rand(g, n) - 0.5),
                      Y * (_rand(g, ns, n) - 0.5))
    elif op == "jacobian":
        state["layout"] = case["layout"]
    elif op == "progress":
        state["what"] = case["what"]
        state["C"] = rho * Y / torch.tensor(mech.molecular_weights,
                                            dtype=_F64, device=_DEV)[:, None]
    return state


def run(s):
    op, gas = s["op"], s["gas"]
    if op == "wdot":
        return gas.get_net_production_rates(s["rho"], s["T"], s["Y"])
    if op == "temperature":
        return gas.get_temperature(s["target"], s["guess"], s["Y"],
                                   s["energy"])
    if op == "backward":
        x = (s["rho"], s["T"], s["Y"])
        w = net_production_rates(gas, *x)
        return w.detach(), torch.autograd.grad(w, x, s["wbar"])
    if op == "jvp":
        return wdot_jvp(gas, s["rho"], s["T"], s["Y"], *s["v"])
    if op == "jacobian":
        return source_jacobian(gas, s["T"], s["p"], s["Y"],
                               layout=s["layout"])
    if op == "progress":
        if s["what"] == "kf":
            return gas.get_fwd_rate_coefficients(s["T"], s["C"])
        return gas.get_net_rates_of_progress(s["T"], s["C"])
    if op == "transport":
        T, Y = s["T"], s["Y"]
        return (gas.get_mixture_viscosity_mixavg(T, Y),
                gas.get_mixture_thermal_conductivity_mixavg(T, Y),
                gas.get_species_mass_diffusivities_mixavg(s["p"], T, Y))
    if op == "newton":
        return s["batch"].newton_update(
            s["phi"], s["chi"], s["vd"], s["tg"], s["p"], s["batch"].modes,
            s["phi_prev"], s["r_prev"], apply=False)
    res = solve_batch(gas, s["problems"], equilibrate_steps=24)
    return {"h": torch.cat([r.state.enthalpy for r in res]),
            "Y": torch.cat([r.state.mass_fractions for r in res], dim=1),
            "T": torch.cat([r.temperature for r in res])}


def work(case):
    mech = bundled(case["mech"])
    f = wdot_flops(mech)
    ns, nr, w = mech.n_species, mech.n_reactions, f["flop_per_cell"]
    nv, op = ns + 1, case["op"]
    if op in ("newton", "solve"):
        pts = sum(_sizes(case))
        # phi, phi_n, R_n, the update; T guess, chi, p, stencil
        by = 8 * (4 * nv + 7)
        # rates and their derivatives, then one block row of block Thomas
        # with scalar couplings
        fl = 3 * w + 2 * nv * nv + 4.67 * nv ** 3 + 8 * nv * nv
        if op == "solve":  # the benchmark's flamelets take 137 updates
            fl *= 137
        return {"bytes": by * pts, "flops": fl * pts}
    per = {
        "wdot": (8 * (2 * ns + 2), w),
        "temperature": (8 * (ns + 3), 12 * ns + 120),
        "backward": (8 * (5 * ns + 6), 3 * w),
        "jvp": (8 * (4 * ns + 4), 2 * w),
        "jacobian": (8 * (nv * nv + ns + 2), 3 * w + 4 * nv * nv),
        "progress": (8 * (ns + 1 + nr),
                     20 * (nr + f["nf"] + 6 * f["n_troe"])
                     if case.get("what") == "kf" else w),
        "transport": (8 * (2 * ns + 4), 26 * ns * ns + 40 * ns),
    }[op]
    return {"bytes": per[0] * case["cells"], "flops": per[1] * case["cells"]}


# ---------------------------------------------------------------------------
# the same formulas in plain torch
# ---------------------------------------------------------------------------
class _Plain:
    """NASA-7 thermodynamics, kinetics and mixture-averaged transport of one
    mechanism as whole-array torch expressions."""

    def __init__(self, name):
        m = self.mech = bundled(name)
        t = lambda a: torch.tensor(np.asarray(a, dtype=float), dtype=_F64,
                                   device=_DEV)
        self.ns, self.nr = m.n_species, m.n_reactions
        self.W = t(m.molecular_weights)[:, None]
        self.lo = t([s.low for s in m.species]).T[:, :, None]
        self.hi = t([s.high for s in m.species]).T[:, :, None]
        self.tmid = t([s.t_mid for s in m.species])[:, None]
        ix = m.species_index
        nu_r = np.zeros((self.nr, self.ns))
        nu_p = np.zeros((self.nr, self.ns))
        # the species of each side, repeated by its coefficient; the index
        # ns stands for a factor of one
        sides = np.full((2, self.nr, 3), self.ns)
        for i, r in enumerate(m.reactions):
            for nu, side, terms in ((nu_r, 0, r.reactants),
                                    (nu_p, 1, r.products)):
                names = []
                for sp, c in terms:
                    nu[i, ix(sp)] += c
                    names += [ix(sp)] * int(c)
                sides[side, i, :len(names)] = names
        self.sides = torch.tensor(sides, device=_DEV)
        self.nu_r, self.nu_p = t(nu_r), t(nu_p)
        self.dnu = t((nu_p - nu_r).sum(1))[:, None]
        self.rev = t([float(r.reversible) for r in m.reactions])[:, None]
        main = [r.high_rate if r.is_falloff else r.rate for r in m.reactions]
        self.fall = [i for i, r in enumerate(m.reactions) if r.is_falloff]
        low = [m.reactions[i].low_rate for i in self.fall]
        arr = lambda rs: tuple(t(v)[:, None] for v in (
            [math.log(a.A) for a in rs], [a.b for a in rs],
            [a.Ea / GAS_CONSTANT for a in rs]))
        self.main, self.low = arr(main), arr(low)
        eff = lambda r: [dict(r.efficiencies).get(s, r.default_efficiency)
                         for s in m.species_names]
        self.body = [i for i, r in enumerate(m.reactions)
                     if r.kind == "three-body"]
        self.eff_b = t([eff(m.reactions[i]) for i in self.body])
        self.eff_f = t([eff(m.reactions[i]) for i in self.fall])

    def _nasa(self, T, f):
        return torch.where(T > self.tmid, f(self.hi), f(self.lo))

    def cp_r(self, T):
        return self._nasa(T, lambda a: a[0] + T * (a[1] + T * (
            a[2] + T * (a[3] + T * a[4]))))

    def h_rt(self, T):
        return self._nasa(T, lambda a: a[0] + T * (a[1] / 2 + T * (
            a[2] / 3 + T * (a[3] / 4 + T * a[4] / 5))) + a[5] / T)

    def s_r(self, T):
        return self._nasa(T, lambda a: a[0] * torch.log(T) + T * (
            a[1] + T * (a[2] / 2 + T * (a[3] / 3 + T * a[4] / 4))) + a[6])

    @staticmethod
    def _arrhenius(p, T):
        return torch.exp(p[0] + p[1] * torch.log(T) - p[2] / T)

    def kf(self, T, C):
        k = self._arrhenius(self.main, T)
        scale = torch.ones_like(k)
        if self.body:
            scale = scale.index_copy(0, torch.tensor(self.body, device=_DEV),
                                     self.eff_b @ C)
        if self.fall:
            idx = torch.tensor(self.fall, device=_DEV)
            pr = (self.eff_f @ C) * self._arrhenius(self.low, T) / k[idx]
            rows = []
            for j, i in enumerate(self.fall):
                r, x = self.mech.reactions[i], pr[j]
                f = x / (1 + x)
                if r.falloff_type == "Troe":
                    q = r.troe
                    fc = ((1 - q[0]) * torch.exp(-T / q[1])
                          + q[0] * torch.exp(-T / q[2]))
                    if len(q) > 3:
                        fc = fc + torch.exp(-q[3] / T)
                    fc = torch.log10(fc)
                    u = torch.log10(x) - 0.4 - 0.67 * fc
                    v = 0.75 - 1.27 * fc - 0.14 * u
                    f = f * 10.0 ** (fc / (1 + (u / v) ** 2))
                rows.append(f)
            scale = scale.index_copy(0, idx, torch.stack(rows))
        return k * scale

    def progress(self, T, C):
        one = torch.cat([C, torch.ones_like(C[:1])])
        prod = lambda s: one[s[:, 0]] * one[s[:, 1]] * one[s[:, 2]]
        g = self.h_rt(T) - self.s_r(T)
        nlk = (self.nu_p - self.nu_r) @ g - self.dnu * torch.log(
            ONE_ATM / (GAS_CONSTANT * T))
        return self.kf(T, C) * (prod(self.sides[0]) - self.rev
                                * torch.exp(nlk) * prod(self.sides[1]))

    def wdot(self, rho, T, Y):
        return (self.nu_p - self.nu_r).T @ self.progress(T, rho * Y / self.W)

    def cp(self, T, Y):
        return GAS_CONSTANT * (self.cp_r(T) * Y / self.W).sum(0)

    def h(self, T, Y, shift=0.0):
        return GAS_CONSTANT * T * ((self.h_rt(T) - shift) * Y
                                   / self.W).sum(0)

    def temperature(self, target, T, Y, energy):
        """Newton from the guess T, each cell until its step is at rounding
        level."""
        shift = 1.0 if energy else 0.0
        inv = GAS_CONSTANT * (Y / self.W).sum(0)
        for _ in range(60):
            d = (target - self.h(T, Y, shift)) / (self.cp(T, Y) - shift * inv)
            T = T + d
            if float(d.abs().max()) < 1e-10:
                break
        return T

    def source(self, h, Y, T0, p):
        """W_k omega_k / rho at (h, Y); T0 is the temperature there, and the
        one Newton step taken from it carries T's derivative."""
        T = T0 + (h - self.h(T0, Y)) / self.cp(T0, Y).detach()
        rho = p / (GAS_CONSTANT * T * (Y / self.W).sum(0))
        return self.W * self.wdot(rho, T, Y) / rho

    def source_jacobian(self, T0, p, Y):
        """dS/d[h; Y] per cell, (n, nv, nv): row 0 is zero without viscous
        dissipation."""
        n, nv = T0.numel(), self.ns + 1
        J = torch.zeros((n, nv, nv), dtype=_F64, device=_DEV)
        h = self.h(T0, Y).detach().requires_grad_()
        Y = Y.detach().clone().requires_grad_()
        S = self.source(h, Y, T0, p)
        for k in range(self.ns):
            gh, gy = torch.autograd.grad(S[k].sum(), (h, Y),
                                         retain_graph=True)
            J[:, k + 1, 0] = gh
            J[:, k + 1, 1:] = gy.T
        return S.detach(), J

    def transport(self, fits, p, T, Y):
        visc, cond, diff = (torch.tensor(f, dtype=_F64, device=_DEV)
                            for f in fits)
        lt = torch.log(T)
        poly = lambda c: c[..., 0, None] + lt * (c[..., 1, None] + lt * (
            c[..., 2, None] + lt * (c[..., 3, None] + lt * c[..., 4, None])))
        mmw = 1.0 / (Y / self.W).sum(0)
        X = Y * mmw / self.W
        rt = torch.sqrt(T)
        mu, lam = rt * poly(visc) ** 2, rt * poly(cond)
        eta = torch.zeros_like(T)
        D = torch.empty_like(Y)
        for k in range(self.ns):
            wk = self.W[k]
            phi = (1 + torch.sqrt(mu[k] / mu * torch.sqrt(self.W / wk))) ** 2 \
                / torch.sqrt(8 * (1 + wk / self.W))
            eta = eta + X[k] * mu[k] / (X * phi).sum(0)
            dk = rt * T * poly(diff[k])
            x = X / dk
            x[k] = 0.0
            D[k] = (mmw - X[k] * wk) / (p * mmw * x.sum(0))
        lam = 0.5 * ((X * lam).sum(0) + 1.0 / (X / lam).sum(0))
        return eta, lam, D


def _by_chunks(f, arrays, chunk, dim=-1):
    """f on chunks of the arrays' last axis, the results joined."""
    n = arrays[0].shape[-1]
    parts = [f(*(a[..., i:i + chunk] for a in arrays))
             for i in range(0, n, chunk)]
    if isinstance(parts[0], tuple):
        return tuple(torch.cat(q, dim=dim) for q in zip(*parts))
    return torch.cat(parts, dim=dim)


def _newton_exact(plain, s):
    """The Crank-Nicolson update by a plain sequential block elimination,
    all flamelets of the batch side by side."""
    b, phi = s["batch"], s["phi"]
    nv, off, sizes = plain.ns + 1, b.offsets_np, b.sizes
    T = plain.temperature(phi[0], s["tg"], phi[1:], False)
    S, J = [], []
    for i in range(0, b.P, 16384):
        sl = slice(i, i + 16384)
        a, c = plain.source_jacobian(T[sl], s["p"][sl], phi[1:, sl])
        S.append(a)
        J.append(c)
    S = torch.cat([torch.zeros((1, b.P), dtype=_F64, device=_DEV),
                   torch.cat(S, 1)])
    J = torch.cat(J)
    ends = torch.zeros(b.P, dtype=torch.bool, device=_DEV)
    ends[torch.as_tensor(off[:-1], device=_DEV)] = True
    ends[torch.as_tensor(off[1:] - 1, device=_DEV)] = True
    zero = torch.zeros_like(b.la)
    la, lc = torch.where(ends, zero, b.la), torch.where(ends, zero, b.lc)
    lap = la * (torch.roll(phi, 1, 1) - phi) + lc * (torch.roll(phi, -1, 1)
                                                     - phi)
    lap = torch.where(ends, b.lb * phi, lap)
    hc = 0.5 * s["chi"]
    R = hc * lap + torch.where(ends, zero, S)
    for side, at in ((0, off[:-1]), (1, off[1:] - 1)):
        R[:, torch.as_tensor(at, device=_DEV)] -= b.bc[:, side].T
    eye = torch.eye(nv, dtype=_F64, device=_DEV)
    J = torch.where(ends[:, None, None], torch.zeros_like(J), J)
    J = J + (hc * b.lb)[:, None, None] * eye
    hdt = 0.5e-5
    rhs = -(phi - s["phi_prev"] - hdt * (R + s["r_prev"])).T
    J = eye - hdt * J
    lower, upper = -hdt * hc * la, -hdt * hc * lc
    # one padded system per flamelet: identity rows past its end
    m, nmax = len(sizes), max(sizes)
    pos = torch.zeros((m, nmax), dtype=torch.int64, device=_DEV)
    live = torch.zeros((m, nmax), dtype=torch.bool, device=_DEV)
    for j, n in enumerate(sizes):
        pos[j, :n] = torch.arange(int(off[j]), int(off[j + 1]), device=_DEV)
        live[j, :n] = True
    G = torch.empty((nmax, m, nv, nv + 1), dtype=_F64, device=_DEV)
    for i in range(nmax):
        q, on = pos[:, i], live[:, i]
        A = torch.where(on[:, None, None], J[q], eye)
        r = torch.where(on[:, None], rhs[q], torch.zeros_like(rhs[q]))
        if i:
            lo = torch.where(on, lower[q], torch.zeros_like(lower[q]))
            A = A - lo[:, None, None] * G[i - 1, :, :, :nv]
            r = r - lo[:, None] * G[i - 1, :, :, nv]
        up = torch.where(on, upper[q], torch.zeros_like(upper[q]))
        G[i] = torch.linalg.solve(A, torch.cat(
            [up[:, None, None] * eye.expand(m, nv, nv), r[:, :, None]], 2))
    x = torch.empty((b.P, nv), dtype=_F64, device=_DEV)
    nxt = torch.zeros((m, nv), dtype=_F64, device=_DEV)
    for i in range(nmax - 1, -1, -1):
        nxt = G[i, :, :, nv] - (G[i, :, :, :nv] * nxt[:, None, :]).sum(2)
        x[pos[:, i][live[:, i]]] = nxt[live[:, i]]
    norm = torch.stack([torch.stack(((v[:, 0] ** 2).sum(),
                                     (v[:, 1:] ** 2).sum()))
                        for v in torch.split(x, sizes)])
    return norm, x


def exact(case, seed):
    op = case["op"]
    if op == "solve":  # minutes of plain iterations
        return None
    s = prepare(case, seed)
    plain = _Plain(case["mech"])
    if op == "newton":
        return _newton_exact(plain, s)
    T, p, Y, rho = s["T"], s["p"], s["Y"], s["rho"]
    if op == "wdot":
        return _by_chunks(plain.wdot, (rho, T, Y), 1 << 18)
    if op == "temperature":
        return _by_chunks(lambda e, g, y: plain.temperature(
            e, g, y, case["energy"]), (s["target"], s["guess"], Y), 1 << 18)
    if op == "backward":
        def back(r, t, y, b):
            x = tuple(a.detach().clone().requires_grad_() for a in (r, t, y))
            w = plain.wdot(*x)
            return (w.detach(),) + torch.autograd.grad(w, x, b)
        w, gr, gt, gy = _by_chunks(back, (rho.detach(), T.detach(),
                                          Y.detach(), s["wbar"]), 1 << 16)
        return w, (gr, gt, gy)
    if op == "jvp":
        def push(r, t, y, *v):
            # the product as the derivative of a reverse pass that is linear
            # in its cotangent
            x = tuple(a.detach().clone().requires_grad_() for a in (r, t, y))
            w = plain.wdot(*x)
            z = torch.zeros_like(w, requires_grad=True)
            g = torch.autograd.grad(w, x, z, create_graph=True)
            dw = torch.autograd.grad(sum((a * c).sum() for a, c in
                                         zip(g, v)), z)[0]
            return w.detach(), dw
        return _by_chunks(push, (rho, T, Y) + tuple(s["v"]), 1 << 15)
    if op == "jacobian":
        J = torch.cat([plain.source_jacobian(T[i:i + 16384], p[i:i + 16384],
                                             Y[:, i:i + 16384])[1]
                       for i in range(0, T.numel(), 16384)])
        return J if case["layout"] == "cell" else J.permute(
            1, 2, 0).contiguous()
    if op == "progress":
        f = plain.kf if case["what"] == "kf" else plain.progress
        return _by_chunks(f, (T, s["C"]), 1 << 18)
    fits = s["gas"].get_transport_fits()
    return _by_chunks(lambda a, t, y: plain.transport(fits, a, t, y),
                      (p, T, Y), 1 << 18)
