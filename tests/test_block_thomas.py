"""Block-Thomas: the oracle against dense solves (CPU) and the batched HIP
kernel against the oracle (GPU).  Tolerance: relative 1e-12 on well-
conditioned systems (block-diagonally dominant or pivoting-stressed)."""
import numpy as np
import pytest

from oracle.flamelet_np import assemble_dense, block_thomas


def _system(rng, n, nv, dominant=True, pivot_stress=False):
    L = rng.normal(size=(max(n - 1, 0), nv, nv))
    U = rng.normal(size=(max(n - 1, 0), nv, nv))
    C = rng.normal(size=(n, nv, nv))
    if dominant:
        C += 4 * nv * np.eye(nv)
    if pivot_stress:
        # zero diagonal entries: elimination without row exchanges fails
        for i in range(n):
            C[i][np.arange(nv), np.arange(nv)] = 0.0
            C[i] += 4 * nv * np.roll(np.eye(nv), 1, axis=1)
    r = rng.normal(size=(n, nv))
    return L, C, U, r


@pytest.mark.parametrize("nv", [1, 3, 10])
def test_oracle_matches_dense_solve(nv):
    rng = np.random.default_rng(nv)
    for n in (1, 2, 9):
        L, C, U, r = _system(rng, n, nv)
        x = block_thomas(L, C, U, r)
        A = assemble_dense(L, C, U) if n > 1 else C[0]
        xd = np.linalg.solve(A, r.ravel())
        assert np.max(np.abs(x.ravel() - xd)) < 1e-12 * np.max(np.abs(xd))


def test_oracle_scalar_thomas():
    """nv = 1 reduces to the textbook Thomas algorithm."""
    rng = np.random.default_rng(0)
    n = 12
    a, c = rng.uniform(-1, 1, n - 1), rng.uniform(-1, 1, n - 1)
    b = rng.uniform(3, 4, n)
    d = rng.normal(size=n)
    cp, dp = np.zeros(n), np.zeros(n)
    cp[0], dp[0] = c[0] / b[0], d[0] / b[0]
    for i in range(1, n):
        m = b[i] - a[i - 1] * cp[i - 1]
        cp[i] = c[i] / m if i < n - 1 else 0.0
        dp[i] = (d[i] - a[i - 1] * dp[i - 1]) / m
    x = np.zeros(n)
    x[-1] = dp[-1]
    for i in range(n - 2, -1, -1):
        x[i] = dp[i] - cp[i] * x[i + 1]
    got = block_thomas(a.reshape(-1, 1, 1), b.reshape(-1, 1, 1),
                       c.reshape(-1, 1, 1), d.reshape(-1, 1))
    assert np.max(np.abs(got[:, 0] - x)) < 1e-14


@pytest.mark.gpu
@pytest.mark.parametrize("nv", [1, 2, 5, 9, 10, 16, 20, 54])
@pytest.mark.parametrize("diag", [False, True])
def test_gpu_batched_ragged(nv, diag, device):
    import torch
    from pyrometheus_amd.flamelets.linear_solver import block_thomas_batched
    rng = np.random.default_rng(100 + nv)
    sizes = [1, 2, 3, 17, 64, 5]
    systems = []
    for j, n in enumerate(sizes):
        L, C, U, r = _system(rng, n, nv, pivot_stress=(j % 2 == 1 and nv > 1))
        if diag:
            lv, uv = rng.normal(size=max(n - 1, 0)), rng.normal(size=max(n - 1, 0))
            L = lv[:, None, None] * np.eye(nv)
            U = uv[:, None, None] * np.eye(nv)
        systems.append((L, C, U, r))
    offs = np.concatenate([[0], np.cumsum(sizes)])
    P = offs[-1]
    if diag:
        Lb, Ub = np.zeros(P), np.zeros(P)
    else:
        Lb, Ub = np.zeros((P, nv, nv)), np.zeros((P, nv, nv))
    Cb, Rb = np.zeros((P, nv, nv)), np.zeros((P, nv))
    for (L, C, U, r), o, n in zip(systems, offs, sizes):
        Cb[o:o + n], Rb[o:o + n] = C, r
        if n > 1:
            if diag:
                Lb[o:o + n - 1], Ub[o:o + n - 1] = L[:, 0, 0], U[:, 0, 0]
            else:
                Lb[o:o + n - 1], Ub[o:o + n - 1] = L, U
    t = lambda a: torch.tensor(a, dtype=torch.float64, device=device)
    x = block_thomas_batched(t(Lb), t(Cb), t(Ub), t(Rb),
                             torch.tensor(offs, device=device), diag=diag,
                             check_singular=True).cpu().numpy()
    for (L, C, U, r), o, n in zip(systems, offs, sizes):
        ref = block_thomas(L, C, U, r)
        err = np.max(np.abs(x[o:o + n] - ref)) / np.max(np.abs(ref))
        assert err < 1e-12, (n, err)


@pytest.mark.gpu
@pytest.mark.parametrize("nv", [3, 10, 54])
def test_gpu_singular_block_reported(nv, device):
    """A system whose first central block is zero meets a zero pivot: with
    check_singular the batched solve raises; the same batch without the
    zero block solves to the oracle."""
    import torch
    from pyrometheus_amd.flamelets.linear_solver import block_thomas_batched
    rng = np.random.default_rng(7 + nv)
    sizes = [4, 6]
    offs = np.concatenate([[0], np.cumsum(sizes)])
    P = offs[-1]
    Lb, Ub = np.zeros(P), np.zeros(P)
    Cb, Rb = np.zeros((P, nv, nv)), np.zeros((P, nv))
    refs = []
    for o, n in zip(offs, sizes):
        L, C, U, r = _system(rng, n, nv)
        lv, uv = 0.1 * rng.normal(size=n - 1), 0.1 * rng.normal(size=n - 1)
        Lb[o:o + n - 1], Ub[o:o + n - 1] = lv, uv
        Cb[o:o + n], Rb[o:o + n] = C, r
        refs.append(block_thomas(lv[:, None, None] * np.eye(nv), C,
                                 uv[:, None, None] * np.eye(nv), r))
    t = lambda a: torch.tensor(a, dtype=torch.float64, device=device)
    offs_t = torch.tensor(offs, device=device)
    x = block_thomas_batched(t(Lb), t(Cb), t(Ub), t(Rb), offs_t, diag=True,
                             check_singular=True).cpu().numpy()
    for ref, o, n in zip(refs, offs, sizes):
        assert np.max(np.abs(x[o:o + n] - ref)) <= 1e-12 * np.max(np.abs(ref))
    Cs = Cb.copy()
    Cs[offs[1]] = 0.0
    with pytest.raises(RuntimeError, match="singular"):
        block_thomas_batched(t(Lb), t(Cs), t(Ub), t(Rb), offs_t, diag=True,
                             check_singular=True)


@pytest.mark.gpu
def test_gpu_drop_in_signature(device):
    import torch
    from pyrometheus_amd.flamelets.linear_solver import block_thomas as bt
    rng = np.random.default_rng(5)
    L, C, U, r = _system(rng, 33, 10)
    t = lambda a: torch.tensor(a, dtype=torch.float64, device=device)
    x = bt(t(L), t(C), t(U), t(r)).cpu().numpy()
    assert np.max(np.abs(x - block_thomas(L, C, U, r))) < 1e-12 * np.max(np.abs(x))


@pytest.mark.gpu
@pytest.mark.parametrize("diag", [False, True])
def test_gpu_badly_scaled_rows(diag, device):
    """Rows scaled by factors from 1e-8 to 1e8, as in the flamelet Jacobian
    whose enthalpy row is in J/kg.  Dense couplings: the row-scaled system
    has the solution of the unscaled one, to 1e-12.  Scalar couplings (which
    cannot carry a row scale): badly scaled central blocks, against the
    oracle on the same system, to 1e-10."""
    import torch
    from pyrometheus_amd.flamelets.linear_solver import block_thomas_batched
    rng = np.random.default_rng(77)
    nv, n = 10, 40
    L, C, U, r = _system(rng, n, nv, pivot_stress=True)
    d = 10.0 ** rng.uniform(-8, 8, size=(n, nv))
    t = lambda a: torch.tensor(a, dtype=torch.float64, device=device)
    offs = torch.tensor([0, n], device=device)
    if diag:
        lv, uv = rng.normal(size=n - 1), rng.normal(size=n - 1)
        L = lv[:, None, None] * np.eye(nv)
        U = uv[:, None, None] * np.eye(nv)
        Cs = C * d[:, :, None]
        ref = block_thomas(L, Cs, U, r)
        x = block_thomas_batched(t(np.append(lv, 0.0)), t(Cs),
                                 t(np.append(uv, 0.0)), t(r), offs,
                                 diag=True).cpu().numpy()
        tol = 1e-10
    else:
        ref = block_thomas(L, C, U, r)
        Lf, Uf = np.zeros((n, nv, nv)), np.zeros((n, nv, nv))
        Lf[:n - 1] = L * d[1:, :, None]
        Uf[:n - 1] = U * d[:-1, :, None]
        x = block_thomas_batched(t(Lf), t(C * d[:, :, None]), t(Uf),
                                 t(r * d), offs, diag=False).cpu().numpy()
        tol = 1e-12
    err = np.max(np.abs(x - ref)) / np.max(np.abs(ref))
    assert err < tol, err


@pytest.mark.gpu
@pytest.mark.parametrize("mech,part_len,sweep", [
    ("sandiego", None, "mfma"), ("sandiego", 2, "mfma"),
    ("sandiego", 3, "mfma"), ("sandiego", 8, "mfma"),
    ("gri30", None, "mfma"), ("gri30", 5, "mfma"), ("gri30", 2, "mfma"),
    ("gri30", None, "rowlane"), ("gri30", 5, "rowlane")])
def test_gpu_partitioned_matches_oracle(mech, part_len, sweep, device):
    """The partitioned flamelet block Thomas (partitions swept from both
    ends, the nv-sized recursion for the interface unknowns, recovery)
    against the oracle on ragged systems with scalar couplings, and against
    the one-wavefront kernel: nv = 10 (four sweeps per wavefront) and
    nv = 54 with both sweep forms (blocked Gauss-Jordan with MFMA trailing
    updates, and one row per lane)."""
    import torch
    from pyrometheus_amd import bundled, get_thermochem_class
    from pyrometheus_amd.flamelets.engine import FlameletBatch
    gas = get_thermochem_class(bundled(mech))(device=device)
    nv = gas.num_species + 1
    sizes = ([3, 4, 17, 64, 250, 1000, 5] if nv <= 16
             else [3, 4, 17, 40, 90, 5])
    rng = np.random.default_rng(19)
    grids = [np.linspace(0, 1, n) for n in sizes]
    y = np.zeros(nv - 1)
    y[-1] = 1.0
    bp = FlameletBatch(gas, grids, y, y, thomas="partitioned",
                       part_len=part_len)
    if bp.has_sweep_forms():
        bp.set_thomas("partitioned", None, part_len, sweep=sweep)
    bs = FlameletBatch(gas, grids, y, y, thomas="sequential")
    assert bp.partitioned and not bs.partitioned
    P = sum(sizes)
    Lb, Ub = np.zeros(P), np.zeros(P)
    Cb, Rb = np.zeros((P, nv, nv)), np.zeros((P, nv))
    systems, o = [], 0
    for j, n in enumerate(sizes):
        _, C, _, r = _system(rng, n, nv, pivot_stress=(j % 2 == 1))
        lv, uv = rng.normal(size=n - 1), rng.normal(size=n - 1)
        Lb[o:o + n - 1], Ub[o:o + n - 1] = lv, uv
        Cb[o:o + n], Rb[o:o + n] = C, r
        systems.append((lv[:, None, None] * np.eye(nv), C,
                        uv[:, None, None] * np.eye(nv), r, o, n))
        o += n
    t = lambda a: torch.tensor(a, dtype=torch.float64, device=device)
    print(f"[partitioned] {mech} part_len={part_len} sweep={sweep}",
          flush=True)
    try:
        for b in (bp, bs):
            b.L.copy_(t(Lb))
            b.U.copy_(t(Ub))
            b.J.copy_(t(Cb))
            b.rhs.copy_(t(Rb))
            b.thomas()
        xp, xs = bp.x.cpu().numpy(), bs.x.cpu().numpy()
    finally:
        if bp.has_sweep_forms():   # the library-wide default again
            bp.set_thomas("partitioned", None, part_len, sweep="mfma")
    for L, C, U, r, o, n in systems:
        ref = block_thomas(L, C, U, r)
        sc = np.max(np.abs(ref))
        assert np.max(np.abs(xp[o:o + n] - ref)) <= 1e-12 * sc, n
        assert np.max(np.abs(xp[o:o + n] - xs[o:o + n])) <= 1e-12 * sc, n


@pytest.mark.gpu
@pytest.mark.parametrize("mech", ["uiuc", "sandiego", "hong", "gri30"])
@pytest.mark.parametrize("weight", [0.0, 0.05, 0.3])
def test_gpu_partitioned_exchanges_rows(mech, weight, device):
    """The partitioned solve where pivots lie in arbitrary rows: each central
    block is 4 nv (Q + weight I) + N(0, 1) with Q a random pairing of the
    rows, so that a block needs exchanges all over (weight 0 and 0.05) or
    keeps a diagonal within the pivot threshold of the largest entry (0.3).
    The blocks' condition is at most about 2; tolerance 1e-12 of the
    solution's largest entry as for the other well-conditioned systems."""
    import torch
    from pyrometheus_amd import bundled, get_thermochem_class
    from pyrometheus_amd.flamelets.engine import FlameletBatch
    gas = get_thermochem_class(bundled(mech))(device=device)
    nv = gas.num_species + 1
    sizes = [3, 9, 41, 33]
    rng = np.random.default_rng(nv)
    y = np.zeros(nv - 1)
    y[-1] = 1.0
    b = FlameletBatch(gas, [np.linspace(0, 1, n) for n in sizes], y, y,
                      thomas="partitioned", part_len=4)
    P = sum(sizes)
    lv, uv = rng.normal(size=P), rng.normal(size=P)
    C, r = rng.normal(size=(P, nv, nv)), rng.normal(size=(P, nv))
    for i in range(P):
        pairs = rng.permutation(nv)[:nv - nv % 2].reshape(-1, 2)
        Q = np.eye(nv)
        Q[pairs[:, 0]], Q[pairs[:, 1]] = (np.eye(nv)[pairs[:, 1]],
                                          np.eye(nv)[pairs[:, 0]])
        C[i] += 4 * nv * (Q + weight * np.eye(nv))
    t = lambda a: torch.tensor(a, dtype=torch.float64, device=device)
    print(f"[exchanges] {mech} weight={weight}", flush=True)
    b.L.copy_(t(lv))
    b.U.copy_(t(uv))
    b.J.copy_(t(C))
    b.rhs.copy_(t(r))
    b.thomas()
    x, o = b.x.cpu().numpy(), 0
    for n in sizes:
        s, k = slice(o, o + n), slice(o, o + n - 1)
        want = block_thomas(lv[k, None, None] * np.eye(nv), C[s],
                            uv[k, None, None] * np.eye(nv), r[s])
        assert np.max(np.abs(x[s] - want)) <= 1e-12 * np.max(np.abs(want)), n
        o += n


@pytest.mark.gpu
def test_gpu_autotuner_schedule(device):
    """The block-Thomas autotuner times the sequential schedule and the
    partitioned one per alpha on a synthetic batch, keeps the fastest for the
    block size, and batches built afterwards use it."""
    from pyrometheus_amd import bundled, get_thermochem_class
    from pyrometheus_amd.flamelets import autotune
    from pyrometheus_amd.flamelets.engine import FlameletBatch
    gas = get_thermochem_class(bundled("sandiego"))(device=device)
    y = np.zeros(gas.num_species)
    y[-1] = 1.0
    try:
        res = autotune.tune_thomas(gas, sizes=[17, 40, 97, 300, 1000],
                                   reps=2)
        assert res["kind"] in ("sequential", "partitioned")
        assert len(res["ms"]) == 1 + len(autotune.ALPHAS)
        assert res["sweep"] == "mfma"   # nv = 10 has one sweep form
        assert all(t > 0.0 for t in res["ms"].values())
        best = min(res["ms"].values())
        name = (res["kind"] if res["kind"] == "sequential"
                else f"partitioned alpha={res['alpha']:.3g}")
        assert res["ms"][name] == best
        sch = autotune.schedule(10, device)
        assert sch["kind"] == res["kind"]
        b = FlameletBatch(gas, [np.linspace(0, 1, n) for n in (30, 200)],
                          y, y)
        assert b.partitioned == (res["kind"] == "partitioned")
    finally:
        autotune.reset()
    assert autotune.schedule(10, device) == autotune.DEFAULT


@pytest.mark.parametrize("part_len,alpha", [(None, None), (2, None),
                                            (8, None), (None, 0.5),
                                            (None, 3.0)])
def test_partition_table_properties(part_len, alpha):
    """Partitions cover every system contiguously in order, lengths within
    a system differ by at most one row, and the interface tables agree:
    interface j of a system lies between its partitions q and q+1."""
    from pyrometheus_amd.flamelets.engine import partition_table
    rng = np.random.default_rng(5)
    sizes = [3, 4, 17, 64, 250, 1000, 5] + list(rng.integers(3, 2049, 40))
    ps, pe, psys, jpart, jb, ja, roff = partition_table(sizes, part_len,
                                                        alpha)
    offs = np.concatenate([[0], np.cumsum(sizes)])
    assert len(roff) == len(sizes) + 1 and roff[0] == 0
    for s, n in enumerate(sizes):
        parts = np.nonzero(psys == s)[0]
        assert parts[0] == roff[s] + s and parts[-1] == roff[s + 1] + s
        assert ps[parts[0]] == offs[s] and pe[parts[-1]] == offs[s + 1]
        assert np.array_equal(ps[parts[1:]], pe[parts[:-1]])
        lens = pe[parts] - ps[parts]
        assert lens.min() >= 1 and lens.max() - lens.min() <= 1
        if part_len is None:
            a = np.sqrt(2.0) if alpha is None else alpha
            m = max(8, int(round(a * np.sqrt(n))))
            assert len(parts) == max(1, -(-n // m))
        nj = len(parts) - 1
        assert roff[s + 1] - roff[s] == nj
        for q, p in enumerate(parts):
            assert jb[p] == (roff[s] + q - 1 if q > 0 else -1)
            assert ja[p] == (roff[s] + q if q < nj else -1)
        assert np.array_equal(jpart[roff[s]:roff[s + 1]], parts[:-1])
