"""The default Euler predictor (one space-time array per node, the first sweep
from one time level, the halves of Kxi) through the deferred per-cell entry
points and on grids: every order it serves, both precisions, one and several
FP64 sweeps, cells that stop after the first sweep, anisotropic cells, and the
agreement with the other contraction forms."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

TOL = 1e-12


def rel(a, b):
    a, b = np.asarray(a).reshape(-1, 5), np.asarray(b).reshape(-1, 5)
    scale = np.abs(b).max(axis=0)
    return (np.abs(a - b).max(axis=0) / np.maximum(scale, 1e-3 * scale.max())).max()


def _state(N, seed):
    """A smooth cell; seed None: a uniform one (the first sweep finds the fixed point)."""
    rng = np.random.default_rng(seed or 0)
    B = N + 1
    x = np.linspace(0, 1, B)
    z, y, x = np.meshgrid(x, x, x, indexing="ij")
    q = np.zeros((B, B, B, 5))
    amp = 0.0 if seed is None else 0.1
    for v, base in enumerate((1.0, 0.3, -0.2, 0.1, 2.5)):
        k = rng.uniform(0.5, 2, 3)
        q[..., v] = base + amp * np.sin(k[0] * x + k[1] * y + k[2] * z + rng.uniform(0, 6))
    return q.ravel()


@pytest.mark.parametrize("gravity", [None, 9.81])
@pytest.mark.parametrize("N", range(5, 10))
def test_staged_first_sweep_vs_oracle(N, gravity):
    """The staged form's one-slice first sweep: a cell that takes several, one
    that stops after it (its averages are then the first iterate's), and the
    gravity source, whose share of the slice carries a weight of its own."""
    import exahype_amd as E
    s = E.ADERDGSolver(N, contraction=E.CONTRACT_STAGED, gravity=gravity)
    c = O.cfg(N) if gravity is None else O.cfg(N, pde=3, grav=gravity)
    for seed, dx in ((1, np.array([1 / 27, 1 / 9, 1 / 20])), (None, np.array([0.1, 0.2, 0.3]))):
        luh = _state(N, seed)
        dt = 0.9 * O.stable_time_step_size(c, luh, dx)
        g, o = s.spaceTimePredictor(luh, dx, dt), O.space_time_predictor(c, luh, dx, dt)
        assert g["iters"] == o["iters"] and (seed is not None or gravity is not None or g["iters"] == 1)
        for k in ("lQi", "lQhi", "lFhi", "lQhbnd", "lFhbnd"):
            assert rel(g[k], o[k]) <= TOL, k


@pytest.mark.parametrize("sweeps", [1, 2, 3])
@pytest.mark.parametrize("N", [5, 8, 9])
def test_staged_mixed_outputs_match_the_debug_form(N, sweeps):
    """The staged mixed form keeps only the time average of a sweep known to be
    its last; the per-cell outputs keep the whole iterate.  Same sums in the
    same order: a few roundings (of fused products) apart, also where a
    uniform cell stops before the last sweep."""
    import exahype_amd as E
    B2, B3 = (N + 1) ** 2, (N + 1) ** 3
    s = E.ADERDGSolver(N, precision=E.PREC_FP32, contraction=E.CONTRACT_STAGED, fp64_sweeps=sweeps)
    dx = np.array([1 / 27, 1 / 9, 1 / 20])
    for seed in (1, None):
        luh = _state(N, seed)
        dt = 0.9 * O.stable_time_step_size(O.cfg(N), luh, dx)
        g = s.spaceTimePredictor(luh, dx, dt)
        o = (np.zeros(6 * B2 * 5), np.zeros(6 * B2 * 5), np.zeros(B3 * 5))
        s.batch_prediction(*o, luh, dx, dt)
        s.batch_flush()
        assert rel(o[0], g["lQhbnd"]) <= 1e-14 * (N + 1)
        assert rel(o[1], g["lFhbnd"]) <= 1e-14 * (N + 1)


@pytest.mark.parametrize("N", range(1, 9))
def test_deferred_predictions_vs_oracle(N):
    import exahype_amd as E
    B2, B3 = (N + 1) ** 2, (N + 1) ** 3
    s = E.ADERDGSolver(N)
    c = O.cfg(N)
    cells = [(_state(N, sd), np.array(dx), f) for sd, dx, f in
             ((1, (1 / 27, 1 / 27, 1 / 27), 0.9), (2, (1 / 9, 1 / 27, 1 / 40), 0.5), (None, (0.1, 0.2, 0.3), 0.9),
              (3, (1 / 27, 1 / 9, 1 / 20), 0.1), (4, (0.2, 0.2, 0.2), 0.9))]
    outs = []
    for luh, dx, f in cells:
        dt = f * O.stable_time_step_size(c, luh, dx)
        o = (np.zeros(6 * B2 * 5), np.zeros(6 * B2 * 5), np.zeros(B3 * 5))
        s.batch_prediction(*o, luh, dx, dt)
        outs.append((o, luh, dx, dt))
    s.batch_flush()
    for o, luh, dx, dt in outs:
        r = O.space_time_predictor(c, luh, dx, dt)
        assert rel(o[0], r["lQhbnd"]) <= TOL
        assert rel(o[1], r["lFhbnd"]) <= TOL
        # the volume integral cancels (zero for the uniform cell): its error against the fluxes it sums
        lduh = O.volume_integral(c, r["lFhi"], dx)
        scale = max(np.abs(lduh).max(), np.abs(r["lFhbnd"]).max() / dx.min())
        assert np.abs(o[2] - lduh).max() <= TOL * scale


@pytest.mark.parametrize("N", range(1, 9))
@pytest.mark.parametrize("precision,sweeps", [(0, 1), (1, 1), (1, 2)])
def test_grid_steps_and_sweep_counts(N, precision, sweeps):
    """A few steps on a grid with uniform and smooth regions against the
    oracle's grid; the FP64 sweep counts cell by cell."""
    import exahype_amd as E
    if E.autotune_recorded(N, precision) != (0, 0):
        pytest.skip("an earlier test's tuning has another form serve this order")
    n = (3, 4, 2)
    kw = dict(xc=(0.3, 0.4, 0.5), L=0.05, amp=0.3, rho_inf=1.0, p_inf=1.0, uinf=(0.4, -0.3, 0.2))
    c = O.cfg(N)
    og = O.OracleGrid(c, *n)
    og.init(O.make_ic(5, **kw))
    s = E.ADERDGSolver(N, precision=precision, fp64_sweeps=sweeps)
    g = E.Grid(s, *n)
    g.upload(og.luh().copy())
    dt = og.stable_dt()
    assert abs(g.compute_dt() - dt) <= 1e-14 * dt
    for _ in range(3):
        g.step(1)
        dt = og.step(dt)
        if precision == 0:
            assert np.array_equal(g.picard_iterations(), og.iters())
    # FP32 sweeps: the iterate's FP32 floor times the contraction of the FP64 sweeps
    assert rel(g.download(), og.luh()) <= (TOL if precision == 0 else 5e-6)


@pytest.mark.parametrize("N", [5, 7])
def test_adaptive_mesh_variant_equals_plain_on_smooth_cells(N):
    """The variant for meshes with uniform cells (FP32 sweeps): on a one-level
    mesh without uniform cells its steps are the plain variant's."""
    import exahype_amd as E
    rng = np.random.default_rng(2)
    ic = E.make_ic(0, xc=(0.5, 0.5, 0.5), L=0.1, eps=5.0, uinf=(1.0, 1.0, 0.0), rho_inf=1.0, p_inf=1.0, amp=1e-2,
                   nmodes=8, k=rng.integers(1, 3, size=(8, 3)).astype(float), a=rng.uniform(-1, 1, 8),
                   phi=rng.uniform(0, 6.28, 8))
    s = E.ADERDGSolver(N, precision=E.PREC_FP32)
    a = E.AMRGrid(s, E.amr_config(3, 1, (0.5, 0.5, 0.5), 0.25, (0.1,), relax=1e3))
    g = E.Grid(s, 3, 3, 3)
    for x in (a, g):
        x.set_initial_conditions(ic)
        x.compute_dt()
        x.step(2)
        x.sync()
    cells = a.cells()
    order = np.argsort((cells[:, 3] * 3 + cells[:, 2]) * 3 + cells[:, 1])
    ua = a.download().reshape(27, -1)[order].ravel()
    # the Riemann problems run in another kernel there: rounding only
    assert rel(ua, g.download()) <= TOL


@pytest.mark.parametrize("N,precision", [(3, 0), (5, 1)])
def test_what_the_autotuner_records_is_known_and_steps(N, precision):
    """The autotuner reports the fastest explicit variant and records it only
    if it beats the default: the record says which, and a grid left at the
    defaults steps with it as the oracle does."""
    import exahype_amd as E
    n = (3, 4, 2)
    w, c, ms = E.autotune(N, precision, 12)
    print(w, c, ms, E.autotune_recorded(N, precision))
    assert E.autotune_recorded(N, precision) in ((0, 0), (w, c))
    with pytest.raises(RuntimeError):
        E.autotune(N, precision, 3)
    assert E.autotune_recorded(N, precision) in ((0, 0), (w, c))  # an error leaves the record
    og = O.OracleGrid(O.cfg(N), *n)
    og.init(O.make_ic(5, xc=(0.3, 0.4, 0.5), L=0.05, amp=0.3, rho_inf=1.0, p_inf=1.0, uinf=(0.4, -0.3, 0.2)))
    g = E.Grid(E.ADERDGSolver(N, precision=precision), *n)
    g.upload(og.luh().copy())
    dt = og.stable_dt()
    g.compute_dt()
    for _ in range(2):
        g.step(1)
        dt = og.step(dt)
    assert rel(g.download(), og.luh()) <= (TOL if precision == 0 else 5e-6)
