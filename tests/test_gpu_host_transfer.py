"""Uploads and downloads through the pinned buffers: every value at its place,
bit for bit, for one short chunk, many chunks with a short last one, single
cells larger than usual, special values, and a transfer behind queued steps."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,n", [(1, (1, 1, 1)), (3, (2, 3, 5)), (2, (31, 30, 29)), (5, (11, 10, 9)), (9, (9, 8, 7))])
def test_grid_roundtrip(N, n):
    import exahype_amd as E
    g = E.Grid(E.ADERDGSolver(N), *n)
    a = np.random.default_rng(N).standard_normal(g.ncells * g.cell_size)
    a[:6] = (np.nan, np.inf, -np.inf, -0.0, 5e-324, 1e308)[:6]
    for k in range(2):  # the second transfer finds the buffers of the first
        g.upload(a + k)
        assert np.array_equal(g.download().view(np.int64), (a + k).view(np.int64))


@pytest.mark.parametrize("dim,P,n", [(2, 10, (7, 5, 1)), (3, 3, (4, 3, 2)), (3, 11, (5, 4, 4))])
def test_fv_roundtrip(dim, P, n):
    import exahype_amd as E
    s = E.FiniteVolumesSolver(dim, P, scheme=E.FV_GODUNOV if dim == 2 else E.FV_MUSCLHANCOCK)
    g = E.FVGrid(s, *n)
    a = np.random.default_rng(P).standard_normal(g.npatch * s.patch_size)
    g.upload(a)
    assert np.array_equal(g.download(), a)


def test_layout_and_order_behind_steps():
    """Device blocks are [v][node]: the initial conditions read back are the
    per-cell entry point's; a download waits for the steps before it."""
    import exahype_amd as E
    s = E.ADERDGSolver(4)
    ic = E.make_ic(5, xc=(0.4, 0.5, 0.6), L=0.05, amp=0.3, rho_inf=1.0, p_inf=1.0, uinf=(0.4, -0.3, 0.2))
    g = E.Grid(s, 12, 11, 10)
    g.set_initial_conditions(ic)
    cells = g.download().reshape(g.ncells, -1)
    dx = np.array([1 / 12, 1 / 11, 1 / 10])
    for c in (0, 13, g.ncells - 1):
        i = np.array([c % 12, c // 12 % 11, c // 132])
        assert np.array_equal(cells[c], s.adjustSolution((i + 0.5) * dx, dx, 0.0, ic))
    g.compute_dt()
    g.use_graph(True)
    g.step(20)
    a = g.download()
    g.sync()
    assert np.array_equal(a, g.download()) and not np.array_equal(a, cells.ravel())


def test_adaptive_grid_and_ensemble():
    import exahype_amd as E
    s = E.ADERDGSolver(3)
    g = E.AMRGrid(s, E.amr_config(3, 2, (0.5, 0.5, 0.5), 0.25, (0.1,)))
    a = np.tile(np.array((1.0, 0.1, -0.2, 0.3, 2.5)), g.ncells * 64)
    a *= 1 + 0.01 * np.random.default_rng(0).random(a.size)
    g.upload(a)
    assert np.array_equal(g.download(), a)
    ic = E.make_ic(5, xc=(0.4, 0.5, 0.6), L=0.05, amp=0.3, rho_inf=1.0, p_inf=1.0, uinf=(0.4, -0.3, 0.2))
    e = E.Ensemble([dict(order=n, cells=(4, 5, 3)) for n in (2, 4, 4)])
    e.set_initial_conditions([ic] * 3)
    for i, n in enumerate((2, 4, 4)):
        o = E.Grid(E.ADERDGSolver(n), 4, 5, 3)
        o.set_initial_conditions(ic)
        assert np.array_equal(e.download(i), o.download())


@pytest.mark.parametrize("dim,P,n", [(2, 10, (60, 50, 1)), (3, 11, (12, 11, 10))])
def test_upload_right_after_creation_of_a_patch_grid(dim, P, n):
    """A new grid's clearing is over when the grid is handed out: what is
    written first on its own stream stays, and a step from it finds the ghost
    layers of the other buffer cleared."""
    import exahype_amd as E
    s = E.FiniteVolumesSolver(dim, P, scheme=E.FV_GODUNOV if dim == 2 else E.FV_MUSCLHANCOCK)
    rng = np.random.default_rng(P)
    a = np.tile(np.array((1.0, 0.1, -0.2, 0.0 if dim == 2 else 0.3, 2.5)), int(np.prod(n)) * s.patch_size // 5)
    a *= 1 + 0.01 * rng.random(a.size)
    first = None
    for _ in range(4):
        g = E.FVGrid(s, *n)
        g.upload(a)
        assert np.array_equal(g.download(), a)
        g.compute_dt()
        g.step(1)
        b = g.download()
        first = b if first is None else first
        assert np.array_equal(b, first)
        ic = E.make_ic(5, xc=(0.4, 0.5, 0.6), L=0.05, amp=0.3, rho_inf=1.0, p_inf=1.0, uinf=(0.4, -0.3, 0.2))
        h = E.FVGrid(s, *n)
        h.set_initial_conditions(ic)
        h = h.download()
        g.set_initial_conditions(ic)  # cleared long ago
        side, gh = s.side, (s.side - P) // 2
        inner = (slice(None),) + (slice(gh, -gh),) * dim
        shape = (int(np.prod(n)),) + (side,) * dim + (5,)
        assert np.array_equal(h.reshape(shape)[inner], g.download().reshape(shape)[inner])


def test_upload_right_after_creation_of_an_adaptive_grid():
    """The clearing of the statuses and patch slots is over when the grid is
    handed out: the limiter's start, which the upload runs, is what a later
    upload of the same state finds."""
    import exahype_amd as E
    s = E.ADERDGSolver(3)
    cfg = E.amr_config(9, 3, (0.5, 0.5, 0.5), 0.25, (0.1, 0.05))
    g = E.AMRGrid(s, cfg)
    a = np.tile(np.array((1.0, 0.1, -0.2, 0.3, 2.5)), g.ncells * 64)
    a *= 1 + 0.01 * np.random.default_rng(0).random(a.size)
    level = g.cells()[:, 0]
    a.reshape(-1, 64, 5)[np.flatnonzero(level == level.max())[::997], 5, 0] = -0.1  # troubled cells
    del g
    for _ in range(4):
        g = E.AMRGrid(s, cfg)
        g.upload(a)
        first = g.limiter_status(), g.patches()
        E.device_synchronize()
        g.upload(a)
        again = g.limiter_status(), g.patches()
        assert np.array_equal(first[0], again[0]) and len(set(first[0])) > 1
        for p in (first, again):
            assert len(set(p[1][0])) == len(p[1][0]) and np.all(p[0][p[1][0]] != 0)
        assert set(first[1][0]) == set(again[1][0])


def _at_once(calls, rounds):
    """Runs the calls in a host thread each, over and over; what they returned."""
    got, gate = [[] for _ in calls], threading.Barrier(len(calls))

    def work(i):
        for _ in range(rounds):
            gate.wait(60)
            got[i].append(calls[i]())

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(calls))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    return got


def test_downloads_of_one_handle_at_once():
    """Host threads that read one object at the same time (the call releases
    the interpreter's lock): members of an ensemble whose buffers differ in
    size, and one grid, of several chunks each."""
    import exahype_amd as E
    ic = E.make_ic(5, xc=(0.4, 0.5, 0.6), L=0.05, amp=0.3, rho_inf=1.0, p_inf=1.0, uinf=(0.4, -0.3, 0.2))
    members = [dict(order=n, cells=c) for n, c in ((3, (9, 9, 9)), (5, (14, 13, 12)), (7, (9, 10, 11)), (5, (13, 14, 11)))]
    e = E.Ensemble(members)
    e.set_initial_conditions([ic] * 4)
    serial = [E.Ensemble([m]) for m in members]
    for s in serial:
        s.set_initial_conditions([ic])
    want = [s.download(0) for s in serial]
    # the ensemble's first transfers: its buffers grow while the others wait
    for got, w in zip(_at_once([lambda i=i: e.download(i) for i in range(4)], 6), want):
        assert all(np.array_equal(g, w) for g in got)
    g = E.Grid(E.ADERDGSolver(5), 14, 13, 12)
    g.set_initial_conditions(ic)
    for got in _at_once([g.download] * 3, 4):
        assert all(np.array_equal(x, want[1]) for x in got)


@pytest.mark.parametrize("up", [False, True])
def test_transfer_behind_steps_leaves_the_cores_idle(up):
    """A transfer that has to wait for queued steps sleeps meanwhile: the
    process may use the calling thread's core and one more, not one per thread
    that will share the copying."""
    import time
    import exahype_amd as E
    g = E.Grid(E.ADERDGSolver(5), 27, 27, 27)
    ic = E.make_ic(5, xc=(0.4, 0.5, 0.6), L=0.05, amp=0.3, rho_inf=1.0, p_inf=1.0, uinf=(0.4, -0.3, 0.2))
    g.set_initial_conditions(ic)
    a = g.download()
    g.compute_dt()
    g.use_graph(True)
    g.step(2)
    g.sync()
    g.step(500)
    t, c = time.perf_counter(), time.process_time()
    if up:
        g.upload(a)
    else:
        a = g.download()
    t, c = time.perf_counter() - t, time.process_time() - c
    assert t > 0.2  # it waited
    assert c < 2.5 * t
