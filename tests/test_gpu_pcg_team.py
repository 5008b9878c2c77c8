"""The PCG solve as one kernel on MI355X: its sums are formed in the order of
the two-kernel loop, so a Newton direction is the same bit for bit whichever
runs it.  A batch of more rows than one launch holds takes the two-kernel
loop, and so does any solve at profile level 3.  Which of the two ran is read
from a profile: one SpMV record and no update record for the one kernel."""
import threading

import numpy as np
import pytest

from idp_amd import driver, scenes

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)


def _scene(nx, ny, nz, seed=5):
    X, tets = scenes.kuhn_block(nx, ny, nz, 0.05)
    rng = np.random.default_rng(seed)
    X = X + rng.normal(0.0, 0.001, X.shape)
    side = 0.05 * min(nx, ny, nz)
    return scenes.Scene(f"bar{nx}x{ny}x{nz}", X, tets, scenes.sinusoid_target(X, side, 4, (0.2, 0.4), (0.5, 1.0), rng))


def _direction(d, sc, level, coarse=-1, X=None):
    """One Newton direction at a profile level; (gradient, direction, PCG
    iterations, one-kernel solves, launches of the update kernel seen)."""
    d.ctx.profile(level)
    g, s, r, it = d.ctx.newton_direction(sc.X if X is None else X, sc.target, sc.h, d.dHat2, d.kappa[0],
                                         pcg_rtol=1e-10, coarse_verts=coarse)
    p = d.ctx.profile_read()
    d.ctx.profile(0)
    assert r <= 1e-10
    return g, s, it, p["pcg_spmv"]["launches"], p["pcg_update"]["launches"]


# rows of the first instance: 8 (less than a wavefront's), 64 and 66 (one
# 64-row block, one and two rows more), 126 and 130 (one workgroup and the
# next), 195 (odd number of 64-row blocks, two workgroups)
@pytest.mark.parametrize("cells", [(1, 1, 1), (3, 3, 3), (10, 2, 1), (6, 5, 2), (12, 4, 1), (12, 4, 2)])
def test_one_kernel_equals_two_kernels(cells):
    sc = _scene(*cells)
    big = _scene(31, 31, 31, seed=6)  # 32,768 rows: the batch no longer fits one launch
    a, b = driver.BatchAnimFix([sc]), driver.BatchAnimFix([sc, big])
    try:
        say(f"[pcg team] {sc.X.shape[0]} rows alone, then beside {big.X.shape[0]}")
        for d in (a, b):
            d.ctx.profile(2)
            d.advance_one_time_step(max_newton=2)
        pa, pb = a.ctx.profile_read(), b.ctx.profile_read()
        assert pa["pcg_spmv"]["launches"] == 2 and pa["pcg_update"]["launches"] == 0
        assert pb["pcg_update"]["launches"] > 0
        Xa, va = a.state(0)
        Xb, vb = b.state(0)
        assert np.array_equal(Xa, Xb) and np.array_equal(va, vb)
    finally:
        a.close()
        b.close()


# 5, 22, 147 and 27 workgroups; 5, 48, 208 and 25 aggregates (the second more
# than two per workgroup, the last a sheet, whose thin direction is one voxel)
@pytest.mark.parametrize("cells,verts", [((20, 4, 4), 144), ((33, 9, 7), 100), ((64, 16, 16), 144), ((40, 40, 1), 144)])
def test_one_kernel_with_coarse_level(cells, verts):
    """The direction agrees with the one without a coarse level to the solves'
    residual, a second solve of the same system gives the same bits, and so do
    the kernels of the two-kernel loop."""
    sc = _scene(*cells)
    d = driver.TetAnimFix(sc)
    try:
        g0, s0, i0, n0, u0 = _direction(d, sc, 2)
        g1, s1, i1, n1, u1 = _direction(d, sc, 2, verts)
        g2, s2, i2, _, _ = _direction(d, sc, 2, verts)
        g3, s3, i3, _, u3 = _direction(d, sc, 3, verts)
        say(f"[pcg team] {sc.X.shape[0]} rows: {i0} iterations without the coarse level, {i1} with it")
        assert (n0, u0) == (n1, u1) == (1, 0) and u3 > 0
        assert np.array_equal(g0, g1) and np.array_equal(s1, s2) and i1 == i2
        assert np.array_equal(g1, g3) and np.array_equal(s1, s3) and i1 == i3
        # |error| <= cond |residual|: 1e-8 holds for systems of condition below 100
        assert np.linalg.norm(s1 - s0) <= 1e-8 * np.linalg.norm(s0)
    finally:
        d.close()


def _plates(nx, nz, n, gap, seed=4):
    """n plates of nx x 1 x nz cells, facing surfaces gap times the contact
    distance apart and shifted by a fraction of a cell, pressed together."""
    P, T = scenes.kuhn_block(nx, 1, nz, 0.05)
    rng = np.random.default_rng(seed)
    g = gap * 1e-3 * 0.05 * np.sqrt((nx + 1) ** 2 + n ** 2 + (nz + 1) ** 2)
    X = np.vstack([P + [rng.uniform(0.01, 0.04), k * (0.05 + g), rng.uniform(0.01, 0.04)] for k in range(n)])
    X[:, [0, 2]] += rng.normal(0.0, 1e-3, (X.shape[0], 2))
    X[:, 1] += rng.uniform(-0.1, 0.1, X.shape[0]) * g
    tets = np.vstack([T + k * P.shape[0] for k in range(n)]).astype(np.int32)
    return scenes.Scene("plates", X, tets, X * [1.0, 0.9, 1.0])


def _hub_ball(level):
    """A ball of one tet per triangle of an icosphere, all around its centre
    (vertex 0): one row coupled with every vertex."""
    X, tris = scenes.icosphere(level, 0.5)
    X = np.vstack([[0.0, 0.0, 0.0], X])
    rng = np.random.default_rng(2)
    X = X + rng.normal(0.0, 1e-4, X.shape)
    tets = np.hstack([np.zeros((tris.shape[0], 1), np.int32), tris + 1]).astype(np.int32)
    return scenes.Scene("ball", X, tets, X * [1.1, 0.95, 1.0])


@pytest.mark.parametrize("coarse", [-1, 144])
@pytest.mark.parametrize("make", [lambda: _plates(24, 21, 3, 0.5), lambda: _plates(30, 30, 2, 0.4),
                                  lambda: _hub_ball(3), lambda: _hub_ball(4)],
                         ids=["plates24x21x3", "plates30x30x2", "ball642", "ball2562"])
def test_long_rows_and_many_columns_equal_two_kernels(make, coarse):
    """Rows of more than the 16 blocks that a workgroup keeps in registers
    (contact; the centre of a ball) and workgroups of more than the 1,024
    columns that it stages."""
    sc = make()
    d = driver.TetAnimFix(sc)
    try:
        g0, s0, i0, n0, u0 = _direction(d, sc, 2, coarse)
        g1, s1, i1, _, u1 = _direction(d, sc, 3, coarse)
        rp, col, _ = d.ctx.get_bsr()
        longest = int(np.diff(rp).max())
        columns = max(np.unique(col[rp[a]:rp[min(a + 128, len(rp) - 1)]]).size for a in range(0, len(rp) - 1, 128))
        say(f"[pcg team] {sc.name}, {sc.X.shape[0]} rows: longest {longest} blocks, {columns} columns of 128 rows")
        assert longest > (16 if "plates" in sc.name else 512)
        if sc.X.shape[0] == 2563:
            assert columns > 1024
        assert (n0, u0) == (1, 0) and u1 > 0
        assert i0 == i1 and np.array_equal(g0, g1) and np.array_equal(s0, s1)
    finally:
        d.close()


def test_batch_of_many_small_meshes_in_one_kernel():
    """Instances of one workgroup each and of several, together and alone."""
    mix = [scenes.cube_sinusoid(n, seed=n) for n in (2, 4, 5, 3, 6, 8, 4, 2)]
    b = driver.BatchAnimFix(mix)
    its, _ = b.advance_one_time_step(max_newton=4)
    for i, sc in enumerate(mix):
        say(f"[pcg team] instance {i} alone ({sc.X.shape[0]} rows)")
        a = driver.BatchAnimFix([sc])
        ia, _ = a.advance_one_time_step(max_newton=4)
        assert ia[0] == its[i]
        Xa, va = a.state(0)
        Xm, vm = b.state(i)
        assert np.array_equal(Xa, Xm) and np.array_equal(va, vm)
        a.close()
    b.close()


def test_a_team_that_does_not_start_leaves_the_solve_to_the_two_kernels(monkeypatch):
    """With no patience at all (a negative number of polls) the workgroups leave
    and the solve runs in the two-kernel loop: same bits."""
    sc = _scene(20, 4, 4)

    def solve(cv):
        d = driver.TetAnimFix(sc)
        r = _direction(d, sc, 2, cv)
        d.close()
        return r

    for cv in (-1, 144):
        g0, s0, i0, _, u0 = solve(cv)
        monkeypatch.setenv("IDP_TEAM_WAIT", "-1")
        say(f"[pcg team] coarse {cv}: no wait for the team")
        g1, s1, i1, _, u1 = solve(cv)
        monkeypatch.delenv("IDP_TEAM_WAIT")
        assert u0 == 0 and u1 > 0
        assert i0 == i1 and np.array_equal(g0, g1) and np.array_equal(s0, s1)


def test_profiles_record_the_solve_that_runs():
    """Levels 1 and 2 record the one-kernel solve of a program that does not
    profile; level 3 runs the two kernels, which are then seen, with the same
    result."""
    sc = _scene(12, 4, 2)
    d = driver.TetAnimFix(sc)
    try:
        runs = {level: _direction(d, sc, level) for level in (1, 2, 3)}
        for level in (1, 2):
            assert runs[level][3:] == (1, 0), (level, runs[level][3:])
        assert runs[3][3] >= 1 and runs[3][4] >= 1
        for level in (2, 3):
            assert runs[level][2] == runs[1][2]
            assert np.array_equal(runs[level][0], runs[1][0]) and np.array_equal(runs[level][1], runs[1][1])
    finally:
        d.close()


def _served(scs, level, max_newton):
    """The scenes started together in one engine: (engine calls, finishing
    order with the call of each, states)."""
    b = driver.BatchAnimFix(scs)
    c = b.ctx
    try:
        c.profile(level)
        c.serve_configure(b.h, pcg_rtol=b.pcg_rtol, max_newton=max_newton)
        ids = list(range(len(scs)))
        c.serve_start(ids, [s.X for s in scs], [s.velocity for s in scs], b.tol[ids], b.dHat2[ids], b.kappa[ids])
        calls, order, left = 0, [], 1
        while left:
            left, fin = c.serve_iterate()
            calls += 1
            order += [(calls, int(i)) for i in np.nonzero(fin)[0]]
        return calls, order, [c.serve_result(i)[:2] for i in ids]
    finally:
        b.close()


def _rest(*cells):
    X, tets = scenes.kuhn_block(*cells, 0.05)
    return scenes.Scene("rest", X, tets, X.copy())


# solves that stop at once beside a long one; solves that stop at different
# looks; more instances, most of them long
HANDOVER = [
    ("stop_at_once", lambda: [_rest(2, 1, 1), _rest(3, 2, 2), scenes.bar_bend(20, 4, 4, 0.05, 0.15, 30.0)], 6),
    ("mix", lambda: [scenes.small_bend(), scenes.cube_sinusoid(4, seed=3), scenes.cube_sinusoid(5, seed=7),
                     scenes.bar_bend(20, 4, 4, 0.05, 0.15, 60.0)], 6),
    ("uneven", lambda: [_rest(1, 1, 1)] + [scenes.cube_sinusoid(n, seed=n) for n in (2, 3, 9, 4, 12, 5, 7)], 5),
]


@pytest.mark.parametrize("name,make,newton", HANDOVER, ids=[h[0] for h in HANDOVER])
def test_handover_points_are_those_of_the_two_kernels(name, make, newton):
    """When solves are handed over decides how many engine calls a batch takes
    and in which order frames finish: both equal the two-kernel loop's, and
    the results are the same bits."""
    scs = make()
    want = _served(scs, 3, newton)
    say(f"[pcg team] {name}: {want[0]} engine calls, finished {want[1]}")
    for _ in range(2):
        got = _served(scs, 0, newton)
        assert got[:2] == want[:2], (got[:2], want[:2])
        for (Xa, va), (Xb, vb) in zip(got[2], want[2]):
            assert np.array_equal(Xa, Xb) and np.array_equal(va, vb)


@pytest.mark.parametrize("contexts", [2, 3])
def test_contexts_on_threads_at_once_equal_alone(contexts):
    """Contexts whose teams do not fit the GPU together (253 and 147
    workgroups) step at the same time on threads of their own: whichever solves
    leave for the two-kernel loop, every context ends as it does alone."""
    scs = [scenes.bar_twist_fold(*dims, 0.05, seed=3, fold_radius=0.35 * dims[1] / 16)
           for dims in ((80, 20, 18), (64, 16, 16), (40, 9, 9))[:contexts]]

    def steps(d, sc, kappa, out):
        for _ in range(2):
            d.kappa[:] = kappa
            d.ctx.set_state(sc.X)
            d.set_target(sc.target)
            d.advance_one_time_step(max_newton=6)
            out.append(d.state())

    def run(together):
        ds = [driver.TetAnimFix(sc) for sc in scs]
        outs = [[] for _ in scs]
        th = [threading.Thread(target=steps, args=(d, sc, d.kappa.copy(), o)) for d, sc, o in zip(ds, scs, outs)]
        for t in th:
            t.start()
            if not together:
                t.join()
        for t in th:
            t.join()
        for d in ds:
            d.close()
        return outs

    say(f"[pcg team] {contexts} contexts at once")
    alone, both = run(False), run(True)
    for a, b in zip(alone, both):
        assert len(a) == len(b) == 2
        for (Xa, va), (Xb, vb) in zip(a, b):
            assert np.array_equal(Xa, Xb) and np.array_equal(va, vb)


def test_a_team_whose_wait_runs_out_starts_the_solve_again(monkeypatch):
    """With one poll per wait a started team gives up at a meet: the call does
    not fail, its solves run again in the two-kernel loop.  A direction starts
    from zero either way, so it is the same bits; a step loses its warm starts
    and ends where the oracle's tolerance says (1e-6 of the diagonal)."""
    def run(make):
        b = make()
        try:
            if isinstance(b, driver.TetAnimFix):
                return [_direction(b, b.scene, 2, cv) for cv in (-1, 144)]
            b.advance_one_time_step()
            return [b.state(i)[0] for i in range(len(b.scenes))]
        finally:
            b.close()

    def bar():
        return driver.TetAnimFix(_scene(33, 9, 7))

    batch = [scenes.small_bend(), scenes.cube_sinusoid(5, seed=7), scenes.small_bend(angle_deg=200.0)]

    def mix():
        return driver.BatchAnimFix(batch)

    want = [run(bar), run(mix)]
    monkeypatch.setenv("IDP_TEAM_SPIN", "1")
    say("[pcg team] one poll per wait")
    got = [run(bar), run(mix)]
    for (g0, s0, i0, _, upd0), (g1, s1, i1, _, upd1) in zip(want[0], got[0]):
        assert upd0 == 0 and upd1 > 0  # the one kernel without the limit, the two kernels with it
        assert i0 == i1 and np.array_equal(g0, g1) and np.array_equal(s0, s1)
    for sc, X0, X1 in zip(batch, want[1], got[1]):
        assert np.abs(X0 - X1).max() <= 1e-6 * sc.diag
