"""The coarse level of the one-mesh PCG preconditioner on MI355X (rigid-body
modes of voxel aggregates added to the cluster block Jacobi): the Newton
direction it gives is the one the solve without it gives, to the solves'
relative residual, in far fewer iterations, and Dirichlet rows of the
direction stay exactly zero (the aggregates leave those nodes out)."""
import numpy as np
import pytest

from idp_amd import capi, driver, scenes

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)


def test_coarse_level_gives_the_same_direction_in_fewer_iterations():
    sc = scenes.config2()
    d = driver.TetAnimFix(sc)
    try:
        Xt = sc.X + sc.h * sc.velocity  # x~ of the step
        # the Newton system after 200 iterations of the twist-and-fold step
        # (folded, in contact: the systems whose solves take thousands of
        # PCG iterations)
        say("[coarse] 64x16x16 bar: 200 Newton iterations")
        d.ctx.advance(sc.h, sc.newton_tol, d.dHat2, d.kappa, max_newton=200, coarse_verts=-1)
        X, _ = d.ctx.get_state()
        say("[coarse] its Newton system without and with the coarse level")
        g0, s0, rel0, it0 = d.ctx.newton_direction(X, Xt, sc.h, d.dHat2, d.kappa[0], pcg_rtol=1e-10,
                                                   coarse_verts=-1)
        g1, s1, rel1, it1 = d.ctx.newton_direction(X, Xt, sc.h, d.dHat2, d.kappa[0], pcg_rtol=1e-10,
                                                   coarse_verts=144)
        say(f"[coarse] PCG iterations {it0} -> {it1}")
        assert np.array_equal(g0, g1)
        assert rel0 <= 1e-10 and rel1 <= 1e-10
        assert np.linalg.norm(s1 - s0) <= 1e-8 * np.linalg.norm(s0)
        assert it1 < 0.6 * it0
    finally:
        d.close()


def test_coarse_level_keeps_dirichlet_rows_zero():
    sc = scenes.config1()  # 525 vertices: above the coarse level's size floor
    d = driver.TetAnimFix(sc)
    try:
        dbc = np.where(sc.X[:, 0] < 1e-9)[0].astype(np.int32)
        assert dbc.size > 0
        d.ctx.set_dbc(dbc)
        X = sc.X
        Xt = X + sc.h * sc.velocity
        say(f"[coarse] 20x4x4 bar with {dbc.size} Dirichlet nodes")
        g, s, rel, it = d.ctx.newton_direction(X, Xt, sc.h, d.dHat2, d.kappa[0], pcg_rtol=1e-10, coarse_verts=48)
        g0, s0, _, it0 = d.ctx.newton_direction(X, Xt, sc.h, d.dHat2, d.kappa[0], pcg_rtol=1e-10, coarse_verts=-1)
        s = s.reshape(-1, 3)
        assert np.all(s[dbc] == 0.0)
        assert np.linalg.norm(s.ravel() - s0) <= 1e-8 * np.linalg.norm(s0)
        say(f"[coarse] PCG iterations {it0} -> {it}")
    finally:
        d.close()


def test_coarse_level_is_deterministic_and_bounded_on_a_large_mesh():
    """The 160x48x48 crumple bar (384k vertices): the aggregates are capped in
    number (the dense A_c^-1 is read by every PCG iteration), and two solves
    of the same system give the same direction bit for bit."""
    sc = scenes.config5()
    d = driver.TetAnimFix(sc)
    try:
        X = sc.X
        Xt = X + 0.5 * sc.h * sc.velocity
        say("[coarse] 160x48x48 bar: two solves of its first Newton system")
        g0, s0, rel0, it0 = d.ctx.newton_direction(X, Xt, sc.h, d.dHat2, d.kappa[0], pcg_rtol=1e-8, coarse_verts=144)
        g1, s1, rel1, it1 = d.ctx.newton_direction(X, Xt, sc.h, d.dHat2, d.kappa[0], pcg_rtol=1e-8, coarse_verts=144)
        say(f"[coarse] PCG iterations {it0}, {it1}")
        assert np.array_equal(s0, s1) and it0 == it1
        assert rel0 <= 1e-8
    finally:
        d.close()


# orders of A_c of 48 (one tile of 64 rows), 108 and 162 (two and three tiles,
# both with a ragged end), 384 (six whole tiles), 750 and 1728
@pytest.mark.parametrize("contrast", [1.0, 1e8, 1e10])
@pytest.mark.parametrize("cells", [(1, 1, 1), (2, 2, 1), (2, 2, 2), (3, 3, 3), (4, 4, 4), (5, 5, 7)])
def test_coarse_inverse_is_exact_when_the_coarse_space_is_everything(cells, contrast):
    """With one vertex per aggregate the coarse space holds every vector, so
    z = (Z + A^-1) r and the preconditioned operator is Z A + I.  Every tet
    touches at most four clusters, so the eigenvalues of Z A lie in (0, 4] and
    those of Z A + I in (1, 5]: CG's error falls by 2 rho^k, rho = (sqrt 5 - 1)
    / (sqrt 5 + 1), and the residual by that times sqrt(cond A).  An inverse
    that is not A's breaks the bound; the cluster preconditioner by itself is
    far from it on these systems (a step of 1 s: stiffness over mass).  A
    contrast makes one tet in eight that much stiffer, which leaves stiff and
    soft directions at the same vertices, as a barrier does: the inverse keeps a
    Cholesky factorization's accuracy there."""
    X, tets = scenes.kuhn_block(*cells, 0.05)
    rng = np.random.default_rng(3)
    X = X + rng.normal(0.0, 5e-4, X.shape)
    Xt, h = X + rng.normal(0.0, 1e-2, X.shape), 1.0
    vol, IB, lam, mu, mass = capi.fem_init(X, tets, scenes.DENSITY, scenes.YOUNGS, scenes.POISSON)
    stiff = rng.uniform(size=tets.shape[0]) < 0.125
    dHat2, kappa = capi.initialize_oipc(1e-4, mass)
    with capi.Context(0) as ctx:
        ctx.set_mesh(X, tets, IB, vol, np.where(stiff, contrast * lam, lam), np.where(stiff, contrast * mu, mu), mass)

        def direction(cv):
            return ctx.newton_direction(X, Xt, h, dHat2, kappa[0], pcg_rtol=1e-10, coarse_verts=cv)

        g, s1, rel, it1 = direction(1)
        rp, col, val = ctx.get_bsr()
        n = len(rp) - 1
        A = np.zeros((n, 3, n, 3))
        for r in range(n):
            for k in range(rp[r], rp[r + 1]):
                A[r, :, col[k], :] += val[k]
        A = A.reshape(3 * n, 3 * n)
        # (the largest eigenvalue's rounding bounds how small the least one can be told from it)
        ev = np.linalg.eigvalsh(0.5 * (A + A.T))
        cond = ev[-1] / max(ev[0], 1e-15 * ev[-1])
        rho = (np.sqrt(5) - 1) / (np.sqrt(5) + 1)
        most = int(np.ceil(np.log(2 * np.sqrt(cond) / 1e-10) / -np.log(rho)))
        say(f"[coarse] {n} vertices, contrast {contrast:.0e}, condition {cond:.1e}: {it1} iterations, at most {most}")
        assert rel <= 1e-10 and it1 <= most
        if contrast == 1.0:
            _, _, _, it0 = direction(-1)
            say(f"[coarse] {it0} iterations without the coarse level")
            if n >= 27:
                assert it0 > 1.5 * most
            # |A s + g| <= 1e-10 |g| up to the residual's own rounding
            assert np.linalg.norm(A @ s1 + g) <= 2e-10 * np.linalg.norm(g) + 1e-15 * ev[-1] * np.linalg.norm(s1) * n
