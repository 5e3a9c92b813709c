"""The field solvers at the sizes where their kernels can go wrong: grids whose
node count is not a multiple of four, whose i-lines are shorter than a group
of four nodes, and grids with more groups of four than threads."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pg():
    import pic_gpu

    return pic_gpu


def _rho(shape, seed):
    rng = np.random.default_rng(seed)
    return 1e-9 * rng.normal(size=shape[0] * shape[1] * shape[2])


@pytest.mark.parametrize("shape", [(3, 3, 3), (5, 4, 3), (3, 3, 30), (7, 6, 5), (33, 17, 9), (103, 101, 103)])
@pytest.mark.parametrize("method,tol", [("SOLVER_PCG", 1e-10), ("SOLVER_PCG_MIXED", 1e-8)])
def test_pcg_residual_by_the_oracle(pg, shape, method, tol):
    L = [1e-2 * (n - 1) for n in shape]
    c = pg.Context(*shape, [0, 0, 0], L)
    c.dirichlet_walls()
    g = O.make_grid(*shape, [0, 0, 0], L)
    rho = _rho(shape, shape[0])
    c.set_field(pg.FIELD_RHO, rho)
    st = c.poisson(getattr(pg, method), tol=tol, tol_kind=pg.TOL_REL, max_it=5000)
    assert st["converged"], st
    r2, b2 = O.residual_dirichlet(g, c.get_field(pg.FIELD_PHI), rho)
    # the device sums the same rows in another order
    assert r2 / b2 <= 1.001 * tol
    c.close()


@pytest.mark.parametrize("shape", [(5, 6, 7), (18, 11, 13), (15, 13, 9)])
@pytest.mark.parametrize("method,tol", [("SOLVER_PCG", 1e-10), ("SOLVER_PCG_MIXED", 1e-8)])
def test_boltzmann_pcg_matches_oracle(pg, shape, method, tol):
    """Newton-Boltzmann on odd grids against the oracle's tight solve; J's
    smallest eigenvalue is at least the walls' pi^2 / L^2 sum and the start
    residual F is b, so a residual of tol leaves phi well within 1e3 tol."""
    L = [1e-2 * (n - 1) for n in shape]
    c = pg.Context(*shape, [0, 0, 0], L)
    c.dirichlet_walls()
    g = O.make_grid(*shape, [0, 0, 0], L)
    rho = np.full(O.nn(g), O.QE * 1.5e12)
    c.set_field(pg.FIELD_RHO, rho)
    st = c.poisson(getattr(pg, method), tol=tol, tol_kind=pg.TOL_REL, max_it=5000, n0=1e12, Te0=2.0)
    assert st["converged"], st
    _, nt = c.node_flags()
    tight, ok, *_ = O.nrpcg(g, np.zeros(O.nn(g), np.int32), nt, np.zeros(O.nn(g)), rho, 0.0, 1e12, 2.0, 5000, 1e-12,
                            axis_swap=False)
    phi = c.get_field(pg.FIELD_PHI)
    assert np.max(np.abs(phi - tight)) <= 1e3 * tol * np.max(np.abs(tight))
    c.close()


@pytest.mark.parametrize("shape", [(21, 18, 19), (40, 33, 29)])
@pytest.mark.parametrize("method,tol", [("SOLVER_PCG", 1e-10), ("SOLVER_PCG_MIXED", 1e-8)])
def test_boltzmann_pcg_with_neumann_sides_matches_oracle(pg, shape, method, tol):
    """An electrode plane and open sides: the PCG kernels that keep s = M g
    (M per row type) against the oracle's Newton-PCG on the same rows."""
    L = [1e-2 * (n - 1) for n in shape]
    rho = _rho(shape, 1) + 1.5e12 * O.QE
    c = pg.Context(*shape, [0, 0, 0], L)
    c.add_rectangle([L[0] / 2, L[1] / 2, 0], [1.1 * L[0], 1.1 * L[1], 0.15 * L[2]], 3.0)
    phi0 = c.get_field(pg.FIELD_PHI)
    oid, nt = c.node_flags()
    c.set_field(pg.FIELD_RHO, rho)
    st = c.poisson(getattr(pg, method), tol=tol, tol_kind=pg.TOL_REL, max_it=5000, n0=1e12, Te0=2.0)
    assert st["converged"], st
    g = O.make_grid(*shape, [0, 0, 0], L)
    tight, ok, *_ = O.nrpcg(g, oid, nt, phi0, rho, 0.0, 1e12, 2.0, 5000, 1e-11, axis_swap=False)
    phi = c.get_field(pg.FIELD_PHI)
    # the electrons' shift P bounds J's smallest eigenvalue from below
    assert np.max(np.abs(phi - tight)) <= 1e3 * tol * np.max(np.abs(tight))
    c.close()


SMALL, LINES, SQUARE = (32, 16, 12), (64, 16, 16), (32, 32, 16)  # nodes of the SOR tiles


def _sor_tile(shape, neumann):
    """the tile that the sweeps of a grid are made on (the solver's rule)"""
    def tiles(t):  # cores of t - 8 nodes, and four more at the ends
        return np.prod([next(m for m in range(1, 999) if (m - 1) * (e - 8) + e >= n) for n, e in zip(shape, t)])

    if tiles(SMALL) <= 400:
        return SMALL
    return LINES if neumann or tiles(LINES) < tiles(SQUARE) else SQUARE


@pytest.mark.parametrize("shape,tile,sides", [
    ((3, 3, 3), SMALL, "walls"), ((3, 3, 3), SMALL, "neumann"), ((4, 3, 5), SMALL, "walls"), ((4, 3, 5), SMALL, "neumann"),
    ((17, 16, 15), SMALL, "walls"), ((17, 16, 15), SMALL, "neumann"), ((31, 33, 32), SMALL, "walls"),
    ((31, 33, 32), SMALL, "neumann"), ((65, 41, 29), SMALL, "walls"), ((65, 41, 29), SMALL, "neumann"),
    ((70, 71, 72), SMALL, "walls"), ((70, 71, 72), SMALL, "neumann"), ((128, 30, 90), SMALL, "walls"),
    ((128, 30, 90), SMALL, "neumann"),
    ((100, 81, 67), SQUARE, "walls"), ((100, 81, 67), LINES, "neumann"), ((128, 65, 64), SQUARE, "walls"),
    ((128, 65, 64), LINES, "neumann"), ((33, 130, 140), SQUARE, "walls"), ((33, 130, 140), LINES, "neumann"),
    ((63, 64, 101), LINES, "walls"), ((63, 64, 101), LINES, "neumann"), ((61, 106, 51), LINES, "walls")])
@pytest.mark.parametrize("n0", [0.0, 1e10])
def test_tiled_sor_sweeps_equal_plain(pg, shape, tile, sides, n0):
    """The tiled sweeps against one launch per colour (PIC_SOLVE_SOR_PLAIN),
    bit for bit, after an odd and an even number of sweeps and with a check
    in between: grids smaller than a tile, with cores that end inside a node
    pair, and of several tiles of each of the three kinds, with ragged ends;
    objects on faces, edges and inside."""
    assert _sor_tile(shape, sides == "neumann") == tile
    L = [1e-2 * (n - 1) for n in shape]
    rng = np.random.default_rng(shape[0])
    rho = 1e-9 * rng.normal(size=shape[0] * shape[1] * shape[2])
    phi0 = 0.1 * rng.normal(size=rho.size)
    for max_it, check in ((1, 25), (2, 25), (25, 9)):
        out = []
        for flags in (0, pg.SOLVE_SOR_PLAIN):
            c = pg.Context(*shape, [0, 0, 0], L)
            if sides == "walls":
                c.dirichlet_walls()
            else:
                c.add_rectangle([L[0] / 2, L[1] / 2, 0], [0.7 * L[0], 1.1 * L[1], 0.3 * L[2]], 3.0)
                c.add_rectangle([0, 0.6 * L[1], 0.7 * L[2]], [0.6 * L[0], 0.3 * L[1], 0.4 * L[2]], -2.0)
            c.set_field(pg.FIELD_RHO, rho)
            c.set_field(pg.FIELD_PHI, phi0)
            st = c.poisson(pg.SOLVER_SOR_RB, tol=1e-300, tol_kind=pg.TOL_REL, max_it=max_it, omega=1.6,
                           check_every=check, n0=n0, Te0=2.0, flags=flags)
            assert st["iterations"] == max_it and not st["converged"]
            out.append((c.get_field(pg.FIELD_PHI), st["rel_residual"]))
            c.close()
        assert np.array_equal(out[0][0], out[1][0], equal_nan=True), max_it
        assert out[0][1] == pytest.approx(out[1][1], rel=1e-11, nan_ok=True)


@pytest.mark.parametrize("check", [2**31 - 1, 2**31 - 7, 31])
@pytest.mark.parametrize("flags", ["SOLVE_SOR_PLAIN", None])
def test_sor_check_interval_beyond_the_sweeps(pg, check, flags):
    """A check interval larger than max_it, up to INT_MAX (only the first sweep
    and the last are checked): all max_it sweeps are made, and the sweep
    count does not overflow."""
    shape = (17, 12, 9)
    L = [1e-2 * (n - 1) for n in shape]
    out = []
    for chk in (check, 1):
        c = pg.Context(*shape, [0, 0, 0], L)
        c.dirichlet_walls()
        c.set_field(pg.FIELD_RHO, _rho(shape, 2))
        st = c.poisson(pg.SOLVER_SOR_RB, tol=1e-300, tol_kind=pg.TOL_REL, max_it=31, omega=1.5, check_every=chk,
                       flags=getattr(pg, flags) if flags else 0)
        assert st["iterations"] == 31 and not st["converged"]
        out.append(c.get_field(pg.FIELD_PHI))
        c.close()
    assert np.array_equal(out[0], out[1])


def test_long_check_interval_costs_nothing_after_convergence(pg):
    """A SOR solve whose first sweep meets the criterion queues a few launches
    behind it and not the whole next interval, whose launches return at once
    but take 2 us each: 4000 sweeps' 4.5 ms against the solve's 45 us."""
    shape = (33, 30, 35)
    L = [1e-2 * (n - 1) for n in shape]
    c = pg.Context(*shape, [0, 0, 0], L)
    c.dirichlet_walls()
    c.set_field(pg.FIELD_RHO, _rho(shape, 4))
    kw = dict(method=pg.SOLVER_SOR_RB, tol=1e-5, tol_kind=pg.TOL_REL, max_it=20000, omega=1.83)
    assert c.poisson(**kw)["converged"]
    best = {}
    for check in (25, 4000) * 6:
        st = c.poisson(**dict(kw, check_every=check))
        assert st["converged"] and st["iterations"] == 1
        best[check] = min(best.get(check, 1.0), st["seconds"])
    assert best[4000] < 2 * best[25] + 2e-4, best
    c.close()


@pytest.mark.parametrize("shape", [(3, 3, 3), (3, 9, 5), (12, 3, 4), (5, 4, 3), (17, 11, 13)])
@pytest.mark.parametrize("objects", [0, 1, 3])
def test_row_types_of_open_boxes(pg, shape, objects):
    """The operator's row of every node (Dirichlet in objects and on flagged
    nodes; a Neumann face copies its neighbour along the first axis it is an end
    of; regular inside): a face node's value after one sweep is that of the node
    its row names, for boxes with open sides and objects on faces and edges."""
    L = np.array([1e-2 * (n - 1) for n in shape])
    c = pg.Context(*shape, [0, 0, 0], L)
    rng = np.random.default_rng(sum(shape) + objects)
    for q in range(objects):
        c.add_rectangle([L, 0 * L, 0.5 * L][q], 0.6 * L, float(q + 1))
    rho = 1e-9 * rng.normal(size=int(np.prod(shape)))
    c.set_field(pg.FIELD_RHO, rho)
    oid, _ = c.node_flags()
    phi0 = c.get_field(pg.FIELD_PHI)
    phi0[oid == 0] = rng.normal(size=int(np.sum(oid == 0)))
    c.set_field(pg.FIELD_PHI, phi0)
    c.poisson(pg.SOLVER_SOR_RB, tol=1e-300, tol_kind=pg.TOL_REL, max_it=1, omega=1.3)
    phi = c.get_field(pg.FIELD_PHI).reshape(shape[::-1])
    oid = oid.reshape(shape[::-1])
    old = phi0.reshape(shape[::-1])
    n = shape[::-1]  # index order k, j, i
    for k in range(n[0]):
        for j in range(n[1]):
            for i in range(n[2]):
                at = [k, j, i]
                if oid[k, j, i] > 0:
                    assert phi[k, j, i] == old[k, j, i]
                    continue
                axis = next((d for d in (2, 1, 0) if at[d] in (0, n[d] - 1)), None)
                if axis is not None:
                    at[axis] += 1 if at[axis] == 0 else -1
                    assert phi[k, j, i] == phi[tuple(at)], (k, j, i)
                else:
                    assert phi[k, j, i] != old[k, j, i]
    c.close()


@pytest.mark.parametrize("shape", [(3, 3, 3), (5, 3, 4), (9, 8, 7), (3, 12, 6)])
def test_dirichlet_walls_flag_every_face_node(pg, shape):
    L = [1e-2 * (n - 1) for n in shape]
    c = pg.Context(*shape, [0, 0, 0], L)
    before = c.node_flags()[1].reshape(shape[::-1])
    c.dirichlet_walls()
    after = c.node_flags()[1].reshape(shape[::-1])
    face = np.ones(shape[::-1], bool)
    face[1:-1, 1:-1, 1:-1] = False
    assert np.all(before[face] == 1) and np.all(after[face] == 2)
    assert np.all(before[~face] == 0) and np.all(after[~face] == 0)
    c.close()
