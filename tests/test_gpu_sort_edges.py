"""Sorts and counts of species in the states where pic_sort chooses its path:
births appended behind a sorted part, nothing appended, removed particles
still in the arrays."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ME, QE, AMU, KB = 9.10938215e-31, 1.602176565e-19, 1.660538921e-27, 1.380648e-23


@pytest.fixture(scope="module")
def pg():
    import pic_gpu

    return pic_gpu


def _rows(p):
    p = np.asarray(p).reshape(-1, 7)
    return p[np.lexsort(p.T)]


def _cells(p, dx, n):
    c = np.floor(p.reshape(-1, 7)[:, :3] / dx + 1e-9).astype(np.int64)
    return (c[:, 2] * (n[1] - 1) + c[:, 1]) * (n[0] - 1) + c[:, 0]


def _gas(pg, table, dt, n_neu, n_ele, E_ion=12.07 * QE):
    n, dx = (20, 18, 33), 1e-4
    L = dx * (np.array(n) - 1)
    box = 0.98 * L
    vol = float(np.prod(box))
    n_gas = 10.0 / (KB * 300.0)
    w_n = n_gas * vol / n_neu
    c = pg.Context(*n, [0, 0, 0], L)
    c.set_dt(dt)
    sn = c.species_add(32 * AMU, 0.0, w_n, 2 * n_neu)
    si = c.species_add(32 * AMU, QE, w_n / 1000, n_ele + 200000)
    se = c.species_add(ME, -QE, w_n / 1000, n_ele + 200000)
    c.load_box_thermal(sn, 0.5 * L, box, n_gas, 300.0, seed=3, mode=0)
    c.load_box_thermal(se, 0.5 * L, box, n_ele * w_n / 1000 / vol, 10.0 * 11604.52, seed=4, mode=0)
    t = np.loadtxt(table)
    m_red = 32 * AMU * ME / (32 * AMU + ME)
    wsv = w_n * float(np.max(t[:, 1] * np.sqrt(2.0 * t[:, 0] * QE / m_red)))
    mid = c.mcc_create(sn, si, se, E_ion, t[:, 0], t[:, 1], wsv_max_init=wsv)
    return c, sn, si, se, mid, dx, n


# 1.2M neutrals: above the size from which appended births are joined; 300k:
# sorted whole
@pytest.mark.parametrize("n_neu,n_ele", [(1_200_000, 60_000), (300_000, 60_000)])
def test_sort_after_births_keeps_every_particle_in_cell_order(pg, sigma_table_path, n_neu, n_ele):
    c, sn, si, se, mid, dx, n = _gas(pg, sigma_table_path, 1e-9, n_neu, n_ele)
    for step in range(3):
        st = c.mcc_apply(mid, 1e-9, 5, step)
    assert st["collisions"] > 0
    for sid in (sn, se, si):
        before = c.download(sid)
        assert c.count(sid) == before.size // 7  # counted while unsorted
        c.sort(sid)
        after = c.download(sid)
        assert np.array_equal(_rows(before), _rows(after))
        cells = _cells(after, dx, n)
        assert np.all(np.diff(cells) >= 0)
        macro = c.species_field(sid, pg.SFIELD_MACRO_COUNT)
        assert np.array_equal(macro, np.bincount(cells, minlength=macro.size))
    c.close()


def test_sort_with_nothing_appended(pg, sigma_table_path):
    """Elastic collisions alone: the electrons get no births, and a sort that
    finds nothing appended leaves them as they are."""
    c, sn, si, se, mid, dx, n = _gas(pg, sigma_table_path, 1e-10, 60_000, 1_100_000, E_ion=1.0)
    c.sort(se)
    st = c.mcc_apply(mid, 1e-10, 5, 0)
    assert st["collisions"] > 0 and st["ionizations"] == 0
    before = c.download(se)
    c.sort(se)
    assert np.array_equal(before, c.download(se))
    assert c.count(se) == before.size // 7
    c.close()


def test_count_leaves_out_removed_particles(pg):
    n, dx = (9, 10, 11), 1e-2
    L = dx * (np.array(n) - 1)
    rng = np.random.default_rng(1)
    for num in (1, 63, 70_001):
        p = np.zeros((num, 7))
        p[:, :3] = rng.uniform(0.01, 0.99, (num, 3)) * L
        p[:, 3:6] = rng.normal(0, 1e6, (num, 3))
        p[:, 6] = 1.0
        c = pg.Context(*n, [0, 0, 0], L)
        sid = c.species_add(ME, 0.0, 1.0, num)
        c.upload(sid, p)
        c.push(sid, 2e-8)  # most leave the box
        live = c.count(sid)
        assert live == c.download(sid).size // 7 and (num < 100 or 0 < live < num)
        c.sort(sid)
        assert c.count(sid) == live
        c.close()


@pytest.mark.parametrize("dt", [1e-10, 3e-8, 1e-6])  # none, most and all of them leave the box
@pytest.mark.parametrize("num", [1, 64, 1000, 130_001])
def test_removed_particles_take_no_place_in_the_sort(pg, dt, num):
    n, dx = (9, 10, 11), 1e-2
    L = dx * (np.array(n) - 1)
    rng = np.random.default_rng(num)
    p = np.zeros((num, 7))
    p[:, :3] = rng.uniform(0.1, 0.9, (num, 3)) * L
    p[:, 3:6] = rng.normal(0, 1e6, (num, 3))
    p[:, 6] = np.arange(num) + 1.0
    out = []
    for fused in (True, False):
        c = pg.Context(*n, [0, 0, 0], L)
        sid = c.species_add(ME, 0.0, 1.0, num)
        c.upload(sid, p)
        c.sort(sid)
        if fused:
            c.push_sort(sid, dt)
        else:
            c.push(sid, dt)
            c.sort(sid)
        q = c.download(sid)
        macro = c.species_field(sid, pg.SFIELD_MACRO_COUNT)
        assert c.count(sid) == q.size // 7 == int(macro.sum())
        if q.size:
            cells = _cells(q, dx, n)
            assert np.all(np.diff(cells) >= 0)
            assert np.array_equal(macro, np.bincount(cells, minlength=macro.size))
        out.append(_rows(q))
        c.close()
    assert np.array_equal(out[0], out[1])
    x = p[:, :3] + dt * p[:, 3:6]
    assert abs(len(out[0]) - np.sum(np.all((x > 0) & (x < L), axis=1))) <= 2 + num // 10000
