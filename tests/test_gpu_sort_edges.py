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


def _charged(pg, num, mass, charge, seed):
    n, dx = (9, 10, 11), 1e-2
    L = dx * (np.array(n) - 1)
    rng = np.random.default_rng(seed)
    c = pg.Context(*n, [0, 0, 0], L)
    c.dirichlet_walls()
    c.set_dt(1e-10)
    p = np.zeros((num, 7))
    p[:, :3] = rng.uniform(0.05, 0.95, (num, 3)) * L
    p[:, 3:6] = rng.normal(0, np.sqrt(1.6e-19 * 2.0 / mass), (num, 3))
    p[:, 6] = np.arange(num) + 1.0
    sid = c.species_add(mass, charge, 1.0, num + 5000)
    c.upload(sid, p)
    c.sort(sid)
    ef = rng.normal(0, 100.0, 3 * c.nn)
    return c, sid, ef


@pytest.mark.parametrize("mass,charge", [(ME, -QE), (16 * AMU, QE), (32 * AMU, 0.0)])
@pytest.mark.parametrize("num", [65, 20_001])
def test_push_sort_chain_equals_push_then_sort(pg, mass, charge, num):
    """Several pic_push_sort in a row, whose histogram pass uses the flags the
    one before left, against pic_push + pic_sort: larger and smaller steps,
    a field that grows within and beyond the flags' bound, and every call
    that changes the particles in between."""
    chains = [_charged(pg, num, mass, charge, 7) for _ in range(2)]
    field = [1.0, 1.5, 2.9, 2.9, 40.0, 40.0, 1.0, 1.0, 1.0, 1.0, 1.0]
    steps = [1e-10, 1e-10, 1e-10, 3e-10, 1e-10, 1e-10, 1e-9, 1e-10, 1e-10, 1e-10, 1e-10]
    for k, (amp, dt) in enumerate(zip(field, steps)):
        rows = []
        for fused, (c, sid, ef) in zip((True, False), chains):
            if amp != (field[k - 1] if k else None):
                c.set_field(pg.FIELD_EF, amp * ef)
            if k == 7:  # other particles
                q = c.download(sid).reshape(-1, 7)
                q = q[np.argsort(q[:, 6])]
                q[:, 3:6] *= -3.0
                c.upload(sid, q)
                c.sort(sid)
            if k == 9:  # moved by another call
                c.push(sid, 5e-10)
                c.sort(sid)
            if fused:
                c.push_sort(sid, dt)
            else:
                c.push(sid, dt)
                c.sort(sid)
            r = c.download(sid)
            macro = c.species_field(sid, pg.SFIELD_MACRO_COUNT)
            cells = _cells(r, 1e-2, (9, 10, 11))
            assert np.all(np.diff(cells) >= 0), k
            assert np.array_equal(macro, np.bincount(cells, minlength=macro.size)), k
            rows.append(_rows(r))
        assert np.array_equal(rows[0], rows[1]), k
    for c, _, _ in chains:
        c.close()


def test_push_sort_flags_after_collisions_and_sources(pg):
    """DSMC_MEX changes velocities in place and a source appends: the next
    pic_push_sort sorts by where the particles really go."""
    c, sid, ef = _charged(pg, 30_000, 32 * AMU, 0.0, 3)
    did = c.dsmc_create(sid)
    src = c.source_create(sid, 0, 4e3, 5e9, 300.0)
    for step in range(6):
        c.push_sort(sid, 5e-7)  # about a tenth of a cell
        r = c.download(sid)
        cells = _cells(r, 1e-2, (9, 10, 11))
        assert np.all(np.diff(cells) >= 0), step
        macro = c.species_field(sid, pg.SFIELD_MACRO_COUNT)
        assert np.array_equal(macro, np.bincount(cells, minlength=macro.size)), step
        if step % 2:
            assert c.dsmc_apply(did, 1e7, 5, step)["collisions"] > 1000
        else:
            assert c.source_sample(src, seed=step) > 0
    c.close()


def _in_cell_order(pg, c, sid, dx, n):
    r = c.download(sid)
    cells = _cells(r, dx, n)
    assert np.all(np.diff(cells) >= 0)
    macro = c.species_field(sid, pg.SFIELD_MACRO_COUNT)
    assert np.array_equal(macro, np.bincount(cells, minlength=macro.size))
    return r.size // 7


def test_push_sort_flags_after_merges(pg):
    """Three pic_push_sort in a row (the second leaves flags, of 99% of the
    particles, and the third uses them), then a merge, which moves particles
    to other members' places and velocities: the next ones sort by where the
    particles really go."""
    n, dx = (9, 10, 11), 1e-2
    c, sid, _ = _charged(pg, 200_000, 16 * AMU, QE, 5)
    left = 200_000
    for step in range(4):
        for _ in range(3):
            c.push_sort(sid, 1e-9)  # 0.03% of a cell
            left = _in_cell_order(pg, c, sid, dx, n)
        st = c.merge(sid, seed=step)
        assert st["removed"] > 1000 or step
        assert _in_cell_order(pg, c, sid, dx, n) == left - st["removed"]
        c.push_sort(sid, 1e-9)
        _in_cell_order(pg, c, sid, dx, n)
    c.close()


def test_push_sort_flags_after_mcc_steps(pg, sigma_table_path):
    """The same with MC_MEX steps in a box without objects: the collisions turn
    electrons and neutrals and append others."""
    c, sn, si, se, mid, dx, n = _gas(pg, sigma_table_path, 1e-9, 300_000, 60_000)
    for step in range(4):
        for sid, dt in ((se, 2e-13), (sn, 5e-10), (si, 5e-10)):
            for _ in range(3):
                c.push_sort(sid, dt)
                _in_cell_order(pg, c, sid, dx, n)
        st = c.mcc_apply(mid, 1e-9, 5, step)
        assert st["collisions"] > 1000 and st["ionizations"] > 0
    c.close()


def test_push_sort_rule_for_flags_in_a_changing_run(pg):
    """Steps that change between those that nearly no particle leaves its cell
    in and those that most do, so that flags are left, left out and left
    again, against pic_push + pic_sort."""
    chains = [_charged(pg, 60_001, 16 * AMU, QE, 11) for _ in range(2)]
    for _, (c, sid, ef) in zip(range(2), chains):
        c.set_field(pg.FIELD_EF, ef)
    for k, dt in enumerate([1e-10] * 4 + [2e-6] * 3 + [1e-10] * 4 + [2e-6, 1e-10, 1e-10, 1e-10]):
        rows = []
        for fused, (c, sid, _) in zip((True, False), chains):
            if fused:
                c.push_sort(sid, dt)
            else:
                c.push(sid, dt)
                c.sort(sid)
            _in_cell_order(pg, c, sid, 1e-2, (9, 10, 11))
            rows.append(_rows(c.download(sid)))
        assert np.array_equal(rows[0], rows[1]), k
    assert len(rows[0]) > 100
    for c, _, _ in chains:
        c.close()


@pytest.mark.parametrize("num", [0, 1, (1 << 20) - 1, 1 << 20, (1 << 20) + 3])
def test_upload_in_pieces(pg, num):
    """uploads of no, one, and just below and above one staging piece"""
    n, dx = (9, 10, 11), 1e-2
    L = dx * (np.array(n) - 1)
    rng = np.random.default_rng(2)
    p = np.zeros((num, 7))
    p[:, :3] = rng.uniform(0.01, 0.99, (num, 3)) * L
    p[:, 3:6] = rng.normal(0, 1e3, (num, 3)).astype(np.float32)
    p[:, 6] = np.arange(num) + 1.0
    c = pg.Context(*n, [0, 0, 0], L)
    sid = c.species_add(ME, -QE, 1.0, max(num, 1))
    c.upload(sid, p)
    q = c.download(sid).reshape(-1, 7)
    assert np.array_equal(q[:, 3:], p[:, 3:])
    # the offset in the cell is stored in FP32
    assert num == 0 or np.max(np.abs(q[:, :3] - p[:, :3])) <= 1e-7 * dx
    c.close()


@pytest.mark.parametrize("shape", [(3, 3, 3), (64, 128, 128), (64, 128, 129), (129, 131, 127)])
def test_velocity_moments_in_pieces(pg, shape):
    """n v of grids of up to one, just over one and over two staging pieces of
    2^20 nodes: with one velocity of powers of two for all particles it is the
    density sum times that velocity, bit for bit."""
    dx = 1e-2
    L = dx * (np.array(shape) - 1)
    rng = np.random.default_rng(4)
    num = 300_000
    p = np.zeros((num, 7))
    p[:, :3] = rng.uniform(0.001, 0.999, (num, 3)) * L
    v = np.array([2.0, -64.0, 0.25])
    p[:, 3:6] = v
    p[:, 6] = rng.uniform(0.5, 2.0, num)
    c = pg.Context(*shape, [0, 0, 0], L)
    sid = c.species_add(ME, 0.0, 1.0, num)
    c.upload(sid, p)
    c.clear_samples(sid)
    c.deposit(sid, pg.DEPOSIT_DENSITY | pg.DEPOSIT_MOMENTS)
    n = c.species_field(sid, pg.SFIELD_NSUM)
    nv = c.species_field(sid, pg.SFIELD_NVSUM).reshape(-1, 3)
    assert n.sum() > 0.99 * p[:, 6].sum()
    assert np.array_equal(nv, n[:, None] * v)
    c.close()


@pytest.mark.parametrize("shape", [(3, 3, 3), (5, 5, 64), (33, 33, 5), (33, 33, 6), (17, 65, 67), (50, 100, 201)])
def test_cell_offsets_at_scan_tile_edges(pg, shape):
    """cell counts below, at and above a scan row (1024) and tile (4096), and
    more tiles than one workgroup has threads"""
    dx = 1e-2
    L = dx * (np.array(shape) - 1)
    ncells = int(np.prod(np.array(shape) - 1))
    rng = np.random.default_rng(ncells)
    num = 20_000
    p = np.zeros((num, 7))
    p[:, :3] = rng.uniform(0.001, 0.999, (num, 3)) * L
    p[:, 6] = np.arange(num) + 1.0
    c = pg.Context(*shape, [0, 0, 0], L)
    sid = c.species_add(ME, 0.0, 1.0, num)
    c.upload(sid, p)
    for sort in (c.sort, lambda s: c.push_sort(s, 1e-12)):
        sort(sid)
        q = c.download(sid)
        assert np.array_equal(np.sort(q.reshape(-1, 7)[:, 6]), p[:, 6])
        cells = _cells(q, dx, shape)
        assert np.all(np.diff(cells) >= 0)
        assert np.array_equal(c.species_field(sid, pg.SFIELD_MACRO_COUNT), np.bincount(cells, minlength=ncells))
    c.close()
