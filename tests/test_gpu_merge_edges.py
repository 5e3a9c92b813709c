"""Merge at the cell sizes where its kernels change: below 10 particles
(untouched), up to 64 (a wave per cell), beyond (a workgroup per cell)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

TAG_MERGE = 0x4D524701


@pytest.mark.parametrize("counts", [[0, 1, 9, 10, 11, 63, 64, 65], [64, 64, 64, 64, 10, 10, 9, 0],
                                    [66, 128, 129, 257, 600, 2, 0, 30], [3000, 0, 64, 0, 65, 0, 12, 12]])
@pytest.mark.parametrize("charge", [0.0, -O.QE])
def test_merge_cell_sizes_match_oracle(counts, charge):
    import pic_gpu as pg

    shape, dx = (3, 5, 2 + 1), 0.01
    L = dx * (np.array(shape) - 1)
    nc = np.array(shape) - 1
    rng = np.random.default_rng(sum(counts))
    p = []
    for c in range(int(np.prod(nc))):  # 16 cells: the counts twice
        n = counts[c % len(counts)]
        i = np.array([c % nc[0], c // nc[0] % nc[1], c // (nc[0] * nc[1])])
        q = np.zeros((n, 7))
        q[:, :3] = (i + rng.uniform(0.05, 0.95, (n, 3))) * dx
        q[:, 3:6] = rng.normal(0, 300, (n, 3)) * (rng.random((n, 1)) < 0.3) + rng.normal(0, 5, (n, 3))
        q[:, 6] = rng.uniform(0.5, 2, n)
        p.append(q)
    p = np.concatenate(p)
    p[:, 3:7] = p[:, 3:7].astype(np.float32).astype(np.float64)
    g = O.make_grid(*shape, [0, 0, 0], L)
    ef = rng.normal(0, 10, 3 * O.nn(g))
    c = pg.Context(*shape, [0, 0, 0], L)
    c.set_dt(2e-9)
    c.set_field(pg.FIELD_EF, ef)
    sid = c.species_add(16 * O.AMU, charge, 1.0, len(p) + 64)
    c.upload(sid, p)
    c.sort(sid)
    before = c.download(sid)
    st = c.merge(sid, seed=404)
    after = c.download(sid).reshape(-1, 7)
    ref, rst = O.merge(g, before, charge, 16 * O.AMU, 2e-9, O.rng_philox(404, 0, TAG_MERGE), ef=ef, gpu_mode=True)
    ref = ref.reshape(-1, 7)
    assert st["bins"] == rst[0] and st["merged"] == rst[1] and st["removed"] == len(p) - len(ref)
    assert len(after) == len(ref)
    ka = np.lexsort(np.round(ref[:, [3, 6, 0, 1, 2]] / [1e-2, 1e-6, 1e-8, 1e-8, 1e-8]).T)
    kb = np.lexsort(np.round(after[:, [3, 6, 0, 1, 2]] / [1e-2, 1e-6, 1e-8, 1e-8, 1e-8]).T)
    a, b = ref[ka], after[kb]
    vs = np.max(np.abs(a[:, 3:6]))
    # positions and velocities are stored in FP32 (6e-8 of a cell, of v)
    assert np.max(np.abs(a[:, :3] - b[:, :3])) < 1e-6 * dx
    assert np.max(np.abs(a[:, 3:6] - b[:, 3:6])) < 1e-5 * vs
    assert np.allclose(a[:, 6], b[:, 6], rtol=1e-6)
    c.close()


def _many_cells(nc, counts, dx, rng):
    """particles of cells 0, 1, ... (i fastest), counts[c] in cell c, away from its faces"""
    cell = np.repeat(np.arange(len(counts)), counts)
    i = np.stack([cell % nc[0], cell // nc[0] % nc[1], cell // (nc[0] * nc[1])], 1)
    p = np.zeros((len(cell), 7))
    p[:, :3] = (i + rng.uniform(0.05, 0.95, (len(cell), 3))) * dx
    p[:, 3:6] = rng.normal(0, 300, (len(cell), 3)) * (rng.random((len(cell), 1)) < 0.3) + rng.normal(0, 5, (len(cell), 3))
    p[:, 6] = rng.uniform(0.5, 2, len(cell))
    p[:, 3:7] = p[:, 3:7].astype(np.float32).astype(np.float64)
    return p


def _by_cell(p, nc, dx):
    """rows by cell, then weight (bit-equal in FP32: the same FP64 sums), then vx (a merged pair has one weight)"""
    p = np.asarray(p).reshape(-1, 7)
    i = np.floor(p[:, :3] / dx).astype(np.int64)
    return p[np.lexsort((p[:, 3], p[:, 6].astype(np.float32), (i[:, 2] * nc[1] + i[:, 1]) * nc[0] + i[:, 0]))]


def test_merge_of_many_cells_matches_oracle():
    """13824 cells, more than the waves and workgroups that walk them: cells
    of every class (no merge, a wave, a workgroup) in consecutive turns of one
    wave or workgroup, and large cells 1024 apart."""
    import pic_gpu as pg

    nc, dx = (24, 24, 24), 0.01
    shape, L = [n + 1 for n in nc], [n * dx for n in nc]
    rng = np.random.default_rng(77)
    counts = rng.choice([0, 3, 9, 10, 12, 20, 40, 64, 65, 70], size=int(np.prod(nc)))
    counts[::1024] = 200
    counts[5000:5100] = 90
    counts[9000:9300] = 4
    p = _many_cells(nc, counts, dx, rng)
    assert np.sum((counts >= 10) & (counts <= 64)) > 2048 * 4 / 2 and np.sum(counts > 64) > 2 * 1024
    g = O.make_grid(*shape, [0, 0, 0], L)
    ef = rng.normal(0, 10, 3 * O.nn(g))
    c = pg.Context(*shape, [0, 0, 0], L)
    c.set_dt(2e-9)
    c.set_field(pg.FIELD_EF, ef)
    sid = c.species_add(16 * O.AMU, -O.QE, 1.0, len(p) + 64)
    c.upload(sid, p)
    c.sort(sid)
    before = c.download(sid)
    st = c.merge(sid, seed=404)
    a = _by_cell(c.download(sid), nc, dx)
    ref, rst = O.merge(g, before, -O.QE, 16 * O.AMU, 2e-9, O.rng_philox(404, 0, TAG_MERGE), ef=ef, gpu_mode=True)
    b = _by_cell(ref, nc, dx)
    assert st["bins"] == rst[0] > 10000 and st["merged"] == rst[1] and st["removed"] == len(p) - len(b)
    assert a.shape == b.shape
    # positions and velocities are stored in FP32 (6e-8 of a cell, of v)
    assert np.max(np.abs(a[:, :3] - b[:, :3])) < 1e-6 * dx
    assert np.max(np.abs(a[:, 3:6] - b[:, 3:6])) < 1e-5 * np.max(np.abs(b[:, 3:6]))
    assert np.allclose(a[:, 6], b[:, 6], rtol=1e-6)
    c.close()


@pytest.mark.parametrize("where", [0, 700, 2999])
def test_cell_beyond_the_merge_bound_leaves_the_others_merged(where):
    """One cell of more than 8192 particles among large and small ones: the
    call fails, that cell is as it was, and every other cell is merged."""
    import pic_gpu as pg

    nc, dx = (10, 15, 20), 0.01
    shape, L = [n + 1 for n in nc], [n * dx for n in nc]
    rng = np.random.default_rng(3)
    counts = rng.choice([0, 5, 30, 100], size=int(np.prod(nc)))
    counts[where] = 8193
    p = _many_cells(nc, counts, dx, rng)
    out = []
    for part in (p, p[np.repeat(np.arange(len(counts)), counts) != where]):
        c = pg.Context(*shape, [0, 0, 0], L)
        c.set_dt(2e-9)
        sid = c.species_add(16 * O.AMU, 0.0, 1.0, len(p) + 64)
        c.upload(sid, part)
        c.sort(sid)
        if len(part) == len(p):
            with pytest.raises(RuntimeError, match="8192"):
                c.merge(sid, seed=9)
        else:
            assert c.merge(sid, seed=9)["bins"] > 100
        q = c.download(sid).reshape(-1, 7)
        i = np.floor(q[:, :3] / dx).astype(np.int64)
        out.append((q, (i[:, 2] * nc[1] + i[:, 1]) * nc[0] + i[:, 0]))
        c.close()
    (q, cell), (r, rc) = out
    assert np.sum(cell == where) == 8193
    assert np.array_equal(np.sort(q[cell == where][:, 6]), np.sort(p[np.repeat(np.arange(len(counts)), counts) == where][:, 6]))
    # the order inside a cell, and with it the sums' rounding, follows the upload's
    per = [np.bincount(x, weights=w, minlength=len(counts)) for x, w in ((cell[cell != where], q[cell != where][:, 6]), (rc, r[:, 6]))]
    assert np.allclose(per[0], per[1], rtol=1e-5)
    assert len(r) == np.sum(cell != where)
