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
