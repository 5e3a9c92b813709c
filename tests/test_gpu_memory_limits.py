"""Calls that work faster with memory they can do without, on a GPU that has
none left: they take their other path and give the same result.  Blocks
take the GPU's free memory but for a rest that the call's buffer does not
fit in."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ME, QE, AMU, KB = 9.10938215e-31, 1.602176565e-19, 1.660538921e-27, 1.380648e-23
MB = 1 << 20


@pytest.fixture(scope="module")
def pg():
    import pic_gpu

    return pic_gpu


class _Hog:
    """all of the GPU's free memory but `rest` bytes, through the HIP runtime
    that the library is linked with"""

    def __init__(self, ctx, rest):
        self.hip, self.rest, self.blocks = ctx.L, rest, []  # (its dependencies' names are found through it)

    def _take(self, size):
        p = C.c_void_p()
        if self.hip.hipMalloc(C.byref(p), C.c_size_t(size)):
            self.hip.hipGetLastError()
            return None
        return p

    def __enter__(self):
        free, total = C.c_size_t(), C.c_size_t()
        assert self.hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        kept = self._take(self.rest)
        assert kept
        size = free.value - self.rest
        while size >= 4 * MB:
            p = self._take(size)
            if p:
                self.blocks.append(p)
            else:
                size //= 2
        assert self.hip.hipFree(kept) == 0
        return self

    def __exit__(self, *a):
        for p in self.blocks:
            assert self.hip.hipFree(p) == 0


def _cells(p, dx, n):
    c = np.floor(p.reshape(-1, 7)[:, :3] / dx + 1e-9).astype(np.int64)
    return (c[:, 2] * (n[1] - 1) + c[:, 1]) * (n[0] - 1) + c[:, 0]


def _rows(p):
    p = np.asarray(p).reshape(-1, 7)
    return p[np.lexsort(p.T)]


def test_sort_without_memory_for_the_index(pg, sigma_table_path):
    """Births behind 1.2M sorted neutrals: pic_sort joins them through an
    index of 4 bytes per particle of the capacity (240 MB here); without room
    for it the species is sorted whole."""
    n, dx = (20, 18, 33), 1e-4
    L = dx * (np.array(n) - 1)
    box, n_neu, n_ele, cap = 0.98 * L, 1_200_000, 60_000, 60_000_000
    vol = float(np.prod(box))
    n_gas = 10.0 / (KB * 300.0)
    w_n = n_gas * vol / n_neu
    c = pg.Context(*n, [0, 0, 0], L)
    c.set_dt(1e-9)
    sn = c.species_add(32 * AMU, 0.0, w_n, cap)
    si = c.species_add(32 * AMU, QE, w_n / 1000, n_ele + 200000)
    se = c.species_add(ME, -QE, w_n / 1000, n_ele + 200000)
    c.load_box_thermal(sn, 0.5 * L, box, n_gas, 300.0, seed=3, mode=0)
    c.load_box_thermal(se, 0.5 * L, box, n_ele * w_n / 1000 / vol, 10.0 * 11604.52, seed=4, mode=0)
    t = np.loadtxt(sigma_table_path)
    m_red = 32 * AMU * ME / (32 * AMU + ME)
    wsv = w_n * float(np.max(t[:, 1] * np.sqrt(2.0 * t[:, 0] * QE / m_red)))
    mid = c.mcc_create(sn, si, se, 12.07 * QE, t[:, 0], t[:, 1], wsv_max_init=wsv)
    assert c.mcc_apply(mid, 1e-9, 5, 0)["collisions"] > 0
    num = c.count(sn)
    assert num > n_neu  # births behind the sorted part
    with _Hog(c, 128 * MB):
        c.sort(sn)
        after = c.download(sn)
        macro = c.species_field(sn, pg.SFIELD_MACRO_COUNT)
    cells = _cells(after, dx, n)
    assert c.count(sn) == num == after.size // 7
    assert np.all(np.diff(cells) >= 0)
    assert np.array_equal(macro, np.bincount(cells, minlength=macro.size))
    # with the memory back, the next births are joined again
    assert c.mcc_apply(mid, 1e-9, 5, 1)["collisions"] > 0
    before = c.download(sn)
    c.sort(sn)
    assert np.array_equal(_rows(before), _rows(c.download(sn)))
    c.close()


def test_species_without_memory_for_the_flags(pg):
    """pic_push_sort keeps a byte per particle of the capacity (60 MB here)
    for its next call; a species that there is no room for them for is
    added all the same and pushed like any other."""
    n, dx, num = (9, 10, 11), 1e-2, 20_001
    L = dx * (np.array(n) - 1)
    rng = np.random.default_rng(7)
    p = np.zeros((num, 7))
    p[:, :3] = rng.uniform(0.05, 0.95, (num, 3)) * L
    p[:, 3:6] = rng.normal(0, 4e3, (num, 3))
    p[:, 6] = np.arange(num) + 1.0
    cap = 60_000_000
    out = []
    for full in (True, False):
        c = pg.Context(*n, [0, 0, 0], L)
        if full:
            with _Hog(c, int(68.5 * cap)):
                sid = c.species_add(16 * AMU, QE, 1.0, cap)
        else:
            sid = c.species_add(16 * AMU, QE, 1.0, num)
        c.set_field(pg.FIELD_EF, np.random.default_rng(1).normal(0, 100.0, 3 * c.nn))
        c.upload(sid, p)
        c.sort(sid)
        for _ in range(5):
            c.push_sort(sid, 2e-8)
        q = c.download(sid)
        assert np.all(np.diff(_cells(q, dx, n)) >= 0)
        out.append(_rows(q))
        c.close()
    assert np.array_equal(out[0], out[1])


def test_sor_without_memory_for_the_second_potential(pg):
    """The tiled sweeps go from one potential to another (49 MB here); without
    room for it they are made in place, with the same values."""
    shape = (190, 180, 180)
    L = [1e-2 * (n - 1) for n in shape]
    rng = np.random.default_rng(2)
    rho = 1e-9 * rng.normal(size=shape[0] * shape[1] * shape[2])
    out = []
    for full in (True, False):
        c = pg.Context(*shape, [0, 0, 0], L)
        c.add_rectangle([L[0] / 2, L[1] / 2, 0], [1.1 * L[0], 1.1 * L[1], 0.2 * L[2]], 3.0)  # open sides
        c.set_field(pg.FIELD_RHO, rho)
        kw = dict(method=pg.SOLVER_SOR_RB, tol=1e-300, tol_kind=pg.TOL_REL, max_it=21, omega=1.7, check_every=8)
        if full:
            with _Hog(c, 24 * MB):
                st = c.poisson(**kw)
        else:
            st = c.poisson(**kw)
        assert st["iterations"] == 21 and not st["converged"]
        out.append(c.get_field(pg.FIELD_PHI))
        c.close()
    assert np.array_equal(out[0], out[1])


def test_velocity_moments_without_memory_for_all_of_them(pg):
    """n v is interleaved on the device in pieces of 25 MB; 24 bytes for every
    node (80 MB here) are not asked for."""
    shape = (150, 150, 150)
    L = 1e-2 * (np.array(shape) - 1)
    c = pg.Context(*shape, [0, 0, 0], L)
    sid = c.species_add(ME, 0.0, 1.0, 100)
    p = np.zeros((100, 7))
    p[:, :3] = 0.5 * L
    p[:, 3:7] = [1.0, 2.0, -4.0, 1.0]
    c.upload(sid, p)
    c.deposit(sid, pg.DEPOSIT_DENSITY | pg.DEPOSIT_MOMENTS)
    with _Hog(c, 48 * MB):
        nv = c.species_field(sid, pg.SFIELD_NVSUM)
    assert np.allclose(nv.reshape(-1, 3).sum(0), [100.0, 200.0, -400.0], rtol=1e-6)
    c.close()
