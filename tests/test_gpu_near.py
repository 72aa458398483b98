"""GPU near field of the PM force (near.hip) against the FP64 oracle and the
periodic FP64 judge: ragged and clustered particle sets (cells holding more
than one tile and more than one LDS key chunk), both pair kernels, a
neighbourhood that covers whole rows (3 cells per side), sparse sets whose
work items span whole columns (the sinks' bounding-box test then skips z, or
every axis), a single sphere packing most particles into one cell,
determinism and the argument checks."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TWO32 = 2 ** 32


@pytest.fixture(autouse=True)
def near_off(ct2):
    """The near-field setting is library state: leave it off for other tests."""
    yield
    ct2.pm_near(0.0)


def f32(v):
    return float(np.float32(v))


def rel(F, J):
    return np.linalg.norm(F - J, axis=0) / np.linalg.norm(J, axis=0)


def load(ct2, x, y, z):
    ct2.particle_allocate(x.size)
    ct2.particles_upload(x, y, z)


def near_only(ct2, rcut_rs):
    """(PM + near) and its near-field part (PM + near - PM), FP64."""
    ct2.pm_near(0.0)
    pm = np.stack(ct2.pm_forces()).astype(np.float64)
    ct2.pm_near(rcut_rs)
    tot = np.stack(ct2.pm_forces()).astype(np.float64)
    return tot, tot - pm


CASES = [
    # name, builder, ng, rs_cells, rcut_rs, kernel, expected cells per side
    ("uniform_ragged", "uniform", 64, 2.0, 6.0, 0, 5),
    ("clustered_3cells", "clustered", 32, 2.0, 5.0, 0, 3),
    ("clustered_ct2_kernel", "clustered", 64, 1.5, 6.0, 1, 7),
    # ~33 particles per (x, y) column: a work item's sinks span the whole
    # column, so the bounding-box test skips z; with rcut = 0.331 box it skips
    # x and y too (half-extent + rcut near half the box)
    ("sparse_whole_columns", "sparse", 32, 2.0, 5.0, 0, 3),
    ("sparse_no_box_test", "sparse", 32, 2.0, 5.3, 0, 3),
    # one compact sphere: ~15,000 particles share a cell, so the (cell, slice,
    # index) order of a very full cell is exercised
    ("dense_cell", "dense", 32, 2.0, 5.0, 0, 3),
]


def build(ct2, kind):
    if kind in ("uniform", "sparse"):
        rng = np.random.default_rng(11)
        n = 4099 if kind == "uniform" else 300
        return tuple(rng.integers(0, TWO32, n, dtype=np.uint64).astype(np.uint32) for _ in range(3))
    if kind == "dense":
        return ct2.ic_plummer_mix(20000, 16000, 1, 0.003, 0.1, 7)
    return ct2.ic_plummer_mix(24000, 16000, 4, 0.01, 0.1, 5)


@pytest.mark.parametrize("name,kind,ng,rs_cells,rcut_rs,kernel,ncell", CASES)
def test_near_field_vs_fp64_oracle(ct2, orc, name, kind, ng, rs_cells, rcut_rs, kernel, ncell):
    x, y, z = build(ct2, kind)
    n = x.size
    load(ct2, x, y, z)
    gm, soft = f32(1.0 / n), f32(2e-3)
    ct2.set_force_options(soft, gm, kernel)
    ct2.pm_init(ng, rs_cells)
    tot, near = near_only(ct2, rcut_rs)
    assert ct2.pm_near_cells() == ncell
    rs = rs_cells / ng
    sinks = np.random.default_rng(2).choice(n, min(n, 2000), replace=False)
    want = np.stack(orc.pm_near(x, y, z, gm, soft, rs, rcut_rs * rs, kernel, sinks=sinks))
    # the FP32 near-field sum against FP64, on the scale of the total force
    e = np.linalg.norm(near[:3, sinks] - want[:3], axis=0) / np.linalg.norm(tot[:3, sinks], axis=0)
    assert np.median(e) < 1e-5 and np.percentile(e, 99) < 2e-4 and e.max() < 2e-3, (np.median(e), e.max())
    ep = np.abs(near[3, sinks] - want[3]) / np.abs(tot[3, sinks])
    assert np.median(ep) < 1e-5 and ep.max() < 1e-3, (np.median(ep), ep.max())


@pytest.mark.parametrize("kernel", [0, 1])
@pytest.mark.parametrize("n", [2, 15, 17, 65, 2000, 2001])
def test_near_field_work_items(ct2, orc, n, kernel):
    """Work items of fewer than 16 sinks, rows of one sink more than whole
    items, and both sides of the density (16 per cell, 5^3 cells) above which
    cells are split in x and y; the tolerance of the cases above."""
    rng = np.random.default_rng(n)
    x, y, z = (rng.integers(0, TWO32, n, dtype=np.uint64).astype(np.uint32) for _ in range(3))
    x[: n // 2] = (x[: n // 2] >> 6) + np.uint32(2 ** 31)  # half of them within a few columns
    y[: n // 2] = (y[: n // 2] >> 6) + np.uint32(2 ** 31)
    load(ct2, x, y, z)
    gm, soft, ng, rs, rcut_rs = f32(1.0 / n), f32(2e-3), 64, 2.0, 6.0
    ct2.set_force_options(soft, gm, kernel)
    ct2.pm_init(ng, rs)
    tot, near = near_only(ct2, rcut_rs)
    assert ct2.pm_near_cells() == 5
    want = np.stack(orc.pm_near(x, y, z, gm, soft, rs / ng, rcut_rs * rs / ng, kernel))
    scale = np.linalg.norm(tot[:3], axis=0) + np.linalg.norm(want[:3], axis=0)
    e = np.linalg.norm(near[:3] - want[:3], axis=0) / scale
    assert np.median(e) < 1e-5 and e.max() < 2e-3, (np.median(e), e.max())
    ep = np.abs(near[3] - want[3]) / (np.abs(tot[3]) + np.abs(want[3]))  # the total passes through zero
    assert np.median(ep) < 1e-5 and ep.max() < 1e-3, (np.median(ep), ep.max())


def test_near_field_is_deterministic(ct2):
    x, y, z = ct2.ic_plummer_mix(30000, 20000, 3, 0.01, 0.1, 9)
    load(ct2, x, y, z)
    ct2.set_force_options(f32(1e-3), f32(1.0 / x.size), 0)
    ct2.pm_init(64, 2.0)
    ct2.pm_near(6.0)
    a = np.stack(ct2.pm_forces())
    b = np.stack(ct2.pm_forces())
    assert np.array_equal(a, b)


def test_pm_plus_near_field_vs_periodic_judge(ct2):
    """Lattice + Gaussian(0.2 cell): PM alone is off by ~100 %; PM + near field
    reaches the periodic FP64 direct sum to the mesh's discretisation error."""
    side = 32
    x, y, z = ct2.ic_lattice(side, 0.2, 1)
    n = x.size
    load(ct2, x, y, z)
    ct2.set_force_options(f32(1.0 / (50 * side)), f32(1.0 / n), 0)
    ct2.pm_init(2 * side, 3.0)
    idx = np.random.default_rng(5).choice(n, 1024, replace=False)
    J = np.stack(ct2.kick_sample_fp64(idx, periodic=True))
    ct2.pm_near(0.0)
    pm = np.stack(ct2.pm_forces())[:, idx]
    ct2.pm_near(6.0)
    tot = np.stack(ct2.pm_forces())[:, idx]
    assert np.median(rel(pm[:3], J[:3])) > 0.5
    e = rel(tot[:3], J[:3])
    assert np.median(e) < 2e-3 and np.percentile(e, 90) < 5e-3, (np.median(e), np.percentile(e, 90))
    assert np.max(np.abs(tot[3] - J[3])) < 1e-3 * np.abs(J[3]).max()


def test_tsc_pm_plus_near_field_vs_periodic_judge(ct2):
    """With TSC assignment the mesh error at a 2-cell split radius is ~10x
    below CIC's: the median force error against the periodic FP64 direct sum
    drops below 1e-3 with a small neighbourhood (cutoff 2.75 lattice spacings)."""
    side = 32
    x, y, z = ct2.ic_lattice(side, 0.2, 1)
    n = x.size
    load(ct2, x, y, z)
    ct2.set_force_options(f32(1.0 / (50 * side)), f32(1.0 / n), 0)
    idx = np.random.default_rng(5).choice(n, 1024, replace=False)
    J = np.stack(ct2.kick_sample_fp64(idx, periodic=True))
    errs = []
    for order in (1, 2):
        ct2.pm_assignment(order)
        ct2.pm_init(2 * side, 2.0)
        ct2.pm_near(5.5)
        tot = np.stack(ct2.pm_forces())[:, idx]
        errs.append(np.median(rel(tot[:3], J[:3])))
    ct2.pm_assignment(1)
    assert errs[1] < 1e-3 and errs[1] < errs[0] / 5, errs


def test_near_field_argument_checks(ct2):
    from ct2_amd._lib import Ct2Error
    x, y, z = ct2.ic_lattice(8, 0.1, 1)
    load(ct2, x, y, z)
    ct2.pm_init(16, 2.0)
    with pytest.raises(Ct2Error):
        ct2.pm_near(3.0)  # rcut = 3 * 2/16 = 0.375 box > 1/3
    with pytest.raises(Ct2Error):
        ct2.pm_near(-1.0)
    ct2.pm_init(16, 0.0)
    with pytest.raises(Ct2Error):
        ct2.pm_near(2.0)  # no Gaussian split
    ct2.pm_near(0.0)


def fill_with_copies(ct2, base, copies):
    """A container of `copies` times the base positions, one after the other; returns its device pointers."""
    import ctypes as C

    from ct2_amd import _lib as L
    m = base[0].size
    ct2.particle_allocate(m * copies)
    ptr = L.ParticlePtrs()
    L.check(L.load().ct2_particles_device_ptrs(C.byref(ptr)))
    for dst, src in zip((ptr.x, ptr.y, ptr.z), base):
        for k in range(copies):
            L.check(L.load().ct2_memcpy_h2d(dst + 4 * m * k, src.ctypes.data_as(C.c_void_p), 4 * m))
    return ptr


def velocities(ptr, first, count):
    import ctypes as C

    from ct2_amd import _lib as L
    v = np.empty((3, count), np.float32)
    for a, p in zip(v, (ptr.vx, ptr.vy, ptr.vz)):
        L.check(L.load().ct2_memcpy_d2h(a.ctypes.data_as(C.c_void_p), p + 4 * first, 4 * count))
    return v.astype(np.float64)


def test_near_field_of_more_work_items_than_a_launch_takes(ct2):
    """2^30 + 2^20 particles, 1,025 copies of 2^20 (a wave per 16 sinks: more than 2^32 threads): every copy's
    velocities after a half-kick equal the first's to the FP32 sums' rounding (about 10^5 terms; 1e-5 of their size),
    and they are those of the same mass in one copy."""
    m, copies = 2 ** 20, 1025
    rng = np.random.default_rng(30)
    base = [rng.integers(0, TWO32, m, dtype=np.uint64).astype(np.uint32) for _ in range(3)]
    kick = ct2.kick_params(ascending=True, top=True, rung=0, t0=2.0)
    soft = f32(1e-3)
    try:
        ct2.pm_init(128, 1.0)
        ct2.pm_near(0.5)
        got = []
        for k in (1, copies):
            ct2.set_force_options(soft, f32(1.0 / (m * k)), ct2.KERNEL_PLUMMER)
            ptr = fill_with_copies(ct2, base, k)
            ct2.kick_pm(kick)
            got.append([velocities(ptr, (j * (k - 1) // 8) * m, m) for j in range(9 if k > 1 else 1)])
        scale = np.sqrt((got[0][0] ** 2).mean())
        for v in got[1]:
            assert np.abs(v - got[1][0]).max() < 1e-4 * scale
            assert np.sqrt(((v - got[0][0]) ** 2).mean()) < 1e-5 * scale
    finally:
        ct2.finalize()  # 90 GB
        ct2.init(0)
        ct2.pm_init(32, 1.0)
