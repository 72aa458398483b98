"""ct2's cell binning of the container (particle_to_grid, particle.cpp:59-114,
349-362) through the C ABI, and the failure path of a device allocation
(ct2 aborts, memory.cpp:7-10; the library reports CT2_ERR_NOMEM and stays
usable)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TWO32 = 2 ** 32


def cell_of(x, y, z, nc):
    x, y, z = (v.astype(np.uint64) for v in (x, y, z))
    return ((x * nc >> 32) * nc + (y * nc >> 32)) * nc + (z * nc >> 32)


@pytest.mark.parametrize("n,nc,minrung", [(1, 1, 0), (1000, 3, 0), (65543, 16, 2), (300000, 37, 1)])
def test_to_grid_is_a_stable_cell_sort(ct2, n, nc, minrung):
    rng = np.random.default_rng(n + nc)
    x, y, z = (rng.integers(0, TWO32, n, dtype=np.uint64).astype(np.uint32) for _ in range(3))
    edge = np.array([0, TWO32 - 1, TWO32 // 2, TWO32 // 2 - 1], np.uint32)
    x[: min(n, 4)] = edge[: min(n, 4)]
    vx = np.arange(n, dtype=np.float32)  # tags (exact below 2^24)
    vy = rng.standard_normal(n).astype(np.float32)
    vz = rng.standard_normal(n).astype(np.float32)
    rung = rng.integers(0, 4, n).astype(np.int8)
    ct2.particle_allocate(n)
    ct2.particles_upload(x, y, z, vx, vy, vz, rung)
    ct2.particle_sort_by_rung(minrung)
    first, last = ct2.particle_current_range()
    p0 = ct2.particles_download()
    starts = ct2.particles_to_grid(nc)
    p = ct2.particles_download()
    # outside the range nothing moves
    for a in ("x", "y", "z", "vx", "vy", "vz", "rung"):
        assert np.array_equal(getattr(p, a)[:first], getattr(p0, a)[:first])
    key0 = cell_of(p0.x[first:], p0.y[first:], p0.z[first:], nc)
    order = np.argsort(key0, kind="stable")
    for a in ("x", "y", "z", "vx", "vy", "vz", "rung"):
        assert np.array_equal(getattr(p, a)[first:], getattr(p0, a)[first:][order]), a
    key = key0[order]
    cells = np.arange(nc ** 3 + 1)
    assert np.array_equal(starts, first + np.searchsorted(key, cells, side="left"))
    assert starts[-1] == last


@pytest.mark.parametrize("n", [2, 2047, 2048, 2049, 4097, 65536, 65537, 2 ** 21 - 1, 2 ** 21 + 8191])
@pytest.mark.parametrize("nc", [1, 2, 13, 64, 129, 162, 256])
@pytest.mark.parametrize("one_cell", [False, True])
def test_cell_sort_tiles_and_passes(ct2, n, nc, one_cell):
    """Records in one tile, in few (their counts summed by the placement) and many,
    full and not; keys of one, two and three passes; all particles but one in a
    cell in the middle (long runs of empty cells before and after it)."""
    rng = np.random.default_rng(n + nc)
    x, y, z = (rng.integers(0, TWO32, n, dtype=np.uint64).astype(np.uint32) for _ in range(3))
    if one_cell:
        x[1:], y[1:], z[1:] = (rng.integers(TWO32 // 2, TWO32 // 2 + 1000, n - 1, dtype=np.uint64).astype(np.uint32)
                               for _ in range(3))
    vx = np.arange(n, dtype=np.float32)
    ct2.particle_allocate(n)
    ct2.particles_upload(x, y, z, vx, -vx, 2 * vx, (np.arange(n) % 5).astype(np.int8))
    ct2.particle_sort_by_rung(0)
    starts = ct2.particles_to_grid(nc)
    p = ct2.particles_download()
    key = cell_of(x, y, z, nc)
    order = np.argsort(key, kind="stable")
    assert np.array_equal(p.vx, vx[order])
    assert np.array_equal(p.vy, -vx[order]) and np.array_equal(p.vz, 2 * vx[order])
    assert np.array_equal(p.rung, order % 5)
    for a, b in ((p.x, x), (p.y, y), (p.z, z)):
        assert np.array_equal(a, b[order])
    assert np.array_equal(starts, np.searchsorted(key[order], np.arange(nc ** 3 + 1), side="left"))


def cell_centres(key, nc):
    return [((2 * (k.astype(np.uint64)) + 1) * TWO32 // (2 * nc)).astype(np.uint32)
            for k in (key // (nc * nc), key // nc % nc, key % nc)]


@pytest.mark.parametrize("occupied", [
    [0], [32767], [1023], [1024], [16384], [1023, 2047], [1024, 2048], [1022, 2047], [1023, 2046, 4000],
    [5, 1028], [5, 1029], [5, 1030], [100, 1123, 2147, 3172, 32000], [0, 15, 31, 48, 1072, 2097, 32767]])
def test_starts_across_long_runs_of_empty_cells(ct2, occupied):
    """32^3 cells, 9,000 particles in a few of them: runs of 15 to 32,767 empty cells, 1,023 to 1,025 of them
    starting and ending at, before and after multiples of 1,024 (starts are then written 1,024 to a wave)."""
    nc, n = 32, 9000
    key = np.array(occupied)[np.random.default_rng(len(occupied)).integers(0, len(occupied), n)]
    ct2.particle_allocate(n)
    ct2.particles_upload(*cell_centres(key, nc))
    starts = ct2.particles_to_grid(nc)
    assert np.array_equal(starts, np.searchsorted(np.sort(key), np.arange(nc ** 3 + 1), side="left"))


def test_to_grid_of_a_set_in_a_corner_takes_no_longer(ct2):
    """2^21 particles on 128^3 cells, in 1/50 of the box along each axis and in all of it: the empty cells' starts
    must not be one wave's work.  About equal times are expected, 3x allowed."""
    import time

    from ct2_amd import _lib as L
    n, nc = 2 ** 21, 128
    rng = np.random.default_rng(4)
    took = []
    for part in (1, 50):
        ct2.particle_allocate(n)
        ct2.particles_upload(*(rng.integers(0, TWO32 // part, n, dtype=np.uint64).astype(np.uint32) for _ in range(3)))
        best = np.inf
        for _ in range(8):
            t = time.perf_counter()
            L.check(L.load().ct2_particles_to_grid(nc, None))
            best = min(best, time.perf_counter() - t)
        took.append(best)
    print(f"all of the box {took[0] * 1e6:.0f} us, a corner {took[1] * 1e6:.0f} us", flush=True)
    assert took[1] < 3 * took[0], took


def test_to_grid_rejects_bad_sizes(ct2):
    from ct2_amd import Ct2Error
    ct2.particle_allocate(10)
    for nc in (0, -1, 1025):
        with pytest.raises(Ct2Error):
            ct2.particles_to_grid(nc)


def test_injected_allocation_failure(ct2):
    """ct2_debug_fail_allocations(after, count) makes device allocations fail
    without calling hipMalloc: the call reports CT2_ERR_NOMEM naming the
    allocation, leaves no half-made container (a failure at any of the
    container's eleven arrays), and the library works once the hook is spent,
    also when the failing allocation is a kernel's scratch buffer."""
    from ct2_amd import Ct2Error
    from ct2_amd import _lib as L
    for after in (0, 4, 10):
        ct2.debug_fail_allocations(after, 1)
        with pytest.raises(Ct2Error) as e:
            ct2.particle_allocate(4096)
        assert e.value.code == L.ERR_NOMEM and "test hook" in str(e.value)
        assert ct2.particle_count() == 0
    ct2.debug_fail_allocations(0, 0)
    # a fresh library state, so that the kick has to allocate its partial sums
    ct2.finalize()
    ct2.init(0)
    x, y, z = ct2.ic_lattice(16, 0.2, 1)
    ct2.particle_allocate(x.size)
    ct2.particles_upload(x, y, z)
    ct2.set_force_options(1e-3, 1.0 / x.size, 0)
    ct2.debug_fail_allocations(0, 1)
    with pytest.raises(Ct2Error) as e:
        ct2.kick(None, ct2.KICK_STORE)
    assert e.value.code == L.ERR_NOMEM
    ct2.kick(None, ct2.KICK_STORE)  # the hook is spent
    fx, fy, fz, pot = ct2.forces_download()
    assert np.isfinite(fx).all() and (pot > 0).all()
