"""GPU parity of the particle-mesh force and of the periodic FP64 judge
against the CPU oracle (particle.cpp:116-271 shape, particle.cpp:141-144
periodic force), through the C ABI."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TWO32 = 2 ** 32


def f32(v):
    return float(np.float32(v))


def load(ct2, x, y, z, vx=None, vy=None, vz=None, rung=None):
    ct2.particle_allocate(x.size)
    ct2.particles_upload(x, y, z, vx, vy, vz, rung)


@pytest.mark.parametrize("ng", [16, 32, 64, 256])
def test_cic_deposit_bit_exact(ct2, orc, ng):
    """Integer atomics make the deposit order-independent: the GPU grid equals
    the CPU restatement bit for bit, clusters (heavy contention) included."""
    x, y, z = ct2.ic_plummer_mix(50000, 30000, 3, 0.005, 0.05, 21)
    load(ct2, x, y, z)
    ct2.set_force_options(1e-3, 1.0 / x.size, 0)
    ct2.pm_init(ng, 1.25)
    ct2.pm_forces()
    got = ct2.pm_density_download()
    want = orc.cic_deposit(x, y, z, ng.bit_length() - 1)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("ng,rs", [(32, 1.25), (64, 1.0), (64, 2.0)])
def test_pm_forces_vs_fp64_oracle(ct2, orc, ng, rs):
    x, y, z = ct2.ic_plummer_mix(30000, 15000, 8, 0.02, 0.2, 4)
    n = x.size
    load(ct2, x, y, z)
    gm = f32(1.0 / n)
    ct2.set_force_options(1e-3, gm, 0)
    ct2.pm_init(ng, rs)
    fx, fy, fz, pot = ct2.pm_forces()
    ox, oy, oz, op = orc.pm_forces(x, y, z, ng.bit_length() - 1, gm, rs)
    F = np.stack([fx, fy, fz])
    O = np.stack([ox, oy, oz])
    rms = np.sqrt(np.mean(O ** 2))
    assert np.max(np.abs(F - O)) < 2e-5 * rms * np.sqrt(ng), np.max(np.abs(F - O)) / rms
    assert np.max(np.abs(pot - op)) < 1e-5 * np.abs(op).max()


@pytest.mark.parametrize("ng", [8, 16, 32, 64, 128, 256, 512])
def test_pm_fields_of_the_density_at_every_grid_size(ct2, ng):
    """The force and potential grids against FP64 transforms of the same
    density: every size of the half-spectrum passes and of the fused x pass
    (its kz = 0 and N/2 columns and its mirrored half).  An FP32 transform
    stays within 1e-6 of the complex grid it transforms (relative L2), forward
    and inverse within 2e-6: Fx + i Fy and Fz + i pot are one grid each."""
    rng = np.random.default_rng(ng)
    n, rs = 4000, 1.0
    x, y, z = (rng.integers(0, TWO32, n, dtype=np.uint64).astype(np.uint32) for _ in range(3))
    load(ct2, x, y, z)
    gm = f32(1.0 / n)
    ct2.set_force_options(1e-3, gm, 0)
    ct2.pm_init(ng, rs)
    ct2.pm_forces()
    hat = np.fft.rfftn(ct2.pm_density_download().astype(np.float64) * 2.0 ** -32)
    m = np.fft.fftfreq(ng, 1.0 / ng)
    k = [2 * np.pi * v for v in np.meshgrid(m, m, np.abs(m[:ng // 2 + 1]), indexing="ij", sparse=True)]
    k2 = sum(v * v for v in k)
    k2[0, 0, 0] = 1.0
    w = 1.0
    for v in k:
        w = w * np.sinc(v / (2 * np.pi * ng)) ** 4
    phi = -4 * np.pi * gm * np.exp(-k2 * (rs / ng) ** 2) / (k2 * w) * hat
    phi[0, 0, 0] = 0.0
    k = [np.where(np.abs(v) > np.pi * ng - 1.0, 0.0, v) for v in k]  # no force from the Nyquist components
    for which, pair in ((0, (-1j * k[0] * phi, -1j * k[1] * phi)), (1, (-1j * k[2] * phi, -phi))):
        re, im = (np.fft.irfftn(f, s=(ng,) * 3, axes=(0, 1, 2)) * float(ng) ** 3 for f in pair)
        want = (re + 1j * im).ravel()
        assert np.linalg.norm(ct2.pm_grid_download(which).ravel() - want) < 2e-6 * np.linalg.norm(want)


def test_pm_force_on_1024(ct2):
    """The largest grid (its own shape of the x pass, real passes of 512 points, planes in ragged groups): particles on
    nodes, so that deposit and interpolation are exact, against the FP64 sum of the Green's function over all wave
    vectors, axis by axis.  FP32 transforms stay within 2e-6 of their grid's rms (2-norm); five times that of the
    fields' largest value at the particles, which are its peaks, is allowed at each."""
    ng, rs = 1024, 1.0
    h = ng // 2
    node = np.array([[3, 5, 7], [4, 5, 7], [1020, 1019, 1022], [500, 511, 512], [3, 517, 1000], [1008, 23, 24]])
    load(ct2, *(np.ascontiguousarray(node[:, a].astype(np.uint32) << 22) for a in range(3)))
    gm = f32(1.0 / len(node))
    ct2.set_force_options(1e-3, gm, 0)
    try:
        ct2.pm_init(ng, rs)
        got = np.stack(ct2.pm_forces()).astype(np.float64)
    finally:
        ct2.pm_init(8, 1.25)  # the large grids are released
    m = np.arange(h + 1)
    k = 2 * np.pi * m
    green = -4 * np.pi * gm / np.maximum(k[:, None, None] ** 2 + k[:, None] ** 2 + k ** 2, 1.0)
    green[0, 0, 0] = 0.0
    axis = np.exp(-(k * rs / ng) ** 2) / np.sinc(m / ng) ** 4 * np.where((m == 0) | (m == h), 1.0, 2.0)
    d = ((node[:, None] - node[None]) % ng).reshape(-1, 3)  # particle minus source
    even = [axis[:, None] * np.cos(2 * np.pi * np.outer(m, v) / ng) for v in d.T]
    odd = [np.where((m == 0) | (m == h), 0.0, k * axis)[:, None] * np.sin(2 * np.pi * np.outer(m, v) / ng) for v in d.T]
    want = []
    for gradient in (0, 1, 2, None):
        f = [odd[a] if a == gradient else even[a] for a in range(3)]
        yz = (green.reshape(-1, h + 1) @ f[2]).reshape(h + 1, h + 1, -1)
        total = np.einsum("xd,yd,xyd->d", f[0], f[1], yz, optimize=True).reshape(len(node), -1).sum(1)
        want.append(total if gradient is not None else -total)
    want = np.stack(want)
    assert (np.abs(got - want).max(1) < 1e-5 * np.abs(want).max(1)).all(), (got, want)


def test_pm_matches_periodic_judge_on_a_single_mode(ct2):
    """Linear single-mode lattice: PM long-range force 4 pi psi exp(-k^2 rs^2),
    the periodic FP64 judge the full 4 pi psi."""
    n, A, rs = 32, 1e-4, 1.0
    q = (np.arange(n) + 0.5) / n
    X, Y, Z = np.meshgrid(q, q, q, indexing="ij")
    psi = A * np.sin(2 * np.pi * X.ravel())
    x = ((X.ravel() + psi) % 1 * TWO32).astype(np.uint64).astype(np.uint32)
    y = (Y.ravel() * TWO32).astype(np.uint64).astype(np.uint32)
    z = (Z.ravel() * TWO32).astype(np.uint64).astype(np.uint32)
    N = n ** 3
    load(ct2, x, y, z)
    ct2.set_force_options(1e-4, 1.0 / N, 0)
    ct2.pm_init(32, rs)
    fx, fy, fz, _ = ct2.pm_forces()
    want = 4 * np.pi * psi
    filt = np.exp(-(2 * np.pi * rs / 32) ** 2)
    assert np.allclose(fx, want * filt, rtol=0, atol=3e-3 * np.abs(want).max())
    idx = np.array([0, 77, np.argmax(psi), 20000])
    jx, jy, jz, _ = ct2.kick_sample_fp64(idx, periodic=True)
    assert np.allclose(jx, want[idx], rtol=0, atol=3e-3 * np.abs(want).max())
    # pairs exactly half a box apart in y take the one-sided int32 minimum
    # image, whose Plummer softening leaves a residue of order GM eps^2 n^2 / s^4
    assert np.max(np.abs(jy)) < 1e-5 * np.abs(want).max()


def test_periodic_judge_vs_cpu_ewald(ct2, orc):
    x, y, z = ct2.ic_plummer_mix(3000, 1500, 4, 0.03, 0.3, 13)
    n = x.size
    load(ct2, x, y, z)
    soft, gm = f32(2e-3), f32(1.0 / n)
    ct2.set_force_options(soft, gm, 0)
    idx = np.arange(0, n, 97)
    g = ct2.kick_sample_fp64(idx, periodic=True)
    c = orc.ewald_kick(x, y, z, gm, soft, sinks=idx)
    for a, b in zip(g, c):
        assert np.allclose(a, b, rtol=1e-9, atol=1e-10 * np.abs(b).max())


def test_periodic_judge_madelung_and_lattice(ct2):
    XI = -2.837297479480620
    n = 8
    q = (np.arange(n) + 0.5) / n
    X, Y, Z = np.meshgrid(q, q, q, indexing="ij")
    f = lambda v: (v.ravel() * TWO32).astype(np.uint64).astype(np.uint32)
    load(ct2, f(X), f(Y), f(Z))
    soft = f32(1e-5)
    ct2.set_force_options(soft, f32(1.0 / n ** 3), 0)
    ax, ay, az, p = ct2.kick_sample_fp64(np.array([0, 100, 511]), periodic=True)
    assert np.max(np.abs([ax, ay, az])) < 1e-9
    gm = f32(1.0 / n ** 3)
    assert np.allclose(p - gm / soft, gm * n * XI, atol=1e-9)


def test_kick_pm_epilogue_bit_exact(ct2, orc):
    x, y, z = ct2.ic_lattice(24, 0.3, 2)
    n = x.size
    rng = np.random.default_rng(5)
    vx, vy, vz = (rng.standard_normal(n).astype(np.float32) * 1e-3 for _ in range(3))
    rung = rng.integers(0, 3, n).astype(np.int8)
    load(ct2, x, y, z, vx, vy, vz, rung)
    ct2.set_force_options(1e-3, 1.0 / n, 0)
    ct2.pm_init(32, 1.25)
    p = ct2.kick_params(ascending=1, descending=1, top=1, first=0, rung=1, t0=0.02, eta=0.1, max_dt=0.01, scale=0.5)
    mr = ct2.kick_pm(p)
    fx, fy, fz, _ = ct2.forces_download()
    after = ct2.particles_download()
    r2 = rung.copy()
    omr = orc.kick_epilogue(fx, fy, fz, vx, vy, vz, r2, orc.KickParams(*[getattr(p, f) for f, _ in p._fields_]),
                            f32(1e-3))
    assert np.array_equal(after.vx, vx) and np.array_equal(after.vz, vz) and np.array_equal(after.rung, r2)
    assert mr == omr


def test_pm_512_cubed_runs_and_conserves_momentum(ct2):
    """The PM grid of the clustered and stepping configurations."""
    x, y, z = ct2.ic_lattice(128, 0.3, 3)
    n = x.size
    load(ct2, x, y, z)
    ct2.set_force_options(1.0 / 6400, 1.0 / n, 0)
    ct2.pm_init(512, 1.25)
    fx, fy, fz, pot = ct2.pm_forces()
    for a in (fx, fy, fz):
        assert np.isfinite(a).all()
        assert abs(a.astype(np.float64).sum()) < 1e-4 * np.abs(a).sum()


@pytest.fixture
def tsc(ct2):
    ct2.pm_assignment(2)
    yield
    ct2.pm_assignment(1)


@pytest.mark.parametrize("ng", [16, 32, 128, 256])
def test_tsc_deposit_bit_exact(ct2, orc, tsc, ng):
    x, y, z = ct2.ic_plummer_mix(50000, 30000, 3, 0.005, 0.05, 22)
    load(ct2, x, y, z)
    ct2.set_force_options(1e-3, 1.0 / x.size, 0)
    ct2.pm_init(ng, 1.25)
    ct2.pm_forces()
    assert np.array_equal(ct2.pm_density_download(), orc.mesh_deposit(x, y, z, ng.bit_length() - 1, 2))


@pytest.mark.parametrize("ng,order", [(128, 1), (512, 2), (1024, 2)])
def test_deposit_binning_by_grid_size_bit_exact(ct2, orc, ng, order):
    """The three ways tiles are counted (512 and 32,768 tiles in LDS, 262,144 by
    global atomics), with several binning workgroups, and particles on every
    face, edge and corner of tiles."""
    rng = np.random.default_rng(ng)
    n, s = 9001, 32 - (ng.bit_length() - 1)
    node = rng.integers(0, ng, (3, n), dtype=np.uint64) // 16 * 16  # the first node of a tile, or next to it
    x, y, z = ((node.astype(np.int64) + rng.integers(-2, 2, (3, n))) % ng * (1 << s) +
               rng.integers(0, 1 << s, (3, n))).astype(np.uint64).astype(np.uint32)
    load(ct2, x, y, z)
    ct2.set_force_options(1e-3, 1.0 / n, 0)
    ct2.pm_assignment(order)
    try:
        ct2.pm_init(ng, 1.25)
        ct2.pm_forces()
        got = ct2.pm_density_download()
    finally:
        ct2.pm_assignment(1)
        ct2.pm_init(8, 1.25)  # the large grids are released
    assert np.array_equal(got.ravel(), orc.mesh_deposit(x, y, z, ng.bit_length() - 1, order).ravel())


@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("ng", [8, 32, 64])
@pytest.mark.parametrize("n", [1, 63, 1037, 4096])
def test_deposit_edge_cases_bit_exact(ct2, orc, order, ng, n):
    """Ragged particle counts (partial waves), lattice order (long runs of
    one tile), and positions on the wrap, on nodes and on half nodes."""
    rng = np.random.default_rng(n * 131 + ng)
    side = int(round(n ** (1 / 3))) + 1
    q = (np.arange(n) % side).astype(np.uint64)
    x = ((q * TWO32) // side).astype(np.uint32)
    y = ((((np.arange(n) // side) % side).astype(np.uint64) * TWO32) // side).astype(np.uint32)
    z = rng.integers(0, TWO32, n, dtype=np.uint64).astype(np.uint32)
    s = 32 - (ng.bit_length() - 1)
    special = np.array([0, 1, TWO32 - 1, 1 << (s - 1), (1 << (s - 1)) - 1, TWO32 - (1 << (s - 1)), 1 << s,
                        TWO32 - (1 << s)], np.uint64).astype(np.uint32)
    k = min(n, special.size)
    x[:k], y[-k:], z[:k] = special[:k], special[:k], special[::-1][:k]
    load(ct2, x, y, z)
    ct2.set_force_options(1e-3, 1.0 / n, 0)
    ct2.pm_assignment(order)
    try:
        ct2.pm_init(ng, 1.25)
        ct2.pm_forces()
        got = ct2.pm_density_download()
    finally:
        ct2.pm_assignment(1)
    assert np.array_equal(got, orc.mesh_deposit(x, y, z, ng.bit_length() - 1, order))


@pytest.mark.parametrize("ng,rs", [(32, 1.25), (64, 2.0)])
def test_tsc_pm_forces_vs_fp64_oracle(ct2, orc, tsc, ng, rs):
    x, y, z = ct2.ic_plummer_mix(30000, 15000, 8, 0.02, 0.2, 4)
    n = x.size
    load(ct2, x, y, z)
    gm = f32(1.0 / n)
    ct2.set_force_options(1e-3, gm, 0)
    ct2.pm_init(ng, rs)
    fx, fy, fz, pot = ct2.pm_forces()
    ox, oy, oz, op = orc.pm_forces(x, y, z, ng.bit_length() - 1, gm, rs, order=2)
    F = np.stack([fx, fy, fz])
    O = np.stack([ox, oy, oz])
    rms = np.sqrt(np.mean(O ** 2))
    assert np.max(np.abs(F - O)) < 2e-5 * rms * np.sqrt(ng), np.max(np.abs(F - O)) / rms
    assert np.max(np.abs(pot - op)) < 1e-5 * np.abs(op).max()


@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("n,ng", [(65, 16), (5000, 64), (40000, 32)])
@pytest.mark.parametrize("descending", [False, True])
def test_kick_pm_applies_the_epilogue_to_the_range(ct2, orc, order, n, ng, descending):
    """The interpolation's own epilogue (the first two) and the separate kernel
    (tiled interpolation), on a rung range that starts inside a wave."""
    rng = np.random.default_rng(n + order)
    x, y, z = (rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32) for _ in range(3))
    rung = rng.integers(0, 3, n).astype(np.int8)
    v = [(0.01 * rng.standard_normal(n)).astype(np.float32) for _ in range(3)]
    ct2.particle_allocate(n)
    ct2.particles_upload(x, y, z, *v, rung)
    gm, soft = float(np.float32(1.0 / n)), float(np.float32(2e-3))
    ct2.set_force_options(soft, gm, ct2.KERNEL_PLUMMER)
    ct2.particle_sort_by_rung(1)
    first, _ = ct2.particle_current_range()
    p0 = ct2.particles_download()
    params = ct2.kick_params(ascending=True, descending=descending, top=True, rung=1, t0=0.01)
    ct2.pm_assignment(order)
    try:
        ct2.pm_init(ng, 1.25)
        mr = ct2.kick_pm(params)
    finally:
        ct2.pm_assignment(1)
    f = ct2.forces_download()
    p1 = ct2.particles_download()
    for a in ("vx", "vy", "vz", "rung"):
        assert np.array_equal(getattr(p1, a)[:first], getattr(p0, a)[:first]), a
    want = [getattr(p0, a)[first:].copy() for a in ("vx", "vy", "vz", "rung")]
    op = orc.KickParams(*[getattr(params, k) for k, _ in params._fields_])
    omr = orc.kick_epilogue(f[0][first:], f[1][first:], f[2][first:], *want, op, soft)
    for a, w in zip(("vx", "vy", "vz", "rung"), want):
        assert np.array_equal(getattr(p1, a)[first:], w), a
    assert mr == omr


@pytest.mark.parametrize("n,ng,order", [(16 * 4096 + 4095, 64, 2), (17 * 4096, 64, 1), (17 * 4096 - 1, 128, 1), (9001, 256, 2)])
def test_deposit_few_binning_counts_bit_exact(ct2, orc, n, ng, order):
    """16 and 17 binning workgroups, 64, 512 and 4,096 tiles: the counts summed by
    the placement or by a kernel of their own."""
    rng = np.random.default_rng(n)
    x, y, z = (rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32) for _ in range(3))
    load(ct2, x, y, z)
    ct2.set_force_options(1e-3, 1.0 / n, 0)
    ct2.pm_assignment(order)
    try:
        ct2.pm_init(ng, 1.25)
        ct2.pm_forces()
    finally:
        ct2.pm_assignment(1)
    assert np.array_equal(ct2.pm_density_download().ravel(), orc.mesh_deposit(x, y, z, ng.bit_length() - 1, order).ravel())


def fill_with_copies(ct2, base, copies):
    """A container of `copies` times the base positions, one after the other."""
    import ctypes as C

    from ct2_amd import _lib as L
    m = base[0].size
    ct2.particle_allocate(m * copies)
    ptr = L.ParticlePtrs()
    L.check(L.load().ct2_particles_device_ptrs(C.byref(ptr)))
    for dst, src in zip((ptr.x, ptr.y, ptr.z), base):
        for k in range(copies):
            L.check(L.load().ct2_memcpy_h2d(dst + 4 * m * k, src.ctypes.data_as(C.c_void_p), 4 * m))


def test_containers_beyond_one_tile_list(ct2):
    """2^28 particles (a tile list counts eight entries of each in an int, so the deposit takes more than one), 1,024
    copies of 2^18 on a 256^3 grid with TSC: density and force are 2^10 times one copy's exactly, whatever the list,
    and take about as long as for one copy fewer, which one list holds (2x allowed: binning runs again before the
    interpolation; one global atomic per particle and node took several times as long)."""
    import time

    from ct2_amd import _lib as L
    m, copies = 2 ** 18, 1024
    rng = np.random.default_rng(28)
    base = [rng.integers(0, 2 ** 32, m, dtype=np.uint64).astype(np.uint32) for _ in range(3)]
    ct2.set_force_options(1e-3, 2.0 ** -28, ct2.KERNEL_PLUMMER)
    ct2.pm_assignment(2)
    try:
        ct2.pm_init(256, 1.5)
        ct2.particle_allocate(m)
        ct2.particles_upload(*base)
        one = ct2.pm_forces()
        w = ct2.pm_density_download()
        took = []
        for k in (copies - 1, copies):
            fill_with_copies(ct2, base, k)
            best = np.inf
            for _ in range(3):
                t = time.perf_counter()
                L.check(L.load().ct2_pm_forces())
                ct2.synchronize()
                best = min(best, time.perf_counter() - t)
            took.append(best)
            print(f"{k} copies: {best * 1e3:.1f} ms", flush=True)
        assert np.array_equal(ct2.pm_density_download(), w * np.uint64(copies))
        for f, g in zip(ct2.forces_download(), one):
            assert (f.reshape(copies, m) == g * np.float32(copies)).all()
    finally:
        ct2.pm_assignment(1)
        ct2.particle_allocate(16)
    assert took[1] < 2 * took[0], took
