"""GPU parity of the 3-D FFT against the FP64 oracle and numpy, through the C
ABI (the transform the PM path needs: fft.hpp:28-29, particle.cpp:230,261)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rel_l2(a, b):
    return np.linalg.norm((a - b).ravel()) / np.linalg.norm(b.ravel())


@pytest.mark.parametrize("n", [8, 16, 32, 64])
def test_fft3d_fp32_vs_oracle(ct2, orc, n):
    rng = np.random.default_rng(n)
    z = rng.standard_normal((n,) * 3) + 1j * rng.standard_normal((n,) * 3)
    for d in (1, -1):
        got = ct2.fft3d(z.astype(np.complex64), d)
        want = orc.fft3d(z, d)
        assert rel_l2(got, want) < 1e-6, (n, d, rel_l2(got, want))


@pytest.mark.parametrize("n", [8, 16, 32, 64])
def test_fft3d_fp64_vs_oracle(ct2, orc, n):
    rng = np.random.default_rng(100 + n)
    z = rng.standard_normal((n,) * 3) + 1j * rng.standard_normal((n,) * 3)
    for d in (1, -1):
        assert rel_l2(ct2.fft3d(z, d), orc.fft3d(z, d)) < 1e-14


def test_fft3d_golden(ct2):
    import os
    g = np.load(os.path.join(os.path.dirname(__file__), "golden", "fft_golden.npz"))
    for n in (8, 16):
        assert rel_l2(ct2.fft3d(g[f"c3d_in_{n}"], 1), g[f"c3d_out_{n}"]) < 1e-14
        assert rel_l2(ct2.fft3d(g[f"c3d_in_{n}"].astype(np.complex64), 1), g[f"c3d_out_{n}"]) < 1e-6


@pytest.mark.parametrize("n", [128, 256])
def test_fft3d_fp32_vs_numpy_fp64(ct2, n):
    """The GPU configuration's gate: 256^3 complex FP32, rel L2 <= 1e-5 against
    an FP64 transform, forward and round trip."""
    rng = np.random.default_rng(256)
    z = (rng.standard_normal((n,) * 3) + 1j * rng.standard_normal((n,) * 3)).astype(np.complex64)
    want = np.fft.fftn(z.astype(np.complex128))
    got = ct2.fft3d(z, 1)
    assert rel_l2(got, want) < 1e-5
    back = ct2.fft3d(got, -1) / n ** 3
    assert rel_l2(back, z.astype(np.complex128)) < 1e-5


@pytest.mark.parametrize("f64", [False, True])
@pytest.mark.parametrize("d", [1, -1])
def test_fft3d_in_groups_of_planes(ct2, f64, d):
    """Cubes of 1 GB and more take their z and y passes by groups of planes (512^3:
    96 or 48 planes, the last group smaller): a product of three random lines,
    whose transform is the product of theirs."""
    n, rng = 512, np.random.default_rng(5)
    a = rng.standard_normal((3, n)) + 1j * rng.standard_normal((3, n))
    t = np.fft.fft(a) if d > 0 else np.fft.ifft(a, norm="forward")
    cube = [(v[0][:, None, None] * v[1][:, None]) * v[2] for v in (a, t)]
    got = ct2.fft3d(cube[0] if f64 else cube[0].astype(np.complex64), d)
    assert rel_l2(got, cube[1]) < (1e-14 if f64 else 1e-6)


def test_fft3d_fp32_of_1024(ct2):
    """1024^3, the largest: 24 planes to a group, the last one of 16.  A product of three random lines forward,
    compared with the product of their FP64 transforms on planes of every group, then back to itself."""
    import ctypes as C

    from ct2_amd import _lib as L
    n, rng = 1024, np.random.default_rng(10)
    a = (rng.standard_normal((3, n)) + 1j * rng.standard_normal((3, n))).astype(np.complex64)
    t = np.fft.fft(a.astype(np.complex128))
    buf = ct2.DeviceBuffer(n ** 3 * 8)
    plane, slab = a[1][:, None] * a[2], np.empty((8, n, n), np.complex64)
    for i in range(0, n, 8):
        for j in range(8):
            np.multiply(plane, a[0][i + j], out=slab[j])
        L.check(L.load().ct2_memcpy_h2d(buf.ptr + i * n * n * 8, slab.ctypes.data_as(C.c_void_p), slab.nbytes))
    some = sorted(set(range(0, n, 23)) | {1, 512, 1007, 1008, 1022, 1023})
    for d, lines in ((1, t), (-1, a.astype(np.complex128) * [[n], [n], [n]])):
        ct2.fft3d_device(buf, n, d)
        plane, err, ref = lines[1][:, None] * lines[2], 0.0, 0.0
        for i in some:
            L.check(L.load().ct2_memcpy_d2h(slab[0].ctypes.data_as(C.c_void_p), buf.ptr + i * n * n * 8, n * n * 8))
            want = lines[0][i] * plane
            err += np.linalg.norm(slab[0] - want) ** 2
            ref += np.linalg.norm(want) ** 2
        assert (err / ref) ** 0.5 < 1e-6, (d, (err / ref) ** 0.5)
    buf.close()


def test_fft3d_512_round_trip_and_delta(ct2):
    """512^3 (the PM grid of the clustered and stepping configurations):
    delta -> constant, and forward/inverse round trip."""
    n = 512
    buf = ct2.DeviceBuffer(n ** 3 * 8)
    z = np.zeros((n,) * 3, np.complex64)
    z[3, 5, 7] = 1.0
    buf.upload(z)
    ct2.fft3d_device(buf, n, 1)
    out = buf.download(np.empty_like(z))
    k = np.arange(n)
    ph = np.exp(-2j * np.pi * 7 * k / n)
    assert np.allclose(out[0, 0, :], ph, atol=1e-5)
    assert np.allclose(np.abs(out[::37, ::41, ::43]), 1.0, atol=1e-5)
    rng = np.random.default_rng(512)
    z = (rng.standard_normal((n,) * 3, dtype=np.float32) + 1j * rng.standard_normal((n,) * 3, dtype=np.float32)).astype(np.complex64)
    buf.upload(z)
    ct2.fft3d_device(buf, n, 1)
    ct2.fft3d_device(buf, n, -1)
    back = buf.download(np.empty_like(z)) / np.float32(n ** 3)
    assert rel_l2(back, z) < 1e-5
    buf.close()


def test_fft3d_rejects_bad_sizes(ct2):
    from ct2_amd import Ct2Error
    buf = ct2.DeviceBuffer(1024)
    for n, d in ((12, 1), (4, 1), (2048, 1), (64, 0)):
        with pytest.raises(Ct2Error):
            ct2.fft3d_device(buf, n, d)
    buf.close()


def test_cfg2_fft_of_the_cic_density(ct2):
    """The GPU configuration's FFT gate on the field it names: the CIC density
    of N = 128^3 lattice + Gaussian(0.2 cell) particles on the 256^3 grid (the
    library's own deposit), as complex FP32, transformed forward and back on
    the device; rel L2 <= 1e-5 against numpy's FP64 transform of the same
    values, for the density and for its contrast (the mean's k = 0 term
    removed, so that the check is not carried by that one mode)."""
    side, ng = 128, 256
    x, y, z = ct2.ic_lattice(side, 0.2, 1)
    ct2.particle_allocate(x.size)
    ct2.particles_upload(x, y, z)
    ct2.set_force_options(float(np.float32(1.0 / (50 * side))), float(np.float32(1.0 / x.size)), 0)
    ct2.pm_assignment(1)
    ct2.pm_init(ng, 1.25)
    ct2.pm_forces()
    W = ct2.pm_density_download()
    rho = (W.astype(np.float64) * 2.0 ** -32).astype(np.float32)  # particles per cell
    assert rho.sum(dtype=np.float64) == pytest.approx(x.size, rel=1e-6)
    for field in (rho, rho / np.float32(rho.mean()) - np.float32(1.0)):
        zc = field.astype(np.complex64)
        want = np.fft.fftn(zc.astype(np.complex128))
        got = ct2.fft3d(zc, 1)
        assert rel_l2(got, want) < 1e-5, rel_l2(got, want)
        back = ct2.fft3d(got, -1) / ng ** 3
        assert rel_l2(back, zc.astype(np.complex128)) < 1e-5
