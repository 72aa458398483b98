"""GPU drop-ins for ct2's own FFT API (fft.hpp:18-29) in ct2's conventions --
bit-reversed 1-D input, half-complex real output, 4-lane interleaving, the
planar 3-D half spectrum -- against the FP64 oracle (itself pinned by numpy
golden vectors and the DFT's invariants)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def relerr(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("N", [2, 8, 32, 256, 1024, 4096])
@pytest.mark.parametrize("lanes", [1, 4])
@pytest.mark.parametrize("dir", [1, -1])
def test_fft_complex_1d(ct2, orc, N, lanes, dir):
    batch = 3
    X = np.random.default_rng(N + lanes).standard_normal(batch * 2 * lanes * N)
    got = ct2.fft_complex(X, N, dir, lanes)
    want = np.concatenate([orc.fft_complex(g, N, dir, lanes) for g in np.split(X, batch)])
    assert relerr(got, want) < 1e-14


@pytest.mark.parametrize("N", [2, 8, 64, 512, 4096])
@pytest.mark.parametrize("lanes", [1, 4])
@pytest.mark.parametrize("dir", [1, -1])
def test_fft_real_1d(ct2, orc, N, lanes, dir):
    batch = 5
    X = np.random.default_rng(7 * N + lanes).standard_normal(batch * lanes * N)
    got = ct2.fft_real(X, N, dir, lanes)
    want = np.concatenate([orc.fft_real(g, N, dir, lanes) for g in np.split(X, batch)])
    assert relerr(got, want) < 1e-14


@pytest.mark.parametrize("N,lanes,batch", [(2, 1, 700), (4, 4, 130), (16, 1, 129), (64, 4, 33), (128, 1, 17), (512, 1, 5),
                                           (1024, 4, 2), (2048, 1, 3), (2048, 4, 3), (4096, 1, 2), (4096, 4, 2)])
@pytest.mark.parametrize("dir", [1, -1])
def test_fft_1d_ragged_batches(ct2, orc, N, lanes, batch, dir):
    """Batches that end inside a workgroup's set of transforms, every radix
    remainder (2, 4, none) and the sizes where a group's lanes share a
    workgroup or split over two.  A transform rounds to a few FP64 ulps per
    step, so 1e-14 bounds log2 N of them."""
    rng = np.random.default_rng(N * lanes + batch)
    scale = np.repeat(10.0 ** rng.integers(-6, 7, batch), lanes * N)  # transforms of unequal size stay apart
    X = rng.standard_normal(batch * lanes * N) * scale
    got, want = ct2.fft_real(X, N, dir, lanes), [orc.fft_real(g, N, dir, lanes) for g in np.split(X, batch)]
    for g, w in zip(np.split(got, batch), want):
        assert relerr(g, w) < 1e-14
    X = rng.standard_normal(2 * batch * lanes * N)
    got, want = ct2.fft_complex(X, N, dir, lanes), [orc.fft_complex(g, N, dir, lanes) for g in np.split(X, batch)]
    for g, w in zip(np.split(got, batch), want):
        assert relerr(g, w) < 1e-14


@pytest.mark.parametrize("N,lanes,batch", [
    (2, 1, 2049), (8, 1, 4097), (16, 4, 129), (32, 4, 128), (32, 4, 129), (64, 1, 2048), (64, 1, 4097), (128, 1, 255),
    (128, 4, 64), (128, 4, 300), (256, 1, 2049), (256, 4, 65), (512, 1, 1025), (512, 4, 33), (1024, 1, 512), (1024, 1, 513),
    (1024, 4, 32), (1024, 4, 33), (2048, 1, 257), (2048, 4, 32), (2048, 4, 65), (4096, 4, 33)])
def test_fft_1d_at_the_edges_of_the_small_batches(ct2, orc, N, lanes, batch):
    """Batches at and past the sizes where a transform has a workgroup of its own, and where a workgroup takes fewer
    transforms than it could (down to a group's lanes, and to single ones).  Bounds as above."""
    rng = np.random.default_rng(N * lanes + batch)
    X = rng.standard_normal(batch * lanes * N)
    Z = rng.standard_normal(2 * batch * lanes * N)
    for dir in (1, -1):
        for got, want in ((ct2.fft_real(X, N, dir, lanes), [orc.fft_real(g, N, dir, lanes) for g in np.split(X, batch)]),
                          (ct2.fft_complex(Z, N, dir, lanes), [orc.fft_complex(g, N, dir, lanes) for g in np.split(Z, batch)])):
            d, w = np.split(got, batch) - np.array(want), np.array(want)
            assert (np.linalg.norm(d, axis=1) < 1e-14 * np.linalg.norm(w, axis=1)).all()


def test_small_1d_batches_take_little_more_than_a_launch(ct2):
    """200 calls in a row: 100 real transforms of 256 points against one of 2 points, which is a launch and little
    else (3.6 us; 4.0 are expected for the batch, 1.8 times the launch allowed)."""
    import ctypes as C
    import time

    from ct2_amd import _lib as L
    buf = C.c_void_p()
    L.check(L.load().ct2_dev_alloc(100 * 256 * 8, C.byref(buf)))
    try:
        zero = np.zeros(100 * 256)
        L.check(L.load().ct2_memcpy_h2d(buf, zero.ctypes.data_as(C.c_void_p), zero.nbytes))
        took = []
        for N, batch in ((2, 1), (256, 100)):
            best = np.inf
            for _ in range(12):
                ct2.synchronize()
                t = time.perf_counter()
                for _ in range(200):
                    L.check(L.load().ct2_fft_real_1d(buf, N, 1, 1, batch))
                ct2.synchronize()
                best = min(best, (time.perf_counter() - t) / 200)
            took.append(best)
    finally:
        L.check(L.load().ct2_dev_free(buf))
    print(f"one of 2: {took[0] * 1e6:.2f} us, 100 of 256: {took[1] * 1e6:.2f} us", flush=True)
    assert took[1] < 1.8 * took[0], took


def test_fft_real_matches_numpy_after_scramble(ct2, orc):
    """End to end in ct2's order of calls (fft_test.cpp:108-127): scramble on
    the device, then fft_real; the half-complex result equals numpy's rfft."""
    N = 1024
    x = np.random.default_rng(3).standard_normal(N)
    Xs = ct2.scramble(x, 1, N, 1)
    assert np.array_equal(Xs, orc.scramble(x, 1, N, 1))
    H = ct2.fft_real(Xs, N)
    F = np.fft.rfft(x)
    assert np.allclose(H[:N // 2 + 1], F.real, atol=1e-11)
    assert np.allclose(H[N - 1:N // 2:-1], F.imag[1:N // 2], atol=1e-11)


@pytest.mark.parametrize("N1,N2,N3", [(1, 16, 1), (3, 64, 5), (2, 1024, 4)])
def test_scramble(ct2, orc, N1, N2, N3):
    X = np.random.default_rng(N2).standard_normal(N1 * N2 * N3)
    assert np.array_equal(ct2.scramble(X, N1, N2, N3), orc.scramble(X, N1, N2, N3))


@pytest.mark.parametrize("N", [4, 16, 32])
def test_transposes(ct2, orc, N):
    X = np.random.default_rng(N).standard_normal(N ** 3)
    assert np.array_equal(ct2.transpose_yz(X, N), orc.transpose_yz(X, N))
    Y = ct2.transpose_r2c(X, N)
    assert np.array_equal(Y, orc.transpose_r2c(X, N))
    assert np.array_equal(ct2.transpose_c2r(Y, N), orc.transpose_c2r(Y, N))


@pytest.mark.parametrize("N", [8, 32, 64])
def test_fft_r2c_c2r_3d(ct2, orc, N):
    X = np.random.default_rng(N).standard_normal(N ** 3)
    Y = ct2.fft_r2c_3d(X)
    assert relerr(Y, orc.fft_r2c_3d(X.reshape(N, N, N))) < 1e-14
    R = np.fft.rfftn(X.reshape(N, N, N))  # [i][j][k<N/2+1]
    h = N * N * (N // 2 + 1)
    assert np.allclose(Y[:h], R.real.ravel(), atol=1e-10 * N ** 1.5)
    assert np.allclose(Y[h:], R.imag.ravel(), atol=1e-10 * N ** 1.5)
    Z = ct2.fft_c2r_3d(Y, N)
    assert relerr(Z, orc.fft_c2r_3d(Y, N).ravel()) < 1e-14
    assert relerr(Z / N ** 3, X) < 1e-14


@pytest.mark.parametrize("N", [8, 16, 128, 256, 512])
def test_fft_r2c_c2r_3d_half_spectrum(ct2, N):
    """Every size class of the half-spectrum passes (one-stage and multi-stage
    rows, 4 to 16 columns per workgroup, the kz = N/2 plane on its own) against
    numpy, with a mean much larger than the fluctuations.  The FP64 transforms
    round to a few ulps per stage: 1e-14."""
    X = np.random.default_rng(N).standard_normal(N ** 3) + 50.0
    Y = ct2.fft_r2c_3d(X)
    R = np.fft.rfftn(X.reshape(N, N, N))
    h = N * N * (N // 2 + 1)
    assert relerr(Y[:h], R.real.ravel()) < 1e-14
    Y[0], R[0, 0, 0] = 0.0, 0.0  # the fluctuations on their own, against the error of the mean
    e = np.hypot(Y[:h] - R.real.ravel(), Y[h:] - R.imag.ravel())
    assert np.linalg.norm(e) < 50.0 * 1e-14 * np.linalg.norm(R) and e[N // 2::N // 2 + 1].max() < 50.0 * 1e-14 * N ** 1.5 * 10
    Z = ct2.fft_c2r_3d(Y, N)
    assert relerr(Z / N ** 3, X - X.mean()) < 50.0 * 1e-14


@pytest.mark.parametrize("N", [8, 32])
def test_fft_c2r_3d_of_any_half_spectrum(ct2, N):
    """A planar spectrum whose kz = 0 and N/2 planes have no Hermitian symmetry:
    the result is the real part of the complex transform, those planes taken as
    they are and the columns above N/2 as the partners' conjugates."""
    h = N // 2 + 1
    Y = np.random.default_rng(N).standard_normal(2 * N * N * h)
    C = (Y[:N * N * h] + 1j * Y[N * N * h:]).reshape(N, N, h)
    full = np.zeros((N, N, N), complex)
    full[:, :, :h] = C
    neg = (-np.arange(N)) % N
    full[:, :, h:] = np.conj(C[neg][:, neg][:, :, h - 2:0:-1])
    want = (np.fft.ifftn(full) * N ** 3).real
    assert relerr(ct2.fft_c2r_3d(Y, N), want.ravel()) < 1e-14


def test_fft_r2c_c2r_3d_in_place(ct2):
    """Input and output in one device buffer (the library reads all of the
    input before it writes)."""
    from ct2_amd import _lib

    N = 32
    h = N * N * (N // 2 + 1)
    X = np.random.default_rng(1).standard_normal(N ** 3)
    buf = ct2.DeviceBuffer(2 * h * 8)
    buf.upload(X)
    _lib.check(_lib.load().ct2_fft_r2c_3d(buf.ptr, buf.ptr, N))
    ct2.synchronize()
    assert np.array_equal(buf.download(np.empty(2 * h)), ct2.fft_r2c_3d(X))
    _lib.check(_lib.load().ct2_fft_c2r_3d(buf.ptr, buf.ptr, N))
    ct2.synchronize()
    assert relerr(buf.download(np.empty(N ** 3)) / N ** 3, X) < 1e-14
    buf.close()


def test_twiddles(ct2, orc):
    for N in (8, 1000, 4096):
        for a, b in zip(ct2.twiddles(N), orc.twiddles(N)):
            assert np.allclose(a, b, rtol=0, atol=1e-15)


def test_argument_checks(ct2):
    from ct2_amd._lib import Ct2Error
    with pytest.raises(Ct2Error):
        ct2.fft_complex(np.zeros(2 * 3000), 3000)
    with pytest.raises(Ct2Error):
        ct2.fft_real(np.zeros(8 * 8192), 8192)
    with pytest.raises(Ct2Error):
        ct2.fft_complex(np.zeros(2 * 3 * 16), 16, lanes=3)
