"""The pieces of the filtered potential that the near-field kernel reads
(ct2_near_potential_table), evaluated as the kernel evaluates them, against the
closed forms of potential and force in FP64 (scipy's erf): values over the whole
range, both ends of it, the r -> 0 limits, and continuity between pieces."""
import numpy as np
import pytest
from scipy.special import erf

from ct2_amd import api

C = 2 / np.sqrt(np.pi)
LAST = 512  # the last piece


def closed(r2, rs):
    u = np.sqrt(r2) / (2 * rs)
    kl = (erf(u) - C * u * np.exp(-u * u)) / u ** 3 / (2 * rs) ** 3
    pl = erf(u) / u / (2 * rs)
    return kl, pl


def evaluate(p4, r2, rc):
    """near_pair's steps: t = r^2 * tscale in FP32, the piece from the low bits of t + 1.5 2^23, then value and
    derivative side by side (here in FP64, so that what is left is the table's and the coordinate's)."""
    tscale = np.float32(LAST / rc ** 2)
    t = r2.astype(np.float32) * tscale
    tm = t + np.float32(1.5 * 2 ** 23)
    i = tm.view(np.int32) - 0x4B400000
    assert i.min() >= 0 and i.max() <= LAST
    f = (t - (tm - np.float32(1.5 * 2 ** 23))).astype(np.float64)
    assert np.abs(f).max() <= 0.5 and (f[i == 0] >= 0).all()
    c = p4.astype(np.float64)[i]
    v = c[:, 3] * f + c[:, 2]
    d = c[:, 3] * f + v
    v = v * f + c[:, 1]
    d = d * f + v
    v = v * f + c[:, 0]
    return -2.0 * tscale * d, v, i


@pytest.mark.parametrize("rs_cells,ng,rcut_rs,force,potential", [
    (1.5, 256, 5.5, 3e-7, 2e-7), (2.5, 512, 5.5, 3e-7, 2e-7), (1.0, 64, 4.0, 3e-7, 2e-7), (4.0, 512, 8.0, 4e-7, 2e-7),
    (1.0, 64, 12.0, 9e-7, 2e-7), (1.0, 64, 20.0, 1.4e-5, 4e-7)])
def test_pieces_match_closed_forms(rs_cells, ng, rcut_rs, force, potential):
    """Bounds: the cubic pieces' own error (6e-9, 5e-8, 6e-7 and 1.3e-5 of the force to 5.5, 8, 12 and 20 rs), FP32
    coefficients (6e-8) and the coordinate's two roundings, 2^-24 of t each, through the slope d ln k / d ln t, at
    most 3/2 (1.8e-7; 1/2 and 6e-8 for the potential)."""
    rs = rs_cells / ng * 2.0 ** 32
    rc = rcut_rs * rs
    p4 = api.near_potential_table(rs, rc)
    rng = np.random.default_rng(3)
    r2 = np.concatenate([rng.uniform(0.0, 1.0, 50000) ** 2, rng.uniform(0.0, 1.0, 50000)]) * rc ** 2
    # around the ends of the pieces and the range (r^2 = rcut^2 may round into piece 512 only)
    ends = (np.arange(LAST) + 0.5) * rc ** 2 / LAST
    r2 = np.concatenate([r2, ends, np.nextafter(ends.astype(np.float32), np.float32(0)), ends * (1 + 1e-6), [rc ** 2]])
    r2 = r2[r2 > (1e-3 * rs) ** 2].astype(np.float32)
    kl, pl, i = evaluate(p4, r2, rc)
    assert set(i) == set(range(LAST + 1))
    wk, wp = closed(r2.astype(np.float64), rs)
    assert np.max(np.abs(kl - wk) / wk) < force
    assert np.max(np.abs(pl - wp) / wp) < potential


def test_limits_at_zero_separation():
    rs = 1.5 / 256 * 2.0 ** 32
    kl, pl, i = evaluate(api.near_potential_table(rs, 5.5 * rs), np.zeros(1, np.float32), 5.5 * rs)
    assert i[0] == 0
    assert kl[0] == pytest.approx(C * (2 / 3) / (2 * rs) ** 3, rel=2e-7)
    assert pl[0] == pytest.approx(C / (2 * rs), rel=1e-7)


def test_pieces_are_continuous():
    """Piece i at f = 1/2 and piece i + 1 at -1/2: FP32 coefficients (value: two half ulps; derivative: the same)."""
    rs = 2.0 / 128 * 2.0 ** 32
    c = api.near_potential_table(rs, 5.5 * rs).astype(np.float64)
    value = lambda c, f: ((c[:, 3] * f + c[:, 2]) * f + c[:, 1]) * f + c[:, 0]
    slope = lambda c, f: (3 * c[:, 3] * f + 2 * c[:, 2]) * f + c[:, 1]
    for fn in (value, slope):
        a, b = fn(c[:-1], 0.5), fn(c[1:], -0.5)
        assert np.max(np.abs(a - b) / np.abs(b)) < 2.5e-7


def test_bad_arguments():
    from ct2_amd._lib import Ct2Error
    with pytest.raises(Ct2Error):
        api.near_potential_table(0.0, 1.0)
    with pytest.raises(Ct2Error):
        api.near_potential_table(1.0, 0.0)
