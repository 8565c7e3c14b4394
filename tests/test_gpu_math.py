"""The division and the Q-weight tests of awp_math.h against IEEE arithmetic
(numpy), over the domain that the header states."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def probe():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from awp_amd import _lib
    lib = _lib.load()

    def run(op, a, b=None):
        a = np.ascontiguousarray(a, np.float32)
        b = a if b is None else np.ascontiguousarray(b, np.float32)
        assert a.shape == b.shape
        da, db = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
        out = torch.empty_like(da)
        lib.awp_math_probe(op, da.data_ptr(), db.data_ptr(), out.data_ptr(), a.size,
                           torch.cuda.current_stream().cuda_stream)
        _lib.check()
        return out.cpu().numpy()

    return run


def _significands(exponent):
    return (np.arange(1 << 23, dtype=np.uint32) | np.uint32((exponent + 127) << 23)).view(np.float32)


def _random(rng, n, lo, hi):
    """Random signs and significands, exponents in [lo, hi]."""
    bits = rng.integers(0, 1 << 23, n, dtype=np.uint32)
    bits |= rng.integers(lo + 127, hi + 128, n, dtype=np.uint32) << np.uint32(23)
    return (bits | rng.integers(0, 2, n, dtype=np.uint32) << np.uint32(31)).view(np.float32)


def _same(got, want):
    bad = np.flatnonzero(got.view(np.uint32) != want.view(np.uint32))
    assert len(bad) == 0, (len(bad), bad[0], got[bad[0]], want[bad[0]])


@pytest.mark.parametrize("exponent", [-124, -60, -1, 0, 1, 37, 124])
def test_reciprocal_of_every_significand(probe, exponent):
    b = _significands(exponent)
    _same(probe(0, b), np.float32(1) / b)
    _same(probe(0, -b), np.float32(-1) / b)


def test_quotients(probe):
    rng = np.random.default_rng(1)
    n = 1 << 24
    for lo, hi in ((-2, 2), (-60, 60)):
        a, b = _random(rng, n, lo, hi), _random(rng, n, lo, hi)
        _same(probe(1, a, b), a / b)
    # every significand by thirds and by the moduli's range; quotients next to
    # a midpoint of two binary32 numbers: a = b (q + half an ulp), rounded
    for b in (3.0, 1.0e11 / 3):
        a = _significands(20)
        _same(probe(1, a, np.full_like(a, b)), a / np.float32(b))
    b, q = _random(rng, n, -30, 30), _random(rng, n, -30, 30)
    a = (b.astype(np.float64) * (q.astype(np.float64) * (1 + 2.0 ** -24))).astype(np.float32)
    _same(probe(1, a, b), a / b)


def test_special_quotients(probe):
    x = np.array([0.0, -0.0, 1.0, -3.0, 1e30, np.inf, -np.inf, np.nan], np.float32)
    a, b = (t.ravel() for t in np.meshgrid(x, x))
    with np.errstate(all="ignore"):
        want = a / b
    got = probe(1, a, b)
    nan = np.isnan(want)
    assert np.isnan(got[nan]).all()
    _same(got[~nan], want[~nan])
    with np.errstate(all="ignore"):
        for c in (1.0, 2.0, 8.0, 16.0):
            want = np.float32(c) / x[:-1]
            _same(probe(2, np.full(7, c, np.float32), x[:-1]), want)


def test_small_numerators_stay_within_two_ulps(probe):
    """Below 2^-100, where the residual is flushed: a RN(1/b) has two roundings
    of 2^-24 each, less than two ulps."""
    rng = np.random.default_rng(2)
    a, b = _random(rng, 1 << 22, -120, -101), _random(rng, 1 << 22, -5, 5)
    got, want = probe(1, a, b), a / b
    ulps = np.abs(got.view(np.int32).astype(np.int64) - want.view(np.int32))
    assert ulps.max() <= 2


def test_powers_of_two_over_a_sum(probe):
    rng = np.random.default_rng(3)
    for c in (1.0, 2.0, 8.0, 16.0):
        b = _random(rng, 1 << 22, -100, 100)
        _same(probe(2, np.full_like(b, c), b), np.float32(c) / b)


def test_q_thresholds(probe):
    """1/(2q) <= 200 in binary64 and binary32, on every float around 0.0025
    and on random ones; -0 and NaN, where both branches agree, are left out."""
    rng = np.random.default_rng(4)
    at = int(np.float32(0.0025).view(np.uint32))
    near = np.arange(at - 5000, at + 5001, dtype=np.uint32).view(np.float32)
    q = np.concatenate([near, -near, _random(rng, 1 << 22, -120, 100),
                        np.array([0.0, np.inf, -np.inf, 1e-30], np.float32)])
    with np.errstate(divide="ignore"):
        low64 = 1.0 / (2.0 * q.astype(np.float64)) <= 200.0
        low32 = np.float32(1) / (np.float32(2) * q) <= np.float32(200)
    assert np.array_equal(probe(3, q) != 0, low64)
    assert np.array_equal(probe(4, q) != 0, low32)
