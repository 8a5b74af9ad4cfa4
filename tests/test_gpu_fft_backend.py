"""GPU: which transform a mesh size takes.  Only the power-of-two sizes 16 .. 1024 have one of the library's own; every
other size goes through rocFFT and is the same bits whether the caller asks for rocFFT (fft = 1) or leaves the choice
to the library: smooth sizes, sizes whose factors include a square of a small prime, and large primes."""
import numpy as np
import pytest

import tigerpm_amd as T

pytestmark = pytest.mark.gpu

SIZES = [19, 25, 27, 38, 49, 61, 93, 97, 100, 101, 152, 202, 216]


@pytest.fixture(scope="module")
def fctx():
    ctx = T.Context(0)
    ctx.set_params(T.baseline_params(32, 32, 2))
    yield ctx
    ctx.close()


@pytest.mark.parametrize("M", SIZES)
def test_transform_is_rocfft_bit_for_bit(fctx, M):
    a = np.random.default_rng(M).standard_normal((M, M, M), dtype=np.float32)
    out = []
    for fft in (0, 1):
        fctx.set_tuning(fft=fft)
        c = fctx.fft3d_r2c(a)
        out.append((c, fctx.fft3d_c2r(c)))
    fctx.set_tuning()
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("interlace", [0, 1])
@pytest.mark.parametrize("M", [38, 61, 93, 100])
def test_potential_is_rocfft_bit_for_bit(fctx, M, interlace):
    rng = np.random.default_rng(M)
    pos = [rng.integers(0, 2 ** 32, 32 ** 3, dtype=np.uint64).astype(np.uint32) for _ in range(3)]
    fctx.set_params(T.baseline_params(32, M, 3, interlace=interlace))
    out = []
    for fft in (0, 1):
        fctx.set_tuning(fft=fft)
        fctx.upload(*pos)
        fctx.gravity_long_compute()
        out.append(np.asarray(fctx.get_phi()))
    fctx.set_tuning()
    assert np.array_equal(out[0], out[1])
