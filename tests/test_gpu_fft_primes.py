"""GPU: the mesh FFTs of sizes with a prime factor between 19 and 101, which are
rocFFT's, as every size that is no power of two: small and large sizes and primes,
one and two large primes, every small radix beside them, odd and even.  Against
numpy's FP64 transforms, with the tolerance of the other FFT tests
(relative rms 2e-6), and bit for bit with itself."""
import numpy as np
import pytest

import tigerpm_amd as T

pytestmark = pytest.mark.gpu

SIZES = [19, 38, 57, 93, 95, 97, 101, 133, 152, 202, 361, 384 - 4]


@pytest.fixture(scope="module")
def fctx():
    ctx = T.Context(0)
    ctx.set_params(T.baseline_params(32, 32, 2))
    yield ctx
    ctx.close()


def rel_rms(a, b):
    return float(np.sqrt((np.abs(a - b) ** 2).sum(dtype=np.float64) / (np.abs(b) ** 2).sum(dtype=np.float64)))


@pytest.mark.parametrize("M", SIZES)
def test_prime_sizes_match_numpy(fctx, M):
    a = np.random.default_rng(M).standard_normal((M, M, M), dtype=np.float32)
    ref = np.fft.rfftn(a.astype(np.float64))
    c = fctx.fft3d_r2c(a)
    assert rel_rms(c, ref) < 2e-6
    assert np.array_equal(c, fctx.fft3d_r2c(a))
    b = fctx.fft3d_c2r(ref.astype(np.complex64))
    assert rel_rms(b, a.astype(np.float64) * M ** 3) < 2e-6


@pytest.mark.parametrize("M", [38, 61, 93])
def test_potential_against_fp64(fctx, M):
    """The PM potential against the FP64 transforms of the same density grid and Green's
    table.  A transform whose error is eps of the spectrum's rms, in every mode
    alike, gives the potential's spectrum an error of eps rms(rho) rms(green), forward, and eps of
    itself, inverse; eps as above."""
    n_side = 32
    rng = np.random.default_rng(M)
    x, y, z = [rng.integers(0, 2 ** 32, n_side ** 3, dtype=np.uint64).astype(np.uint32) for _ in range(3)]
    fctx.set_params(T.baseline_params(n_side, M, 3))
    fctx.upload(x, y, z)
    fctx.gravity_long_compute()
    phi = np.asarray(fctx.get_phi(), np.float64).ravel()
    rho = fctx.get_density().view(np.int64).astype(np.float64).reshape(M, M, M) * 2.0 ** -32
    green = np.asarray(fctx.get_green(), np.float64).reshape(M, M, M // 2 + 1)
    spec = np.fft.rfftn(rho)
    ref = np.fft.irfftn(spec * green, s=(M, M, M), axes=(0, 1, 2)).ravel() * M ** 3
    eps = 2e-6
    rms = lambda a: float(np.sqrt((np.abs(a) ** 2).mean()))
    bound = eps * (1.0 + rms(spec) * rms(green) / rms(spec * green))
    assert rms(phi - ref) < bound * rms(ref)


@pytest.mark.parametrize("graph", [0, 1])
def test_batch_same_bits_as_single_box(graph):
    """Boxes on prime meshes in a batch, its step launched and replayed as a graph,
    against tpm_kick_treepm over three steps."""
    sides = [19, 38, 31]
    total = sum(n ** 3 for n in sides)
    t0 = 2.0 ** -12
    with T.Batch(max_particles=total, max_mesh_nodes=total, max_boxes=len(sides), order=4) as bt:
        bt.set_tuning(graph=graph)
        ids = [bt.add_zeldovich(T.box_spec(T.baseline_params(n, n, 4), t0=t0), n, 50 + n, 0.8) for n in sides]
        ctxs = []
        for i in ids:
            c = T.Context(0)
            bt.to_ctx(i, c)
            ctxs.append(c)
        for k in range(3):
            bt.step(0)
            for i, c in zip(ids, ctxs):
                c.kick_treepm(min_rung=0, scale=1.0, t0=t0, first_call=(k == 0))
                a, b = bt.download(i), c.download()
                for key in ("vx", "vy", "vz", "gx", "gy", "gz", "pot"):
                    assert np.array_equal(a[key], b[key]), (k, i, key)
        for c in ctxs:
            c.close()
