"""GPU: the chain-mesh order on both sides of the sizes where the sort changes its algorithm (one workgroup, merge sort,
onesweep from 2^17 particles on), with few and many key bits, equals the oracle's bit for bit."""
import numpy as np
import pytest

import oracle as orc
import tigerpm_amd as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C", [3, 23, 91])
@pytest.mark.parametrize("n", [1, 2, 1023, 1025, 4097, 2 ** 17 - 1, 2 ** 17, 2 ** 17 + 1, 2 ** 20])
def test_order_equals_oracle(gpu_ctx, n, C):
    rng = np.random.default_rng(n + C)
    p = T.baseline_params(32, 6 * C, 3, n_total=n)
    p.chain_dim = C
    # a third of the particles share 100 positions
    x, y, z = [rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32) for _ in range(3)]
    k = rng.integers(0, min(n, 100), n // 3)
    x[: n // 3], y[: n // 3], z[: n // 3] = x[k], y[k], z[k]
    gpu_ctx.set_params(p)
    gpu_ctx.upload(x, y, z)
    gpu_ctx.chainmesh_create()
    perm, cells = orc.chainmesh_sort(x, y, z, C)
    assert np.array_equal(gpu_ctx.chainmesh_perm(), perm)
    assert np.array_equal(gpu_ctx.chainmesh_cells(), cells)
    d = gpu_ctx.download()
    assert np.array_equal(d["x"], x[perm]) and np.array_equal(d["y"], y[perm]) and np.array_equal(d["z"], z[perm])
