"""Deposit blocks shared by several workgroups: boxes of few blocks with many particles give the oracle's integer
grid, whatever the number of shares (the sums are integers, so equality is exact)."""
import numpy as np
import pytest

import oracle as O
import tigerpm_amd as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [2, 3, 4])
@pytest.mark.parametrize("n,mesh,chain_dim", [(700, 20, 3), (1500, 20, 3), (30011, 20, 3), (200003, 30, 5), (65536, 64, 11)])
def test_shared_blocks_give_the_oracles_grid(gpu_ctx, order, n, mesh, chain_dim):
    rng = np.random.default_rng(n + order)
    x, y, z = [rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32) for _ in range(3)]
    x[: n // 2] //= 8  # half of the particles in a corner: blocks of very different counts, empty ones among them
    y[: n // 2] //= 8
    z[: n // 2] //= 8
    p = T.baseline_params(mesh, mesh, order, n_total=n)
    assert p.chain_dim == chain_dim
    gpu_ctx.set_params(p)
    gpu_ctx.upload(x, y, z)
    gpu_ctx.chainmesh_create()
    gpu_ctx.gravity_long_compute()
    got = gpu_ctx.get_density()
    assert np.array_equal(got, O.deposit(x, y, z, mesh, order).ravel())


def test_shared_blocks_in_a_batch():
    """A crowded box beside a small one: the same potential, bit for bit, as alone."""
    rng = np.random.default_rng(5)
    n = 40000
    x, y, z = [rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32) for _ in range(3)]
    spec = T.box_spec(T.baseline_params(20, 20, 4, n_total=n), t0=2.0 ** -12)
    small = T.box_spec(T.baseline_params(18, 18, 4, n_total=500), t0=2.0 ** -12)
    with T.Batch(n + 500, 20 ** 3 + 18 ** 3 + 1000, 2, 4) as bt:
        i = bt.add(spec, x, y, z)
        bt.add(small, x[:500], y[:500], z[:500])
        with T.Context(0) as c:
            bt.to_ctx(i, c)
            bt.step(0)
            c.kick_treepm(0, 1.0, 2.0 ** -12, True)
            a, b = bt.download(i), c.download()
    for k in ("gx", "gy", "gz", "pot"):
        assert np.array_equal(a[k], b[k]), k
