"""GPU: the scan of the cells' tile counts on both sides of its chunk (2048 cells) and of the number of cells that one
workgroup takes (16384): every active particle is in exactly one tile, seen from its force and potential, against the
oracle's FP64 sums with the bound of the other tile tests (2e-5 of the rms force); the counts that a kick reports."""
import numpy as np
import pytest

import tigerpm_amd as T
from test_gpu_tiles import forces, truth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C", [3, 4, 6, 12, 13, 20, 25, 26, 30])
@pytest.mark.parametrize("n", [1, 300, 20000])
def test_scan_sizes(gpu_ctx, C, n):
    rng = np.random.default_rng(C + n)
    mesh = 6 * C
    p = T.baseline_params(mesh, mesh, 3, n_total=n)
    p.chain_dim = C
    x, y, z = [rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32) for _ in range(3)]
    rung = rng.integers(0, 2, n).astype(np.int8)
    gpu_ctx.set_params(p)
    gpu_ctx.upload(x, y, z, rung=rung)
    gpu_ctx.chainmesh_create()
    cells = gpu_ctx.chainmesh_cells()
    for min_rung in (1, 0):
        st = gpu_ctx.kick(min_rung=min_rung, flags=T.TPM_SKIP_PM | T.TPM_SKIP_KICK)
        d = gpu_ctx.download()
        g, pot = forces(gpu_ctx)
        act = d["rung"] >= min_rung
        assert np.array_equal((g != 0).any(1) | (pot != 0), act)
    g64, _ = truth(p, d["x"], d["y"], d["z"], cells, np.arange(n))
    norm = np.sqrt((g64 ** 2).sum(1).mean())
    assert np.sqrt(((g - g64) ** 2).sum(1).mean()) <= 2e-5 * norm
    count = np.diff(cells).reshape(C, C, C)
    near = sum(np.roll(count, s, (0, 1, 2)) for s in np.ndindex(3, 3, 3)) if C > 3 else count.sum()
    near = np.roll(near, (-1, -1, -1), (0, 1, 2)) if C > 3 else near
    assert st.candidate_pairs == (count * near).sum()
    assert st.n_tiles == ((count + 15) // 16).sum()
