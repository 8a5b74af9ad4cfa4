"""GPU: the direct kernel leaves out neighbour cells and sources that are out of reach of a tile's box, round the box's
edges too: random particles with a few close groups across the edges, chain meshes from the coarsest (where offsets
wrap, C < 5) to the finest the cutoff allows, against the oracle's FP64 sums with the bound of the other tile tests
(2e-5 of the rms force); and what is left out is not evaluated."""
import numpy as np
import pytest

import tigerpm_amd as T
from test_gpu_tiles import forces, truth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", [8, 16, 64])
@pytest.mark.parametrize("mesh,C", [(18, 3), (64, 3), (64, 4), (64, 5), (64, 7), (64, 11), (256, 3), (256, 45)])
def test_cells_out_of_reach(gpu_ctx, tile, mesh, C):
    n = 6000
    rng = np.random.default_rng(mesh + C)
    p = T.baseline_params(mesh, mesh, 3, n_total=n)
    p.chain_dim = C
    pos = rng.uniform(0, 1, (n, 3))
    # groups within the cutoff of a corner, an edge and a face of the box and of a cell
    for k, at in enumerate(([0, 0, 0], [0, 0.3, 1], [0.5, 1, 0.2], [1 / C, 1 / C, 1 / C], [1 - 1 / C, 0.5, 0.999])):
        pos[200 * k : 200 * (k + 1)] = np.array(at) + p.rcut * rng.uniform(-1, 1, (200, 3))
    x, y, z = [np.floor((pos[:, d] % 1.0) * 2.0 ** 32).astype(np.uint64).astype(np.uint32) for d in range(3)]
    prev = gpu_ctx.get_tuning()
    try:
        gpu_ctx.set_params(p)
        gpu_ctx.set_tuning(tile_sinks=tile)
        gpu_ctx.upload(x, y, z)
        gpu_ctx.chainmesh_create()
        st = gpu_ctx.kick(flags=T.TPM_SKIP_PM | T.TPM_SKIP_KICK)
        cells = gpu_ctx.chainmesh_cells()
        d = gpu_ctx.download()
        g64, _ = truth(p, d["x"], d["y"], d["z"], cells, np.arange(n))
        g, _ = forces(gpu_ctx)
        norm = np.sqrt((g64 ** 2).sum(1).mean())
        assert np.sqrt(((g - g64) ** 2).sum(1).mean()) < 2e-5 * norm
        if mesh / C > 20:  # cells of 3.6 rcut and more
            assert st.executed_pairs < 0.5 * st.candidate_pairs
    finally:
        gpu_ctx.set_tuning(**prev)
