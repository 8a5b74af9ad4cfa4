"""GPU: a chain cell far more crowded than the others.  Its tiles are made by many waves: forces against the oracle's
FP64 sums with the bound of the other tile tests (2e-5 of the rms force), for every law and subset that makes tiles its own way, and
the kick alone, whose time does not depend on how the particles are spread over the cells."""
import numpy as np
import pytest

import tigerpm_amd as T
from test_gpu_tiles import forces, truth

pytestmark = pytest.mark.gpu


def crowded(n_cell, n_rest, C, seed):
    """n_cell particles in cell (C // 2)^3, n_rest over the whole box."""
    rng = np.random.default_rng(seed)
    a = (C // 2 + rng.uniform(0.01, 0.99, (n_cell, 3))) / C
    pos = np.concatenate([a, rng.uniform(0, 1, (n_rest, 3))])
    rng.shuffle(pos)
    return [np.floor(pos[:, d] * 2.0 ** 32).astype(np.uint64).astype(np.uint32) for d in range(3)]


@pytest.mark.parametrize("tile", [8, 16, 64])
@pytest.mark.parametrize("n_cell,n_rest", [(1100, 3000), (9001, 3000), (20000, 2 ** 19)])
def test_forces_of_a_crowded_cell(gpu_ctx, tile, n_cell, n_rest):
    C = 11
    p = T.baseline_params(64, 64, 3, n_total=n_cell + n_rest)
    assert p.chain_dim == C
    x, y, z = crowded(n_cell, n_rest, C, n_cell)
    rng = np.random.default_rng(tile)
    rung = (rng.uniform(size=len(x)) < 0.6).astype(np.int8)
    prev = gpu_ctx.get_tuning()
    try:
        gpu_ctx.set_params(p)
        gpu_ctx.set_tuning(tile_sinks=tile)
        gpu_ctx.upload(x, y, z, rung=rung)
        gpu_ctx.chainmesh_create()
        cells = gpu_ctx.chainmesh_cells()
        d = gpu_ctx.download()
        c = (C // 2 * C + C // 2) * C + C // 2
        sinks = rng.integers(cells[c], cells[c + 1], 200)
        g64, _ = truth(p, d["x"], d["y"], d["z"], cells, sinks)
        norm = np.sqrt((g64 ** 2).sum(1).mean())
        for min_rung, newton in ((0, 0), (1, 0), (0, 1)):
            gpu_ctx.set_tuning(tile_sinks=tile, pp_newton=newton)
            gpu_ctx.upload(x, y, z, rung=rung)  # clears the forces
            gpu_ctx.chainmesh_create()
            gpu_ctx.kick(min_rung=min_rung, flags=T.TPM_SKIP_PM | T.TPM_SKIP_KICK)
            g, pot = forces(gpu_ctx)
            act = d["rung"][sinks] >= min_rung
            assert np.sqrt(((g[sinks] - g64)[act] ** 2).sum(1).mean()) < 2e-5 * norm, (min_rung, newton)
            # every active sink has a tile, no other
            assert np.array_equal((g != 0).any(1) | (pot != 0), d["rung"] >= min_rung)
    finally:
        gpu_ctx.set_tuning(**prev)


@pytest.mark.parametrize("n_cell", [2047, 2049, 9000])
@pytest.mark.parametrize("lo,hi", [((0, 0, 0), (11, 11, 11)), ((5, 5, 5), (6, 6, 6)), ((0, 0, 0), (11, 11, 5))])
def test_kick_alone_of_a_crowded_cell(gpu_ctx, n_cell, lo, hi):
    """The kick without forces leaves v but for the potential's constant: every active particle of the box's cells is visited once
    (rung and potential set), no other."""
    C = 11
    p = T.baseline_params(64, 64, 3, n_total=n_cell + 3000)
    x, y, z = crowded(n_cell, 3000, C, n_cell)
    rung = (np.random.default_rng(1).uniform(size=len(x)) < 0.6).astype(np.int8)
    gpu_ctx.set_params(p)
    gpu_ctx.upload(x, y, z, rung=rung)
    gpu_ctx.chainmesh_create()
    d = gpu_ctx.download()
    gpu_ctx.kick_box(lo, hi, min_rung=1, flags=T.TPM_SKIP_PP | T.TPM_SKIP_PM | T.TPM_SKIP_KICK)
    pot = gpu_ctx.download()["pot"]
    cell = np.stack([np.floor(d[k] / 2.0 ** 32 * C) for k in "xyz"], 1)
    inside = np.all((cell >= lo) & (cell < hi), 1)
    assert np.array_equal(pot != 0, inside & (d["rung"] >= 1))


def test_kick_alone_time_of_a_crowded_cell(gpu_ctx):
    """10^5 particles in one cell against the same number over all 125: the kick alone does the same work for both."""
    C = 5
    p = T.baseline_params(512, 512, 3, n_total=10 ** 5)
    p.chain_dim = C
    gpu_ctx.set_params(p)
    ms = []
    for n_cell in (10 ** 5, 0):
        x, y, z = crowded(n_cell, 10 ** 5 - n_cell, C, 3)
        gpu_ctx.upload(x, y, z)
        gpu_ctx.chainmesh_create()
        flags = T.TPM_SKIP_PP | T.TPM_SKIP_PM | T.TPM_SKIP_KICK
        ms.append(min(gpu_ctx.kick(flags=flags).ms_pp for _ in range(5)))
    assert ms[0] < 5 * ms[1]
