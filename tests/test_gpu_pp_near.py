"""GPU: the direct kernel's near pairs.  Boxes whose sources are mostly near ones (halos of r^-2 profile, the near radius
beyond the cutoff, a softening length of half the cutoff and beyond it) against the oracle's FP64 sums, with the bound of the other tile
tests (2e-5 of the rms force); near sources beyond the cutoff are not evaluated; and the near pairs at the cutoff are
decided on exact integer offsets, two at a time in a tile that holds both."""
import numpy as np
import pytest

import tigerpm_amd as T
from test_gpu_tiles import forces, truth

pytestmark = pytest.mark.gpu
TWO32 = 2.0 ** 32


def raw(pos):
    return [np.floor((pos[:, d] % 1.0) * TWO32).astype(np.uint64).astype(np.uint32) for d in range(3)]


def halos(n, seed):
    rng = np.random.default_rng(seed)
    size = (rng.pareto(1.2, 40) + 1)
    size = (size / size.sum() * 0.8 * n).astype(int)
    pos = [rng.uniform(0, 1, (n - size.sum(), 3))]
    for s in size:
        u = rng.standard_normal((s, 3))
        r = 0.03 * (s / size.max()) ** (1 / 3) * rng.uniform(0, 1, (s, 1))
        pos.append(rng.uniform(0, 1, 3) + r * u / np.linalg.norm(u, axis=1, keepdims=True))
    return np.concatenate(pos)


@pytest.mark.parametrize("tile", [8, 16, 32, 64])
@pytest.mark.parametrize("kind", ["halos", "near radius beyond rcut", "soft", "softer than rcut"])
@pytest.mark.parametrize("C", [4, 5, 11])
def test_mostly_near(gpu_ctx, tile, kind, C):
    n = 12000
    p = T.baseline_params(64, 64, 3, n_total=n)
    p.chain_dim = C
    pos = halos(n, C) if kind == "halos" else np.random.default_rng(C).uniform(0, 1, (n, 3))
    if kind == "near radius beyond rcut":
        p.rs = p.rcut
    elif kind == "soft":
        p.hsoft = 0.5 * p.rcut
    elif kind == "softer than rcut":
        p.hsoft = 1.1 * p.rcut
    prev = gpu_ctx.get_tuning()
    try:
        gpu_ctx.set_params(p)
        gpu_ctx.set_tuning(tile_sinks=tile)
        gpu_ctx.upload(*raw(pos))
        gpu_ctx.chainmesh_create()
        st = gpu_ctx.kick(flags=T.TPM_SKIP_PM | T.TPM_SKIP_KICK)
        cells = gpu_ctx.chainmesh_cells()
        d = gpu_ctx.download()
        sinks = np.random.default_rng(1).choice(n, 4000, replace=False)
        g, _ = forces(gpu_ctx)
        if kind != "softer than rcut":  # (a softened pair beyond the cutoff counts if its source is staged)
            g64, _ = truth(p, d["x"], d["y"], d["z"], cells, sinks)
            norm = np.sqrt((g64 ** 2).sum(1).mean())
            assert np.sqrt(((g[sinks] - g64) ** 2).sum(1).mean()) < 2e-5 * norm
        else:
            assert np.isfinite(g).all()
        if kind == "near radius beyond rcut" and C == 4:
            assert st.executed_pairs < 0.7 * st.candidate_pairs
    finally:
        gpu_ctx.set_tuning(**prev)


@pytest.mark.parametrize("tile", [8, 16, 32, 64])
def test_near_cutoff_is_exact(gpu_ctx, tile):
    """Two particles of one cell, one tile: its box spans both, so the pair is a near one."""
    p = T.baseline_params(64, 64, 3, n_total=2)
    p.chain_dim = 4
    rc2 = (p.rcut * TWO32) ** 2
    rng = np.random.default_rng(tile)
    prev = gpu_ctx.get_tuning()
    try:
        gpu_ctx.set_tuning(tile_sinks=tile)
        for trial in range(8):
            a = np.floor((rng.integers(0, 4, 3) + rng.uniform(0.3, 0.6, 3)) / 4 * TWO32).astype(np.int64)
            u = np.abs(rng.standard_normal(3))
            d = np.rint(p.rcut * TWO32 * u / np.linalg.norm(u)).astype(np.int64)
            k = int(np.argmax(d))
            for step in (-60, -3, -1, 0, 1, 3, 60):
                e = d.copy()
                e[k] += step
                inside = sum(int(v) ** 2 for v in e) < rc2
                q = np.stack([a, a + e]).astype(np.uint64).astype(np.uint32)
                gpu_ctx.set_params(p)
                gpu_ctx.upload(*[np.ascontiguousarray(q[:, i]) for i in range(3)])
                gpu_ctx.chainmesh_create()
                gpu_ctx.kick(flags=T.TPM_SKIP_PM | T.TPM_SKIP_KICK)
                g, _ = forces(gpu_ctx)
                assert np.all((g != 0).any(1) == inside), (trial, step)
                assert np.array_equal(g[0], -g[1])
    finally:
        gpu_ctx.set_tuning(**prev)
