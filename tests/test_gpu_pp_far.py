"""The direct kernel's far pairs: the cutoff decided on exact integer offsets, and the one-polynomial law.

The law's bounds: its polynomial is within 5e-8 of erfc, its FP32 evaluation (about ten roundings) within 1e-6 of
each factor; a pair's offset is rounded to 2^-24 of up to two cells, so a component of a pair's force is off by at
most about 2e-6 of the pair's force."""
import numpy as np
import pytest
from scipy.special import erfc

import tigerpm_amd as T

pytestmark = pytest.mark.gpu


def kick_pair(ctx, raw, p, tile, flags=0):
    prev = ctx.get_tuning()
    try:
        ctx.set_params(p)
        ctx.set_tuning(tile_sinks=tile)
        ctx.upload(*[np.array(c, np.uint64).astype(np.uint32) for c in raw])
        ctx.chainmesh_create()
        ctx.kick(flags=T.TPM_SKIP_PM | T.TPM_SKIP_KICK | flags)
        return ctx.download()
    finally:
        ctx.set_tuning(**prev)


@pytest.mark.parametrize("tile", [8, 16, 32, 64])
@pytest.mark.parametrize("n_side,chain_dim", [(20, 3), (26, 4), (32, 5), (48, 8), (200, 35)])
def test_cutoff_is_exact(gpu_ctx, tile, n_side, chain_dim):
    """Two particles a few raw units inside and outside rcut: the pair acts if and only if its squared integer
    offset is below (rcut 2^32)^2, whichever way the offset points and wherever the tile lies."""
    p = T.baseline_params(n_side, n_side, 3, n_total=2)
    assert p.chain_dim == chain_dim
    rc2 = (p.rcut * 2.0 ** 32) ** 2
    rng = np.random.default_rng(n_side + tile)
    for trial in range(6):
        a = rng.integers(0, 2 ** 32, 3)
        u = rng.standard_normal(3)
        if trial == 0:
            u = np.array([1.0, 0.0, 0.0])
        d = np.rint(p.rcut * 2.0 ** 32 * u / np.linalg.norm(u)).astype(np.int64)
        k = int(np.argmax(np.abs(d)))
        for step in (-3, -1, 0, 1, 3):
            e = d.copy()
            e[k] += step
            inside = sum(int(v) ** 2 for v in e) < rc2
            g = kick_pair(gpu_ctx, np.stack([a, (a + e) % 2 ** 32], 1), p, tile)
            acts = np.any(np.stack([g["gx"], g["gy"], g["gz"]]) != 0.0)
            assert acts == inside, (trial, step)


@pytest.mark.parametrize("tile", [8, 16, 64])
@pytest.mark.parametrize("n_side,flags", [(20, 0), (32, 0), (200, 0), (20, T.TPM_KICK_PME), (32, T.TPM_KICK_PME)])
def test_pair_law_over_its_range(gpu_ctx, tile, n_side, flags):
    """One pair at distances from below the near radius to the cutoff (kick_pme: to the end of the 27 cells)."""
    p = T.baseline_params(n_side, n_side, 3, n_total=2)
    far = 0.99 * p.rcut if flags == 0 else 0.99 / p.chain_dim
    rng = np.random.default_rng(7 * n_side + tile)
    for r in np.linspace(0.2 * 2 * p.rs, far, 12):
        u = rng.standard_normal(3)
        e = np.rint(r * 2.0 ** 32 * u / np.linalg.norm(u)).astype(np.int64)
        a = rng.integers(0, 2 ** 32, 3)
        g = kick_pair(gpu_ctx, np.stack([a, (a + e) % 2 ** 32], 1), p, tile, flags)
        off = e / 2.0 ** 32
        d = np.sqrt((off ** 2).sum())
        x = d / (2 * p.rs)
        f = (erfc(x) + 2 * x / np.sqrt(np.pi) * np.exp(-x * x)) / d ** 2 * p.GM
        first = 0 if g["x"][0] == np.uint32(a[0]) and g["y"][0] == np.uint32(a[1]) else 1
        got = np.array([g["gx"][first], g["gy"][first], g["gz"][first]], np.float64)
        # A&S 7.1.26 below the near radius: 1.5e-7 of erfc
        tol = 2e-6 * f + 3e-7 / d ** 2 * p.GM
        assert np.abs(got - f * off / d).max() < tol, r
        other = np.array([g["gx"][1 - first], g["gy"][1 - first], g["gz"][1 - first]], np.float64)
        assert np.abs(other + f * off / d).max() < tol, r
