"""GPU: kick_pme's forces are those that the library has always given: the general law on exact integer differences,
summed in the cells' order.  Without a cutoff a sink's sum is a small difference of large parts, so another law or
another order moves it by more than either is off by (2e-5 of the z force's rms, with small displacements, for a far
law three times nearer to FP64).

golden/pme_forces.npz: forces and potentials of every 149th particle (device order) of the boxes below, 16-sink tiles,
from commit 33439ae.  The same operations in the same order give the same bits; held to 1e-6 (norm per component)."""
import os

import numpy as np
import pytest

import tigerpm_amd as T

pytestmark = pytest.mark.gpu
GOLDEN = os.path.join(os.path.dirname(__file__), "golden", "pme_forces.npz")
KEYS = ["gx", "gy", "gz", "pot"]


def lattice(n):
    """n^3 lattice points displaced by 0.3 cells rms, by nine plane waves per axis."""
    g = (np.arange(n) + 0.5) / n
    q = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    rng = np.random.default_rng(n)
    d = np.zeros_like(q)
    for _ in range(9):
        k = rng.integers(1, 5, 3)
        for axis in range(3):
            d[:, axis] += np.sin(2 * np.pi * (q @ k + rng.uniform()))
    d *= 0.3 / n / np.sqrt((d ** 2).sum(1).mean())
    return [np.floor(((q + d)[:, i] % 1.0) * 2.0 ** 32).astype(np.uint64).astype(np.uint32) for i in range(3)]


def pme_forces(ctx, n):
    p = T.reference_params(n)
    p.GM = 1.0 / n ** 3
    ctx.set_params(p)
    ctx.upload(*lattice(n))
    ctx.chainmesh_create()
    ctx.kick(flags=T.TPM_SKIP_PM | T.TPM_SKIP_KICK | T.TPM_KICK_PME)
    d = ctx.download()
    return {k: d[k][::149].copy() for k in KEYS}


@pytest.mark.parametrize("n", [45, 60])
def test_pme_forces_unchanged(gpu_ctx, n):
    gold = np.load(GOLDEN)
    got = pme_forces(gpu_ctx, n)
    for k in KEYS:
        want = gold["%s_%d" % (k, n)].astype(np.float64)
        assert np.linalg.norm(got[k] - want) < 1e-6 * np.linalg.norm(want), k
