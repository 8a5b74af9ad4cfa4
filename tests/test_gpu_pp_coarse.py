"""GPU: the short-range pairs where the chain mesh is much coarser than the cutoff (cells of 164 rs), and the tree
walk's far pairs at the cutoff and over the law's range.

Each chain cell holds one close pair (a, b), a in the cell's lower half and b below it on every axis, and two guards in
the upper corner, further away than the cutoff, so that every force is one pair's.  With only a active the sinks' box
is a point and b is a far source; with the guards active too the box is nearly as wide as the cell and b lies outside.

Bound of the pair's force F at x = r / (2 rs) in [0.74, 1.2]: the offset, r^2, u, the exponential, the reciprocal
root and the polynomial are about fifteen roundings of 2^-24 (rms 3.4e-8 each) of which those of u count x^2 times, and
the two laws are within 1.5e-7 of erfc: less than 2.5e-7 (1 + x^2) F, rms.  Held to 5e-7; offsets rounded to 2^-24 of
a cell give 2e-6 and more."""
import numpy as np
import pytest
from scipy.special import erfc

import tigerpm_amd as T

pytestmark = pytest.mark.gpu
TWO32 = 2.0 ** 32


def law(r, rs):
    x = r / (2 * rs)
    return (erfc(x) + 2 * x / np.sqrt(np.pi) * np.exp(-x * x)) / r ** 2


def pairs_in_cells(C, rs, lo, hi, rng):
    """Raw positions (C^3, 4, 3) of a, b and two guards."""
    k = np.arange(C ** 3)
    centre = (np.stack([k % C, (k // C) % C, k // (C * C)], 1) + 0.5) / C
    a = centre + rng.uniform(-0.4, -0.1, centre.shape) / C
    u = -np.abs(rng.standard_normal(a.shape))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    b = a + u * rng.uniform(lo, hi, (len(a), 1)) * 2 * rs
    guards = [centre + np.array(s) * 0.49 / C for s in ((1, 1, 1), (0.9, 1, 1))]
    pos = np.stack([a, b] + guards, 1)
    return np.floor(pos * TWO32).astype(np.uint64).astype(np.uint32)


@pytest.mark.parametrize("tree", [False, True])
@pytest.mark.parametrize("active", ["one", "wide"])
@pytest.mark.parametrize("tile", [8, 16, 64])
def test_pair_force_in_coarse_cells(gpu_ctx, tree, active, tile):
    C, M = 5, 1024
    p = T.baseline_params(M, M, 3)  # hsoft far below the distances
    p.chain_dim, p.GM = C, 1.0
    prev = gpu_ctx.get_tuning()
    err = []
    try:
        gpu_ctx.set_tuning(tile_sinks=tile)
        for seed in range(4):
            raw = pairs_in_cells(C, p.rs, 0.74, 1.2, np.random.default_rng(seed))
            rung = np.zeros(raw.shape[:2], np.int8)
            rung[:, 0] = 1
            if active == "wide":
                rung[:, 2:] = 1
            gpu_ctx.set_params(p)
            flat = raw.reshape(-1, 3)
            gpu_ctx.upload(*[np.ascontiguousarray(flat[:, d]) for d in range(3)], rung=rung.reshape(-1))
            gpu_ctx.chainmesh_create()
            gpu_ctx.kick(min_rung=1, flags=T.TPM_SKIP_PM | T.TPM_SKIP_KICK | (T.TPM_KICK_TREE if tree else 0))
            d = gpu_ctx.download()
            at = {tuple(q): i for i, q in enumerate(zip(d["x"], d["y"], d["z"]))}
            for cell in raw:
                i = at[tuple(cell[0])]
                off = (cell[1].astype(np.int64) - cell[0].astype(np.int64)) / TWO32
                r = np.sqrt((off ** 2).sum())
                f = law(r, p.rs)
                got = np.array([d["gx"][i], d["gy"][i], d["gz"][i]], np.float64)
                err.append(np.linalg.norm(got - f * off / r) / f / (1 + (r / (2 * p.rs)) ** 2))
    finally:
        gpu_ctx.set_tuning(**prev)
    assert np.sqrt(np.mean(np.square(err))) < 5e-7


def test_tree_far_pairs(gpu_ctx):
    """The walk's far pairs, a the only active particle of its bucket: at the cutoff the pair acts if and only if its
    squared integer offset is below (rcut 2^32)^2; from below the near radius to the cutoff the force is the law's (bounds of
    the direct kernel's test of the same)."""
    C = 5
    p = T.baseline_params(64, 64, 3, n_total=4)
    p.chain_dim, p.GM = C, 1.0
    rng = np.random.default_rng(3)
    rc2 = (p.rcut * TWO32) ** 2

    def force(a, e):
        guards = np.array([[0.59, 0.59, 0.59], [0.41, 0.59, 0.59]]) * TWO32
        raw = np.concatenate([[a, a + e], guards]).astype(np.uint64).astype(np.uint32)
        gpu_ctx.set_params(p)
        gpu_ctx.upload(*[np.ascontiguousarray(raw[:, d]) for d in range(3)], rung=np.array([1, 0, 0, 0], np.int8))
        gpu_ctx.chainmesh_create()
        gpu_ctx.kick(min_rung=1, flags=T.TPM_SKIP_PM | T.TPM_SKIP_KICK | T.TPM_KICK_TREE)
        d = gpu_ctx.download()
        i = int(np.nonzero(d["rung"] == 1)[0][0])
        return np.array([d["gx"][i], d["gy"][i], d["gz"][i]], np.float64)

    def draw(r):
        a = np.floor(rng.uniform(0.41, 0.43, 3) * TWO32).astype(np.int64)
        u = np.abs(rng.standard_normal(3))
        return a, np.rint(r * TWO32 * u / np.linalg.norm(u)).astype(np.int64)

    for trial in range(6):
        a, d = draw(p.rcut)
        k = int(np.argmax(np.abs(d)))
        for step in (-3, -1, 0, 1, 3):
            e = d.copy()
            e[k] += step
            inside = sum(int(v) ** 2 for v in e) < rc2
            assert np.any(force(a, e) != 0.0) == inside, (trial, step)
    for r in np.linspace(0.2 * 2 * p.rs, 0.99 * p.rcut, 16):
        a, e = draw(r)
        off = e / TWO32
        d = np.sqrt((off ** 2).sum())
        f = law(d, p.rs)
        assert np.abs(force(a, e) - f * off / d).max() < 2e-6 * f + 3e-7 / d ** 2, r
