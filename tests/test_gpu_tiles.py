"""GPU: the direct kernel's sink tiles where their making can go wrong: cells
whose active particles fill a chunk of the build (128 in a small box, 256 from
2^19 particles on) exactly, one less or one more, several chunks, cells that
fit one tile, coinciding coordinates (the split's ties), subsets of active
particles and box kicks.  Every sink against the oracle's FP64 sums with the
bound of the other pair tests (1e-5 rms; 2e-5 against FP64), and, in the large
box, tile sizes against each other to FP32 summation order (5e-6)."""
import numpy as np
import pytest

import oracle as orc
import tigerpm_amd as T
from test_gpu_parity import cells_with, oparams

pytestmark = pytest.mark.gpu

COUNTS = [1, 7, 8, 9, 15, 16, 17, 63, 64, 65, 127, 128, 129, 255, 256, 257, 300, 385, 513]


def rel_rms(a, b):
    return float(np.sqrt(((a - b) ** 2).sum() / (b ** 2).sum()))


def truth(p, x, y, z, cell_begin, sinks):
    (gx, gy, gz, ph), _ = orc.pp_sum(oparams(p), x, y, z, cell_begin, sinks, fp64=True)
    phi0 = p.n_total * 4 * np.pi * p.rs ** 2 + (35.0 / 16.0) / p.hsoft
    # the FP64 self pair takes the limit of (erfc(x) - 1) / r too, which the
    # reference's formula (and the kernel) leave out at r = 0
    phi0 -= 2.0 / np.sqrt(np.pi) / (2.0 * p.rs)
    g = np.stack([gx, gy, gz], 1).astype(np.float64) * p.GM
    return g, (ph.astype(np.float64) + phi0) * p.GM


def forces(ctx):
    d = ctx.download()
    return np.stack([d[k] for k in ("gx", "gy", "gz")], 1).astype(np.float64), d["pot"].astype(np.float64)


@pytest.mark.parametrize("tile", [8, 16, 32, 64])
@pytest.mark.parametrize("ties", [False, True])
def test_chunk_edges_vs_oracle(gpu_ctx, tile, ties):
    C = 6
    p = T.baseline_params(34, 34, 3)
    assert p.chain_dim == C
    x, y, z = cells_with(dict(zip([(k % C, (k // C) % C, k // (C * C)) for k in range(0, 11 * len(COUNTS), 11)],
                                  COUNTS)), C, 5)
    if ties:  # a cell's particles on four lines, so that most coordinates are shared
        cell = [np.floor(c / 2.0 ** 32 * C) for c in (x, z)]
        x = ((cell[0] + 0.5) / C * 2.0 ** 32).astype(np.uint32)
        z = ((cell[1] + (0.5 + np.arange(len(z)) % 4) / 4) / C * 2.0 ** 32).astype(np.uint32)
    n = len(x)
    p.n_total, p.GM = float(n), 1.0 / n
    rng = np.random.default_rng(tile)
    rung = rng.integers(0, 3, n).astype(np.int8)
    prev = gpu_ctx.get_tuning()
    try:
        gpu_ctx.set_params(p)
        gpu_ctx.set_tuning(tile_sinks=tile)
        gpu_ctx.upload(x, y, z, rung=rung)
        gpu_ctx.chainmesh_create()
        d = gpu_ctx.download()
        xs, ys, zs, rs = d["x"], d["y"], d["z"], d["rung"]
        perm, cb = orc.chainmesh_sort(x, y, z, C)
        g64, pot64 = truth(p, xs, ys, zs, cb, np.arange(n))
        norm = np.sqrt((g64 ** 2).sum(1).mean())
        for min_rung in (0, 1, 2):
            gpu_ctx.kick(min_rung=min_rung, flags=T.TPM_SKIP_PM | T.TPM_SKIP_KICK)
            g, pot = forces(gpu_ctx)
            act = rs >= min_rung
            assert np.sqrt(((g - g64)[act] ** 2).sum(1).mean()) < 2e-5 * norm
            assert rel_rms(pot[act], pot64[act]) < 2e-5
        # the sinks of a box of cells alone: the same sums
        lo, hi = (1, 0, 1), (4, 6, 5)
        gpu_ctx.kick_box(lo, hi, flags=T.TPM_SKIP_PM | T.TPM_SKIP_KICK)
        gb, _ = forces(gpu_ctx)
        assert np.sqrt(((gb - g64) ** 2).sum(1).mean()) < 2e-5 * norm
    finally:
        gpu_ctx.set_tuning(**prev)


@pytest.mark.parametrize("n", [2 ** 19 - 1, 2 ** 19])
def test_chunk_size_boundary(gpu_ctx, n):
    """Cells of ~1000 particles on both sides of the box size where the chunks double (forces; a
    uniform box's potential is a small difference of large sums)."""
    rng = np.random.default_rng(n)
    p = T.baseline_params(48, 48, 3, n_total=n)
    x, y, z = [rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32) for _ in range(3)]
    prev = gpu_ctx.get_tuning()
    try:
        gpu_ctx.set_params(p)
        out = []
        for tile in (16, 64):
            gpu_ctx.set_tuning(tile_sinks=tile)
            gpu_ctx.upload(x, y, z)
            gpu_ctx.chainmesh_create()
            gpu_ctx.kick(flags=T.TPM_SKIP_PM | T.TPM_SKIP_KICK)
            out.append(forces(gpu_ctx)[0])
        assert rel_rms(out[0], out[1]) < 5e-6
        cells = gpu_ctx.chainmesh_cells()
        d = gpu_ctx.download()
        sinks = rng.choice(n, 300, replace=False)
        g64, _ = truth(p, d["x"], d["y"], d["z"], cells, sinks)
        assert rel_rms(out[1][sinks], g64) < 2e-5
    finally:
        gpu_ctx.set_tuning(**prev)
