"""GPU: sink tiles of boxes with many cells and few particles each, where a lane makes the tile of a cell: cells with
none, one, 64 and 65 particles, one tile exactly filled and one more, a crowded cell among them; subsets of active particles, cell boxes,
the law without cutoff, the pair-once kernel and batches.  Forces against the oracle's FP64 sums with the bound of the other tile tests
(2e-5 of the rms force), every active sink in a tile and no other."""
import numpy as np
import pytest

import tigerpm_amd as T
from test_gpu_parity import cells_with
from test_gpu_tiles import forces, truth

pytestmark = pytest.mark.gpu
C = 45


def sparse_box(seed):
    counts = [1, 2, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 66, 130, 3000]
    rng = np.random.default_rng(seed)
    cells = rng.choice(C ** 3, 4 * len(counts), replace=False)
    want = {(int(k) % C, int(k) // C % C, int(k) // C ** 2): counts[i % len(counts)] for i, k in enumerate(cells)}
    x, y, z = cells_with(want, C, seed)
    extra = [rng.integers(0, 2 ** 32, 20000, dtype=np.uint64).astype(np.uint32) for _ in range(3)]
    return [np.concatenate(p) for p in zip((x, y, z), extra)]


def check(ctx, p, min_rung, sinks_rng, lo=None, hi=None):
    cells = ctx.chainmesh_cells()
    d = ctx.download()
    g, pot = forces(ctx)
    act = d["rung"] >= min_rung
    if lo is not None:
        at = np.repeat(np.arange(C ** 3), np.diff(cells))
        xyz = np.stack([at % C, at // C % C, at // C ** 2], 1)
        act &= np.all((xyz >= lo) & (xyz < hi), 1)
    assert np.array_equal((g != 0).any(1) | (pot != 0), act)
    sinks = sinks_rng.choice(np.nonzero(act)[0], 3000)
    g64, _ = truth(p, d["x"], d["y"], d["z"], cells, sinks)
    norm = np.sqrt((g64 ** 2).sum(1).mean())
    assert np.sqrt(((g[sinks] - g64) ** 2).sum(1).mean()) < 2e-5 * norm


@pytest.mark.parametrize("tile", [8, 16, 64])
def test_sparse_cells(gpu_ctx, tile):
    x, y, z = sparse_box(3)
    n = len(x)
    p = T.baseline_params(256, 256, 3, n_total=n)
    assert p.chain_dim == C and n < 8 * C ** 3
    rng = np.random.default_rng(tile)
    rung = rng.integers(0, 3, n).astype(np.int8)
    prev = gpu_ctx.get_tuning()
    flags = T.TPM_SKIP_PM | T.TPM_SKIP_KICK
    try:
        gpu_ctx.set_params(p)
        for min_rung, newton, lo, hi in ((0, 0, None, None), (1, 0, None, None), (2, 0, None, None), (0, 1, None, None),
                                         (1, 0, (0, 3, 10), (45, 44, 30)), (0, 0, (7, 8, 9), (8, 20, 45))):
            gpu_ctx.set_tuning(tile_sinks=tile, pp_newton=newton)
            gpu_ctx.upload(x, y, z, rung=rung)
            gpu_ctx.chainmesh_create()
            if lo is None:
                gpu_ctx.kick(min_rung=min_rung, flags=flags)
            else:
                gpu_ctx.kick_box(lo, hi, min_rung=min_rung, flags=flags)
            check(gpu_ctx, p, min_rung, rng, lo, hi)
        # kick_pme: the sums of a subset are those of the whole bit for bit (tiles of all particles)
        gpu_ctx.set_tuning(tile_sinks=tile)
        got = []
        for min_rung in (0, 1):
            gpu_ctx.upload(x, y, z, rung=rung)
            gpu_ctx.chainmesh_create()
            gpu_ctx.kick(min_rung=min_rung, flags=flags | T.TPM_KICK_PME)
            got.append((forces(gpu_ctx)[0], gpu_ctx.download()["rung"]))
        act = got[1][1] >= 1
        assert np.array_equal(got[0][0][act], got[1][0][act])
        assert (got[1][0][~act] == 0).all()
    finally:
        gpu_ctx.set_tuning(**prev)


def test_sparse_batch_equals_single_boxes(gpu_ctx):
    boxes = [(sparse_box(5), 256), ([a[:9000] for a in sparse_box(6)], 256)]
    total = sum(len(b[0]) for b, _ in boxes)
    t0 = 2.0 ** -12
    with T.Batch(max_particles=total, max_mesh_nodes=2 * 256 ** 3, max_boxes=2, order=3) as bt:
        ids = [bt.add(T.box_spec(T.baseline_params(M, M, 3, n_total=len(b[0])), t0=t0), *b) for b, M in boxes]
        ctxs = []
        for i in ids:
            c = T.Context(0)
            bt.to_ctx(i, c)
            ctxs.append(c)
        for k in range(2):
            bt.step(0)
            for i, c in zip(ids, ctxs):
                c.kick_treepm(min_rung=0, scale=1.0, t0=t0, first_call=(k == 0))
                a, b = bt.download(i), c.download()
                for key in ("vx", "gx", "gy", "gz", "pot"):
                    assert np.array_equal(a[key], b[key]), (k, i, key)
        for c in ctxs:
            c.close()
