"""The work a user of this library has it do, as cases that can be timed.

A case is one box (or one set of boxes) and the calls a program makes on it:

  step    particles resident on the device, one tpm_kick_treepm (chain mesh, PM, short range + kick), then the
          updated state read back into page-locked buffers that the program keeps
  active  the forces of the particles on the finer time-step rungs only (block time steps)
  mesh    the long-range force alone (the reference's kick_pm)
  pme     kick_pme's pair law: every pair of the 27 neighbour cells
  tree    the reference's own short-range algorithm, per-cell trees with multipoles
  batch   an ensemble of independent boxes kicked together, the step replayed as a graph
  host    the drop-in call: particles in host arrays in the reference's order; upload, kick, download

Particles are uniform or a Zel'dovich lattice displaced by a few tenths to a few cells, masses 1/N, as in the
benchmark and the tests.  The global time step is short enough that every particle stays on rung 0, so that the
integer outputs do not hang on the last bit of a force.
"""
import ctypes
import math

import numpy as np
import torch

import tigerpm_amd as T

T0 = 2.0 ** -12
TWO32 = 4294967296.0


def listed():
    return [
        # the smallest box the serving loop takes: launches and underfilled kernels count
        dict(name="box32_cloud4", kind="step", n=32, mesh=32, order=4, interlace=0, rms=1.0, setup="baseline"),
        # benchmark configuration 1: a uniform 64^3 box, CIC
        dict(name="uniform64_cic", kind="step", n=64, mesh=64, order=2, interlace=0, rms=0.0, setup="baseline"),
        # a box of no convenient size with the interlaced mesh (accuracy runs): ragged cells and tiles, a mesh
        # that is no power of two
        dict(name="odd93_interlaced", kind="step", n=93, mesh=93, order=3, interlace=1, rms=1.0, setup="baseline"),
        # benchmark configurations 2 and 3, the second the headline one
        dict(name="zeldovich256_tsc", kind="step", n=256, mesh=256, order=3, interlace=0, rms=0.5, setup="baseline"),
        dict(name="zeldovich512_tsc", kind="step", n=512, mesh=512, order=3, interlace=0, rms=2.0, setup="baseline"),
        # the reference's default ratios (mesh spacing 3 particle spacings, 15^3 particles per chain cell)
        dict(name="reference120", kind="step", n=120, mesh=40, order=4, interlace=0, rms=1.0, setup="reference"),
        # block time steps: the densest eighth of the particles is due
        dict(name="active256", kind="active", n=256, mesh=256, order=3, interlace=0, rms=2.0, setup="baseline"),
        # the long-range force alone
        dict(name="mesh256", kind="mesh", n=256, mesh=256, order=4, interlace=0, rms=1.0, setup="baseline"),
        # the reference's second kernel at its default ratios, on a small box
        dict(name="pme60", kind="pme", n=60, mesh=20, order=4, interlace=0, rms=1.0, setup="reference"),
        # the reference's tree walk
        dict(name="tree128", kind="tree", n=128, mesh=128, order=3, interlace=0, rms=1.0, setup="baseline"),
        # an ensemble as in the benchmark's, smaller
        dict(name="ensemble24", kind="batch", boxes=24, lo=32, hi=80, order=4),
        # the call as the reference makes it, host arrays in and out
        dict(name="host100", kind="host", n=100, mesh=100, order=4, interlace=0, rms=1.0, setup="baseline"),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["step", "step", "step", "step", "reference", "active", "mesh", "pme", "tree", "batch", "host"])
    rms = rng.choice([0.0, round(rng.uniform(0.3, 2.0), 3)])
    if kind == "batch":
        lo = rng.randint(32, 44)
        return dict(kind="batch", boxes=rng.randint(6, 40), lo=lo, hi=rng.randint(lo + 8, 96), order=rng.choice([2, 3, 4]))
    if kind in ("reference", "pme"):
        n = 15 * (rng.randint(4, 8) if kind == "reference" else rng.randint(3, 5))
        return dict(kind="step" if kind == "reference" else "pme", n=n, mesh=n // 3, order=4, interlace=0, rms=rms,
                    setup="reference")
    if kind == "step":
        n = size(32, 320)
        mesh = rng.choice([n, n, n, size(max(32, 0.7 * n), 1.2 * n)])
    elif kind == "active":
        n = mesh = size(96, 288)
    elif kind == "mesh":
        n = mesh = size(64, 300)
    elif kind == "tree":
        n = mesh = size(40, 160)
    else:
        n = mesh = size(40, 144)
    return dict(kind=kind, n=n, mesh=mesh, order=rng.choice([2, 3, 3, 4]), interlace=rng.choice([0, 0, 1]), rms=rms,
                setup="baseline")


# ------------------------------------------------------------------------------------------------------ inputs

def params_of(case):
    if case["setup"] == "reference":
        p = T.reference_params(case["n"])
        p.GM = 1.0 / float(case["n"]) ** 3
        return p
    return T.baseline_params(case["n"], case["mesh"], case["order"], interlace=case["interlace"])


def to_u32(x):
    """Box positions in FP64 (any period) as raw 32-bit fixed point."""
    r = torch.floor((x - torch.floor(x)) * TWO32).to(torch.int64)
    return r.to(torch.int32).cpu().numpy().view(np.uint32)


def particles(n, rms, seed):
    """n^3 particles: raw positions, velocities along the displacement, and the overdensity at each particle.
    rms = 0: uniform; else a lattice displaced by a Gaussian field (power k^-2, cut at the Nyquist wave number)
    of that rms displacement in lattice cells."""
    dev = torch.device("cuda")
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    if rms == 0.0:
        pos = [to_u32(torch.rand(n ** 3, generator=g, device=dev, dtype=torch.float64)) for _ in range(3)]
        vel = [(1e-3 * torch.randn(n ** 3, generator=g, device=dev)).cpu().numpy() for _ in range(3)]
        return pos, vel, torch.rand(n ** 3, generator=g, device=dev)
    k1 = torch.fft.fftfreq(n, 1.0 / n, device=dev)
    ks = [k1[:, None, None], k1[None, :, None], torch.fft.rfftfreq(n, 1.0 / n, device=dev)[None, None, :]]
    k2 = ks[0] ** 2 + ks[1] ** 2 + ks[2] ** 2
    k2[0, 0, 0] = 1.0
    delta = torch.fft.rfftn(torch.randn(n, n, n, generator=g, device=dev))
    delta *= torch.exp(-2.0 * k2 / n ** 2) / torch.sqrt(k2)
    delta[0, 0, 0] = 0.0
    psi, norm = [], 0.0
    for d in range(3):
        f = torch.fft.irfftn(1j * ks[d] / k2 * delta, s=(n, n, n))
        norm += float((f.double() ** 2).mean())
        psi.append(f)
    a = rms / n / math.sqrt(norm)
    lattice = (torch.arange(n, device=dev, dtype=torch.float64) + 0.5) / n
    pos, vel = [], []
    for d in range(3):
        shape = [1, 1, 1]
        shape[d] = n
        pos.append(to_u32((lattice.view(shape) + a * psi[d].double()).reshape(-1)))
        vel.append((0.1 * a * psi[d]).reshape(-1).cpu().numpy())
    return pos, vel, torch.fft.irfftn(delta, s=(n, n, n)).reshape(-1)


def case_particles(case, seed):
    """The box's host arrays: x, y, z, vx, vy, vz, rung."""
    pos, vel, dense = particles(case["n"], case["rms"], seed)
    rung = np.zeros(case["n"] ** 3, np.int8)
    if case["kind"] == "active":
        top = torch.topk(dense, dense.numel() // 8).indices
        rung[top.cpu().numpy()] = 1
    return pos + vel + [rung]


def ensemble(case):
    """Side and rms displacement of each box: sizes log-spaced, displacements spread over [0.3, 2] cells."""
    b, lo, hi = case["boxes"], case["lo"], case["hi"]
    return [(int(round(lo * (hi / lo) ** (k / (b - 1)))), 0.3 + 1.7 * (k * 7 % b) / b) for k in range(b)]


# ------------------------------------------------------------------------------------------------------- calls

FIELDS = ["x", "y", "z", "vx", "vy", "vz", "rung", "gx", "gy", "gz", "pot"]


class Readback:
    """Page-locked host buffers for some of the particle arrays, and their pointers in the order of FIELDS."""

    def __init__(self, n, names):
        self.t = {k: torch.empty(n, dtype=torch.int8 if k == "rung" else torch.float32, pin_memory=True) for k in names}

    def pointers(self, first=0):
        return [ctypes.c_void_p(self.t[k].data_ptr() + first * self.t[k].element_size()) if k in self.t else None
                for k in FIELDS]


UPDATED = ["vx", "vy", "vz", "rung", "gx", "gy", "gz", "pot"]
FORCES = ["gx", "gy", "gz", "pot"]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        boxes = ensemble(case)
        total = sum(n ** 3 for n, _ in boxes)
        bt = T.Batch(total, total, len(boxes), case["order"])
        ids = []
        for k, (n, rms) in enumerate(boxes):
            pos, vel, _ = particles(n, rms, seed * 1000 + k)
            ids.append(bt.add(T.box_spec(T.baseline_params(n, n, case["order"]), t0=T0), *pos, *vel))
        bt.set_tuning(graph=1)
        for _ in range(2):
            bt.step(0, stats=False)
        bt.sync()
        return dict(kind=kind, bt=bt, ids=ids, sizes=[n ** 3 for n, _ in boxes], out=Readback(total, UPDATED))
    ctx = T.Context(0)
    ctx.set_params(params_of(case))
    data = case_particles(case, seed)
    if kind == "host":
        ctx.set_host_order(T.TPM_ORDER_REFERENCE)
        return dict(kind=kind, ctx=ctx, data=data)
    ctx.upload(*data)
    state = dict(kind=kind, ctx=ctx, out=Readback(len(data[0]), UPDATED if kind == "step" else FORCES))
    ctx._keep = None
    # the step before: plans, tables and buffers are made, the particles lie in chain-mesh order
    if kind == "step":
        ctx.kick_treepm(0, 1.0, T0, True, stats=False)
    else:
        ctx.chainmesh_create()
        ctx.gravity_long_compute()
    ctx.sync()
    return state


FLAGS = {"active": T.TPM_SKIP_KICK, "mesh": T.TPM_SKIP_KICK | T.TPM_SKIP_PP, "pme": T.TPM_SKIP_KICK | T.TPM_KICK_PME,
         "tree": T.TPM_SKIP_KICK | T.TPM_KICK_TREE}


def run(state):
    kind, lib = state["kind"], T.lib()
    if kind == "batch":
        bt, first = state["bt"], 0
        bt.step(0, stats=False)
        for box, n in zip(state["ids"], state["sizes"]):
            if lib.tpm_batch_download(bt._h, box, *state["out"].pointers(first)) != 0:
                raise RuntimeError("tpm_batch_download")
            first += n
        return state["out"].t
    ctx = state["ctx"]
    if kind == "host":
        ctx.upload(*state["data"])
        ctx.kick_treepm(0, 1.0, T0, True)
        return ctx.download()
    if kind == "step":
        ctx.kick_treepm(0, 1.0, T0, False, stats=False)
    else:
        ctx.chainmesh_create()
        ctx.gravity_long_compute()
        ctx.kick(1 if kind == "active" else 0, 1.0, T0, True, flags=FLAGS[kind])
    if lib.tpm_particles_download(ctx._h, *state["out"].pointers()) != 0:
        raise RuntimeError("tpm_particles_download")
    return state["out"].t


# ------------------------------------------------------------------------------------------------- what it takes

def box_work(n, p, kind):
    """Bytes and operations of one box: particles read and written once, the pairs within the cutoff at 44
    operations each, the assignment and interpolation stencils, two transforms of the mesh."""
    N, M = float(n) ** 3, float(p.mesh_dim)
    C = p.chain_dim or int(math.floor(1.0 / p.rcut))
    sinks = N / 8 if kind == "active" else N
    pairs = sinks * N * (27.0 / C ** 3 if kind == "pme" else 4.0 / 3.0 * math.pi * p.rcut ** 3)
    if kind == "mesh":
        pairs = 0.0
    fft = 2 * 2.5 * M ** 3 * math.log2(M ** 3)
    stencils = N * p.order ** 3 * 2 * (1 + p.interlace) + sinks * 216 * 4
    moved = 12 * N + (13 * 2 + 16) * sinks if kind in ("step", "batch", "host") else 12 * N + 16 * sinks
    if kind == "host":
        moved += (25 + 41) * N
    return moved + 4 * M ** 3, 44 * pairs + fft + stencils


def work(case):
    if case["kind"] == "batch":
        parts = [box_work(n, T.baseline_params(n, n, case["order"]), "batch") for n, _ in ensemble(case)]
    else:
        parts = [box_work(case["n"], params_of(case), case["kind"])]
    return {"bytes": sum(b for b, _ in parts), "flops": sum(f for _, f in parts)}


# ----------------------------------------------------------------------------------------------- 64-bit results

def cell_coords(raw, C):
    """Chain cell and quarter of a cell per coordinate: split planes at floor(2^32 (k (1 / C)))."""
    r = raw.astype(np.uint64)
    planes = np.array([int(TWO32 * (k * (1.0 / C))) for k in range(C)], np.uint64)
    k = np.searchsorted(planes, r, side="right") - 1
    prod = r * np.uint64(C)
    kk = (prod >> np.uint64(32)).astype(np.int64)
    sub = ((prod >> np.uint64(30)) & np.uint64(3)).astype(np.int64)
    return k, np.where(k > kk, 0, np.where(k < kk, 3, sub))


def cell_ids(pos, C):
    (cx, sx), (cy, sy), (cz, sz) = [cell_coords(a, C) for a in pos]
    code = np.zeros(len(cx), np.int64)
    for shift, b in ((5, sz >> 1), (4, sy >> 1), (3, sx >> 1), (2, sz & 1), (1, sy & 1), (0, sx & 1)):
        code |= b << shift
    return (cz * C + cy) * C + cx, code


def reference_order(cid, C):
    """The order in which the reference's recursive two-pointer partition leaves the particles."""
    perm = np.arange(len(cid))
    start = np.concatenate([[0], np.cumsum(np.bincount(cid, minlength=C ** 3))])
    stack = [(0, C, 0, C, 0, C)]
    while stack:
        z0, z1, y0, y1, x0, x1 = stack.pop()
        a = (z0 * C + y0) * C + x0
        if z1 - z0 > 1:
            mid, stride = z0 + (z1 - z0) // 2, C * C
            stack += [(z0, mid, y0, y1, x0, x1), (mid, z1, y0, y1, x0, x1)]
            b, e = mid * stride, z1 * stride
        elif y1 - y0 > 1:
            mid = y0 + (y1 - y0) // 2
            stack += [(z0, z1, y0, mid, x0, x1), (z0, z1, mid, y1, x0, x1)]
            b, e = (z0 * C + mid) * C, (z0 * C + y1) * C
        elif x1 - x0 > 1:
            mid = x0 + (x1 - x0) // 2
            stack += [(z0, z1, y0, y1, x0, mid), (z0, z1, y0, y1, mid, x1)]
            b, e = (z0 * C + y0) * C + mid, (z0 * C + y0) * C + x1
        else:
            continue
        s, m, t = start[a], start[b], start[e]
        c = cid[perm[s:t]]
        up = s + np.nonzero(c[:m - s] >= b)[0]
        down = (m + np.nonzero(c[m - s:] < b)[0])[::-1]
        perm[up], perm[down] = perm[down], perm[up]
    return perm


def mesh_potential(pos, p):
    """The PM potential on the mesh, FP64: assignment, Green's function with deconvolution, transforms."""
    M, order = p.mesh_dim, p.order
    dev = pos[0].device

    def assign(shift):
        axes = []
        for x in pos:
            P = x * (M / TWO32) + shift
            if order == 2:
                b = torch.floor(P)
                t = P - b
                w = [1 - t, t]
            elif order == 3:
                b = torch.floor(P + 0.5)
                d = P - b
                w = [0.5 * (0.5 - d) ** 2, 0.75 - d * d, 0.5 * (0.5 + d) ** 2]
                b = b - 1
            else:
                b = torch.floor(P)
                t = P - b
                u = 1 - t
                w = [u ** 3 / 6, (4 - 6 * t * t + 3 * t ** 3) / 6, (4 - 6 * u * u + 3 * u ** 3) / 6, t ** 3 / 6]
                b = b - 1
            axes.append((b.to(torch.int64), w))
        rho = torch.zeros(M ** 3, dtype=torch.float64, device=dev)
        for a in range(order):
            ix = torch.remainder(axes[0][0] + a, M) * M * M
            for b in range(order):
                ixy = ix + torch.remainder(axes[1][0] + b, M) * M
                wxy = axes[0][1][a] * axes[1][1][b]
                for c in range(order):
                    rho.index_add_(0, ixy + torch.remainder(axes[2][0] + c, M), wxy * axes[2][1][c])
        return torch.fft.rfftn(rho.view(M, M, M))

    f = torch.arange(M, device=dev, dtype=torch.float64)
    f = torch.where(2 * f < M, f, f - M) * (2 * math.pi / M)
    kx, ky, kz = f[:, None, None], f[None, :, None], f[None, None, :M // 2 + 1]
    spec = assign(0.0)
    if p.interlace:
        spec = 0.5 * (spec + torch.exp(0.5j * (kx + ky + kz)) * assign(0.5))
    k2 = kx * kx + ky * ky + kz * kz
    k2[0, 0, 0] = 1.0
    s = torch.sinc(kx / (2 * math.pi)) * torch.sinc(ky / (2 * math.pi)) * torch.sinc(kz / (2 * math.pi))
    G = -4 * math.pi * M / k2 * torch.exp(-k2 * (p.rs * M) ** 2) * s ** (-order)
    G[0, 0, 0] = 0.0
    return torch.fft.irfftn(spec * G, s=(M, M, M)).reshape(-1)


def poly(x, coef):
    """Coefficients from the constant term up, over 24ths."""
    r = torch.zeros_like(x)
    for c in reversed(coef):
        r = r * x + c / 24.0
    return r


# The 6-point quintic interpolation weights over 24, powers of x from the constant term up.
QUINTIC = [[0, 2, -1, -9, 13, -5], [0, -16, 16, 39, -64, 25], [24, 0, -30, -70, 126, -50],
           [0, 16, 16, 66, -124, 50], [0, -2, -1, -33, 61, -25], [0, 0, 0, 7, -12, 5]]


def mesh_force(phi, pos, M):
    """Unit-mass mesh force and potential at each position."""
    out = [torch.zeros_like(pos[0]) for _ in range(4)]
    for lo in range(0, len(pos[0]), 1 << 21):
        sl = slice(lo, lo + (1 << 21))
        base, w, dw = [], [], []
        for x in pos:
            P = x[sl] * (M / TWO32)
            b = torch.floor(P)
            t = P - b
            base.append(b.to(torch.int64) - 2)
            w.append([poly(t, c) for c in QUINTIC])
            dw.append([poly(t, [k * c[k] for k in range(1, 6)]) for c in QUINTIC])
        for a in range(6):
            ix = torch.remainder(base[0] + a, M) * M * M
            sums = [0.0, 0.0, 0.0]
            for b in range(6):
                ixy = ix + torch.remainder(base[1] + b, M) * M
                s0, s1 = 0.0, 0.0
                for c in range(6):
                    v = phi[ixy + torch.remainder(base[2] + c, M)]
                    s0 = s0 + w[2][c] * v
                    s1 = s1 + dw[2][c] * v
                sums[0] = sums[0] + w[1][b] * s0
                sums[1] = sums[1] + dw[1][b] * s0
                sums[2] = sums[2] + w[1][b] * s1
            out[0][sl] -= M * dw[0][a] * sums[0]
            out[1][sl] -= M * w[0][a] * sums[1]
            out[2][sl] -= M * w[0][a] * sums[2]
            out[3][sl] += w[0][a] * sums[0]
    return out


def pair_sums(pos, cid, active, p, pme):
    """Unit-mass short-range force and potential of the active particles (sorted by cell) from the 27 neighbour
    cells, FP64."""
    C = p.chain_dim or int(math.floor(1.0 / p.rcut))
    dev = pos[0].device
    count = torch.bincount(cid, minlength=C ** 3)
    start = torch.cumsum(count, 0) - count
    X = torch.stack(pos, 1).to(torch.int64)
    sinks = torch.nonzero(active).reshape(-1)
    g = torch.zeros(len(cid), 4, dtype=torch.float64, device=dev)
    rc2, h = p.rcut ** 2, p.hsoft
    inv2rs, tsp = 0.5 / p.rs, 2.0 / math.sqrt(math.pi)
    for nb in range(27):
        c = cid[sinks]
        cx = torch.remainder(c % C + nb % 3 - 1, C)
        cy = torch.remainder((c // C) % C + (nb // 3) % 3 - 1, C)
        cz = torch.remainder(c // (C * C) + nb // 9 - 1, C)
        c2 = (cz * C + cy) * C + cx
        order = torch.argsort(count[c2])  # sinks with as many sources together
        si, b, m = sinks[order], start[c2][order], count[c2][order]
        sizes = m.cpu().numpy()
        lo = 0
        while lo < len(si):
            hi = min(len(si), lo + max(1, (1 << 24) // max(1, int(sizes[lo]))))
            if int(sizes[hi - 1]) > 2 * max(8, int(sizes[lo])):
                hi = max(lo + 1, int(np.searchsorted(sizes, 2 * max(8, int(sizes[lo])), side="right")))
            hi = max(lo + 1, min(hi, lo + max(1, (1 << 25) // max(1, int(sizes[hi - 1])))))
            w = int(sizes[hi - 1])
            if w:
                j = torch.arange(w, device=dev)[None, :]
                have = j < m[lo:hi, None]
                src = torch.where(have, b[lo:hi, None] + j, 0)
                d = (X[si[lo:hi]][:, None, :] - X[src]).to(torch.int32).to(torch.float64) / TWO32
                r2 = (d * d).sum(2)
                near = have & (r2 <= h * h)
                far = have & (r2 > h * h)
                if not pme:
                    far &= r2 < rc2
                r = torch.sqrt(torch.where(far, r2, 1.0))
                x = r * inv2rs
                e = torch.erfc(x) / r
                f = torch.where(far, (e + tsp * inv2rs * torch.exp(-x * x)) / (r * r), 0.0)
                q = torch.where(far, e, 0.0)
                if bool(near.any()):
                    rn2 = r2[near]
                    q2 = rn2 / h ** 2
                    d1 = ((15 / 8 * q2 - 21 / 4) * q2 + 35 / 8) / h ** 3
                    d0 = (((-5 / 16 * q2 + 21 / 16) * q2 - 35 / 16) * q2 + 35 / 16) / h
                    if not pme:
                        rn = torch.sqrt(rn2)
                        pos_r = rn > 0
                        xs = rn * inv2rs
                        # (erf(x) - 2 x exp(-x^2) / sqrt(pi)) / r^3 and erf(x) / r, by series below x = 0.05
                        one = torch.where(pos_r, rn, 1.0)
                        u = xs * xs
                        t3 = tsp * inv2rs ** 3 * (2 / 3 - 2 * u / 5 + u * u / 7 - u ** 3 / 27)
                        t3 = torch.where(xs < 0.05, t3, (torch.erf(xs) - tsp * xs * torch.exp(-u)) / one ** 3)
                        d1 = torch.where(pos_r, d1 - t3, d1)
                        d0 = torch.where(pos_r, d0 - torch.erf(xs) / one, d0)
                    f[near] = d1
                    q[near] = d0
                g[si[lo:hi], :3] -= (d * f[:, :, None]).sum(1)
                g[si[lo:hi], 3] -= q.sum(1)
            lo = hi
    return g


def exact_box(pos, vel, rung, p, kind, passes):
    """The arrays of a box after `passes` kicks from velocities vel (the first one a first call), in chain-mesh
    order; the permutation and the cell of each particle before it."""
    C = p.chain_dim or int(math.floor(1.0 / p.rcut))
    cid, code = cell_ids(pos, C)
    perm = np.argsort(cid * 64 + code, kind="stable")
    dev = torch.device("cuda")
    q = [torch.from_numpy(a[perm].astype(np.float64)).to(dev) for a in pos]
    mf = mesh_force(mesh_potential(q, p), q, p.mesh_dim)
    active = torch.from_numpy(rung[perm] >= (1 if kind == "active" else 0)).to(dev)
    g = torch.stack(mf, 1)
    phi0 = 0.0
    if kind != "pme":
        phi0 = p.n_total * 4 * math.pi * p.rs ** 2 + 35 / 16 / p.hsoft
    if kind != "mesh":
        g += pair_sums(q, torch.from_numpy(cid[perm]).to(dev), active, p, kind == "pme")
    g[:, 3] += phi0
    g *= p.GM
    g[~active] = 0.0
    out = {k: g[:, i].cpu().numpy() for i, k in enumerate(FORCES)}
    for i, k in enumerate(["vx", "vy", "vz"]):
        out[k] = vel[i][perm].astype(np.float64) + (passes - 0.5) * T0 * out["g" + "xyz"[i]]
    return out, perm, cid


def exact(case, seed):
    kind = case["kind"]
    if kind == "tree":
        return None  # the multipoles are part of that algorithm
    if kind == "batch":
        parts = []
        for k, (n, rms) in enumerate(ensemble(case)):
            pos, vel, _ = particles(n, rms, seed * 1000 + k)
            p = T.baseline_params(n, n, case["order"])
            parts.append(exact_box(pos, vel, np.zeros(n ** 3, np.int8), p, "step", 3)[0])
        out = {k: np.concatenate([q[k] for q in parts]) for k in UPDATED if k != "rung"}
        return dict(out, rung=None)
    p = params_of(case)
    C = p.chain_dim or int(math.floor(1.0 / p.rcut))
    n = float(case["n"]) ** 3
    pairs = 0.0 if kind == "mesh" else n * n * 27.0 / C ** 3
    if pairs > 2.5e10 or n > 300.0 ** 3:
        return None  # over about 20 seconds
    data = case_particles(case, seed)
    pos, vel, rung = data[:3], data[3:6], data[6]
    out, perm, cid = exact_box(pos, vel, rung, p, kind, 2 if kind == "step" else 1)
    if kind == "host":
        back = np.empty_like(perm)
        back[perm] = np.arange(len(perm))
        order = back[reference_order(cid, C)]
        return {k: out[k][order] if k in out else None for k in FIELDS}
    return {k: out.get(k) for k in (UPDATED if kind == "step" else FORCES)}
