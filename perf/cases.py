"""Timed cases: what programs have libmdk do, through megadock_amd's public entry points.

Inputs are synthetic proteins made from the seed: atoms on a jittered lattice in a ball at
the density of a protein's heavy atoms, with the radii, charges and contact energies the
CHARMM and ACE tables hold.  The receptor grids are built here as the host layer builds them
(rPSC shape with contact energies, distance-dependent electrostatics), so exact() shares
them; the ligand is voxelized in exact() with the library's float32 rounding (which voxels
an atom covers is a discrete choice) and everything after that is computed in 64 bits.

Kinds of case:
  dock       Context.dock: rotations given and results taken on the host, one call a batch
  search     the rotation loop of one pair that stays resident: dock_range, then topn
  pair       a job of a job table: new receptor grids and ligand, dock_range, topn
  spectral   hard-voxel score and its translation gradient for poses off the grid
  companion  trilinear score of poses with translation and rotation gradients
  receptor   receptor grids built on the device from the atoms, and read back
"""
import math

import numpy as np
import torch

import megadock_amd as M

GW = 1.2  # voxel pitch (A), the default
REC_CORE = -45.0
OPEN = -7777.0
# even sizes of the default FFT size table
SIZES = [64, 66, 70, 72, 80, 84, 88, 90, 96, 98, 100, 108, 110, 112, 120, 126, 128, 132, 140, 144, 150, 154, 160, 162,
         168, 176, 180, 192, 196, 198, 200, 210, 216, 220, 224, 240, 242, 250, 252, 256, 264, 270, 280, 288, 294, 300,
         308, 320]
# sizes without kernels of their own: multiples of 13 and very large proteins
OTHER_SIZES = [78, 104, 130, 156, 182, 208, 260, 324, 330, 336, 350, 352, 360]


def listed():
    return [
        # one orientation scored on request (the smallest call: launches and latency)
        dict(name="one_rotation_80", kind="dock", nf=80, t=1, rotations=1, batch=1),
        # the FFTProcess class: a device batch of rotations, host to host
        dict(name="class_batch_100", kind="dock", nf=100, t=1, rotations=128, batch=128),
        # one job of an all-to-all table, small proteins: 3600 rotations, best 2000 decoys
        dict(name="pair_96", kind="pair", nf=96, t=1, rotations=3600, batch=256, best=2000),
        # the same with a ragged grid (odd ng) of a mid-sized pair
        dict(name="pair_126", kind="pair", nf=126, t=1, rotations=3600, batch=256, best=2000),
        # the medium search (600 / 250 residues), three results per rotation; a sixth of the
        # 54000-rotation set
        dict(name="search_144", kind="search", nf=144, t=3, rotations=9000, batch=128, best=2000),
        # a large pair between the powers of two
        dict(name="search_216", kind="search", nf=216, t=1, rotations=768, batch=192, best=500),
        # the large search (2000 / 1000 residues)
        dict(name="search_256", kind="search", nf=256, t=3, rotations=768, batch=96, best=2000),
        # a very large receptor: a size without kernels of its own
        dict(name="search_360", kind="search", nf=360, t=1, rotations=32, batch=16, best=32),
        # many results per rotation, above what the inverse pass keeps in registers
        dict(name="ranks_112", kind="search", nf=112, t=64, rotations=1024, batch=128, best=5000),
        # refinement: hard-voxel score and translation gradient of a batch of decoys
        dict(name="spectral_144", kind="spectral", nf=144, poses=512, batch=128),
        # refinement: companion score with pose gradients of the 2000 best decoys
        dict(name="companion_144", kind="companion", nf=144, poses=2000, batch=128),
        # a receptor of 600 residues set up on the device
        dict(name="receptor_144", kind="receptor", nf=144, atoms=4993),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi, sizes=SIZES):
    x = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min((n for n in sizes if lo <= n <= hi), key=lambda n: abs(n - x))


def _batch(nf, rotations):
    """Rotations a device batch, as the host layer chooses them (at most 20 GB of buffers)."""
    return max(1, min(rotations, 256 if nf <= 128 else 128 if nf <= 192 else int(8.0e8 / nf ** 3 * 2)))


def draw(rng):
    kind = rng.choice(["dock", "dock", "search", "search", "search", "pair", "pair", "other", "ranks", "spectral",
                       "companion", "receptor"])
    if kind == "dock":
        n = _log_int(rng, 1, 256)
        return dict(kind=kind, nf=_size(rng, 64, 200), t=rng.choice([1, 1, 2, 3, 5]), rotations=n, batch=n)
    if kind in ("search", "pair"):
        nf = _size(rng, 64, 320 if kind == "search" else 160)
        n = max(20, min(9000, int(_log_int(rng, 10 ** 9, 10 ** 10) / nf ** 3)))
        t = rng.choice([1, 1, 3, 4]) if kind == "search" else 1
        return dict(kind=kind, nf=nf, t=t, rotations=n, batch=_batch(nf, n), best=min(2000, n * t))
    if kind == "other":
        nf = _size(rng, 78, 360, OTHER_SIZES)
        n = max(8, min(1000, int(_log_int(rng, 4 * 10 ** 8, 10 ** 9) / nf ** 3)))
        return dict(kind="search", nf=nf, t=1, rotations=n, batch=min(n, 16), best=n)
    if kind == "ranks":
        nf = _size(rng, 64, 160)
        n = max(32, min(2000, int(_log_int(rng, 2 * 10 ** 8, 10 ** 9) / nf ** 3)))
        return dict(kind="search", nf=nf, t=_log_int(rng, 17, 200), rotations=n, batch=min(n, 128), best=2000)
    if kind == "spectral":
        return dict(kind=kind, nf=_size(rng, 64, 200), poses=_log_int(rng, 1, 512), batch=64)
    if kind == "companion":
        return dict(kind=kind, nf=_size(rng, 64, 256), poses=_log_int(rng, 1, 4000), batch=64)
    nf = _size(rng, 64, 200)
    return dict(kind=kind, nf=nf, atoms=int(0.0016 * nf ** 3 * rng.uniform(0.6, 1.0)))


# ------------------------------------------------------------------ inputs
def _gpu(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


def _protein(rng, n):
    """n heavy atoms centred on the origin: xyz, radius, charge, contact energy (float32)."""
    a = 20.0 ** (1.0 / 3.0)  # 20 A^3 an atom
    m = int(math.ceil((3.0 * n / (4.0 * math.pi)) ** (1.0 / 3.0))) + 2
    g = np.stack(np.meshgrid(*[np.arange(-m, m + 1)] * 3, indexing="ij"), -1).reshape(-1, 3) * a
    g = g[np.argsort((g ** 2).sum(1), kind="stable")[:n]] + rng.uniform(-0.6, 0.6, (n, 3))
    radius = rng.choice([1.63, 1.75, 1.87, 1.95, 2.03, 2.1], n)
    charge = rng.choice([0.0, 0.0, 0.1, -0.15, -0.25, 0.25, 0.33, -0.55, -0.57, 0.6], n)
    ace = rng.choice([0.0, 0.061, -0.079, 0.232, -0.353, -0.432, -0.553, 0.933], n)
    g -= g.mean(0)
    return [v.astype(np.float32) for v in (g, radius, charge, ace)]


def _rotations(rng, n):
    q = rng.normal(size=(n, 4))
    w, x, y, z = (q / np.linalg.norm(q, axis=1, keepdims=True)).T
    r = np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                  2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                  2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], 1)
    return r.astype(np.float32)


def _grid_coord(ng):
    return np.array([np.float32(GW) * np.float32(ng) * (-0.5 + (0.5 + i) / ng) for i in range(ng)], np.float32)


def _boxes(cell, reach, ng):
    """For atoms in cells (n, 3): voxel indices (n, w) of their boxes and whether in the grid."""
    o = torch.arange(-reach, reach + 1, device=cell.device)
    ijk = [cell[:, a, None] + o for a in range(3)]
    ok = [(v >= 0) & (v < ng) for v in ijk]
    vox = ((ijk[0].clamp(0, ng - 1)[:, :, None, None] * ng + ijk[1].clamp(0, ng - 1)[:, None, :, None]) * ng
           + ijk[2].clamp(0, ng - 1)[:, None, None, :])
    inside = ok[0][:, :, None, None] & ok[1][:, None, :, None] & ok[2][:, None, None, :]
    return [v.clamp(0, ng - 1) for v in ijk], vox.flatten(1), inside.flatten(1)


def _dist2(xyz, gc, ijk):
    """((dx^2 + dy^2) + dz^2) of every box voxel, rounded after each operation."""
    d = [(xyz[:, a, None] - gc[ijk[a]]) for a in range(3)]
    d = [v * v for v in d]
    return ((d[0][:, :, None, None] + d[1][:, None, :, None]) + d[2][:, None, None, :]).flatten(1)


def _receptor_grids(atoms, ng):
    """Shape and electrostatic grids (ng^3, float64 on the GPU) of a centred receptor, summed
    in whole units (1e-4 and 2^-30) so that no order of the sums shows."""
    xyz, radius, charge, ace = [_gpu(a) for a in atoms]
    gc = _gpu(_grid_coord(ng))
    n3 = ng ** 3

    def cells(p, gw):
        return (p / torch.tensor(gw, dtype=torch.float32, device="cuda") + ng // 2).to(torch.int64)

    core = torch.zeros(n3, dtype=torch.bool, device="cuda")
    cell = cells(xyz, GW)
    for s in range(0, len(xyz), 20000):
        e = slice(s, s + 20000)
        ijk, vox, ok = _boxes(cell[e], int((2.4 + GW - 0.01) / GW), ng)
        hit = ok & (_dist2(xyz[e], gc, ijk) < (radius[e] * radius[e] * 1.5)[:, None])
        core[vox[hit]] = True
    # open space: what the six rays of each grid line reach before the first core voxel, then
    # two ordered sweeps (a voxel spreads to its zero neighbours if it is open when reached)
    c = core.view(ng, ng, ng)
    free = torch.zeros_like(c)
    for a in range(3):
        free |= torch.cumsum(c.int(), a) == 0
        free |= torch.flip(torch.cumsum(torch.flip(c, [a]).int(), a), [a]) == 0
    free, core_h = free.cpu().numpy(), c.cpu().numpy()
    i, j, k = np.meshgrid(*[np.arange(ng)] * 3, indexing="ij")
    plane = (i + j + k).ravel()
    swept = ((i >= 1) & (i <= ng - 2) & (j >= 2) & (j <= ng - 2) & (k >= 2) & (k <= ng - 2)).ravel()
    order = np.argsort(plane, kind="stable")
    bounds = np.searchsorted(plane[order], np.arange(3 * ng - 1))
    free, solid = free.ravel(), core_h.ravel()
    for _ in range(2):
        seen = np.zeros(n3 + ng * ng, bool)  # shifted by ng^2: predecessors of the first plane read 0
        for s in range(3 * ng - 2):
            v = order[bounds[s]:bounds[s + 1]]
            v = v[swept[v] & ~solid[v]]
            seen[v + ng * ng] = free[v] | seen[v + ng * ng - 1] | seen[v + ng * ng - ng] | seen[v]
        seen = seen[ng * ng:].reshape(ng, ng, ng)
        spread = np.zeros((ng, ng, ng), bool)
        for a in range(3):
            lo, hi = [slice(None)] * 3, [slice(None)] * 3
            lo[a], hi[a] = slice(None, -1), slice(1, None)
            spread[tuple(lo)] |= seen[tuple(hi)]
            spread[tuple(hi)] |= seen[tuple(lo)]
        free = free | (spread.ravel() & ~solid)
    inner = _gpu(solid | ~free)  # core and enclosed cavities
    surf = torch.zeros(n3, dtype=torch.int64, device="cuda")
    reach = int((float(radius.max()) + 3.6) / GW) + 2
    for s in range(0, len(xyz), 5000):
        e = slice(s, s + 5000)
        ijk, vox, ok = _boxes(cell[e], reach, ng)
        rj = (radius[e] + 3.6) * (radius[e] + 3.6)
        hit = ok & (_dist2(xyz[e], gc, ijk) < rj[:, None])
        add = torch.round(1e4 * (1.0 - 0.8 * ace[e].double())).long()[:, None].expand(vox.shape)
        surf.index_add_(0, vox[hit], add[hit])
    shape = torch.where(inner, REC_CORE, surf.double() / 1e4)
    elec = torch.zeros(n3, dtype=torch.int64, device="cuda")
    gwl = float(np.float32(_grid_coord(ng)[1] - _grid_coord(ng)[0]))
    per_cell = np.float32(np.float32(gwl) * np.float32(80.0) / np.float32(2800.0))
    q = charge.cpu().numpy()
    for value in np.unique(q[np.abs(q) > 1e-6]):
        aq = np.float32(abs(value))
        reach = 4 if aq < 0.07 else 5 if aq < 0.21 else int(aq / per_cell)
        sel = _gpu(np.flatnonzero(q == value))
        step = max(1, 40000000 // (2 * reach + 1) ** 3)
        for s in range(0, len(sel), step):
            p = xyz[sel[s:s + step]]
            ijk, vox, ok = _boxes(cells(p, gwl), reach, ng)
            d = _dist2(p, gc, ijk).double().sqrt()
            er = torch.where(d >= 8.0, 80.0, torch.where(d > 6.0, 38.0 * d - 224.0, 4.0))
            ok &= ~(shape < 0)[vox]
            elec.index_add_(0, vox[ok], torch.round(-2800.0 * 2.0 ** 30 * float(value) / er / d)[ok].long())
    return shape, elec.double() / 2.0 ** 30


def _inputs(case, seed):
    """Atoms, rotations and poses of a case: everything that the seed decides."""
    rng = np.random.default_rng([seed, case["nf"]])
    ng = case["nf"] // 2
    n_rec = case.get("atoms") or min(20000, int(0.0125 * ng ** 3 * rng.uniform(0.8, 1.0)))
    rec, lig = _protein(rng, n_rec), _protein(rng, max(60, int(0.42 * n_rec)))
    out = dict(ng=ng, nf=case["nf"], rec=rec, lig=lig)
    n = case.get("rotations", case.get("poses", 0))
    if n:
        out["rot"] = _rotations(rng, n)
    if "poses" in case:  # near contact: within the receptor's radius of the centre
        out["trans"] = (rng.uniform(-0.35, 0.35, (n, 3)) * ng % case["nf"]).astype(np.float32)
    return out


def _set_ligand(ctx, lig, ng):
    ctx.set_ligand(lig[0], np.zeros(3, np.float32), lig[1], lig[2], _grid_coord(ng), GW)


def prepare(case, seed):
    x = _inputs(case, seed)
    kind, ng = case["kind"], x["ng"]
    ctx = M.Context(case["nf"], ng, len(x["lig"][0]), t=case.get("t", 1), max_batch=case.get("batch", 1))
    state = dict(x, kind=kind, ctx=ctx, best=case.get("best", 0), coord=_grid_coord(ng))
    if kind != "receptor":
        grids = [g.float().cpu().numpy() for g in _receptor_grids(x["rec"], ng)]
        if kind == "pair":
            state["grids"] = grids
        else:
            ctx.set_receptor(*grids)
            _set_ligand(ctx, x["lig"], ng)
    if kind in ("search", "pair"):
        ctx.set_rotations(x["rot"])
    if kind == "dock":
        state["ids"] = np.arange(len(x["rot"]), dtype=np.int32)
    return state


def run(state):
    ctx, kind = state["ctx"], state["kind"]
    if kind == "dock":
        r = ctx.dock(state["rot"], state["ids"])
    elif kind in ("search", "pair"):
        if kind == "pair":
            ctx.set_receptor(*state["grids"])
            _set_ligand(ctx, state["lig"], state["ng"])
        ctx.dock_range(0, len(state["rot"]))
        r = ctx.topn(len(state["rot"]), state["best"])
    elif kind == "spectral":
        return {"value": ctx.score_spectral(state["rot"], state["trans"])}
    elif kind == "companion":
        return {"value": ctx.score_companion(state["rot"], state["trans"])}
    else:
        ctx.set_receptor_atoms(*state["rec"], state["coord"])
        return dict(zip(("shape", "elec"), ctx.receptor_grids()))
    return {"score": r["score"], "index": r["index"]}


# ------------------------------------------------------------------ the least work
def work(case):
    nf = case["nf"]
    ng, n3 = nf // 2, nf ** 3
    n = case.get("rotations", case.get("poses", 0))
    atoms = case.get("atoms") or min(20000, 0.0112 * ng ** 3)
    lig = max(60, 0.42 * atoms)
    line = 5.0 * nf * math.log2(nf)  # operations of one complex transform of a grid line
    spectrum = (ng * ng + ng * nf + nf * nf) * line  # the ligand fills an eighth of the grid
    if case["kind"] == "receptor":
        # each atom's surface sphere, and the field of the charged ones, at every voxel in reach
        return {"bytes": 24.0 * atoms + 16.0 * ng ** 3, "flops": atoms * (8.0 * 700 + 0.8 * 12.0 * 8000)}
    if case["kind"] == "companion":
        return {"bytes": 8.0 * ng ** 3 + 24.0 * lig + 76.0 * n, "flops": n * lig * 200.0}
    if case["kind"] == "spectral":
        return {"bytes": 8.0 * n3 + 20.0 * lig + 64.0 * n, "flops": n * (spectrum + 11.0 * n3)}
    # per rotation: forward transform, product and its Hermitian half, inverse of the half
    flops = n * (spectrum + 9.0 * n3 + 0.5 * 3 * nf * nf * line)
    size = 8.0 * n3 + 20.0 * lig + 36.0 * n + 20.0 * n * case["t"]
    return {"bytes": size + (8.0 * ng ** 3 if case["kind"] == "pair" else 0.0), "flops": flops}


# ------------------------------------------------------------------ the same in 64 bits
def _ligand_grids(lig, rot, ng):
    """Shape + i charge (complex128, (n, ng, ng, ng)) of the ligand under n rotations."""
    xyz, radius, charge = [_gpu(a) for a in lig[:3]]
    gc, r = _gpu(_grid_coord(ng)), _gpu(rot)
    gw = torch.tensor(GW, dtype=torch.float32, device="cuda")
    n, na, n3 = len(rot), len(xyz), ng ** 3
    p = torch.stack([(r[:, 3 * a, None] * xyz[:, 0] + r[:, 3 * a + 1, None] * xyz[:, 1]) + r[:, 3 * a + 2, None] * xyz[:, 2]
                     for a in range(3)], -1).reshape(n * na, 3)
    base = (torch.arange(n, device="cuda") * n3).repeat_interleave(na)
    ijk, vox, ok = _boxes((p / gw + float(ng // 2)).to(torch.int64), 2, ng)
    d2, r2 = _dist2(p, gc, ijk), (radius * radius).repeat(n)[:, None]
    vox = vox + base[:, None]
    core = torch.zeros(n * n3, dtype=torch.bool, device="cuda")
    surf = torch.zeros_like(core)
    core[vox[ok & (d2 < r2 * 1.5)]] = True
    surf[vox[ok & (d2 < r2)]] = True
    core, surf = core.view(n, ng, ng, ng), surf.view(n, ng, ng, ng)
    shape = (core | surf).double()
    # interior core voxels with a neighbour outside the core lose the core value
    ins = core[:, 1:-1, 1:-1, 1:-1]
    closed = ins.clone()
    for a in range(3):
        for w in (slice(None, -2), slice(2, None)):
            at = [slice(None)] + [slice(1, -1)] * 3
            at[a + 1] = w
            closed &= core[tuple(at)]
    lost = ins & ~closed & ~surf[:, 1:-1, 1:-1, 1:-1]
    shape[:, 1:-1, 1:-1, 1:-1][lost] = 0.0
    pad = float(np.float32(ng) * np.float32(GW) / np.float32(2))
    c = ((p + pad) / gw).to(torch.int64).clamp(0, ng - 1)
    q = torch.zeros(n * n3, dtype=torch.float64, device="cuda")
    q.index_add_(0, base + (c[:, 0] * ng + c[:, 1]) * ng + c[:, 2], charge.double().repeat(n))
    return torch.complex(shape, q.view(n, ng, ng, ng))


def _embed(g, nf):
    ng = nf // 2
    nd = (nf - ng) // 2
    out = torch.zeros(g.shape[:-3] + (nf, nf, nf), dtype=torch.complex128, device="cuda")
    out[..., nd:nd + ng, nd:nd + ng, nd:nd + ng] = g
    return out


def _signed(nf, n):
    k = torch.arange(n, device="cuda")
    return torch.where(k < nf // 2, k, k - nf).double()


def _companion(x, shape, elec):
    """(s, ds/dt' (3), ds/dw (3)) of every pose by trilinear interpolation."""
    ng, nf = x["ng"], x["nf"]
    xyz, radius, charge = [_gpu(a).double() for a in x["lig"][:3]]
    pad = torch.zeros((2, ng + 4, ng + 4, ng + 4), dtype=torch.float64, device="cuda")
    pad[:, 2:-2, 2:-2, 2:-2] = torch.stack([shape, elec]).view(2, ng, ng, ng).float().double()
    pad = pad.view(2, -1)
    gw = float(np.float32(GW))
    weight = 4.0 / 3.0 * math.pi * radius ** 3 / gw ** 3
    rows = []
    for s in range(0, len(x["rot"]), 256):
        r = _gpu(x["rot"][s:s + 256]).double().view(-1, 3, 3)
        t = _gpu(x["trans"][s:s + 256]).double()
        t = torch.where(t < 0.5 * nf, t, t - nf)
        X = (r[:, None] * xyz[None, :, None, :]).sum(-1)
        u = ((X - gw * t[:, None]) / gw + 0.5 * ng - 0.5).clamp(-1.5, ng + 0.5)
        lo = torch.floor(u)
        f, o = u - lo, lo.long() + 2
        g = [torch.zeros_like(u[..., 0]) for _ in range(4)]
        for corner in range(8):
            bit = [corner >> 2, corner >> 1 & 1, corner & 1]
            v = ((o[..., 0] + bit[0]) * (ng + 4) + o[..., 1] + bit[1]) * (ng + 4) + o[..., 2] + bit[2]
            val = weight * pad[0][v] + charge * pad[1][v]
            w = [f[..., a] if bit[a] else 1 - f[..., a] for a in range(3)]
            sg = [1.0 if b else -1.0 for b in bit]
            g[0] += w[0] * w[1] * w[2] * val
            g[1] += sg[0] * w[1] * w[2] * val / gw
            g[2] += sg[1] * w[0] * w[2] * val / gw
            g[3] += sg[2] * w[0] * w[1] * val / gw
        G = torch.stack(g[1:], -1)
        rows.append(torch.cat([g[0].sum(1, keepdim=True), -gw * G.sum(1), torch.cross(X, G, dim=-1).sum(1)], 1))
    return torch.cat(rows)


def exact(case, seed):
    nf, n = case["nf"], case.get("rotations", case.get("poses", 0))
    if case["kind"] not in ("receptor", "companion") and n * nf ** 3 > 4e10:
        return None
    x = _inputs(case, seed)
    ng = x["ng"]
    shape, elec = _receptor_grids(x["rec"], ng)
    if case["kind"] == "receptor":
        return {"shape": shape, "elec": elec}
    if case["kind"] == "companion":
        return {"value": _companion(x, shape, elec)}
    rec = torch.fft.fftn(_embed(torch.complex(shape.float().double(), elec.float().double()).view(ng, ng, ng), nf)).conj()
    spectral, t = case["kind"] == "spectral", case.get("t", 1)
    best, step = [], max(1, min(32, int(2e8 / nf ** 3)))
    kx, kz = _signed(nf, nf), _signed(nf, nf // 2 + 1)
    weight = torch.full((nf // 2 + 1,), 2.0, dtype=torch.float64, device="cuda")
    weight[0] = weight[-1] = 1.0
    for s in range(0, n, step):
        grids = _embed(_ligand_grids(x["lig"], x["rot"][s:s + step], ng), nf)
        maps = torch.fft.ifftn(torch.fft.fftn(grids, dim=(1, 2, 3)) * rec, dim=(1, 2, 3)).real
        if not spectral:
            top = torch.topk(maps.reshape(len(maps), -1), t, dim=1).values
            best.append(top.clamp(min=0.0) if t == 1 else top)
            continue
        for m, at in zip(maps, _gpu(x["trans"][s:s + step]).double()):
            Q = torch.fft.rfftn(m).reshape(nf * nf, -1)
            ex, ey = [torch.exp(2j * math.pi * kx * at[a] / nf) for a in (0, 1)]
            ez = torch.exp(2j * math.pi * kz * at[2] / nf) * weight
            Z = (Q @ torch.stack([ez, kz * ez], 1)).view(nf, nf, 2)
            Y = [Z[..., 0] @ ey, Z[..., 0] @ (kx * ey), Z[..., 1] @ ey]
            g = -2.0 * math.pi / nf
            best.append(torch.stack([(ex @ Y[0]).real, g * (kx * ex @ Y[0]).imag, g * (ex @ Y[1]).imag,
                                     g * (ex @ Y[2]).imag]) / nf ** 3)
    if spectral:
        return {"value": torch.stack(best)}
    score = torch.cat(best).reshape(-1)
    if case["kind"] != "dock":
        score = torch.sort(score, descending=True).values[:min(case["best"], len(score))]
    return {"score": score, "index": None}
