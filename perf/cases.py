"""The work that a user of this library has it do, as measurable cases.

A case names a molecule, a precision and sizes; `prepare` builds what the
user's program holds before the call (a context with its densities, points,
planes or a network), `run` is one pass through the public entry points, and
`exact` restates the result in plain 64-bit torch.

FP64 is the default of every entry point, of the driver and of the pygimic
class, so most cases run it; the mixed path is what large fields and scans
opt into.  Molecules are the seeded ones of gimic_amd.synth: ring12 (nbf 114),
sheet30 (312), cage60 (1800) and the open-shell sheet200 (2620).
"""
import functools
import math

import numpy as np
import torch

from gimic_amd import flux, grid, lib, surrogate, synth

SCREENING = 1e-8  # lib.Context's default


def listed():
    return [
        # pygimic: one tensor at one point per call, latency only
        dict(name="point", kind="points", mol="ring12", n=1, precision="fp64"),
        # a small molecule's field on a 40^3 cube, host arrays as the driver's
        # cdens run passes them
        dict(name="ring_field", kind="points", mol="ring12", n=64000, precision="fp64"),
        # the driver's integral run: one bond plane (20 x 30 blocks of order
        # 7), current, modulus and ACID from the same tensors
        dict(name="bond_plane", kind="planes", mol="sheet30", planes=1, n1=140, n2=210,
             precision="fp64", graph=False),
        # an integration scan, planes of uneven size in one call
        dict(name="scan_fp64", kind="scan", mol="sheet30", planes=256, precision="fp64",
             graph=False),
        # the same scan opted into mixed precision and one graph launch
        dict(name="scan_mixed", kind="scan", mol="sheet30", planes=256, precision="mixed",
             graph=True),
        # a field on a ragged cube around a 60-atom cage, points resident on
        # the GPU, in the default precision
        dict(name="cage_fp64", kind="cube", mol="cage60", side=95, precision="fp64"),
        # the dense visualisation grid of the same molecule in mixed precision
        dict(name="cage_mixed", kind="cube", mol="cage60", side=128, precision="mixed"),
        # open shell, two density sets of 2620 functions: charge and spin
        # current from one pass over the basis
        dict(name="open_shell", kind="spin", mol="sheet200", n1=96, n2=96, n3=47,
             precision="mixed"),
        # shielding of every nucleus and the magnetizability on per-atom grids
        dict(name="shielding", kind="property", mol="sheet30", nr=24, nt=12, precision="fp64"),
        # a whole run on one molecule: context from arrays, densities, one
        # plane, context closed again
        dict(name="cage_job", kind="job", mol="cage60", n1=140, n2=140, precision="fp64"),
        # the learned field on a 256^3 visualisation grid
        dict(name="net_grid", kind="predict", n=256 ** 3),
        # 16 training steps of the learned field between two checkpoints of
        # its parameters, at the batch size of Surrogate.fit
        dict(name="net_train", kind="train", batch=16384, steps=16),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["points", "points", "cube", "cube", "planes", "scan", "property", "job",
                       "predict", "train"])
    mol = rng.choice(["ring12", "sheet30", "cage60"])
    prec = rng.choice(["fp64", "fp64", "mixed"])
    if kind == "points":
        return dict(kind=kind, mol=mol, n=_log_int(rng, 1, 60000), precision=prec)
    if kind == "cube":
        return dict(kind=kind, mol=mol, side=_log_int(rng, 11, 80), precision=prec)
    if kind == "planes":
        return dict(kind=kind, mol=mol, planes=rng.randint(1, 9), n1=7 * rng.randint(1, 30),
                    n2=7 * rng.randint(1, 30), precision=prec, graph=rng.random() < 0.5)
    if kind == "scan":
        return dict(kind=kind, mol="sheet30", planes=_log_int(rng, 4, 250), precision=prec,
                    graph=rng.random() < 0.5)
    if kind == "property":
        return dict(kind=kind, mol=mol, nr=rng.randint(5, 20), nt=rng.randint(4, 12),
                    precision="fp64")
    if kind == "job":
        return dict(kind=kind, mol=mol, n1=7 * rng.randint(1, 30), n2=7 * rng.randint(1, 30),
                    precision="fp64")
    if kind == "predict":
        return dict(kind=kind, n=_log_int(rng, 100, 10_000_000))
    return dict(kind=kind, batch=_log_int(rng, 300, 60000), steps=rng.randint(4, 20))


# ------------------------------------------------------------------ inputs


@functools.lru_cache(maxsize=None)
def molecule(name):
    return getattr(synth, name)()


def _context(case):
    ctx = molecule(case["mol"]).context(screening=SCREENING)
    if case.get("graph"):
        ctx.set_graph(True)
    return ctx


def _rng(seed):
    return np.random.default_rng([int(seed), 77])


def _half_box(system):
    return float(np.abs(np.asarray(system.coords)).max()) + 3.0


def _points(case, seed):
    """(N, 3) host points of a points, cube or spin case"""
    rng, s = _rng(seed), molecule(case["mol"])
    if case["kind"] == "points":
        # half spread over the box, half along the atoms, as lines and small
        # sets of probe points are
        n, box = case["n"], _half_box(s)
        u = rng.uniform(-box, box, (n, 3))
        a = np.asarray(s.coords)[rng.integers(0, s.natoms, n)] + rng.normal(0.0, 1.0, (n, 3))
        return np.where((np.arange(n) % 2 == 0)[:, None], u, a)
    if case["kind"] == "cube":
        # a regular grid over the molecule, x fastest, shifted by less than a step
        side, box = case["side"], 7.62 if case["mol"] == "cage60" else _half_box(s)
        h = 2.0 * box / max(side - 1, 1)
        return synth.cube_grid(side, h, -box) + h * rng.uniform(-0.5, 0.5, 3)
    n = (case["n1"], case["n2"], case["n3"])
    ax = [0.2 * (np.arange(k) - 0.5 * (k - 1)) * 192.0 / case["n1"] for k in n]
    z, y, x = np.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    p = np.stack([x.ravel(), y.ravel(), z.ravel()], axis=1)
    return p + 0.2 * rng.uniform(-0.5, 0.5, 3)


def _grids(case, seed):
    """[(Grid, B)] of a planes, scan or job case: planes across the first
    bond, moved along it by an offset of the seed's"""
    rng, s = _rng(seed), molecule(case["mol"])
    c = np.asarray(s.coords)
    d = np.linalg.norm(c - c[0], axis=1)
    d[0] = np.inf
    j = int(np.argmin(d))
    fix = [0.0, 0.0, 0.0] if case["mol"] == "cage60" else [0.0, 0.0, 10.0]
    k = case.get("planes", 1)
    if case["kind"] == "scan":
        # the same sizes whatever the seed: a moved scan, not another one
        offs = np.linspace(-6.0, 6.0, k) + rng.uniform(-0.02, 0.02)
        fixed = np.random.default_rng(7)
        sizes = [(int(fixed.integers(40, 121)), int(fixed.integers(60, 201))) for _ in range(k)]
    else:
        offs = rng.uniform(-0.5, 0.5, k)
        sizes = [(case["n1"], case["n2"])] * k
    out = []
    for off, (n1, n2) in zip(offs, sizes):
        kw = {"_arg": "bond", "type": "lobatto", "gauss_order": 7, "bond": [1, j + 1],
              "fixcoord": fix, "distance": float(d[j] / 2 + off), "height": [-8.0, 8.0],
              "width": [-10.0, 10.0], "grid_points": [n1, n2, 0]}
        g = grid.new_grid(kw, c)
        out.append((g, grid.get_magnet(g, "X")))
    return out


def _atom_grids(case, seed):
    """points, weights and block sizes of per-atom product grids: Gauss in r
    and cos(theta), trapezoid in phi, turned by an angle of the seed's"""
    c, nr, nt, rmax = np.asarray(molecule(case["mol"]).coords), case["nr"], case["nt"], 6.0
    x, w = np.polynomial.legendre.leggauss(nr)
    r = 0.5 * rmax * (x + 1.0)
    w = 0.5 * rmax * w * r * r
    ct, wt = np.polynomial.legendre.leggauss(nt)
    ph = 2.0 * np.pi * (np.arange(2 * nt) + _rng(seed).uniform()) / (2 * nt)
    R, C, P = np.meshgrid(r, ct, ph, indexing="ij")
    W = np.broadcast_to(w[:, None, None] * wt[None, :, None] * (np.pi / nt), R.shape).reshape(-1)
    S = np.sqrt(1.0 - C * C)
    local = np.stack([R * S * np.cos(P), R * S * np.sin(P), R * C], axis=-1).reshape(-1, 3)
    pts = np.concatenate([local + a for a in c])
    return pts, np.tile(W, len(c)), np.full(len(c), len(local))


NET = dict(sigma=3.0, center_scale=[0.0, 0.0, 0.0, 8.0], out_scale=np.linspace(0.5, 1.5, 9), seed=3)
NET_LR, NET_EPS = 2e-4, 1e-3


def _net_points(n, seed):
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    return 16.0 * torch.rand((n, 3), generator=g, dtype=torch.float64, device="cuda") - 8.0


def _net_targets(r):
    """a smooth field that decays over the box, the shape J has"""
    k = torch.arange(1, 10, dtype=torch.float64, device=r.device)
    a = 0.3 * torch.outer(r[:, 0], k) + 0.2 * torch.outer(r[:, 1], 10 - k) + 0.5 * r[:, 2:]
    return torch.sin(a) * torch.exp(-0.4 * r.norm(dim=1, keepdim=True))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "points":
        return dict(case=case, ctx=_context(case), points=_points(case, seed))
    if kind in ("cube", "spin"):
        pts = torch.as_tensor(_points(case, seed)).cuda()
        return dict(case=case, ctx=_context(case), points=pts)
    if kind in ("planes", "scan"):
        g = _grids(case, seed)
        return dict(case=case, ctx=_context(case), grids=[a for a, _ in g], fields=[b for _, b in g])
    if kind == "property":
        return dict(case=case, ctx=_context(case), grid=_atom_grids(case, seed),
                    nuclei=np.asarray(molecule(case["mol"]).coords))
    if kind == "job":
        s = molecule(case["mol"])
        return dict(case=case, arrays=s.arrays(), dens=s.dens, grid=_grids(case, seed)[0])
    net = surrogate.Network(**NET)
    if kind == "predict":
        return dict(case=case, net=net, points=_net_points(case["n"], seed))
    r = _net_points(case["steps"] * case["batch"], seed).reshape(case["steps"], case["batch"], 3)
    return dict(case=case, net=net, points=r, targets=torch.stack([_net_targets(x) for x in r]))


# -------------------------------------------------------------- one pass


def run(state):
    case = state["case"]
    kind, prec = case["kind"], case.get("precision")
    if kind == "points":
        return state["ctx"].jtensor(state["points"], precision=prec)
    if kind == "cube":
        return state["ctx"].jtensor_device(state["points"], precision=prec)
    if kind == "spin":
        return state["ctx"].jtensor_multi_device(state["points"], ["total", "spindens"],
                                                 precision=prec)
    if kind == "planes":
        return state["ctx"].flux_plane_grids(state["grids"], state["fields"], precision=prec,
                                             modulus=True, acid=True)
    if kind == "scan":
        return flux.integrate_planes(state["ctx"], state["grids"], state["fields"], precision=prec)
    if kind == "property":
        pts, w, sizes = state["grid"]
        return state["ctx"].properties(pts, w, sizes, state["nuclei"], precision=prec)
    if kind == "job":
        a, (g, b) = state["arrays"], state["grid"]
        with lib.Context.from_arrays(a["coords"], a["shell_atom"], a["shell_l"], a["shell_nprim"],
                                     a["shell_poff"], a["exps"], a["coefs"], spherical=True,
                                     screening=SCREENING) as ctx:
            ctx.set_density(state["dens"])
            return np.array(flux.integrate_current(ctx, g, b, precision=prec))
    if kind == "predict":
        return state["net"].predict(state["points"])
    loss = None
    for i in range(case["steps"]):
        loss = state["net"].train_step(state["points"][i], state["targets"][i], NET_EPS, NET_LR,
                                       want_loss=i == case["steps"] - 1)
    return dict(loss=loss, params=state["net"].params())


# ------------------------------------------------------------------- work


def _counts(case):
    """(points, mean square of the functions that reach a point)"""
    kind = case["kind"]
    if kind in ("points", "cube", "spin"):
        pts = _points(case, 1)
    elif kind == "property":
        pts = _atom_grids(case, 1)[0]
    else:
        pts = np.concatenate([_plane_points(g)[0] for g, _ in _grids(case, 1)])
    s = molecule(case["mol"])
    x = pts[np.random.default_rng(1).integers(0, len(pts), 512)]
    d = np.linalg.norm(x[:, None] - np.asarray(s.coords)[None], axis=2)
    live = np.zeros(len(x))
    for a, l, n, o in zip(s.shell_atom, s.shell_l, s.shell_nprim, s.shell_poff):
        live += (2 * l + 1) * (d[:, a] <= _radius(l, s.exps[o:o + n]))
    return len(pts), float((live * live).mean())


def work(case):
    kind = case["kind"]
    if kind in ("predict", "train"):
        macs = 160 * 128 + 3 * 128 * 128 + 128 * 16
        if kind == "predict":
            return dict(bytes=case["n"] * 96.0, flops=2.0 * macs * case["n"])
        p = case["batch"] * case["steps"]
        return dict(bytes=p * 96.0 + case["steps"] * macs * 28.0, flops=6.0 * macs * p)
    n = molecule(case["mol"]).nbf
    npts, live2 = _counts(case)
    sets = 2 if kind == "spin" else 1
    out = {"points": 72, "cube": 72, "spin": 144}.get(kind, 0)
    # the densities are read once, the points once; seven products over the
    # functions that reach a point
    return dict(bytes=npts * (24.0 + out) + 32.0 * sets * n * n, flops=14.0 * sets * live2 * npts)


# ------------------------------------------------- the results in 64 bits

# rows m = -l..l of the real solid harmonics as {(a, b, c): coefficient} of
# x^a y^b z^c, before normalisation (l = 1: x, y, z)
_HARMONICS = {
    0: [{(0, 0, 0): 1.0}],
    1: [{(1, 0, 0): 1.0}, {(0, 1, 0): 1.0}, {(0, 0, 1): 1.0}],
    2: [{(1, 1, 0): 1.0}, {(0, 1, 1): 1.0}, {(0, 0, 2): 2.0, (2, 0, 0): -1.0, (0, 2, 0): -1.0},
        {(1, 0, 1): 1.0}, {(2, 0, 0): 1.0, (0, 2, 0): -1.0}],
    3: [{(2, 1, 0): 3.0, (0, 3, 0): -1.0}, {(1, 1, 1): 1.0},
        {(0, 1, 2): 4.0, (2, 1, 0): -1.0, (0, 3, 0): -1.0},
        {(0, 0, 3): 2.0, (2, 0, 1): -3.0, (0, 2, 1): -3.0},
        {(1, 0, 2): 4.0, (3, 0, 0): -1.0, (1, 2, 0): -1.0},
        {(2, 0, 1): 1.0, (0, 2, 1): -1.0}, {(3, 0, 0): 1.0, (1, 2, 0): -3.0}],
}


def _moment(k):
    return 0.0 if k % 2 else float(np.prod(np.arange(k - 1, 0, -2))) if k > 0 else 1.0


def _harmonics(l):
    rows = []
    for row in _HARMONICS[l]:
        norm = sum(u * v * math.prod(_moment(i + j) for i, j in zip(p, q))
                   for p, u in row.items() for q, v in row.items())
        rows.append({p: u / math.sqrt(norm) for p, u in row.items()})
    return rows


def _radius(l, exps):
    """the first multiple of 0.25 bohr where t^l exp(-alpha_min t^2) is down
    to the screening threshold"""
    t = 0.0
    while True:
        t += 0.25
        if t ** l * math.exp(-min(exps) * t * t) <= SCREENING:
            return t


def _basis(s, r):
    """phi (P, n) and gradient (3, P, n) of every function at r (P, 3)"""
    atoms = torch.as_tensor(np.asarray(s.coords), device=r.device)
    out = torch.zeros((4, r.shape[0], s.nbf), dtype=torch.float64, device=r.device)
    groups, col = {}, 0
    for a, l, n, o in zip(s.shell_atom, s.shell_l, s.shell_nprim, s.shell_poff):
        key = (l, tuple(s.exps[o:o + n]), tuple(s.coefs[o:o + n]))
        groups.setdefault(key, ([], []))
        groups[key][0].append(a)
        groups[key][1].append(col)
        col += 2 * l + 1
    for (l, exps, coefs), (at, cols) in groups.items():
        al, c = np.array(exps), np.array(coefs)
        t = 2.0 * np.sqrt(np.outer(al, al)) / (al[:, None] + al)
        c = c / math.sqrt((np.outer(c, c) * t ** (l + 1.5)).sum())
        c = c * (4.0 * al) ** (0.5 * l + 0.75) * (0.5 / math.pi) ** 0.75
        d = r[:, None, :] - atoms[at][None]
        s2 = (d * d).sum(dim=2)
        live = s2.sqrt() <= _radius(l, exps)
        g, h = torch.zeros_like(s2), torch.zeros_like(s2)
        for x, w in zip(al, c):
            e = torch.where(live, w * torch.exp(-x * s2), 0.0)
            g += e
            h += x * e
        pw = [[torch.ones_like(s2)] for _ in range(3)]
        for k in range(3):
            for _ in range(l):
                pw[k].append(pw[k][-1] * d[:, :, k])
        idx = torch.as_tensor(cols, device=r.device)
        for i, row in enumerate(_harmonics(l)):
            val = [torch.zeros_like(s2) for _ in range(4)]
            for p, u in row.items():
                val[0] += u * pw[0][p[0]] * pw[1][p[1]] * pw[2][p[2]]
                for k in range(3):
                    if p[k]:
                        q = [p[j] - (j == k) for j in range(3)]
                        val[1 + k] += u * p[k] * pw[0][q[0]] * pw[1][q[1]] * pw[2][q[2]]
            out[0][:, idx + i] = val[0] * g
            for k in range(3):
                out[1 + k][:, idx + i] = val[1 + k] * g - 2.0 * d[:, :, k] * val[0] * h
    return out[0], out[1:]


def _cyclic(i, j, k):
    return (i - j) * (j - k) * (k - i) / 2.0


def _tensors(mol, pts, spin="total"):
    """J (N, 9) at pts, element m + 3b = J(m, b), on the GPU"""
    s = molecule(mol)
    dens = np.asarray(s.dens)
    if len(dens) == 2:
        dens = dens[0] - dens[1] if spin == "spindens" else dens[0] + dens[1]
    else:
        dens = dens[0]
    D = torch.as_tensor(dens).cuda()
    at = [a for a, l in zip(s.shell_atom, s.shell_l) for _ in range(2 * l + 1)]
    R = torch.as_tensor(np.asarray(s.coords)[at]).cuda()
    W = [D[0] * (R[None, :, d] - R[:, None, d]) for d in range(3)]
    pts = torch.as_tensor(pts).cuda()
    out = torch.empty((len(pts), 9), dtype=torch.float64, device="cuda")
    step = max(1024, int(6e7 / s.nbf))
    for p0 in range(0, len(pts), step):
        r = pts[p0:p0 + step]
        phi, G = _basis(s, r)
        y = (phi @ D[0]) * phi
        E = [(y * (r[:, d:d + 1] - R[None, :, d])).sum(dim=1) for d in range(3)]
        A = [[(G[m] * Y).sum(dim=1) for m in range(3)] for Y in (phi @ D[1 + b] for b in range(3))]
        Q = [[(G[m] * Y).sum(dim=1) for m in range(3)] for Y in (phi @ W[d] for d in range(3))]
        for b in range(3):
            for m in range(3):
                v = A[b][m].clone()
                for c in range(3):
                    for d in range(3):
                        if _cyclic(b, c, d):
                            v += _cyclic(b, c, d) * r[:, c] * Q[d][m]
                for d in range(3):
                    if _cyclic(m, b, d):
                        v += _cyclic(m, b, d) * E[d]
                out[p0:p0 + step, m + 3 * b] = 0.5 * v
    return out


def _plane_points(g):
    """points and weights of a one-layer product grid from its 1-D rules"""
    v = np.asarray(g.basv)
    p = [np.asarray(x) for x in g.pts]
    w = [np.asarray(x) for x in g.wgt]
    r = (np.asarray(g.origin) + p[0][None, :, None] * v[:, 0] + p[1][:, None, None] * v[:, 1]
         + p[2][0] * v[:, 2])
    return r.reshape(-1, 3), (w[2][0] * w[1][:, None] * w[0][None, :]).reshape(-1)


def _signed_sums(v):
    return [v.sum(), v[v > 0].sum(), v[v <= 0].sum()]


def _plane_sums(mol, grids):
    parts = [_plane_points(g) for g, _ in grids]
    J = _tensors(mol, np.concatenate([p for p, _ in parts])).cpu().numpy().reshape(-1, 3, 3)
    cur, mod, acid, at = [], [], [], 0
    for (g, b), (p, w) in zip(grids, parts):
        T = J[at:at + len(p)].transpose(0, 2, 1)  # T[:, m, b]
        at += len(p)
        v = np.asarray(g.basv)
        corner = [np.asarray(g.origin) + g.pts[0][i] * v[:, 0] + g.pts[1][j] * v[:, 1]
                  + g.pts[2][0] * v[:, 2] for i, j in ((-1, 0), (0, -1))]
        w = np.where(np.linalg.norm(p - 0.5 * (corner[0] + corner[1]), axis=1) > g.radius, 0.0, w)
        jv = T @ np.asarray(b, dtype=np.float64)
        dot = jv @ v[:, 2]
        cur.append(_signed_sums(w * dot))
        sgn = np.where(np.abs(dot) < 1e-12, 0.0, np.sign(dot))
        mod.append(_signed_sums(w * sgn * np.linalg.norm(jv, axis=1)))
        dd = (T[:, 0, 0] - T[:, 1, 1]) ** 2 + (T[:, 1, 1] - T[:, 2, 2]) ** 2 \
            + (T[:, 2, 2] - T[:, 0, 0]) ** 2
        oo = (T[:, 0, 1] + T[:, 1, 0]) ** 2 + (T[:, 0, 2] + T[:, 2, 0]) ** 2 \
            + (T[:, 1, 2] + T[:, 2, 1]) ** 2
        acid.append((w * (0.3333333 * dd + 0.5 * oo)).sum())
    return np.array(cur), np.array(mod), np.array(acid)


def _properties(case, seed):
    pts, w, sizes = _atom_grids(case, seed)
    J = _tensors(case["mol"], pts)
    r, w = torch.as_tensor(pts).cuda(), torch.as_tensor(w).cuda()
    edge = np.concatenate([[0], np.cumsum(sizes)])

    def blocks(d, f):
        t = [f * (d[:, (b + 2) % 3] * J[:, (b + 1) % 3 + 3 * b]
                  - d[:, (b + 1) % 3] * J[:, (b + 2) % 3 + 3 * b]) * w for b in range(3)]
        tot = t[0] + t[1] + t[2]
        cols = t + [tot.clamp(min=0.0), tot.clamp(max=0.0)]
        return [[float(c[i:j].sum()) for c in cols] for i, j in zip(edge[:-1], edge[1:])]

    shield = []
    for R in torch.as_tensor(np.asarray(molecule(case["mol"]).coords)).cuda():
        d = r - R
        shield.append(blocks(d, -1e6 / (d.norm(dim=1) ** 3 * 137.0359998 ** 2)))
    return dict(shield=np.array(shield), magnet=np.array(blocks(r, 0.5)))


def _net():
    """the network's layers in 64 bits (its weights and frequencies as the
    handle reports them)"""
    net = surrogate.Network(**NET)
    p = torch.as_tensor(net.params()).cuda().double()
    sizes, at, layers = [(160, 128)] + [(128, 128)] * 3 + [(128, 16)], 0, []
    for k, n in sizes:
        layers += [p[at:at + n * k].reshape(n, k), p[at + n * k:at + n * k + n]]
        at += n * k + n
    return layers, torch.as_tensor(net.freqs()).cuda().double().reshape(-1, 3)


def _net_forward(layers, freqs, r):
    u = (r - torch.tensor(NET["center_scale"][:3], dtype=torch.float64, device="cuda")) \
        / NET["center_scale"][3]
    t = 2.0 * math.pi * u @ freqs.T
    x = torch.cat([torch.sin(t), torch.cos(t), u,
                   torch.zeros((len(r), 29), dtype=torch.float64, device="cuda")], dim=1)
    for i in range(4):
        x = torch.nn.functional.silu(x @ layers[2 * i].T + layers[2 * i + 1])
    return x @ layers[8].T + layers[9]


def _train(case, seed):
    layers, freqs = _net()
    layers = [x.requires_grad_(True) for x in layers]
    adam = torch.optim.Adam(layers, lr=NET_LR, betas=(0.9, 0.999), eps=1e-8)
    scale = torch.as_tensor(NET["out_scale"]).cuda()
    r = _net_points(case["steps"] * case["batch"], seed).reshape(case["steps"], case["batch"], 3)
    loss = None
    for x in r:
        t = _net_targets(x) / scale
        n = ((t * t).sum(dim=1) + NET_EPS ** 2).sqrt()
        y = _net_forward(layers, freqs, x)
        loss = (((y[:, :9] - t / n[:, None]) ** 2).sum(dim=1) + (y[:, 9] - n.log()) ** 2).mean()
        adam.zero_grad()
        loss.backward()
        adam.step()
    return dict(loss=float(loss), params=torch.cat([x.detach().reshape(-1) for x in layers]).cpu().numpy())


def exact(case, seed):
    kind = case["kind"]
    if kind in ("points", "cube"):
        J = _tensors(case["mol"], _points(case, seed))
        return J.cpu().numpy() if kind == "points" else J
    if kind == "spin":
        pts = _points(case, seed)
        return torch.stack([_tensors(case["mol"], pts, s) for s in ("total", "spindens")])
    if kind == "planes":
        return _plane_sums(case["mol"], _grids(case, seed))
    if kind == "scan":
        return _plane_sums(case["mol"], _grids(case, seed))[0]
    if kind == "property":
        return _properties(case, seed)
    if kind == "job":
        return _plane_sums(case["mol"], _grids(case, seed))[0][0]
    if kind == "predict":
        layers, freqs = _net()
        r, s = _net_points(case["n"], seed), torch.as_tensor(NET["out_scale"]).cuda()
        out = torch.empty((case["n"], 9), dtype=torch.float64, device="cuda")
        for i in range(0, case["n"], 1 << 20):
            y = _net_forward(layers, freqs, r[i:i + (1 << 20)])
            out[i:i + (1 << 20)] = y[:, :9] * torch.exp(y[:, 9:10].clamp(max=60.0)) * s
        return out
    return _train(case, seed)
