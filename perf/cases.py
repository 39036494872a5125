"""Cases of the short-range force framework: what its users run, at the sizes they run it.

Each case is a dict of plain values; ``prepare`` makes its inputs and the handle a
program keeps (a Context, a ForceSolver, a Particles object), ``run`` makes one pass
through the public entry points, ``exact`` gives the outputs in 64 bits with plain
torch where they have such a value, ``work`` states what a pass cannot do without.

Particles are those of the framework's own loads (haccsr.ics): a Plummer mix (70 %
uniform, 30 % in clumps) and a clustered load (Zel'dovich displacements of a k^-2
field and NFW halos), one particle per unit cell on average, generated here on the
device; ghosts within a shell of 3.2 around the periodic box; cell order, as
Particles::resortParticles leaves them.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(ROOT, "hacc-coral_amd")
if _PKG not in sys.path:
    sys.path.insert(1, _PKG)

from haccsr import _lib, autograd, forcetree  # noqa: E402
from haccsr.particles import Particles, TimeStepperValues  # noqa: E402

DEV = "cuda:0"
SHELL = 3.2        # ghost shell width
RC, RSM = 3.12, 0.1
P5 = (0.269327, -0.0750978, 0.0114808, -0.00109313, 0.0000605491, -0.00000147177)
P6 = (0.271431, -0.0783394, 0.0133122, -0.00159485, 0.000132336, -0.00000663394, 0.000000147305)
FLOPS_PAIR = 30    # of one pair: difference, s, rsqrt, cube, polynomial, mass, accumulation
ARRAYS = ("x", "y", "z", "vx", "vy", "vz", "mass", "phi", "id", "mask")


def listed():
    return [
        # the smallest calls: one rank's step on a small box, where latency and launches count
        {"name": "step_16", "kind": "step", "load": "plummer", "side": 16, "nd": 32,
         "law": "step16", "tdpts": 1, "graph": False},
        # the 64^3 Plummer mix at the constructor's usual leaf size
        {"name": "step_64", "kind": "step", "load": "plummer", "side": 64, "nd": 128,
         "law": "step16", "tdpts": 1, "graph": False},
        # the headline step of bench.py: 256^3 clustered, the tuned leaf size and kernel shape
        {"name": "step_256", "kind": "step", "load": "clustered", "side": 256, "nd": 512,
         "law": "step16", "tdpts": 1, "graph": True},
        # the quadrupole tree on an odd-sized box
        {"name": "quad_61", "kind": "step", "load": "plummer", "side": 61, "nd": 100,
         "law": "poly6", "tdpts": 12, "graph": False},
        # forces of an isolated group in the caller's own order with the reference's default
        # law, ForceLawSR over the fitted grid force (FGridEvalFit)
        {"name": "fit_60", "kind": "forces", "load": "plummer", "side": 60, "nd": 128,
         "law": "fit"},
        # the drop-in constructor on a caller's host arrays (RCBMonopoleForceTree)
        {"name": "dropin_48", "kind": "dropin", "load": "clustered", "side": 48, "nd": 128,
         "law": "poly6"},
        # forward and backward of the differentiable force, a group small enough to check
        {"name": "grad_50", "kind": "grad", "load": "plummer", "side": 50, "nd": 128,
         "images": False},
        # the same at the 128^3 differentiation load, ghosts included
        {"name": "grad_128", "kind": "grad", "load": "clustered", "side": 128, "nd": 256,
         "images": True},
        # an ensemble of boxes of mixed sizes in one build, one list pass, one launch
        {"name": "ensemble_24", "kind": "ensemble", "boxes": 24, "side_min": 20, "side_max": 64,
         "nd": 256},
        # one sub-step of Particles::subCycle with resident particles: stream, resort, tree,
        # lists, kick, stream (one: the order after a kick depends on its rounding)
        {"name": "substep_128", "kind": "substep", "load": "clustered", "side": 128, "nd": 256},
        # the particle-grid steps of a long step: deposit, then three interpolations
        {"name": "pm_256", "kind": "pm", "load": "clustered", "side": 256},
        # the one-rank overload refresh of a long step
        {"name": "refresh_160", "kind": "refresh", "load": "clustered", "side": 160},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "forces", "dropin", "grad", "ensemble", "substep",
                       "pm", "refresh"])
    load = rng.choice(["plummer", "clustered"])
    c = {"kind": kind}
    if kind == "ensemble":
        lo = rng.randint(14, 32)
        return dict(c, boxes=rng.randint(2, 24), side_min=lo, side_max=rng.randint(lo, 64),
                    nd=_log_int(rng, 64, 512))
    c["load"] = load

    def leaf(side, hi):  # small leaves where the box is small
        return _log_int(rng, 24 if side <= 40 else 100, hi)

    if kind == "step":
        tdpts = rng.choice([1, 1, 1, 12])
        side = _log_int(rng, 12, 180 if tdpts == 1 else 96)
        c.update(side=side, nd=leaf(side, 700),
                 law=rng.choice(["step16", "step16", "poly5", "poly6", "interp"]),
                 tdpts=tdpts, graph=rng.random() < 0.5)
    elif kind == "forces":
        side = _log_int(rng, 10, 64)
        c.update(side=side, nd=leaf(side, 512),
                 law=rng.choice(["step16", "poly6", "fit", "fit", "interp"]))
    elif kind == "dropin":
        side = _log_int(rng, 10, 64)
        c.update(side=side, nd=leaf(side, 512),
                 law=rng.choice(["step16", "poly5", "poly6", "fit", "interp"]))
    elif kind == "grad":
        images = rng.random() < 0.5
        side = _log_int(rng, 10, 128 if images else 50)
        c.update(side=side, nd=leaf(side, 512), images=images)
    elif kind == "substep":
        side = _log_int(rng, 12, 160)
        c.update(side=side, nd=leaf(side, 640))
    else:
        c.update(side=_log_int(rng, 16, 256))
    return c


# ---------------------------------------------------------------- particles

def _plummer(side, g):
    n = side ** 3
    n_uni = int(round(0.7 * n))
    pos = torch.rand((n, 3), generator=g, device=DEV, dtype=torch.float64) * side
    centres = torch.rand((20, 3), generator=g, device=DEV, dtype=torch.float64) * side
    which = torch.randint(0, 20, (n - n_uni,), generator=g, device=DEV)
    u = torch.rand(n - n_uni, generator=g, device=DEV, dtype=torch.float64).clamp(1e-12, 1 - 1e-12)
    r = (0.5 / torch.sqrt(u ** (-2.0 / 3.0) - 1.0)).clamp(max=0.45 * side)
    d = torch.randn((n - n_uni, 3), generator=g, device=DEV, dtype=torch.float64)
    pos[n_uni:] = centres[which] + r[:, None] * d / d.norm(dim=1, keepdim=True)
    return pos


def _clustered(side, g):
    n = side ** 3
    k = torch.fft.fftfreq(side, d=1.0 / side, device=DEV) * (2 * math.pi / side)
    kr = torch.fft.rfftfreq(side, d=1.0 / side, device=DEV) * (2 * math.pi / side)
    ks = (k[:, None, None], k[None, :, None], kr[None, None, :])
    k2 = ks[0] ** 2 + ks[1] ** 2 + ks[2] ** 2
    k2[0, 0, 0] = 1.0
    dk = torch.fft.rfftn(torch.randn((side,) * 3, generator=g, device=DEV)) / torch.sqrt(k2)
    dk[0, 0, 0] = 0
    disp = torch.stack([torch.fft.irfftn(1j * kk / k2 * dk, s=(side,) * 3) for kk in ks], -1)
    disp *= 2.0 / torch.sqrt((disp.double() ** 2).sum(-1).mean()).float()
    q = torch.arange(side, device=DEV, dtype=torch.float64) + 0.5
    pos = torch.stack(torch.meshgrid(q, q, q, indexing="ij"), -1) + disp.double()
    pos = pos.reshape(n, 3)
    # NFW halos of 1e3..1e5 particles replace field particles
    halos = max(1, round(500 * (side / 256) ** 3))
    size = torch.exp(torch.rand(halos, generator=g, device=DEV, dtype=torch.float64) * math.log(100.0)
                     + math.log(1e3))
    size = (size * min(1.0, 0.5 * n / float(size.sum()))).long()
    h = torch.repeat_interleave(torch.arange(halos, device=DEV), size)
    conc = 5.0 + 10.0 * torch.rand(halos, generator=g, device=DEV, dtype=torch.float64)
    r200 = (3.0 * size.double() / (800.0 * math.pi)) ** (1.0 / 3.0)
    centre = torch.rand((halos, 3), generator=g, device=DEV, dtype=torch.float64) * side
    mu = torch.log1p(conc) - conc / (1 + conc)
    u = torch.rand(h.numel(), generator=g, device=DEV, dtype=torch.float64)
    # inverse of the enclosed mass, from a table over x = c r / r200
    xt = torch.logspace(-6, math.log10(15.0), 20000, device=DEV, dtype=torch.float64)
    mt = torch.log1p(xt) - xt / (1 + xt)
    x = xt[torch.searchsorted(mt, u * mu[h]).clamp(max=xt.numel() - 1)]
    d = torch.randn((h.numel(), 3), generator=g, device=DEV, dtype=torch.float64)
    halo = centre[h] + (x * (r200 / conc)[h])[:, None] * d / d.norm(dim=1, keepdim=True)
    pos[torch.randperm(n, generator=g, device=DEV)[: h.numel()]] = halo
    return pos


def _positions(load, side, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    pos = (_plummer if load == "plummer" else _clustered)(side, g)
    pos = torch.remainder(pos, side).float()
    pos[pos >= side] = 0.0
    return pos, g


def _ghosts(pos, side):
    """Periodic images within SHELL of the box, then a shift by +SHELL; the
    first entries are the box's own particles.  Returns positions and the
    index each entry images."""
    idx = [torch.arange(pos.shape[0], device=DEV)]
    out = [pos]
    for sx in (-1, 0, 1):
        for sy in (-1, 0, 1):
            for sz in (-1, 0, 1):
                if not (sx or sy or sz):
                    continue
                sel = torch.ones(pos.shape[0], dtype=torch.bool, device=DEV)
                for a, s in enumerate((sx, sy, sz)):
                    if s == 1:
                        sel &= pos[:, a] < SHELL
                    elif s == -1:
                        sel &= pos[:, a] >= side - SHELL
                i = torch.nonzero(sel).flatten()
                idx.append(i)
                out.append(pos[i] + torch.tensor([sx, sy, sz], device=DEV, dtype=torch.float32) * side)
    return torch.cat(out) + SHELL, torch.cat(idx)


def _cell_order(pos, ng):
    c = pos.floor().long()
    inside = ((c >= 0) & (c < ng)).all(1)
    key = torch.where(inside, (c[:, 0] * ng + c[:, 1]) * ng + c[:, 2], ng ** 3)
    return torch.argsort(key, stable=True)


def _capacity(side):
    """Particles a rank's arrays hold: half as many again as its unit cells."""
    return int(1.5 * (side + 2 * SHELL) ** 3)


def _rank(load, side, seed):
    """One rank's particles in cell order, with the ghosts its arrays have room
    for; and the generator."""
    pos, g = _positions(load, side, seed)
    pos, _ = _ghosts(pos, side)
    pos = pos[: _capacity(side)]
    return pos[_cell_order(pos, math.ceil(side + 2 * SHELL))], g


def _arrays(pos, g, cap):
    """The ten arrays of `cap` entries, the first len(pos) in use."""
    d, n = _ten(pos, g), pos.shape[0]
    return {k: torch.cat([v, v.new_zeros(cap - n)]) for k, v in d.items()}, n


def _ten(pos, g):
    n = pos.shape[0]
    d = {"x": pos[:, 0].contiguous(), "y": pos[:, 1].contiguous(), "z": pos[:, 2].contiguous()}
    for k in ("vx", "vy", "vz"):
        d[k] = 5.0 * torch.randn(n, generator=g, device=DEV)
    d["mass"] = torch.ones(n, device=DEV)
    d["phi"] = torch.zeros(n, device=DEV)
    d["id"] = torch.arange(n, dtype=torch.int64, device=DEV)
    d["mask"] = torch.zeros(n, dtype=torch.int16, device=DEV)
    return d


def _law(name):
    return {"step16": _lib.LAW_STEP16, "poly5": _lib.LAW_SR_POLY5, "poly6": _lib.LAW_SR_POLY6,
            "fit": _lib.LAW_SR_FIT, "interp": _lib.LAW_SR_INTERP}[name]


def _context(case, tdpts=1, graph=False):
    law = case.get("law", "step16")
    table = forcetree.FGridEvalInterp(forcetree.FGrid(), 2048).table() if law == "interp" else None
    ctx = _lib.Context(nd=case["nd"], fsrrmax=RC, rsm=RSM, oa=0.1, law=_law(law), tdpts=tdpts,
                       interp_table=table)
    if graph:  # bench.py's settings: the tuned kernel shape, the force phase as one graph
        shape = {} if law == "interp" else {"i_per_lane": 2, "unroll": 2, "tile": 128}
        ctx.set_tuning(use_graph=1, **shape)
    return ctx


def _boxes(side, shell):
    hi = side + 2 * shell
    return ([0.0] * 3, [hi] * 3), ([shell] * 3, [side + shell] * 3)


def _open_boxes(side):
    """The boxes of an isolated group: every leaf is listed."""
    return ([0.0] * 3, [float(side)] * 3), ([-1.0] * 3, [side + 1.0] * 3)


def _sides(case):
    r = np.random.RandomState(case["boxes"] * 1009 + case["side_min"])
    lo, hi = math.log(case["side_min"]), math.log(case["side_max"])
    return [int(round(math.exp(v))) for v in r.uniform(lo, hi, case["boxes"])]


# ----------------------------------------------------------------- prepare

def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "kind": kind}
    if kind == "ensemble":
        s.update(_prepare_ensemble(case, seed))
    elif kind == "step":
        side = case["side"]
        pos, g = _rank(case["load"], side, seed)
        s["src"], s["n"] = _arrays(pos, g, _capacity(side))
        s["buf"] = {k: v.clone() for k, v in s["src"].items()}
        s["tree"], s["force"] = _boxes(side, SHELL)
        s["ctx"] = _context(case, case["tdpts"], case["graph"])
    elif kind == "forces":
        side = case["side"]
        s["pos"], _ = _group(case, seed)
        s["tree"], s["force"] = _open_boxes(side)
        s["ctx"] = _context(case)
    elif kind == "dropin":
        side = case["side"]
        pos, g = _rank(case["load"], side, seed)
        src, s["n"] = _arrays(pos, g, _capacity(side))
        s["src"] = {k: v.cpu().numpy() for k, v in src.items()}
        s["src"]["mask"] = s["src"]["mask"].view(np.uint16)
        s["buf"] = {k: v.copy() for k, v in s["src"].items()}
        s["tree"], s["force"] = _boxes(side, SHELL)
        fg = forcetree.FGrid()
        ev = {"fit": lambda: forcetree.FGridEvalFit(fg),
              "interp": lambda: forcetree.FGridEvalInterp(fg, 2048),
              "poly5": lambda: forcetree.FGridEvalPoly(fg, 5)}.get(
                  case["law"], lambda: forcetree.FGridEvalPoly(fg, 6))()
        s["fl"] = forcetree.ForceLawSR(ev, RSM)
    elif kind == "grad":
        s.update(_prepare_grad(case, seed))
    elif kind == "substep":
        side = case["side"]
        pos, g = _rank(case["load"], side, seed)
        s["src"], s["n"] = _arrays(pos, g, _capacity(side))
        s["buf"] = {k: v.clone() for k, v in s["src"].items()}
        P = Particles([math.ceil(side + 2 * SHELL)] * 3, alpha=1.0, gpscal=1.0, edge=SHELL, nsub=1,
                      rcb_tree_ppn=case["nd"])
        P.set_particles(*(s["buf"][k][: s["n"]] for k in ARRAYS))
        s["P"] = P
        s["ts"] = TimeStepperValues(pp=0.5, tau=0.004, tau2=0.004, adot=1.3, fscal=1.1)
    elif kind == "pm":
        s["ng"], s["xyz"], s["grad"], s["v0"] = _grid_inputs(case, seed)
        s["rho"] = torch.empty(s["ng"][0] ** 3 + 1, device=DEV)
        s["n"] = s["xyz"][0].shape[0]
        s["v"] = [v.clone() for v in s["v0"]]
        s["ctx"] = _lib.Context()
    else:
        assert kind == "refresh", kind
        side = case["side"]
        dom = _lib.domain(side, SHELL, side)
        pos, g = _rank(case["load"], side, seed)
        pos = pos + (dom.ng_overload - SHELL)
        s["dom"] = dom
        # room for the copies of the wider shell whole cells make
        s["src"], s["n"] = _arrays(pos, g, 2 * _capacity(side))
        s["buf"] = {k: v.clone() for k, v in s["src"].items()}
        s["ctx"] = _lib.Context()
    torch.cuda.synchronize()
    return s


def _prepare_ensemble(case, seed):
    sides = _sides(case)
    parts, off, tree, force = [], [0], ([], []), ([], [])
    for b, side in enumerate(sides):
        pos, g = _rank("clustered", side, seed * 1000 + b)
        parts.append(pos)
        off.append(off[-1] + pos.shape[0])
        (tlo, thi), (flo, fhi) = _boxes(side, SHELL)
        tree[0].append(tlo)
        tree[1].append(thi)
        force[0].append(flo)
        force[1].append(fhi)
    src, n = _arrays(torch.cat(parts), g, sum(_capacity(side) for side in sides))
    return {"src": src, "n": n, "buf": {k: v.clone() for k, v in src.items()},
            "off": np.array(off, np.int64), "tree": tree, "force": force, "ctx": _context(case)}


def _grid_inputs(case, seed):
    """Grid, positions, the gradient of the potential per component, and the
    velocities it kicks."""
    pos, g = _rank(case["load"], case["side"], seed)
    ng = math.ceil(case["side"] + 2 * SHELL)
    xyz = [pos[:, k].contiguous() for k in range(3)]
    grad = [torch.randn(ng ** 3 + 1, generator=g, device=DEV) for _ in range(3)]
    v0 = [torch.zeros(_capacity(case["side"]), device=DEV) for _ in range(3)]
    for v in v0:
        v[: pos.shape[0]].normal_(generator=g)
    return [ng] * 3, xyz, grad, v0


def _group(case, seed):
    """An isolated group in cell order, and the cotangent of its forces."""
    pos, g = _positions(case["load"], case["side"], seed)
    pos = pos[_cell_order(pos, case["side"])]
    return pos, torch.randn(pos.shape, generator=g, device=DEV)


def _prepare_grad(case, seed):
    side = case["side"]
    images = None
    if case["images"]:
        pos, g = _positions(case["load"], side, seed)
        full, idx = _ghosts(pos, side)
        order = _cell_order(full, math.ceil(side + 2 * SHELL))
        # the box's own particles first, as the overload layout has them
        order = torch.cat([order[order < pos.shape[0]], order[order >= pos.shape[0]]])
        rank = torch.empty_like(order)
        own = order[: pos.shape[0]]
        rank[own] = torch.arange(pos.shape[0], device=DEV)
        base = pos[own]
        full, idx = full[order], rank[idx[order]]
        images = autograd.Images(idx, full - base[idx], pos.shape[0])
        pos, lam = base, torch.randn(base.shape, generator=g, device=DEV)
        tree, force = _boxes(side, SHELL)
    else:
        pos, lam = _group(case, seed)
        tree, force = _open_boxes(side)
    solver = autograd.ForceSolver(*tree, *force, nd=case["nd"], fsrrmax=RC, rsm=RSM)
    return {"pos": pos, "images": images, "solver": solver, "lam": lam}


# --------------------------------------------------------------------- run

def _restore(s):
    """The particles in the caller's arrays as its last step left them."""
    n = s["n"]
    b = {k: s["buf"][k][:n] for k in ARRAYS}
    for k in ARRAYS:
        b[k].copy_(s["src"][k][:n])
    torch.cuda.synchronize()  # the context launches on a stream of its own
    return b


def run(s):
    kind = s["kind"]
    if kind == "step":
        b, ctx = _restore(s), s["ctx"]
        ctx.build(b["x"], b["y"], b["z"], b["mass"], b["vx"], b["vy"], b["vz"], b["phi"], b["id"],
                  b["mask"], min_loc=s["tree"][0], max_loc=s["tree"][1], device_ptrs=True)
        ctx.lists(*s["force"])
        ctx.kick(0.01)
        return s["buf"]
    if kind == "forces":
        return _run_forces(s)
    if kind == "dropin":
        n = s["n"]
        b = {k: s["buf"][k][:n] for k in ARRAYS}
        for k in ARRAYS:
            np.copyto(b[k], s["src"][k][:n])
        forcetree.RCBMonopoleForceTree(
            s["tree"][0], s["tree"][1], s["force"][0], s["force"][1], n,
            *(b[k] for k in ARRAYS), 1.0, RC, RSM, 0.1, nd=s["case"]["nd"], fl=s["fl"],
            fcoeff=0.01, kernel="step16" if s["case"]["law"] == "step16" else "sr")
        return s["buf"]
    if kind == "grad":
        pos = s["pos"].detach().clone().requires_grad_(True)
        im = s["images"]
        full = pos if im is None else pos[im.index] + im.shift
        F = autograd.ShortRangeForce.apply(full, s["solver"])
        F = F if im is None else F[: im.n_alive]
        F.backward(s["lam"])
        return {"force": F.detach(), "grad": pos.grad}
    if kind == "ensemble":
        b, ctx = _restore(s), s["ctx"]
        ctx.build_many(s["off"], b["x"], b["y"], b["z"], b["mass"], *s["tree"], vx=b["vx"],
                       vy=b["vy"], vz=b["vz"], phi=b["phi"], ids=b["id"], mask=b["mask"],
                       device_ptrs=True)
        ctx.lists_many(*s["force"])
        ctx.kick(0.01)
        return s["buf"]
    if kind == "substep":
        _restore(s)
        s["P"].subCycle(s["ts"])
        return s["buf"]
    if kind == "pm":
        for v, v0 in zip(s["v"], s["v0"]):
            v.copy_(v0)
        torch.cuda.synchronize()
        ctx, xyz, ng = s["ctx"], s["xyz"], s["ng"]
        ctx.cic(*xyz, ng, 1.0, s["rho"], device_ptrs=True)
        for grid, v in zip(s["grad"], s["v"]):
            ctx.inverse_cic(*xyz, ng, grid, 0.01, 1.1, v[: s["n"]], device_ptrs=True)
        return {"rho": s["rho"], "v": s["v"]}
    _restore(s)
    n, inside = s["ctx"].refresh(s["dom"], 0.8, s["n"], *(s["buf"][k] for k in ARRAYS),
                                 device_ptrs=True)
    return {"n": n, "inside": inside, **s["buf"]}


def _run_forces(s):
    pos, ctx = s["pos"], s["ctx"]
    n = pos.shape[0]
    x, y, z = (pos[:, k].contiguous() for k in range(3))
    m = torch.ones(n, device=DEV)
    ids = torch.arange(n, dtype=torch.int64, device=DEV)
    f = [torch.empty(n, device=DEV) for _ in range(3)]
    torch.cuda.synchronize()
    ctx.build(x, y, z, m, ids=ids, min_loc=s["tree"][0], max_loc=s["tree"][1], device_ptrs=True)
    ctx.lists(*s["force"])
    ctx.forces(*f, device_ptrs=True)
    out = torch.empty((n, 3), device=DEV)
    out[ids] = torch.stack(f, 1)
    return {"force": out, "order": ids}


# ------------------------------------------------------------------- exact

def _weight(law, r2):
    """w(r2) of the pair force w (x_j - x_i), and its derivative's polynomial
    part where the gradient needs it (step16), masked by the cutoff."""
    rsm2 = float(np.float32(RSM) * np.float32(RSM))
    y = (r2 + rsm2) ** -1.5
    if law in ("step16", "poly5", "poly6"):
        c = [float(np.float32(v)) for v in (P6 if law == "poly6" else P5)]
        p = torch.zeros_like(r2)
        for v in reversed(c):
            p = p * r2 + v
        w = y - p
    else:  # FGrid::fgor
        b, cc, d, e, ff, g, h, l = (float(np.float32(v)) for v in
                                    (0.72, 0.01, 0.27, 0.0001, 360.0, 100.0, 0.67, 17.0))
        r = r2.sqrt()
        t = torch.tanh(b * r) - b * r / torch.cosh(b * r) ** 2 \
            + cc * r * r2 * (1 + d * r2) * torch.exp(-d * r2) \
            + e * r2 * (ff * r2 + g * r2 ** 2 + l * r2 ** 3) * torch.exp(-h * r2)
        # below r = 1e-3 the limit is within 1e-6 of the value
        w = y - torch.where(r < 1e-3, torch.full_like(r, cc + 2.0 / 3.0 * b ** 3), t / r.clamp(min=1e-3) ** 3)
    rc2 = float(np.float32(RC) * np.float32(RC))
    if law != "step16":
        rc2 = min(rc2, float(np.float32(3.116326355) * np.float32(3.116326355)))
    return torch.where(r2 < rc2, w, torch.zeros_like(w))


def _dweight(r2):
    """dw/dr2 of the step16 weight."""
    rsm2 = float(np.float32(RSM) * np.float32(RSM))
    c = [k * float(np.float32(v)) for k, v in enumerate(P5)][1:]
    p = torch.zeros_like(r2)
    for v in reversed(c):
        p = p * r2 + v
    rc2 = float(np.float32(RC) * np.float32(RC))
    return torch.where(r2 < rc2, -1.5 * (r2 + rsm2) ** -2.5 - p, torch.zeros_like(r2))


def _near(pos):
    """Index blocks of particles and of all particles within RC of the block's
    box: (targets, sources) of a direct sum."""
    n = pos.shape[0]
    side = pos.max(0).values.clamp(min=1.0)
    key = (pos / 4.0).floor().long()
    ng = int((float(side.max()) / 4.0)) + 1
    order = torch.argsort((key[:, 0] * ng + key[:, 1]) * ng + key[:, 2])
    for a in range(0, n, 2048):
        i = order[a: a + 2048]
        lo, hi = pos[i].min(0).values - RC, pos[i].max(0).values + RC
        j = torch.nonzero(((pos >= lo) & (pos <= hi)).all(1)).flatten()
        yield i, j


def _direct_force(pos, law):
    out = torch.zeros_like(pos)
    for i, j in _near(pos):
        d = [pos[j, k][None, :] - pos[i, k][:, None] for k in range(3)]
        w = _weight(law, d[0] ** 2 + d[1] ** 2 + d[2] ** 2)
        for k in range(3):
            out[i, k] = (w * d[k]).sum(1)
    return out


def _direct_grad(pos, lam):
    """d(sum lam . F)/dx of the direct sum of the step16 force."""
    out = torch.zeros_like(pos)
    for i, j in _near(pos):
        d = [pos[j, k][None, :] - pos[i, k][:, None] for k in range(3)]
        r2 = d[0] ** 2 + d[1] ** 2 + d[2] ** 2
        dl = [lam[j, k][None, :] - lam[i, k][:, None] for k in range(3)]
        w = _weight("step16", r2)
        t = 2.0 * _dweight(r2) * (dl[0] * d[0] + dl[1] * d[1] + dl[2] * d[2])
        for k in range(3):
            out[i, k] = (w * dl[k] + t * d[k]).sum(1)
    return out


def _cic_terms(xyz, ng):
    """Cells (the slot after the last for those outside) and weights of the
    eight corners."""
    p = [v.double() for v in xyz]
    b = [v.floor() for v in p]
    w = [(1.0 - (v - f), v - f) for v, f in zip(p, b)]
    for cx in (0, 1):
        for cy in (0, 1):
            for cz in (0, 1):
                c = [f.long() + o for f, o in zip(b, (cx, cy, cz))]
                ok = (c[0] >= 0) & (c[0] < ng) & (c[1] >= 0) & (c[1] < ng) & (c[2] >= 0) & (c[2] < ng)
                cell = torch.where(ok, (c[0] * ng + c[1]) * ng + c[2], ng ** 3)
                yield cell, w[0][cx] * w[1][cy] * w[2][cz], ok


def exact(case, seed):
    kind = case["kind"]
    if kind == "forces":
        if case["law"] == "interp":
            return None
        pos, _ = _group(case, seed)
        return {"force": _direct_force(pos.double(), case["law"]), "order": None}
    if kind == "grad" and not case["images"]:
        pos, lam = (v.double() for v in _group(case, seed))
        return {"force": _direct_force(pos, "step16"), "grad": _direct_grad(pos, lam)}
    if kind == "pm":
        (ng, _, _), xyz, grad, v0 = _grid_inputs(case, seed)
        rho = torch.zeros(ng ** 3 + 1, dtype=torch.float64, device=DEV)
        v = [a.double() for a in v0]
        c = float(np.float32(1.1)) * float(np.float32(0.01))
        for cell, w, ok in _cic_terms(xyz, ng):
            rho.index_add_(0, cell, w)
            for a, grid in zip(v, grad):
                a[: w.numel()] += c * w * torch.where(ok, grid[cell].double(), torch.zeros_like(w))
        return {"rho": rho, "v": v}
    return None


# -------------------------------------------------------------------- work

def _pairs(pos, lo, hi):
    """Pairs (i inside [lo, hi), any j) closer than the cutoff, from a sample
    of targets."""
    g = torch.Generator(device=DEV)
    g.manual_seed(3)
    tgt = torch.nonzero(((pos >= lo) & (pos < hi)).all(1)).flatten()
    k = min(tgt.numel(), 1024)
    if k == 0:
        return 0.0
    pick = tgt[torch.randint(0, tgt.numel(), (k,), generator=g, device=DEV)]
    x, total = pos[pick], 0
    for a in range(0, pos.shape[0], 1 << 18):
        y = pos[a: a + (1 << 18)]
        r2 = sum((x[:, k][:, None] - y[:, k][None, :]) ** 2 for k in range(3))
        total += int((r2 < RC * RC).sum())
    return tgt.numel() * total / k


def work(case):
    """Bytes: the arrays a pass takes, read once, and gives, written once.
    Flops: FLOPS_PAIR for each pair inside the cutoff (three times that with
    the backward pass), and what each particle's eight corners take in the
    particle-grid steps."""
    kind = case["kind"]
    if kind == "ensemble":
        flops = n = 0
        for b, side in enumerate(_sides(case)):
            pos, _ = _rank("clustered", side, 5000 + b)
            n += pos.shape[0]
            flops += FLOPS_PAIR * _pairs(pos, SHELL, side + SHELL)
        return {"bytes": 84 * n, "flops": flops}
    side = case["side"]
    if kind == "forces" or kind == "grad" and not case["images"]:
        pos, _ = _positions(case["load"], side, 5000)
        n, p = pos.shape[0], _pairs(pos, -1.0, side + 1.0)
    else:
        pos, _ = _rank(case["load"], side, 5000)
        n = pos.shape[0]
        p = 0.0 if kind in ("pm", "refresh") else _pairs(pos, SHELL, side + SHELL)
    if kind == "forces":
        return {"bytes": 32 * n, "flops": FLOPS_PAIR * p}
    if kind == "grad":
        return {"bytes": 48 * n, "flops": 3 * FLOPS_PAIR * p}
    if kind == "pm":
        ng = math.ceil(side + 2 * SHELL)
        return {"bytes": 36 * n + 16 * ng ** 3, "flops": 80 * n}
    if kind == "refresh":
        return {"bytes": 84 * n, "flops": 12 * n}
    return {"bytes": 84 * n, "flops": FLOPS_PAIR * p}
