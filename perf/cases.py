"""Performance cases: what a user of this package has it do, over the real range of sizes.

``listed()`` holds the fixed cases, ``draw(rng)`` gives further ones of the same ranges.  Each goes through the
package's public entry points:

* ``mc``       marching_cubes on a UniformGrid (either method, any level)
* ``mc_grad``  differentiable marching cubes of a dense grid, forward and backward
* ``dc``       dual_contouring on a UniformGrid (intersections and normals found on the way)
* ``dc_norm``  get_intersection, set_normals with the caller's normals, dual_contouring
* ``dc_grad``  differentiable dual contouring, forward and backward
* ``sparse``   differentiable marching cubes of a narrow-band SparseGrid, forward and backward
* ``batch``    a ragged batch of requests as a server gets them: marching cubes and dual contouring
* ``sdf``      marching cubes of an SDF tree that is never stored as a grid

Fields are unions of random spheres (the benchmark's and the server's field), a box with a drilled hole united with
spheres (sharp edges), and a sphere with Fourier noise in a narrow band.  They are made with plain torch operations,
in the float operation order sqrt((dx*dx + dy*dy) + dz*dz) - r, so that ``exact`` sees the same float32 values.

The shapes in a field are the case's (``field``); the seed gives every grid point its own measurement noise, a factor
on its distance, so that meshes of two seeds have the same size and other coordinates.  Distances below TINY cells
are widened to it, as meshes of one size need: closer, two crossings can round to one vertex.  ``snapped`` points at
the surface lie exactly on the level, as clipped or quantised data do; their vertices coincide and are welded.  A
field that is never stored takes its seed as its scale (a power of two) and its spheres' order.
"""

import math

import numpy as np
import torch

import isoext_amd as iso
from isoext_amd import autograd as iso_grad
from isoext_amd.batch import GridJob, dc_batch, mc_batch
from isoext_amd.csg import SdfProgram
from isoext_amd.fused import marching_cubes_sdf
from isoext_amd.sdf import CuboidSDF, CylinderSDF, IntersectionOp, NegationOp, SphereSDF, TranslationOp, UnionOp

DEV = "cuda"
REG = 1e-2   # dual_contouring's default regularisation
BOX, DRILL = 0.6, 0.3   # half-extent of the box and radius of the hole of the drilled box
AMP, AMP_DC = 0.05, 0.01   # measurement noise, as a part of the distance
TINY = 5e-4   # smallest distance to the level, in cells
BAND, NOISE_R, NOISE_AMP = 2.0, 0.7, 0.02   # narrow band: |d| < BAND cells around a sphere with noise


def listed():
    return [
        # the smallest call: the 64^3 grid of the first examples, where launches and waits are the time
        {"name": "mc_64", "kind": "mc", "x": 64, "y": 64, "z": 64, "spheres": 1, "field": 1, "level": 0.0, "method": "nagae"},
        # a small ragged grid, off-level, with the other triangle tables: rows neither aligned nor whole words
        {"name": "mc_ragged_lorensen", "kind": "mc", "x": 97, "y": 131, "z": 75, "spheres": 5, "field": 3, "level": 0.02,
         "method": "lorensen"},
        # the ordinary call: one 256^3 grid
        {"name": "mc_256", "kind": "mc", "x": 256, "y": 256, "z": 256, "spheres": 16, "field": 4, "level": 0.0,
         "method": "nagae"},
        # a scanned volume: large, odd in every direction, unaligned rows
        {"name": "mc_509x387x451", "kind": "mc", "x": 509, "y": 387, "z": 451, "spheres": 32, "field": 5, "level": 0.0,
         "method": "nagae"},
        # the headline workload: 1024^3, 64 spheres, a few points of which lie on the level
        {"name": "mc_1024", "kind": "mc", "x": 1024, "y": 1024, "z": 1024, "spheres": 64, "field": 0, "level": 0.0,
         "method": "nagae", "snapped": 400},
        # one step of an optimisation through a dense grid
        {"name": "mc_grad_128", "kind": "mc_grad", "x": 128, "y": 128, "z": 128, "spheres": 8, "field": 7, "level": 0.0},
        # dual contouring of a plain grid, ragged
        {"name": "dc_200x161x130", "kind": "dc", "x": 200, "y": 161, "z": 130, "spheres": 12, "field": 8, "level": 0.0},
        # dual contouring of sharp features with the caller's analytic normals, the 256^3 benchmark workload
        {"name": "dc_norm_256", "kind": "dc_norm", "x": 256, "y": 256, "z": 256, "spheres": 16, "field": 9, "level": 0.0},
        # one step of an optimisation through dual contouring
        {"name": "dc_grad_96", "kind": "dc_grad", "x": 96, "y": 96, "z": 96, "spheres": 8, "field": 10, "level": 0.0},
        # the narrow band at 2048^3 effective resolution, forward and backward
        {"name": "sparse_2048", "kind": "sparse", "n": 2048, "field": 0, "level": 0.0},
        # 24 requests of the serving mix: sides log-uniform in [32, 512], four of five marching cubes
        {"name": "batch_24", "kind": "batch", "requests": 24, "lo": 32, "hi": 512, "field": 1},
        # a modelling program's field, extracted without a grid
        {"name": "sdf_256", "kind": "sdf", "x": 256, "y": 256, "z": 256, "spheres": 16, "field": 11, "level": 0.0},
    ]


def draw(rng):
    kind = rng.choice(["mc", "mc", "mc", "mc_grad", "dc", "dc", "dc_norm", "dc_grad", "sparse", "batch", "sdf"])

    def log_uniform(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    if kind == "sparse":
        return {"kind": kind, "n": int(log_uniform(256, 1600)), "field": rng.randint(1, 1 << 20), "level": 0.0}
    if kind == "batch":
        return {"kind": kind, "requests": rng.randint(6, 24), "lo": 32, "hi": int(log_uniform(96, 512)),
                "field": rng.randint(2, 1 << 20)}
    lo, hi = {"mc": (32, 720), "mc_grad": (32, 288), "dc": (32, 384), "dc_norm": (32, 320), "dc_grad": (32, 192),
              "sdf": (48, 512)}[kind]
    s = log_uniform(lo, hi)
    c = {"kind": kind, **{a: max(24, int(s * rng.uniform(0.7, 1.3))) for a in "xyz"},
         "spheres": int(log_uniform(1, 64.99)), "field": rng.randint(1, 1 << 20), "level": rng.choice([0.0, 0.0, rng.uniform(-0.02, 0.04)])}
    if rng.random() < 0.3:   # an aligned size of the kind that programs like
        c["z"] = max(64, c["z"] // 64 * 64)
    if kind == "mc":
        c["method"] = rng.choice(["nagae", "nagae", "lorensen"])
        c["snapped"] = rng.choice([0, 0, int(log_uniform(1, 400))])
    return c


# ---- fields ---------------------------------------------------------------------------------------------------

def _spheres(n, seed, drilled=False):
    """n seeded spheres; the first one is large and central, so that no field is without a surface."""
    rng = np.random.default_rng(seed)
    if drilled:
        return (rng.uniform(-0.8, 0.8, (n, 3)).astype(np.float32), rng.uniform(0.05, 0.15, n).astype(np.float32))
    c, r = rng.uniform(-0.8, 0.8, (n, 3)), rng.uniform(0.05, 0.25, n)
    c[0], r[0] = rng.uniform(-0.2, 0.2, 3), rng.uniform(0.3, 0.7 if n == 1 else 0.4)
    return c.astype(np.float32), r.astype(np.float32)


def _axis(n, dtype=torch.float32):
    return -1.0 + torch.arange(n, device=DEV, dtype=dtype) / (n - 1) * 2.0


def _sphere_field(shape, c, r, dtype=torch.float32, base=None):
    """min over the spheres (and `base`), in slabs that stay in cache."""
    X, Y, Z = shape
    ax, ay, az = (_axis(n, dtype) for n in shape)
    out = torch.empty(shape, dtype=dtype, device=DEV) if base is None else base
    ct, rt = c.astype(np.float64), r.astype(np.float64)   # the float32 values; python floats do not change an op's type
    step = max(1, (1 << 23) // (Y * Z))
    for x0 in range(0, X, step):
        xs, o = ax[x0:x0 + step], out[x0:x0 + step]
        for k in range(len(rt)):
            dx, dy, dz = xs - float(ct[k, 0]), ay - float(ct[k, 1]), az - float(ct[k, 2])
            t = ((dx * dx)[:, None] + (dy * dy)[None])[:, :, None] + (dz * dz)
            t.sqrt_().sub_(float(rt[k]))
            if k == 0 and base is None:
                o.copy_(t)
            else:
                torch.minimum(o, t, out=o)
    return out


def _drilled(shape, c, r, dtype=torch.float32):
    """Box minus a z-cylinder, united with the spheres."""
    ax, ay, az = (_axis(n, dtype) for n in shape)
    qx, qy, qz = (a.abs() - float(np.float32(2 * BOX) / np.float32(2)) for a in (ax, ay, az))
    m = torch.maximum(torch.maximum(qx[:, None], qy[None])[:, :, None], qz).clamp_(max=0)
    px, py, pz = qx.clamp(min=0), qy.clamp(min=0), qz.clamp(min=0)
    box = (((px * px)[:, None] + (py * py)[None])[:, :, None] + pz * pz).sqrt_().add_(m)
    cyl = ((ax * ax)[:, None] + (ay * ay)[None]).sqrt_() - float(np.float32(DRILL))
    return _sphere_field(shape, c, r, dtype, torch.maximum(box, -cyl[:, :, None]))


def _drilled_normals(p, c, r):
    """Unit gradients of the drilled field at points p (N, 3) by its active branch."""
    q = p.abs() - BOX
    box = q.clamp(min=0).norm(dim=-1) + q.max(dim=-1).values.clamp(max=0)
    n_box = torch.where((q > 0).any(-1, keepdim=True), q.clamp(min=0), (q == q.max(dim=-1, keepdim=True).values).to(p))
    n_box = n_box * p.sign()
    cyl = DRILL - p[:, :2].norm(dim=-1)
    n_cyl = torch.cat([-p[:, :2], torch.zeros_like(p[:, :1])], -1)
    d, n = torch.maximum(box, cyl), torch.where((cyl > box)[:, None], n_cyl, n_box)
    for k in range(len(r)):
        w = p - torch.from_numpy(c[k]).to(p)
        dk = w.norm(dim=-1) - float(r[k])
        n, d = torch.where((dk < d)[:, None], w, n), torch.minimum(d, dk)
    return torch.nn.functional.normalize(n, dim=-1).contiguous()


def _shape(case):
    return case["x"], case["y"], case["z"]


def _noisy(d, level, seed, amp, cell):
    """In place: distance d from the level to a value, with a seeded factor on each point's distance."""
    g = torch.Generator(device=DEV).manual_seed(_int(seed))
    step = max(1, (1 << 25) // d[0].numel())
    for o in d.split(step):
        o.sub_(level).mul_(torch.rand(o.shape, device=DEV, generator=g).mul_(2 * amp).add_(1 - amp))
        small = o.abs() < TINY * cell
        o.copy_(torch.where(small, torch.where(o < 0, -TINY * cell, TINY * cell).to(o), o)).add_(level)
    return d


def _int(seed):
    return int(np.random.default_rng(seed).integers(1 << 40))


def _snap(vals, level, count):
    """`count` outside points with an inside neighbour along z, spread over the grid, put exactly on the level."""
    got = []
    for x0 in range(0, vals.shape[0], 64):
        a = _inside(vals[x0:x0 + 64], level)
        got.append(torch.nonzero((~a[:, :, :-1]) & a[:, :, 1:]) + torch.tensor([x0, 0, 0], device=DEV))
    at = torch.cat(got)
    at = at[torch.linspace(0, len(at) - 1, min(count, len(at)), device=DEV, dtype=F8).long()]
    vals[at[:, 0], at[:, 1], at[:, 2]] = level


def _field(case, seed):
    shape, drilled = _shape(case), case["kind"] == "dc_norm"
    c, r = _spheres(case["spheres"], case["field"], drilled)
    d = _drilled(shape, c, r) if drilled else _sphere_field(shape, c, r)
    amp = AMP_DC if case["kind"].startswith("dc") else AMP
    v = _noisy(d, case["level"], seed, amp, 2.0 / (max(shape) - 1))
    if case.get("snapped"):
        _snap(v, case["level"], case["snapped"])
    return v


def _model(case, seed):
    """Scale and spheres (in their order) of a field that is never stored."""
    c, r = _spheres(case["spheres"], case["field"], True)
    order = np.random.default_rng(seed).permutation(len(r))
    return 2.0 ** (int(seed) % 7 - 3), c[order], r[order]


def _noisy_sphere(seed):
    rng = np.random.default_rng(seed)
    ks = [(rng.normal(size=3) * (4.0 * 2 ** o), rng.uniform(0, 2 * np.pi)) for o in range(3)]

    def f(p):
        d = ((p[..., 0] * p[..., 0] + p[..., 1] * p[..., 1]) + p[..., 2] * p[..., 2]).sqrt() - NOISE_R
        for o, (k, phi) in enumerate(ks):
            d = d + (NOISE_AMP / 2 ** o) * torch.sin((p[..., 0] * k[0] + p[..., 1] * k[1]) + p[..., 2] * k[2] + phi)
        return d
    return f


def _band(case, seed):
    """Sorted ids of the cells whose centre lies within BAND cells of the noisy sphere, and their (N, 8) corner
    values (a point's value is the same in every cell that has it)."""
    n = case["n"]
    f, nc, B = _noisy_sphere(case["field"]), n - 1, 16
    mix = np.random.default_rng(seed).integers(1, 1 << 31, 2).tolist()
    h, nb = 2.0 / nc, -(-nc // B)
    bc = -1.0 + (torch.arange(nb, device=DEV) * B + B / 2) * h
    P = torch.stack(torch.meshgrid(bc, bc, bc, indexing="ij"), -1).reshape(-1, 3)
    blocks = torch.cat([torch.nonzero(f(q).abs() < BAND * h + math.sqrt(3) * B * h).flatten() + i * (1 << 20)
                        for i, q in enumerate(P.split(1 << 20))])
    o = torch.arange(B ** 3, device=DEV)
    ids = []
    for b in blocks.split(4096):
        x = ((b // (nb * nb)) * B)[:, None] + (o // (B * B))
        y = ((b // nb % nb) * B)[:, None] + (o // B % B)
        z = ((b % nb) * B)[:, None] + (o % B)
        ctr = torch.stack([-1.0 + (t + 0.5) * h for t in (x, y, z)], -1)
        keep = (f(ctr).abs() < BAND * h) & (x < nc) & (y < nc) & (z < nc)
        ids.append((((x * nc + y) * nc) + z)[keep])
    ids = torch.sort(torch.cat(ids)).values
    vals = torch.empty((ids.numel(), 8), device=DEV)
    ax = _axis(n)
    for s in range(0, ids.numel(), 1 << 22):
        i = ids[s:s + (1 << 22)]
        x, y, z = i // (nc * nc), i // nc % nc, i % nc
        for k in range(8):
            px, py, pz = x + (k >> 2), y + ((k >> 1) & 1), z + (k & 1)
            d = f(torch.stack([ax[px], ax[py], ax[pz]], -1)) - case["level"]
            u = ((px * n + py) * n + pz + mix[0]) * 2654435761 % (1 << 32)
            u = ((u ^ (u >> 15)) * mix[1] % (1 << 32)).float() / (1 << 32)
            d = d * (1 + AMP * (2 * u - 1))
            d = torch.where(d.abs() < TINY * h, torch.where(d < 0, -TINY * h, TINY * h).to(d), d)
            vals[s:s + (1 << 22), k] = d + case["level"]
    return ids, vals


def _requests(case):
    """(shape, spheres, is dual contouring) of each request of a batch."""
    rng = np.random.default_rng([case["field"], 77])
    got = []
    for i in range(case["requests"]):
        side = math.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"])))
        shape = tuple(max(24, int(side * k)) for k in rng.uniform(0.8, 1.0, 3))
        got.append((shape, int(rng.integers(1, 65)), i % 5 == 4))
    return got


def _batch_fields(case, seed):
    for i, (shape, n, dc) in enumerate(_requests(case)):
        d = _sphere_field(shape, *_spheres(n, [case["field"], i]))
        yield _noisy(d, 0.0, [seed, i], AMP_DC if dc else AMP, 2.0 / (max(shape) - 1)), dc


# ---- the cases --------------------------------------------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        mc, dc = [], []
        for v, is_dc in _batch_fields(case, seed):
            (dc if is_dc else mc).append(GridJob(v))
        return {"kind": kind, "mc": mc, "dc": dc}
    if kind == "sdf":
        k, c, r = _model(case, seed)
        body = IntersectionOp([CuboidSDF([2 * BOX * k] * 3), NegationOp(CylinderSDF(DRILL * k))])
        tree = UnionOp([body] + [TranslationOp(SphereSDF(float(r[i] * k)), [float(t * k) for t in c[i]])
                                 for i in range(len(r))])
        return {"kind": kind, "program": SdfProgram(tree, DEV), "shape": _shape(case), "level": case["level"] * k,
                "box": ((-k,) * 3, (k,) * 3)}
    if kind == "sparse":
        ids, vals = _band(case, seed)
        grid = iso.SparseGrid([case["n"]] * 3)
        grid.add_cells(ids)
        grid.set_values(vals)
        return {"kind": kind, "grid": grid, "values": vals.requires_grad_(), "level": case["level"]}
    vals = _field(case, seed)
    grid = iso.UniformGrid(list(_shape(case)))
    grid.set_values(vals)
    state = {"kind": kind, "grid": grid, "level": case["level"]}
    if kind == "mc":
        state["method"] = case["method"]
    elif kind in ("mc_grad", "dc_grad"):
        state["values"] = vals.requires_grad_()
    elif kind == "dc_norm":   # the caller's model gives the normals at the intersection points
        state["normals"] = _drilled_normals(_crossed(vals, case["level"])[0].float(),
                                            *_spheres(case["spheres"], case["field"], True))
    return state


def run(state):
    kind = state["kind"]
    if kind == "mc":
        return iso.marching_cubes(state["grid"], state["level"], state["method"])
    if kind == "dc":
        return iso.dual_contouring(state["grid"], state["level"])
    if kind == "dc_norm":
        its = iso.get_intersection(state["grid"], state["level"])
        its.set_normals(state["normals"])
        return its.get_points(), iso.dual_contouring(state["grid"], state["level"], its)
    if kind == "batch":
        return mc_batch(state["mc"]), dc_batch(state["dc"])
    if kind == "sdf":
        return marching_cubes_sdf(state["program"], state["shape"], state["level"], aabb_min=state["box"][0],
                                  aabb_max=state["box"][1])
    # an optimisation step whose loss is half the sum of squares of the vertex coordinates
    step = iso_grad.dual_contouring if kind == "dc_grad" else iso_grad.marching_cubes
    v, f = step(state["grid"], state["values"], level=state["level"])
    (g,) = torch.autograd.grad(v, state["values"], v.detach())
    return v, f, g


# ---- what a pass cannot do without --------------------------------------------------------------------------------

def _crossings(shape, c, r, level, drilled=False):
    """Crossing grid edges of a field, from a coarse grid scaled by each axis's number of lines."""
    m = 49
    a = np.linspace(-1, 1, m, dtype=np.float32)
    P = np.stack(np.meshgrid(a, a, a, indexing="ij"), -1)
    d = np.full((m, m, m), np.inf, np.float32)
    if drilled:
        q = np.abs(P) - BOX
        box = np.sqrt((np.maximum(q, 0) ** 2).sum(-1)) + np.minimum(q.max(-1), 0)
        d = np.maximum(box, DRILL - np.sqrt((P[..., :2] ** 2).sum(-1)))
    for k in range(len(r)):
        d = np.minimum(d, np.sqrt(((P - c[k]) ** 2).sum(-1)) - r[k])
    i = d < level
    n = [np.count_nonzero(np.diff(i, axis=k)) / (m * m) for k in range(3)]
    X, Y, Z = shape
    return n[0] * Y * Z + n[1] * X * Z + n[2] * X * Y


def work(case):
    """Each value read once and each output written once.  A closed mesh has about one vertex per crossing edge and
    two triangles per vertex; a dual mesh one vertex per crossing edge's quad.  Operations: about 20 a vertex for the
    interpolation, about 1,000 a dual vertex (four crossings with normals, the 3x3 solve)."""
    kind = case["kind"]
    if kind == "sparse":
        n2 = (case["n"] - 1.0) ** 2 / 4
        area = 4 * math.pi * NOISE_R ** 2
        cells, v = area * 2 * BAND * n2, 1.5 * area * n2
        return {"bytes": 40 * cells + 36 * v + 12 * v + 32 * cells, "flops": 60 * v}
    if kind == "batch":
        total = {"bytes": 0.0, "flops": 0.0}
        for i, (shape, n, dc) in enumerate(_requests(case)):
            v = _crossings(shape, *_spheres(n, [case["field"], i]), 0.0)
            total["bytes"] += 4 * math.prod(shape) + 36 * v
            total["flops"] += (1000 if dc else 20) * v
        return total
    shape, drilled = _shape(case), kind in ("dc_norm", "sdf")
    v = _crossings(shape, *_spheres(case["spheres"], case["field"], drilled), case["level"], drilled)
    N = math.prod(shape)
    if kind == "sdf":   # each corner of a cell at the surface evaluated once: about two points a vertex
        return {"bytes": 36 * v, "flops": 20 * v + 2 * v * (30 + 10 * case["spheres"])}
    if kind == "mc":
        return {"bytes": 4 * N + 36 * v, "flops": 20 * v}
    if kind == "mc_grad":   # the vertex gradients read, the gradient of the values written
        return {"bytes": 8 * N + 48 * v, "flops": 60 * v}
    if kind == "dc":
        return {"bytes": 4 * N + 36 * v, "flops": 1000 * v}
    if kind == "dc_norm":   # four intersections a cell: normals read, points written
        return {"bytes": 4 * N + 36 * v + 96 * v, "flops": 600 * v}
    return {"bytes": 8 * N + 48 * v, "flops": 2500 * v}   # dc_grad


def tolerance(case):
    """Vertices are one interpolation in float32 (about 1e-7 off float64) and faces are exact.  Gradients carry the
    interpolation's cancellation (3e-6 off float64, 2e-5 through the dual solve) and are short sums in any order.
    Dual vertices come from a float32 solve with float64 refinement, about 1e-7 off as well; the shorter diagonal of
    a quad may flip where both are equally long."""
    kind = case["kind"]
    if kind in ("mc", "sdf"):
        return {"rel": 5e-7, "max": 1e-5, "differ": 0.0}
    if kind in ("mc_grad", "sparse"):
        return {"rel": 1e-5, "max": 1e-3, "differ": 0.0}
    if kind == "dc_grad":
        return {"rel": 1e-4, "max": 1e-2, "differ": 1e-3}
    return {"rel": 1e-6, "max": 1e-4, "differ": 1e-3}


# ---- the same in 64 bits ------------------------------------------------------------------------------------------

EA = (0, 1, 2, 0, 4, 5, 6, 4, 0, 1, 3, 2)   # corners of a cell's twelve edges; corner k at (k>>2, k>>1&1, k&1)
EB = (1, 3, 3, 2, 5, 7, 7, 6, 4, 5, 7, 6)
F8 = torch.float64


def _inside(v, level):
    return (v - level) < 0


def _mc_exact(vals, level, grad=False, v64=None, weld=False):
    """Crossing points of the grid's edges in float64, by owner point, then axis; with `grad`, the gradient of half
    the sum of their squares with respect to the values.  With `weld`, vertices at one grid point on the level are
    one, the first of them, and the last vertices take the places of the others."""
    shape = vals.shape
    axes = [_axis(n, F8) for n in shape]
    ins = _inside(vals, level)
    v64 = vals if v64 is None else v64
    g = torch.zeros(vals.numel(), dtype=F8, device=DEV) if grad else None
    X, Y, Z = shape
    stride = (Y * Z, Z, 1)
    got, spots = [], []
    step = max(1, (1 << 27) // (Y * Z))
    for x0 in range(0, X, step):
        a = ins[x0:x0 + step]
        cross = torch.zeros((*a.shape, 3), dtype=torch.bool, device=DEV)
        nx = ins[x0 + 1:x0 + 1 + step]
        cross[:nx.shape[0], :, :, 0] = a[:nx.shape[0]] ^ nx
        cross[:, :-1, :, 1] = a[:, :-1] ^ a[:, 1:]
        cross[:, :, :-1, 2] = a[:, :, :-1] ^ a[:, :, 1:]
        i = torch.nonzero(cross.view(-1)).flatten()
        axis, pt = i % 3, i // 3 + x0 * Y * Z
        del cross
        pb = pt + torch.tensor(stride, device=DEV)[axis]
        va, vb = v64.reshape(-1)[pt].to(F8), v64.reshape(-1)[pb].to(F8)
        t = (level - va) / (vb - va)
        ids = (pt // (Y * Z), pt // Z % Y, pt % Z)
        p = torch.stack([axes[k][ids[k]] for k in range(3)], -1)
        h = torch.tensor([2.0 / (n - 1) for n in shape], dtype=F8, device=DEV)[axis]
        along = p.gather(1, axis[:, None])[:, 0] + t * h
        p.scatter_(1, axis[:, None], along[:, None])
        got.append(p)
        if weld:
            spots.append(torch.where(t == 0, pt, torch.where(t == 1, pb, -1)))
        if grad:
            w = along * h / (vb - va) ** 2
            g.index_add_(0, pt, w * (level - vb))
            g.index_add_(0, pb, -w * (level - va))
    v = torch.cat(got)
    if weld:
        spot = torch.cat(spots)
        at = torch.nonzero(spot >= 0).flatten()
        key, order = torch.sort(spot[at], stable=True)
        gone = torch.zeros(len(v), dtype=torch.bool, device=DEV)
        gone[at[order[1:][key[1:] == key[:-1]]]] = True
        n = len(v) - int(gone.sum())
        v[:n][gone[:n]] = v[n:][~gone[n:]]
        v = v[:n]
    return (v, g.view(shape)) if grad else v


def _tri(t, c):
    a = 1 - t[:, 2]
    c00, c01 = c[:, 0] * a + c[:, 1] * t[:, 2], c[:, 2] * a + c[:, 3] * t[:, 2]
    c10, c11 = c[:, 4] * a + c[:, 5] * t[:, 2], c[:, 6] * a + c[:, 7] * t[:, 2]
    b = 1 - t[:, 1]
    return (c00 * b + c01 * t[:, 1]) * (1 - t[:, 0]) + (c10 * b + c11 * t[:, 1]) * t[:, 0]


def _crossed(vals, level, grad=False):
    """The active cells of a grid in ascending order and their crossing edges (by cell, then edge), with the
    intersection points in float64."""
    X, Y, Z = vals.shape
    ins = _inside(vals, level)

    def corner(t, k):
        dx, dy, dz = k >> 2, (k >> 1) & 1, k & 1
        return t[dx:X - 1 + dx, dy:Y - 1 + dy, dz:Z - 1 + dz]

    some, every = corner(ins, 0).clone(), corner(ins, 0).clone()
    for k in range(1, 8):
        some |= corner(ins, k)
        every &= corner(ins, k)
    cell = torch.nonzero(some & ~every)
    axes = [_axis(m, F8) for m in vals.shape]
    lo = torch.stack([axes[k][cell[:, k]] for k in range(3)], -1)
    hi = torch.stack([axes[k][cell[:, k] + 1] for k in range(3)], -1)
    flat = vals.detach().reshape(-1).to(F8).requires_grad_(grad)
    pid = torch.stack([((cell[:, 0] + (k >> 2)) * Y + cell[:, 1] + ((k >> 1) & 1)) * Z + cell[:, 2] + (k & 1)
                       for k in range(8)], -1)
    cv, ci = flat[pid], ins.reshape(-1)[pid]
    ea, eb = torch.tensor(EA, device=vals.device), torch.tensor(EB, device=vals.device)
    row, e = torch.nonzero(ci[:, ea] ^ ci[:, eb], as_tuple=True)
    ca, cb = ea[e], eb[e]
    va, vb = cv[row, ca], cv[row, cb]
    t = ((level - va) / (vb - va))[:, None]

    def place(k):
        o = torch.stack([k >> 2, (k >> 1) & 1, k & 1], -1)
        return torch.where(o > 0, hi[row], lo[row]), o
    (pa, oa), (pb, ob) = place(ca), place(cb)
    return (1 - t) * pa + t * pb, row, oa, ob, cell, lo, hi, cv, flat


def _dc_exact(vals, level, normals=None, grad=False):
    """Intersection points in entry order and the dual vertices of the cells that a quad uses, in float64; with
    `grad`, the gradient of half the sum of the dual vertices' squares with respect to the values (normals held).
    Coinciding dual vertices are not merged."""
    X, Y, Z = vals.shape
    p, row, oa, ob, cell, lo, hi, cv, flat = _crossed(vals, level, grad)
    n = cell.shape[0]
    if normals is None:
        with torch.no_grad():
            c, size, eps = cv[row], (hi - lo)[row], 0.02
            u = ((p - lo[row]) / size).clamp(0.01, 0.99)
            d = []
            for k in range(3):
                up, dn = u.clone(), u.clone()
                up[:, k] = (u[:, k] + eps).clamp(max=0.99)
                dn[:, k] = (u[:, k] - eps).clamp(min=0.01)
                d.append((_tri(up, c) - _tri(dn, c)) / ((up[:, k] - dn[:, k]) * size[:, k]))
            normals = torch.nn.functional.normalize(torch.stack(d, -1), dim=-1)
    nn = normals.to(F8)
    count = torch.zeros(n, dtype=F8, device=DEV).index_add_(0, row, torch.ones_like(p[:, 0]))
    eye = torch.eye(3, dtype=F8, device=DEV) * REG
    M = torch.zeros((n, 3, 3), dtype=F8, device=DEV).index_add_(0, row, nn[:, :, None] * nn[:, None, :]) + eye
    b = torch.zeros((n, 3), dtype=F8, device=DEV).index_add(0, row, nn * (nn * p).sum(-1, keepdim=True))
    mean = torch.zeros((n, 3), dtype=F8, device=DEV).index_add(0, row, p) / count[:, None]
    b = b + REG * mean
    m = M.reshape(n, 9)   # the symmetric 3x3 inverse by cofactors
    cof = torch.stack([m[:, 4] * m[:, 8] - m[:, 5] * m[:, 7], m[:, 2] * m[:, 7] - m[:, 1] * m[:, 8],
                       m[:, 1] * m[:, 5] - m[:, 2] * m[:, 4], m[:, 5] * m[:, 6] - m[:, 3] * m[:, 8],
                       m[:, 0] * m[:, 8] - m[:, 2] * m[:, 6], m[:, 2] * m[:, 3] - m[:, 0] * m[:, 5],
                       m[:, 3] * m[:, 7] - m[:, 4] * m[:, 6], m[:, 1] * m[:, 6] - m[:, 0] * m[:, 7],
                       m[:, 0] * m[:, 4] - m[:, 1] * m[:, 3]], -1)
    det = m[:, 0] * cof[:, 0] + m[:, 1] * cof[:, 3] + m[:, 2] * cof[:, 6]
    x = (cof.reshape(n, 3, 3) * b[:, None, :]).sum(-1) / det[:, None]
    x = torch.minimum(torch.maximum(x, lo), hi)
    # a crossing edge gives a quad when its four cells exist: its other two coordinates are inside the grid
    o = cell[row] + torch.minimum(oa, ob)
    last = torch.tensor([X - 1, Y - 1, Z - 1], device=DEV)
    inner = ((o > 0) & (o < last)) | (oa != ob)
    used = torch.zeros(n, dtype=torch.bool, device=DEV)
    used[row[inner.all(-1)]] = True
    v = x[used]
    if grad:
        (g,) = torch.autograd.grad((v * v).sum() / 2, flat)
        return p.detach(), v.detach(), g.view(vals.shape)
    return p, v


def _sparse_exact(case, seed):
    """Crossing points in the order of the first cell that has them, and the gradient of half the sum of their
    squares at that cell's corner values."""
    ids, vals = _band(case, seed)
    n, level = case["n"], float(np.float32(case["level"]))
    nc, N = n - 1, ids.numel()
    ins = _inside(vals, level)
    ea, eb = torch.tensor(EA, device=DEV), torch.tensor(EB, device=DEV)
    inst = torch.cat([torch.nonzero((i[:, ea] ^ i[:, eb]).reshape(-1)).flatten() + 12 * s
                      for s, i in ((s, ins[s:s + (1 << 23)]) for s in range(0, N, 1 << 23))])
    slot, e = inst // 12, inst % 12
    ca, cb = ea[e], eb[e]
    i = ids[slot]
    pt = (((i // (nc * nc)) + (ca >> 2)) * n + (i // nc % nc) + ((ca >> 1) & 1)) * n + i % nc + (ca & 1)
    axis = 2 - ((cb - ca) >> 1)   # corner steps 4, 2, 1 along x, y, z
    key, order = torch.sort(pt * 3 + axis, stable=True)
    first = torch.ones_like(key, dtype=torch.bool)
    first[1:] = key[1:] != key[:-1]
    rep = torch.sort(order[first]).values
    slot, axis, pt, ca, cb = slot[rep], axis[rep], pt[rep], ca[rep], cb[rep]
    va, vb = vals[slot, ca].to(F8), vals[slot, cb].to(F8)
    t, h, ax = (level - va) / (vb - va), 2.0 / nc, _axis(n, F8)
    v = torch.stack([ax[pt // (n * n)], ax[pt // n % n], ax[pt % n]], -1)
    along = v.gather(1, axis[:, None])[:, 0] + t * h
    v.scatter_(1, axis[:, None], along[:, None])
    g = torch.zeros(8 * N, dtype=F8, device=DEV)
    w = along * h / (vb - va) ** 2
    g.index_add_(0, 8 * slot + ca, w * (level - vb))
    g.index_add_(0, 8 * slot + cb, -w * (level - va))
    return v, None, g.view(N, 8)


@torch.no_grad()
def exact(case, seed):
    kind, level = case["kind"], float(np.float32(case.get("level", 0.0)))   # the entry points take float32
    if kind == "sparse":
        return _sparse_exact(case, seed)
    if kind == "batch":
        mc, dc = [], []
        for v, is_dc in _batch_fields(case, seed):
            if is_dc:
                dc.append((_dc_exact(v, 0.0)[1], None))
            else:
                mc.append((_mc_exact(v, 0.0), None))
        return mc, dc
    if kind == "sdf":
        k, c, r = _model(case, seed)
        return _mc_exact(_drilled(_shape(case), c, r), level, v64=_drilled(_shape(case), c, r, F8)) * k, None
    vals = _field(case, seed)
    if kind == "mc":
        return _mc_exact(vals, level, weld=bool(case.get("snapped"))), None
    if kind == "mc_grad":
        v, g = _mc_exact(vals, level, grad=True)
        return v, None, g
    if kind == "dc":
        return _dc_exact(vals, level)[1], None
    if kind == "dc_norm":
        normals = _drilled_normals(_crossed(vals, level)[0].float(), *_spheres(case["spheres"], case["field"], True))
        p, v = _dc_exact(vals, level, normals)
        return p, (v, None)
    with torch.enable_grad():
        _, v, g = _dc_exact(vals, level, grad=True)
    return v, None, g
