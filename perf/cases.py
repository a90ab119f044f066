"""Performance cases: the builds, traces and differentiable steps a program runs on this package.

A case is a dict of plain values; `kind` says which entry points a pass calls:

  build   BVHBuilder.rebuild of a scene and a first trace on the new tree, as
          for geometry that moves from frame to frame
  trace   HipTracer.trace or trace_sort of one ray set on a standing tree
  ao      one ambient-occlusion pass: RayGen.ao, sorted any-hit trace,
          reconstruct_occlusion
  diff    DifferentiableTracer forward and backward (refit, trace, adjoint)
  batch   HipBatch over many meshes: rebuild, trace, recompute_hits, backward

`listed` holds the named cases, `draw` makes more of the same ranges,
`prepare` makes a case's inputs and handles, `run` is one pass, `exact` the
same outputs in 64 bits by plain torch.
"""
import functools
import math
import random

import torch

import hippie_amd as hx
from hippie_amd import raygen
from hippie_amd.diff import DifferentiableTracer

DEV = "cuda"


def listed():
    return [
        # A small dynamic object in a frame loop: rebuild it, trace a 64x64
        # tile of rays.  All launches and latency.
        dict(name="frame_4k", kind="build", method="lbvh", layout="bin", n=4099, geometry="uniform", bits=60,
             presplit=0.0, rays=4096),
        # One ordinary mesh rebuilt every frame with short Morton keys.
        dict(name="lbvh30_64k", kind="build", method="lbvh", layout="bin", n=65536, geometry="uniform", bits=30,
             presplit=0.0, rays=16384),
        # The benchmark's scene: a whole world rebuilt.
        dict(name="lbvh60_16m", kind="build", method="lbvh", layout="bin", n=16777216, geometry="mixture", bits=60,
             presplit=0.0, rays=262144),
        # A better tree for a model that will be traced for a while.
        dict(name="ploc25_1m", kind="build", method="ploc", layout="bin", n=1000003, geometry="mixture", bits=60,
             presplit=0.0, rays=65536),
        # Treelet restructuring of a model.
        dict(name="atr9_1m", kind="build", method="atr", layout="bin", n=1048576, geometry="mixture", bits=60,
             presplit=0.0, rays=65536),
        # The best tree for a small static asset.
        dict(name="insertion_100k", kind="build", method="insertion", layout="bin", n=100003, geometry="uniform",
             bits=60, presplit=0.0, rays=16384),
        # Presplit references collapsed to four-wide nodes.
        dict(name="presplit_quad_500k", kind="build", method="lbvh", layout="quad", n=500009, geometry="mixture",
             bits=60, presplit=0.3, rays=65536),
        # A 1024x1024 view of a small scene, rays in pixel order.
        dict(name="primary_1m", kind="trace", layout="bin", n=65536, geometry="uniform", rays="primary", count=1048576,
             sort=False, any_hit=False),
        # Diffuse bounces in the benchmark's scene, sorted by ray key.
        dict(name="diffuse_16m", kind="trace", layout="bin", n=16777216, geometry="mixture", rays="diffuse",
             count=16777216, sort=True, any_hit=False),
        # Ambient occlusion of a 500x500 view, 8 samples a pixel.
        dict(name="ao_2m", kind="ao", n=1000003, geometry="mixture", width=500, samples=8),
        # Mesh optimisation: 1.31M triangles seen by 16 cameras of 512x512.
        dict(name="diff_4m", kind="diff", k=330, cameras=16, res=512),
        # A training set of 1024 meshes rebuilt and traced in one step.
        dict(name="batch_1024", kind="batch", meshes=1024, lo=64, hi=32768, rays_per_1k=256),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["build", "build", "build", "trace", "trace", "ao", "diff", "batch"])
    geometry = rng.choice(["uniform", "mixture"])
    if kind == "build":
        method = rng.choice(["lbvh", "lbvh", "ploc", "atr", "insertion"])
        hi = {"lbvh": 8000000, "ploc": 2000000, "atr": 2000000, "insertion": 150000}[method]
        lo = 1000 if method == "lbvh" else 5000
        presplit = rng.choice([0.0, 0.3]) if method == "lbvh" else 0.0
        return dict(kind=kind, method=method, layout=rng.choice(["bin", "bin", "quad"]) if method == "lbvh" else "bin",
                    n=_log_int(rng, lo, hi), geometry=geometry, bits=rng.choice([30, 60]), presplit=presplit,
                    rays=_log_int(rng, 1000, 100000))
    if kind == "trace":
        return dict(kind=kind, layout=rng.choice(["bin", "bin", "quad"]), n=_log_int(rng, 4000, 4000000),
                    geometry=geometry, rays=rng.choice(["primary", "diffuse", "random"]),
                    count=_log_int(rng, 4000, 4000000), sort=rng.choice([True, False]),
                    any_hit=rng.choice([False, False, True]))
    if kind == "ao":
        return dict(kind=kind, n=_log_int(rng, 10000, 2000000), geometry=geometry, width=rng.randint(64, 700),
                    samples=rng.choice([1, 4, 8]))
    if kind == "diff":
        return dict(kind=kind, k=rng.randint(20, 330), cameras=rng.randint(1, 16), res=rng.randint(64, 512))
    return dict(kind=kind, meshes=rng.randint(32, 1024), lo=64, hi=_log_int(rng, 512, 32768),
                rays_per_1k=rng.choice([64, 256]))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _soup(c, g):
    n = c.shape[0]
    s = 0.001 + 0.019 * torch.rand((n, 1, 1), generator=g, device=DEV)
    v = c[:, None, :] + s * (torch.rand((n, 3, 3), generator=g, device=DEV) - 0.5)
    return v.reshape(-1, 3), torch.arange(3 * n, dtype=torch.int32, device=DEV).reshape(-1, 3)


def _geometry(kind, n, g):
    """uniform: n small triangles over the unit box.  mixture: half of them
    drawn from 64 Gaussian clusters, half a ground grid (the rest of n, where
    the grid is not a whole square, goes to the clusters)."""
    if kind == "uniform":
        return _soup(torch.rand((n, 3), generator=g, device=DEV), g)
    cells = int(math.isqrt(n // 4))
    m = n - 2 * cells * cells
    mu = torch.rand((64, 3), generator=g, device=DEV)
    sigma = 0.01 + 0.09 * torch.rand((64, 1), generator=g, device=DEV)
    comp = torch.randint(0, 64, (m,), generator=g, device=DEV)
    v, t = _soup(mu[comp] + sigma[comp] * torch.randn((m, 3), generator=g, device=DEV), g)
    lin = torch.linspace(0.0, 1.0, cells + 1, device=DEV)
    zz, xx = torch.meshgrid(lin, lin, indexing="ij")
    gv = torch.stack([xx.reshape(-1), torch.zeros((cells + 1) ** 2, device=DEV), zz.reshape(-1)], 1)
    i = torch.arange(cells, dtype=torch.int32, device=DEV)
    v00 = (i[:, None] * (cells + 1) + i[None, :]).reshape(-1) + v.shape[0]
    v10, v01 = v00 + 1, v00 + cells + 1
    v11 = v01 + 1
    gt = torch.stack([torch.stack([v00, v10, v11], 1), torch.stack([v00, v11, v01], 1)], 1).reshape(-1, 3)
    return torch.cat([v, gv]).contiguous(), torch.cat([t, gt]).contiguous()


def _unit(d):
    return d / d.norm(dim=1, keepdim=True)


def _rays(o, d, tmax):
    r = torch.zeros((d.shape[0], 8), dtype=torch.float32, device=DEV)
    r[:, 0:3] = o
    r[:, 4:7] = d
    r[:, 7] = tmax
    return r


def _pinhole(count, origin, forward, fov):
    """`count` rays of a square image in row order (the last row may be cut short)."""
    w = math.isqrt(max(count - 1, 0)) + 1
    i = torch.arange(count, device=DEV)
    f = torch.tensor(forward, dtype=torch.float32, device=DEV)
    f = f / f.norm()
    up = torch.tensor([0.0, 1.0, 0.0] if abs(float(f[1])) < 0.99 else [1.0, 0.0, 0.0], device=DEV)
    r = torch.linalg.cross(up, f)
    r = r / r.norm()
    u = torch.linalg.cross(f, r)
    tan = math.tan(math.radians(fov) * 0.5)
    x = (2.0 * (i % w).float() / w - 1.0) * tan
    y = (2.0 * (i // w).float() / w - 1.0) * tan
    d = _unit(x[:, None] * r + y[:, None] * u + f)
    return _rays(torch.tensor(origin, dtype=torch.float32, device=DEV), d, 3.0)


def _primary(geometry, count, g):
    """A view from outside the uniform box, or from inside the mixture scene, jittered by the seed."""
    j = (0.02 * (torch.rand(3, generator=g, device=DEV) - 0.5)).tolist()
    if geometry == "uniform":
        return _pinhole(count, (0.5 + j[0], 0.5 + j[1], -1.5 + j[2]), (0.0, 0.0, 1.0), 60.0)
    return _pinhole(count, (0.5 + j[0], 0.6 + j[1], 0.02 + j[2]), (0.0, -0.35, 1.0), 60.0)


def _random_rays(count, g):
    o = -0.5 + 2.0 * torch.rand((count, 3), generator=g, device=DEV)
    t = torch.rand((count, 3), generator=g, device=DEV)
    return _rays(o, _unit(t - o), 3.0)


def _diffuse(ctx, bvh, v, t, primary, g):
    """Cosine-hemisphere bounces from the primary hits; misses become dead rays (tmax -1)."""
    res = hx.HipTracer(ctx, bvh).trace(hx.RayBuffer(primary))
    n = primary.shape[0]
    hit = res[:, 0] >= 0
    tri = t[res[:, 0].clamp(min=0).long()].long()
    nrm = torch.linalg.cross(v[tri[:, 1]] - v[tri[:, 0]], v[tri[:, 2]] - v[tri[:, 0]])
    nrm = nrm / nrm.norm(dim=1, keepdim=True).clamp(min=1e-30)
    d = primary[:, 4:7]
    nrm = torch.where((nrm * d).sum(1, keepdim=True) > 0, -nrm, nrm)
    o = primary[:, 0:3] + (res[:, 1].view(torch.float32) - 1e-4)[:, None] * d
    phi = 2.0 * math.pi * torch.rand(n, generator=g, device=DEV)
    r2 = torch.rand(n, generator=g, device=DEV)
    sr = r2.sqrt()
    ex = torch.tensor([[1.0, 0.0, 0.0]], device=DEV)
    ey = torch.tensor([[0.0, 1.0, 0.0]], device=DEV)
    tx = _unit(torch.linalg.cross(torch.where(nrm[:, 0:1].abs() > 0.9, ey, ex).expand(n, 3), nrm))
    ty = torch.linalg.cross(nrm, tx)
    w = (sr * phi.cos())[:, None] * tx + (sr * phi.sin())[:, None] * ty + (1.0 - r2).clamp(min=0.0).sqrt()[:, None] * nrm
    out = _rays(o, w, 3.0)
    out[~hit] = primary[~hit]
    out[~hit, 7] = -1.0
    return out.contiguous()


@functools.lru_cache(maxsize=64)
def _cube_sphere(k):
    """Unit sphere of 12 k^2 triangles: six k x k grids of quads, vertices shared within a face."""
    lin = torch.linspace(-0.25 * math.pi, 0.25 * math.pi, k + 1, device=DEV).tan()
    b, a = torch.meshgrid(lin, lin, indexing="ij")
    a, b, one = a.reshape(-1), b.reshape(-1), torch.ones((k + 1) ** 2, device=DEV)
    faces = [(one, a, b), (-one, b, a), (b, one, a), (a, -one, b), (a, b, one), (b, a, -one)]
    v = _unit(torch.cat([torch.stack(f, 1) for f in faces]))
    i = torch.arange(k, dtype=torch.int32, device=DEV)
    v00 = (i[:, None] * (k + 1) + i[None, :]).reshape(-1)
    quad = torch.stack([torch.stack([v00, v00 + 1, v00 + k + 2], 1), torch.stack([v00, v00 + k + 2, v00 + k + 1], 1)], 1)
    t = torch.cat([quad.reshape(-1, 3) + f * (k + 1) ** 2 for f in range(6)])
    return v, t.contiguous()


def _bumpy_sphere(k, g):
    v, t = _cube_sphere(k)
    w = 2.0 + 4.0 * torch.rand((4, 3), generator=g, device=DEV)
    p = 6.283 * torch.rand((4, 3), generator=g, device=DEV)
    r = 1.0 + 0.03 * sum(torch.prod(torch.sin(v * w[q] + p[q]), dim=1) for q in range(4))
    return (v * r[:, None]).contiguous(), t


def _orbit(cameras, res, g):
    """res x res pixel-centre rays from each camera of a Fibonacci sphere of radius 3."""
    i = torch.arange(cameras, device=DEV) + 0.5
    phi = torch.acos(1.0 - 2.0 * i / cameras)
    theta = math.pi * (1.0 + 5 ** 0.5) * i + 6.283 * torch.rand(1, generator=g, device=DEV)
    pos = 3.0 * torch.stack([theta.cos() * phi.sin(), theta.sin() * phi.sin(), phi.cos()], 1)
    f = _unit(-pos)
    up = torch.where(f[:, 1:2].abs() < 0.99, torch.tensor([[0.0, 1.0, 0.0]], device=DEV),
                     torch.tensor([[1.0, 0.0, 0.0]], device=DEV))
    r = _unit(torch.linalg.cross(up, f))
    u = torch.linalg.cross(f, r)
    x = (2.0 * (torch.arange(res, device=DEV) + 0.5) / res - 1.0) * math.tan(math.radians(15.0))
    d = (x[None, None, :, None] * r[:, None, None, :] + x[None, :, None, None] * u[:, None, None, :]
         + f[:, None, None, :]).reshape(-1, 3)
    return _rays(pos.repeat_interleave(res * res, 0), _unit(d), 10.0)


class _Memory:
    """Device memory of a BVH, for torch.as_tensor (no copy); keeps the BVH."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (int(ptr), False),
                                         "version": 3, "strides": None}


def _woop(bvh):
    """The Woop rows of a BVH, in leaf order, as a tensor over its own buffer
    (which every rebuild of the same scene writes again)."""
    w = bvh.view()
    return torch.as_tensor(_Memory(bvh, w.woop, (w.n_references, 12), "<f4"), device=DEV)


BUILDERS = {"lbvh": hx.LBVHBuilder, "ploc": hx.PLOCBuilder, "atr": hx.ATRBuilder, "insertion": hx.InsertionBuilder}
METHOD_PARAMS = {"lbvh": {}, "ploc": {"ploc_radius": 25}, "atr": {"atr_treelet_size": 9}, "insertion": {}}


def prepare(case, seed):
    g = _gen(seed)
    ctx = hx.Context.default()
    kind = case["kind"]
    if kind == "build":
        v, t = _geometry(case["geometry"], case["n"], g)
        params = dict(METHOD_PARAMS[case["method"]], morton_bits=case["bits"], layout=case["layout"])
        if case["presplit"]:
            params.update(presplitting=1, presplitter_beta=case["presplit"])
        builder = BUILDERS[case["method"]](ctx, **params)
        scene = hx.Scene(v, t)
        bvh = builder.build(scene)
        # Leaf order shows in the Woop rows and in the ids of the hits, nodes in
        # the hits.  A presplit scene's reference count is its own, so those
        # trees are seen through the hits alone.
        return dict(case=case, builder=builder, bvh=bvh, tree={} if case["presplit"] else {"woop": _woop(bvh)},
                    tracer=hx.HipTracer(ctx, bvh), rays=hx.RayBuffer(_primary(case["geometry"], case["rays"], g)))
    if kind == "trace":
        v, t = _geometry(case["geometry"], case["n"], g)
        bvh = hx.LBVHBuilder(ctx, morton_bits=60, layout=case["layout"]).build(hx.Scene(v, t))
        if case["rays"] == "random":
            r = _random_rays(case["count"], g)
        else:
            r = _primary(case["geometry"], case["count"], g)
            if case["rays"] == "diffuse":
                r = _diffuse(ctx, bvh, v, t, r, g)
        return dict(case=case, tracer=hx.HipTracer(ctx, bvh), rays=hx.RayBuffer(r, closest_hit=not case["any_hit"]))
    if kind == "ao":
        v, t = _geometry(case["geometry"], case["n"], g)
        scene = hx.Scene(v, t)
        bvh = hx.LBVHBuilder(ctx, morton_bits=60).build(scene)
        w, k = case["width"], case["samples"]
        j = (0.02 * (torch.rand(3, generator=g, device=DEV) - 0.5)).tolist()
        cam = raygen.Camera((0.5 + j[0], 0.6 + j[1], 0.02 + j[2]), (0.0, -0.35, 1.0), size=(w, w))
        rg = raygen.RayGen(ctx)
        primary, itp = rg.primary(cam)
        tracer = hx.HipTracer(ctx, bvh)
        results = tracer.trace(hx.RayBuffer(primary)).clone()
        seeds = raygen.init_seeds(ctx, w * w, frame_index=int(seed) & 0xFFFF)
        rays = torch.empty((w * w * k, 8), dtype=torch.float32, device=DEV)
        rb = hx.RayBuffer.wrap(rays, torch.zeros((w * w * k, 4), dtype=torch.int32, device=DEV), closest_hit=False)
        shade = torch.rand((w * w, 4), generator=g, device=DEV)
        return dict(case=case, ctx=ctx, rg=rg, scene=scene, tracer=tracer, primary=primary, results=results, itp=itp,
                    seeds=seeds, rb=rb, shade=shade, image=torch.zeros_like(shade))
    if kind == "diff":
        v, t = _bumpy_sphere(case["k"], g)
        r = _orbit(case["cameras"], case["res"], g)
        dt = DifferentiableTracer(v, t)
        moved = (v * (1.0 + 0.002 * torch.sin(9.0 * v[:, :1]))).contiguous().requires_grad_()
        return dict(case=case, tracer=dt, verts=moved, rays=hx.RayBuffer(r))
    w = _batch(case, g)
    hb = hx.HipBatch(ctx, hx.MeshBatch(w["V"], w["T"], w["offs"]), morton_bits=60)
    return dict(case=case, batch=hb, rays=w["rays"], owner=w["owner"], target=w["target"], grad=torch.zeros_like(w["V"]),
                results=torch.zeros((w["rays"].shape[0], 4), dtype=torch.int32, device=DEV))


def _batch(case, g):
    """Meshes of log-uniform triangle counts (the case's own), every second one
    a bumpy sphere topped up with a soup, the others soups, each in the unit
    box, and rays from a sphere around the box aimed inside it, grouped by mesh."""
    pick = random.Random(case["meshes"] * 1000003 + case["hi"])
    counts = [int(round(math.exp(pick.uniform(math.log(case["lo"]), math.log(case["hi"]))))) for _ in range(case["meshes"])]
    edge = [math.isqrt(c // 12) if m % 2 else 0 for m, c in enumerate(counts)]
    loose = [c - 12 * k * k for c, k in zip(counts, edge)]
    soup, _ = _soup(torch.rand((sum(loose), 3), generator=g, device=DEV), g)
    verts, tris, offs, vbase, at = [], [], [0], [0], 0
    for c, k, f in zip(counts, edge, loose):
        v = soup[3 * at:3 * (at + f)]
        t = torch.arange(3 * f, dtype=torch.int32, device=DEV).reshape(-1, 3)
        at += f
        if k:
            sv, st = _bumpy_sphere(k, g)
            v, t = torch.cat([0.5 + 0.45 * sv, v]), torch.cat([st, t + sv.shape[0]])
        verts.append(v)
        tris.append(t)
        offs.append(offs[-1] + c)
        vbase.append(vbase[-1] + v.shape[0])
    per = [max(1, round(case["rays_per_1k"] * c / 1000.0)) for c in counts]
    owner = torch.repeat_interleave(torch.arange(len(counts), dtype=torch.int32, device=DEV),
                                    torch.tensor(per, device=DEV))
    n = owner.shape[0]
    o = 0.5 + 1.3 * _unit(torch.randn((n, 3), generator=g, device=DEV))
    d = _unit(torch.rand((n, 3), generator=g, device=DEV) - o)
    return dict(V=torch.cat(verts).contiguous(), T=torch.cat([t + b for t, b in zip(tris, vbase)]).contiguous(),
                tris=tris, offs=offs, vbase=vbase, per=per, owner=owner, rays=_rays(o, d, 4.0),
                target=torch.rand(n, generator=g, device=DEV))


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------

def _hits(res):
    f = res.view(torch.float32)
    return {"id": res[:, 0], "t": f[:, 1], "u": f[:, 2], "v": f[:, 3]}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "build":
        state["builder"].rebuild(state["bvh"])
        return dict(state["tree"], hits=_hits(state["tracer"].trace(state["rays"])))
    if kind == "trace":
        if case["sort"]:
            hits = _hits(state["tracer"].trace_sort(state["rays"]))
            return {"hits": hits, "order": state["rays"].indices}
        return {"hits": _hits(state["tracer"].trace(state["rays"]))}
    if kind == "ao":
        k = case["samples"]
        rb = state["rb"]
        state["rg"].ao(state["primary"], state["results"], state["seeds"], k, 0.2, state["scene"], out=rb.rays)
        state["tracer"].trace_sort(rb)
        raygen.reconstruct_occlusion(state["ctx"], rb.results, state["itp"], k, state["shade"], state["image"])
        return {"rays": rb.rays, "occluder": rb.results[:, 0], "image": state["image"]}
    if kind == "diff":
        verts = state["verts"]
        t, u, v, ids = state["tracer"](verts, state["rays"])
        loss = torch.where(ids >= 0, (t - 2.0) ** 2 + 0.1 * u * v, torch.zeros_like(t)).sum()
        grad, = torch.autograd.grad(loss, verts)
        return {"t": t.detach(), "u": u.detach(), "v": v.detach(), "id": ids, "grad": grad}
    hb, rays, owner, res, grad = (state[x] for x in ("batch", "rays", "owner", "results", "grad"))
    hb.rebuild()
    hb.trace(rays, owner, results=res)
    t, u, v = hb.recompute_hits(rays, owner, res)
    dl_dt = torch.where(res[:, 0] >= 0, 2.0 * (t - state["target"]), torch.zeros_like(t))
    grad.zero_()
    hb.backward(rays, owner, res, dl_dt=dl_dt, out=grad)
    return {"id": res[:, 0], "t": t, "u": u, "v": v, "grad": grad}


# ---------------------------------------------------------------------------
# What a pass cannot do without, and how far another correct one may be off
# ---------------------------------------------------------------------------

def _scene_bytes(case):
    """Vertices and triangles read once: a soup triangle has three vertices of its own, a grid triangle half of one."""
    n = case["n"]
    per = 36.0 if case["geometry"] == "uniform" else 0.5 * 36.0 + 0.5 * 6.0
    return n * (12.0 + per)


def _ray_flops(rays, n):
    """One root-to-leaf path of two box tests a level (12 fused multiply-adds
    and 14 comparisons) and one triangle test: the least any hit takes."""
    return rays * (38.0 * math.log2(max(n, 2)) + 40.0)


def work(case):
    kind = case["kind"]
    if kind == "build":
        refs = case["n"] * (1.0 + case["presplit"])
        # Woop row, triangle id and one 64-byte node for each reference.
        b = _scene_bytes(case) + refs * (48.0 + 4.0 + 64.0)
        return {"bytes": b + 48.0 * case["rays"], "flops": 150.0 * refs + _ray_flops(case["rays"], case["n"])}
    if kind == "trace":
        b = 48.0 * case["count"] + (4.0 * case["count"] if case["sort"] else 0.0)
        return {"bytes": b + min(116.0 * case["n"], 160.0 * case["count"]),
                "flops": _ray_flops(case["count"], case["n"])}
    if kind == "ao":
        px, r = case["width"] ** 2, case["width"] ** 2 * case["samples"]
        return {"bytes": 100.0 * px + 48.0 * r + min(116.0 * case["n"], 160.0 * r),
                "flops": _ray_flops(r, case["n"])}
    if kind == "diff":
        n, r = 12 * case["k"] ** 2, case["cameras"] * case["res"] ** 2
        # Refit of every box and Woop row, hits, and the vertex gradients.
        return {"bytes": n * (12.0 + 6.0 + 48.0 + 64.0 + 6.0) + r * (32.0 + 16.0 + 12.0 + 12.0),
                "flops": 100.0 * n + _ray_flops(r, n) + 120.0 * r}
    n = case["meshes"] * (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"])
    r = n * case["rays_per_1k"] / 1000.0
    return {"bytes": n * (12.0 + 27.0 + 116.0 + 27.0) + r * (36.0 + 16.0 + 12.0 + 12.0),
            "flops": 150.0 * n + _ray_flops(r, case["hi"]) + 120.0 * r}


def tolerance(case):
    """Trees, hits and ray orders are whole numbers and FP32 values with one
    right answer; vertex gradients are FP32 sums of up to hundreds of rays in
    the order the atomics land."""
    if case["kind"] in ("diff", "batch"):
        return {"rel": 1e-6, "max": 1e-5, "differ": 0.0}
    return "exact"


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------

def _brute(rays, v, t):
    """Closest hit of every ray over every triangle in float64: (triangle or
    -1, t, u, v) with u and v the weights of the first and second vertex."""
    V = v.double()
    a, b, c = V[t[:, 0].long()], V[t[:, 1].long()], V[t[:, 2].long()]
    e1, e2 = a - c, b - c
    n = torch.linalg.cross(e1, e2)
    s = (n * n).sum(1, keepdim=True).clamp(min=1e-300)
    gu, gv = torch.linalg.cross(e2, n) / s, torch.linalg.cross(n, e1) / s
    off = [-(m * c).sum(1) for m in (n, gu, gv)]
    R = rays.double()
    count, best = R.shape[0], []
    step = max(1, int(3e7 // max(1, t.shape[0])))
    for i in range(0, count, step):
        o, d = R[i:i + step, 0:3], R[i:i + step, 4:7]
        lo, hi = R[i:i + step, 3:4], R[i:i + step, 7:8]
        h = -(o @ n.T + off[0]) / (d @ n.T)
        p = o @ gu.T + off[1] + h * (d @ gu.T)
        q = o @ gv.T + off[2] + h * (d @ gv.T)
        ok = (h > lo) & (h <= hi) & (p >= 0) & (q >= 0) & (p + q <= 1)
        h = torch.where(ok, h, torch.full_like(h, math.inf))
        m, k = h.min(1)
        miss = torch.isinf(m)
        rows = torch.arange(k.shape[0], device=DEV)
        best.append((torch.where(miss, -1, k), torch.where(miss, hi[:, 0], m),
                     torch.where(miss, 0.0, p[rows, k]), torch.where(miss, 0.0, q[rows, k])))
    return [torch.cat(x) for x in zip(*best)]


def _solve(rays, V, tri):
    """t, u, v of each ray's hit on its own triangle, as a function of the float64 vertices V."""
    a, b, c = V[tri[:, 0]], V[tri[:, 1]], V[tri[:, 2]]
    o, d = rays[:, 0:3].double(), rays[:, 4:7].double()
    e1, e2 = a - c, b - c
    n = torch.linalg.cross(e1, e2)
    h = ((c - o) * n).sum(1) / (d * n).sum(1)
    w = o + h[:, None] * d - c
    s = (n * n).sum(1)
    return h, (torch.linalg.cross(e2, n) * w).sum(1) / s, (torch.linalg.cross(n, e1) * w).sum(1) / s


MOST_PAIRS = 8e10


def exact(case, seed):
    kind = case["kind"]
    if kind == "build":
        if case["n"] * case["rays"] > MOST_PAIRS:
            return None
        g = _gen(seed)
        v, t = _geometry(case["geometry"], case["n"], g)
        _, h, p, q = _brute(_primary(case["geometry"], case["rays"], g), v, t)
        tree = {} if case["presplit"] else {"woop": None}
        return {**tree, "hits": {"id": None, "t": h, "u": p, "v": q}}
    if kind == "trace":
        if case["any_hit"] or case["rays"] == "diffuse" or case["n"] * case["count"] > MOST_PAIRS:
            return None
        g = _gen(seed)
        v, t = _geometry(case["geometry"], case["n"], g)
        r = _random_rays(case["count"], g) if case["rays"] == "random" else _primary(case["geometry"], case["count"], g)
        _, h, p, q = _brute(r, v, t)
        return {"hits": {"id": None, "t": h, "u": p, "v": q}, "order": None}
    if kind == "diff":
        if 12.0 * case["k"] ** 2 * case["cameras"] * case["res"] ** 2 > MOST_PAIRS:
            return None
        g = _gen(seed)
        v, t = _bumpy_sphere(case["k"], g)
        r = _orbit(case["cameras"], case["res"], g)
        v = (v * (1.0 + 0.002 * torch.sin(9.0 * v[:, :1]))).contiguous()
        k, h, p, q = _brute(r, v, t)
        V = v.double().requires_grad_()
        hit = k >= 0
        H, P, Q = _solve(r[hit], V, t.long()[k[hit]])
        grad, = torch.autograd.grad(((H - 2.0) ** 2 + 0.1 * P * Q).sum(), V)
        return {"t": h, "u": p, "v": q, "id": None, "grad": grad}
    if kind == "batch":
        pairs = case["meshes"] * case["hi"] ** 2 / (2.0 * math.log(case["hi"] / case["lo"]))
        if pairs * case["rays_per_1k"] / 1000.0 > MOST_PAIRS:
            return None
        w = _batch(case, _gen(seed))
        target = w["target"].double()
        grad = torch.zeros(w["V"].shape, dtype=torch.float64, device=DEV)
        out, hi = [], 0
        for m, t in enumerate(w["tris"]):
            vs = slice(w["vbase"][m], w["vbase"][m + 1])
            lo, hi = hi, hi + w["per"][m]
            r = w["rays"][lo:hi]
            k, h, p, q = _brute(r, w["V"][vs], t)
            out.append((h, p, q))
            hit = k >= 0
            V = w["V"][vs].double().requires_grad_()
            H, _, _ = _solve(r[hit], V, t.long()[k[hit]])
            grad[vs], = torch.autograd.grad(((H - target[lo:hi][hit]) ** 2).sum(), V)
        h, p, q = (torch.cat(x) for x in zip(*out))
        return {"id": None, "t": h, "u": p, "v": q, "grad": grad}
    return None
