"""The work whose speed this framework is judged by: cases drawn from what a
program that uses it has it do, each through the public entry points of
`tensorray_amd` (the ctypes layer over the C ABI, `multiview.MultiView`).

A case is a dict of plain values; its "kind" says which of the uses below it
stands for, the other entries are the sizes and options of that use:

  rays        ray casting against a resident mesh (trc_intersect): a batch of
              incoherent rays as a mesh-processing or visibility program
              queries them, closest hit, or any hit (whose answer is a mask).
  forward     an image, nothing else (preview, validation): trc_render_fwd.
  step        one optimization step's rendering: image with path checkpoint,
              dL/dI = image - target, gradient of vertices and materials.
  replay      the same without a checkpoint (the memory-saving form the
              reference has): trc_render_fwd, then trc_render_adj.
  views       many views of one textured mesh, forward and adjoint in one
              launch each (MultiView).
  edges       the boundary terms of the gradient of one view.
  deriv       forward-mode derivative images of a translation (the check the
              reference's validation runs).
  largesteps  the LargeSteps optimizer step of a mesh: two solves with
              I + lambda L and a uniform Adam step.
  update      a mesh that moved: scene update with refit, then a look at it.

Sizes come from the configurations of bench.py, tensorray_amd/inverse.py and
the tests, or lie between them.
"""
import functools
import math

import numpy as np
import torch

from tensorray_amd import _capi, inverse, multiview, scenes


def listed():
    return [
        # 2M incoherent rays (an odd number) against a 200,000-triangle mesh
        dict(name="rays_2m", kind="rays", rays=2_000_003, freq=100, any=False),
        # the smallest call: the 64 x 64 Lambertian sphere of 320 triangles,
        # where launches and latency count
        dict(name="forward_64", kind="forward", width=64, height=64, spp=16, bounces=1, scene="sphere", freq=4,
             material="diffuse"),
        # a closed room rendered with the longest paths, ragged image, rough
        # conductor: inter-reflection-heavy preview
        dict(name="forward_room", kind="forward", width=203, height=151, spp=24, bounces=8, scene="room", freq=24,
             material="conductor"),
        # bench.py's headline step: 512 x 512, 16 spp, depth 4, 20,480 triangles
        dict(name="step_512", kind="step", width=512, height=512, spp=16, bounces=3, scene="sphere", freq=32,
             material="microfacet"),
        # a view of the inverse-rendering loop: a large mesh between two
        # lights, many samples, depth 8
        dict(name="step_mesh", kind="step", width=384, height=384, spp=64, bounces=7, scene="shape", freq=140,
             material="diffuse"),
        # smooth shading and a ground texture, an odd image, no checkpoint
        dict(name="replay_smooth", kind="replay", width=301, height=211, spp=16, bounces=3, scene="textured", freq=32,
             material="microfacet"),
        # eight views of uneven odd sizes of a textured 80,000-triangle mesh
        dict(name="views_8", kind="views", views=8, low=97, high=257, spp=8, bounces=3, freq=63, texture=512),
        # silhouettes and pixel boundaries of one view of the headline scene
        dict(name="edges_camera", kind="edges", width=512, height=512, spp=4, bounces=3, scene="sphere", freq=32,
             material="microfacet", terms="primary,pixel", guided=False),
        # shadow edges with guiding, and indirect edges, in the closed room
        dict(name="edges_room", kind="edges", width=252, height=252, spp=8, bounces=4, scene="room", freq=16,
             material="microfacet", terms="direct,indirect", guided=True),
        # derivative images of a translation: interior and silhouette terms
        dict(name="deriv_128", kind="deriv", width=128, height=128, spp=16, bounces=2, scene="sphere", freq=16,
             material="diffuse", terms="interior,primary"),
        # optimizer step of a 100,002-vertex mesh
        dict(name="largesteps_100k", kind="largesteps", freq=100, lmbda=20.0),
        # a 200,000-triangle mesh moved, updated in place and looked at
        dict(name="update_200k", kind="update", freq=100, width=320, height=240, spp=2, bounces=1),
    ]


def draw(rng):
    def logi(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    def image(paths, spp):
        """An image of about `paths` / `spp` pixels, 4:3 to 1:1, odd sizes."""
        px = max(256.0, paths / spp)
        ratio = rng.uniform(0.75, 1.34)
        w = max(16, int(math.sqrt(px * ratio)))
        return w, max(16, int(px / w))

    kind = rng.choice(["rays", "forward", "step", "step", "replay", "views", "edges", "edges", "deriv", "largesteps",
                       "update"])
    mat = rng.choice(["diffuse", "microfacet", "conductor"])
    if kind == "rays":
        return dict(kind=kind, rays=logi(1000, 2_000_000), freq=logi(4, 100), any=rng.random() < 0.4)
    if kind == "largesteps":
        return dict(kind=kind, freq=logi(8, 120), lmbda=rng.choice([5.0, 20.0]))
    if kind == "update":
        return dict(kind=kind, freq=logi(8, 120), width=rng.randrange(64, 320), height=rng.randrange(64, 240),
                    spp=rng.randrange(1, 4), bounces=rng.randrange(1, 4))
    if kind == "views":
        low = rng.randrange(64, 160)
        return dict(kind=kind, views=rng.randrange(2, 10), low=low, high=low + rng.randrange(1, 120),
                    spp=rng.choice([2, 4, 8]), bounces=rng.randrange(1, 5), freq=logi(8, 64),
                    texture=rng.choice([64, 256, 512]))
    scene = rng.choice(["sphere", "room", "textured", "shape"])
    freq = logi(4, 64)
    if kind == "forward":
        spp, bounces, top = rng.choice([1, 3, 8, 16]), rng.randrange(1, 9), 1_500_000
    elif kind == "step":
        spp, bounces, top = rng.choice([2, 8, 16, 31]), rng.randrange(1, 8), 4_000_000
    elif kind == "replay":
        spp, bounces, top = rng.choice([1, 4, 16]), rng.randrange(1, 6), 1_000_000
    elif kind == "edges":
        spp, bounces, top = rng.choice([1, 4, 8]), rng.randrange(1, 5), 1_000_000
    else:
        spp, bounces, top = rng.choice([1, 4, 16]), rng.randrange(1, 5), 400_000
    w, h = image(logi(20_000, top), spp)
    c = dict(kind=kind, width=w, height=h, spp=spp, bounces=bounces, scene=scene, freq=freq, material=mat)
    if kind == "edges":
        c["width"], c["height"] = (w + 1) // 2 * 2, (h + 1) // 2 * 2  # the pixel term takes multiples of 4 samples
        c["terms"] = rng.choice(["primary", "pixel", "direct", "indirect", "primary,pixel", "direct,indirect"])
        c["guided"] = rng.random() < 0.5
    if kind == "deriv":
        c["width"], c["height"] = (w + 1) // 2 * 2, (h + 1) // 2 * 2
        c["terms"] = rng.choice(["interior", "interior,primary", "pixel", "direct", "indirect"])
    return c


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _context():
    return _capi.Context(torch.cuda.current_device())


@functools.lru_cache(maxsize=64)
def _sphere(freq):
    return scenes.geodesic_sphere(freq)


def _material(name):
    if name == "conductor":
        return scenes.Material(scenes.MAT_ROUGHCONDUCTOR, albedo=(0.2, 0.92, 1.1), spec=(3.9, 2.45, 2.14),
                               roughness=0.25)
    if name == "microfacet":
        return scenes.Material(scenes.MAT_MICROFACET, albedo=(0.2, 0.15, 0.1), spec=(0.04, 0.04, 0.04), roughness=0.3)
    return scenes.Material(scenes.MAT_DIFFUSE, albedo=(0.5, 0.5, 0.5))


def _spec(scene, freq, material, seed):
    """The scene of a case, its mesh displaced by noise of `seed`, and a
    camera for it."""
    rng = np.random.default_rng([seed, 11])
    mat = _material(material)
    pos, idx = _sphere(freq)
    move = rng.uniform(-0.05, 0.05, 3)
    if scene == "room":
        spec = scenes.box_scene(subdiv=0, material=mat)
        p = pos * np.float32(0.6) + np.array([0.0, -0.6, 0.0], np.float32)
        spec.meshes[0].pos = scenes.displace(p, 0.03, seed, center=(0.0, -0.6, 0.0))
        spec.meshes[0].idx = idx
        cam = dict(scenes.BOX_CAMERA)
    elif scene == "shape":
        spec = inverse.shape_scene(scenes.displace(pos, 0.1, seed), idx)
        spec.materials[0] = mat
        cam = scenes.fibonacci_cameras(16, radius=3.0, seed=seed)[int(rng.integers(16))]
    else:
        smooth = scene == "textured"
        spec = scenes.sphere_scene(subdiv=0, material=mat, smooth=smooth, texture_res=128 if smooth else 0)
        spec.meshes[0].pos = scenes.displace(pos, 0.05, seed)
        spec.meshes[0].idx = idx
        cam = dict(scenes.CAMERA_DEFAULT)
    cam["pos"] = tuple(float(a + b) for a, b in zip(cam["pos"], move))
    return spec, cam


class _State:
    """What a program holds between calls; gives its scene back when dropped."""

    def __init__(self, case, seed, spec=None):
        self.case = case
        self.seed = seed
        self.ctx = _context()
        self.ds = _capi.DeviceScene(self.ctx, spec) if spec is not None else None
        self.info = self.ds.info() if spec is not None else None
        self.held = []

    def __del__(self):
        try:
            torch.cuda.synchronize()
            for h in self.held:
                h.close()
            if self.ds is not None:
                self.ds.close()
        except Exception:
            pass


def _image_grad(seed, n):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 7919 + 5)
    return torch.rand(3, n, generator=g, device="cuda") - 0.3


def _rays(n, seed):
    """Incoherent rays from a sphere around the unit sphere's mesh to points
    in and beside it: about three in four hit."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 7919 + 3)
    a = torch.randn(n, 3, generator=g, device="cuda")
    b = torch.randn(n, 3, generator=g, device="cuda")
    o = a / a.norm(dim=1, keepdim=True) * 1.8
    to = b * 0.6
    d = to - o
    d = d / d.norm(dim=1, keepdim=True)
    tmin = torch.full((n, 1), 1e-2, device="cuda")
    tmax = torch.full((n, 1), 1e32, device="cuda")
    return torch.cat([o, tmin, d, tmax], 1).contiguous()


def _camera_options(case, seed, cam, **more):
    c = _capi.make_camera(case["width"], case["height"], **cam)
    o = _capi.make_options(seed=1234 + seed, max_bounces=case["bounces"], spp=case["spp"], **more)
    return c, o


def prepare(case, seed):
    kind = case["kind"]
    if kind == "rays":
        spec, _ = _spec("sphere", case["freq"], "diffuse", seed)
        s = _State(case, seed, spec)
        s.rays = _rays(case["rays"], seed)
        s.tri = torch.empty(case["rays"], dtype=torch.int32, device="cuda")
        s.uvt = torch.empty(case["rays"], 3, device="cuda")
    elif kind == "largesteps":
        s = _State(case, seed)
        pos, idx = _sphere(case["freq"])
        x = scenes.displace(pos, 0.1, seed)
        s.n = len(x)
        s.solver = s.ctx.lsolver(idx, s.n, case["lmbda"])
        s.held.append(s.solver)
        g = torch.Generator(device="cuda")
        g.manual_seed(seed * 7919 + 9)
        s.x0 = torch.from_numpy(x).cuda()
        # a vertex gradient as rendering gives it: heavy noise, zero where no view looks
        s.grad = torch.randn(s.n, 3, generator=g, device="cuda") * 1e-3
        s.grad *= (torch.rand(s.n, 1, generator=g, device="cuda") < 0.6)
        s.u0 = torch.empty_like(s.x0)
        s.solver.apply(s.x0.data_ptr(), s.u0.data_ptr())
        s.m0 = torch.randn(s.n, 3, generator=g, device="cuda") * 1e-5
        s.v0 = s.m0.square() * 0.5
        s.x, s.u, s.m, s.v, s.gu = (torch.empty_like(s.x0) for _ in range(5))
        s.gu0 = torch.zeros_like(s.x0)
    elif kind == "update":
        pos, idx = _sphere(case["freq"])
        spec = inverse.shape_scene(scenes.displace(pos, 0.05, seed), idx)
        s = _State(case, seed, spec)
        start = torch.from_numpy(s.ds.vertices()).cuda()
        n = len(pos)
        # two positions of the mesh that the passes go between
        wave = 1.0 + 0.01 * torch.sin(5.0 * start[:n, :1] + seed)
        s.moved = [start.clone(), start.clone()]
        s.moved[0][:n] *= wave
        s.moved[1][:n] *= 2.0 - wave
        s.turn = 0
        cam = scenes.fibonacci_cameras(16, radius=3.0, seed=seed)[4]
        s.cam, s.opt = _camera_options(case, seed, cam)
        s.films = [torch.empty(3, case["width"] * case["height"], device="cuda") for _ in range(2)]
    elif kind == "views":
        spec = scenes.multiview_scene(freq=case["freq"], amplitude=0.0, texture_res=case["texture"])
        spec.meshes[0].pos = scenes.displace(spec.meshes[0].pos, 0.05, seed)
        s = _State(case, seed, spec)
        cams = scenes.fibonacci_cameras(case["views"], radius=3.0, seed=seed)
        sides = [case["low"] + round(k * (case["high"] - case["low"]) / max(1, case["views"] - 1))
                 for k in range(case["views"])]
        views = [multiview.View(width=w, height=w, spp=case["spp"], max_bounces=case["bounces"], seed=seed + k,
                                cam=c) for k, (w, c) in enumerate(zip(sides, cams))]
        s.mv = multiview.MultiView(s.ctx, s.ds, views)
        s.held.append(s.mv)
    else:
        spec, cam = _spec(case["scene"], case["freq"], case["material"], seed)
        s = _State(case, seed, spec)
        n = case["spp"]
        if kind == "edges":
            s.cam, s.opt = _camera_options(case, seed, cam, sppe=n, sppe0=n, sppse0=n, sppse1=n,
                                           g_direct=case["guided"], g_direct_max_size=3 * s.info.num_triangles)
        elif kind == "deriv":
            s.cam, s.opt = _camera_options(case, seed, cam, sppe=n, sppe0=n, sppse0=n, sppse1=n)
        else:
            s.cam, s.opt = _camera_options(case, seed, cam)
        wh = case["width"] * case["height"]
        s.film = torch.empty(3, wh, device="cuda")
        s.dldi = _image_grad(seed, wh)
        s.target = 0.2 + 0.1 * _image_grad(seed + 1, wh)
        s.dpos = torch.zeros(s.info.num_vertices, 3, device="cuda")
        s.dmat = torch.zeros(s.info.num_materials, 8, device="cuda")
        s.dtex = torch.zeros(max(1, s.info.texture_floats), device="cuda")
        if kind == "step":
            s.ckpt = torch.empty(s.ds.checkpoint_bytes(s.cam, s.opt), dtype=torch.uint8, device="cuda")
        if kind == "deriv":
            # translation of the mesh along a direction
            d = torch.tensor(np.random.default_rng([seed, 17]).normal(size=3), dtype=torch.float32)
            s.tpos = torch.zeros(s.info.num_vertices, 3)
            s.tpos[:len(spec.meshes[0].pos)] = d / d.norm()
            s.tpos = s.tpos.cuda()
            s.dimg = torch.zeros(3, wh, device="cuda")
    torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(s):
    kind = s.case["kind"]
    st = torch.cuda.current_stream()
    if kind == "rays":
        s.ds.intersect(s.rays.data_ptr(), s.case["rays"], s.tri.data_ptr(), s.uvt.data_ptr(), s.case["any"], st)
        if s.case["any"]:
            return s.tri >= 0  # which hit an occlusion query names is not specified
        return s.tri, s.uvt
    if kind == "largesteps":
        for a, b in ((s.x, s.x0), (s.u, s.u0), (s.m, s.m0), (s.v, s.v0), (s.gu, s.gu0)):
            a.copy_(b)
        s.solver.solve(s.grad.data_ptr(), s.gu.data_ptr(), 400, 1e-5, st)
        s.ctx.adam_uniform_step(s.u.data_ptr(), s.gu.data_ptr(), s.m.data_ptr(), s.v.data_ptr(), 3 * s.n, 10, 1e-3,
                                stream=st)
        s.solver.solve(s.u.data_ptr(), s.x.data_ptr(), 400, 1e-6, st)
        return dict(gu=s.gu, u=s.u, x=s.x, m=s.m, v=s.v)
    if kind == "update":
        for k in range(2):
            s.ds.set_vertices(s.moved[k].data_ptr(), s.info.num_vertices, True, st)
            s.ds.render_fwd(s.cam, s.opt, s.films[k].data_ptr(), st)
        return tuple(s.films)
    if kind == "views":
        s.mv.step_eager()
        return dict(films=s.mv.film, dpos=s.mv.dpos, dmat=s.mv.dmat, dtex=s.mv.dtex)
    if kind == "forward":
        s.ds.render_fwd(s.cam, s.opt, s.film.data_ptr(), st)
        return s.film
    if kind == "deriv":
        s.dimg.zero_()
        for term in s.case["terms"].split(","):
            s.ds.render_deriv(s.cam, s.opt, term, s.tpos.data_ptr(), None, s.dimg.data_ptr(), st)
        return s.dimg
    s.dpos.zero_()
    if kind == "edges":
        for term in s.case["terms"].split(","):
            s.ds.render_boundary(s.cam, s.opt, term, s.dldi.data_ptr(), s.dpos.data_ptr(), st)
        return s.dpos
    s.dmat.zero_()
    s.dtex.zero_()
    dtex = s.dtex.data_ptr() if s.info.texture_floats else None
    if kind == "step":
        s.ds.render_fwd_ckpt(s.cam, s.opt, s.film.data_ptr(), s.ckpt.data_ptr(), s.ckpt.numel(), st)
        torch.sub(s.film, s.target, out=s.dldi)
        s.ds.render_adj_ckpt(s.cam, s.opt, s.ckpt.data_ptr(), s.ckpt.numel(), s.dldi.data_ptr(), s.dpos.data_ptr(),
                             s.dmat.data_ptr(), dtex, st)
    else:
        s.ds.render_fwd(s.cam, s.opt, s.film.data_ptr(), st)
        torch.sub(s.film, s.target, out=s.dldi)
        s.ds.render_adj(s.cam, s.opt, s.dldi.data_ptr(), s.dpos.data_ptr(), s.dmat.data_ptr(), st, dtex)
    return dict(film=s.film, dpos=s.dpos, dmat=s.dmat, dtex=s.dtex)


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
# Operations of the estimator, counted from its definition: a ray query in a
# 4-wide tree over T triangles opens about log2(T) nodes of 4 boxes (each 6
# subtractions, 6 products, 11 comparisons) and tests 3 triangles (45
# operations each); a shading point costs about 350 (frame, light sample,
# two BSDF values, their weights and the draws), its adjoint twice that.
def _query_flops(tris):
    return max(3.0, math.log2(tris)) * 4 * 23 + 3 * 45


_SHADE = 350.0
_VERTEX_STEPS = dict(sphere=1.1, textured=1.1, shape=0.75, room=None, mesh=0.7)  # bounces a path lives, on average


def _path_flops(case, scene, tris, adjoint):
    live = _VERTEX_STEPS[scene]
    b = case["bounces"] if live is None else min(case["bounces"], live)
    f = (1 + 2 * b) * _query_flops(tris) + (1 + b) * _SHADE
    return f + (2 * (1 + b) * _SHADE if adjoint else 0.0)


def _scene_size(case):
    t = 20 * case["freq"] ** 2 + 12
    v = t // 2 + 30
    # positions, indices, shading records, triangle records, tree
    return t, v, 12 * v + 12 * t + 32 * t + 48 * t + 43 * t


def work(case):
    kind = case["kind"]
    t, v, scene = _scene_size(case)
    if kind == "rays":
        n = case["rays"]
        return {"bytes": scene + n * (32 + 4 + 12), "flops": n * _query_flops(t)}
    if kind == "largesteps":
        # conjugate gradients: condition 1 + 12 lambda, residual 1e-5 and 1e-6;
        # the matrix is the mesh's edges and stays in cache between iterations,
        # so only the vectors of a step count as bytes
        iters = 0.5 * math.sqrt(1 + 12 * case["lmbda"]) * (math.log(2e5) + math.log(2e6))
        return {"bytes": 12 * v * 12 + 7 * 4 * v, "flops": iters * v * 3 * (2 * 7 + 12)}
    if kind == "update":
        px = case["width"] * case["height"]
        f = _path_flops(case, "shape", t, False) * px * case["spp"] + t * 200
        return {"bytes": 2 * (24 * v + 2 * scene + 12 * px), "flops": 2 * f}
    if kind == "views":
        sides = [case["low"] + round(k * (case["high"] - case["low"]) / max(1, case["views"] - 1))
                 for k in range(case["views"])]
        px = sum(w * w for w in sides)
        f = _path_flops(case, "mesh", t, True) * px * case["spp"]
        return {"bytes": scene + 24 * v + 24 * case["texture"] ** 2 + 24 * px, "flops": f}
    px = case["width"] * case["height"]
    n = px * case["spp"]
    if kind == "forward":
        return {"bytes": scene + 12 * px, "flops": n * _path_flops(case, case["scene"], t, False)}
    terms = case.get("terms", "interior").split(",")
    if kind == "edges":
        # a sample's two rays and its geometry; the survivors' paths
        share = dict(primary=0.1, pixel=0.8, direct=0.01, indirect=0.13)
        f = sum(n * (2 * _query_flops(t) + 200 + share[k] * _path_flops(case, case["scene"], t, False)) for k in terms)
        return {"bytes": scene + 12 * px + 12 * v, "flops": f}
    if kind == "deriv":
        f = sum(n * (_path_flops(case, case["scene"], t, True) if k == "interior" else 2 * _query_flops(t) + 200)
                for k in terms)
        return {"bytes": scene + 12 * px + 12 * v, "flops": f}
    return {"bytes": scene + 36 * px + 12 * v, "flops": n * _path_flops(case, case["scene"], t, True)}


# ---------------------------------------------------------------------------
# The same in 64 bits, where it has a value that plain torch can give: the
# estimators are random walks whose draws and discrete decisions are part of
# the result, so only the ray queries and the optimizer step do.
# ---------------------------------------------------------------------------
def exact(case, seed):
    kind = case["kind"]
    if kind == "rays":
        t, _, _ = _scene_size(case)
        if case["any"] or case["rays"] * t > 4e9:
            return None
        return None, _exact_hits(case, seed)
    if kind == "largesteps":
        return _exact_largesteps(case, seed)
    return None


def _exact_hits(case, seed):
    """(u, v, t) of the closest hit by testing every triangle."""
    spec, _ = _spec("sphere", case["freq"], "diffuse", seed)
    flat = spec.flat()
    p = torch.from_numpy(flat["pos"]).cuda().double()[torch.from_numpy(flat["idx"].astype(np.int64)).cuda()]
    p0, e1, e2 = p[:, 0], p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]
    nrm = torch.linalg.cross(e1, e2)
    rays = _rays(case["rays"], seed).double()
    out = []
    for r in rays.split(max(1, 20_000_000 // len(p0))):
        o, d = r[:, None, :3], r[:, None, 4:7]
        det = -(d * nrm).sum(2)
        s = o - p0
        q = torch.linalg.cross(s, d.expand_as(s))
        u = (e2 * q).sum(2) / det
        v = -(e1 * q).sum(2) / det
        t = (s * nrm).sum(2) / det
        ok = (u >= 0) & (v >= 0) & (u + v <= 1) & (t > r[:, None, 3]) & (t < r[:, None, 7])
        t = torch.where(ok, t, torch.full_like(t, math.inf))
        best, k = t.min(1)
        uvt = torch.stack([u.gather(1, k[:, None])[:, 0], v.gather(1, k[:, None])[:, 0], best], 1)
        miss = torch.tensor([0.0, 0.0, -1.0], dtype=torch.float64, device="cuda")
        out.append(torch.where(torch.isinf(best)[:, None], miss, uvt))
    return torch.cat(out)


def _exact_largesteps(case, seed):
    s = prepare(case, seed)
    _, idx = _sphere(case["freq"])
    f = torch.from_numpy(idx.astype(np.int64)).cuda()
    e = torch.cat([f[:, [0, 1]], f[:, [1, 2]], f[:, [2, 0]]])
    e = torch.unique(torch.cat([e, e.flip(1)]), dim=0)
    deg = torch.bincount(e[:, 0], minlength=s.n).double()
    lam = float(np.float32(case["lmbda"]))

    def mul(x):
        y = torch.zeros_like(x).index_add_(0, e[:, 0], x[e[:, 1]])
        return x + lam * (deg[:, None] * x - y)

    def solve(b):
        x = torch.zeros_like(b)
        r = b.clone()
        p = r.clone()
        rr = r.square().sum(0)
        for _ in range(400):
            ap = mul(p)
            a = rr / (p * ap).sum(0).clamp_min(1e-300)
            x += a * p
            r -= a * ap
            new = r.square().sum(0)
            p = r + new / rr.clamp_min(1e-300) * p
            rr = new
            if bool((rr <= 1e-28 * b.square().sum(0)).all()):
                break
        return x

    gu = solve(s.grad.double())
    m = 0.9 * s.m0.double() + 0.1 * gu
    v = 0.999 * s.v0.double() + 0.001 * gu.square()
    scale = 1e-3 / ((1 - 0.9 ** 10) * torch.sqrt(v.max() / (1 - 0.999 ** 10)))
    u = s.u0.double() - scale * m
    return dict(gu=gu, u=u, x=solve(u), m=m, v=v)
