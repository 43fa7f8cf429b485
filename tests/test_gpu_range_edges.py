"""Sizes at the edges of the kernels' tiles, blocks, windows and segments.

Forward radiance is compared bit for bit with the oracle; gradients within the
bound of float sums in another order (relative 1e-3 of an entry plus 1e-5 of the
largest one: 2^-24 times the square root of some thousand summands, with room),
solves within 1e-4 of a dense solve in float64 (tolerance 1e-6 of the residual
times the system's condition number, below 50 here).
"""
import numpy as np
import pytest

from tensorray_amd import _capi, scenes

pytestmark = pytest.mark.gpu


def _close(got, ref):
    scale = np.abs(ref).max()
    assert scale > 0
    err = np.abs(got - ref) / (1e-3 * np.abs(ref) + 1e-5 * scale)
    assert (err <= 1).all(), err.max()


# blocks of 8 x 8 pixels: whole, ragged, too ragged to be used; one path; no bounce
@pytest.mark.parametrize("W,H,spp,B", [(1, 1, 1, 0), (7, 9, 1, 1), (8, 8, 2, 0), (63, 65, 2, 2), (72, 8, 3, 1),
                                       (129, 64, 1, 2)])
def test_path_order(gpu_ctx, oracle_mod, W, H, spp, B):
    import torch
    spec = scenes.box_scene(subdiv=2)
    ds = _capi.DeviceScene(gpu_ctx, spec)
    cam = _capi.make_camera(W, H, **scenes.BOX_CAMERA)
    opt = _capi.make_options(seed=7, max_bounces=B, spp=spp)
    n = W * H * spp
    paths = torch.full((n, 3), -1.0, device="cuda")
    ds.render_paths(cam, opt, paths.data_ptr())
    torch.cuda.synchronize()
    ref = oracle_mod.Scene(spec).render_paths(scenes.BOX_CAMERA, W, H, 7, B, 0, n)
    assert np.array_equal(paths.cpu().numpy(), ref)
    ds.close()


# trees whose stack spills out of LDS, and one that needs all of its 80 entries
@pytest.mark.parametrize("levels,per,ratio", [(40, 4, 0.5), (60, 4, 0.25)])
def test_deep_tree(gpu_ctx, oracle_mod, levels, per, ratio):
    import torch
    spec = scenes.chain_scene(levels, per, ratio)
    ds = _capi.DeviceScene(gpu_ctx, spec)
    assert 40 <= ds.info().bvh_stack_need <= 80
    rng = np.random.default_rng(9)
    n = 20000
    # along the chain, from its far end and from its tip, and across it
    pos = spec.meshes[0].pos
    to = pos[rng.integers(0, len(pos), n)].astype(np.float64)
    o = np.where(rng.random((n, 1)) < 0.5, rng.normal(size=(n, 3)) * 1e-3, np.array([1.5, 0.0, 0.0]) * rng.uniform(0.7, 1, (n, 1)))
    o[::5] = rng.normal(size=(len(o[::5]), 3))
    rays = np.concatenate([o, np.full((n, 1), 1e-9), to - o, np.full((n, 1), 1e30)], 1).astype(np.float32)
    rd = torch.from_numpy(rays).cuda()
    tri, uvt = torch.empty(n, dtype=torch.int32, device="cuda"), torch.empty(n, 3, device="cuda")
    ds.intersect(rd.data_ptr(), n, tri.data_ptr(), uvt.data_ptr())
    torch.cuda.synchronize()
    want_tri, want_uvt = oracle_mod.Scene(spec).intersect(rays, brute=True)
    assert np.array_equal(tri.cpu().numpy(), want_tri)
    assert np.array_equal(uvt.cpu().numpy(), want_uvt)  # rays through vertices: zeros of either sign
    cam = _capi.make_camera(24, 20, pos=(1.3, 0.05, 0.0), target=(0.0, 0.0, 0.0))
    opt = _capi.make_options(seed=2, max_bounces=2, spp=2)
    paths = torch.zeros(960, 3, device="cuda")
    ds.render_paths(cam, opt, paths.data_ptr())
    torch.cuda.synchronize()
    ref = oracle_mod.Scene(spec).render_paths(dict(scenes.CAMERA_DEFAULT, pos=(1.3, 0.05, 0.0), target=(0.0, 0.0, 0.0)),
                                              24, 20, 2, 2, 0, 960)
    assert np.array_equal(paths.cpu().numpy(), ref)
    ds.close()


# one sample group; ragged and whole blocks; more samples than a chunk of 2^22
@pytest.mark.parametrize("W,H,spp", [(5, 4, 4), (64, 64, 4), (70, 50, 8), (256, 256, 68)])
def test_pixel_boundary(gpu_ctx, oracle_mod, W, H, spp):
    import torch
    spec = scenes.box_scene(subdiv=2)
    ds = _capi.DeviceScene(gpu_ctx, spec)
    cam = _capi.make_camera(W, H, **scenes.BOX_CAMERA)
    opt = _capi.make_options(seed=31, max_bounces=2, spp=1, sppe0=spp)
    dl = np.random.default_rng(2).uniform(0.2, 1.0, (3, W * H)).astype(np.float32)
    dpos = torch.zeros(ds.info().num_vertices, 3, device="cuda")
    ds.render_boundary(cam, opt, "pixel", torch.from_numpy(dl).cuda().data_ptr(), dpos.data_ptr())
    torch.cuda.synchronize()
    ref = oracle_mod.boundary_adj(oracle_mod.Scene(spec), scenes.BOX_CAMERA, W, H, 31, 2, "pixel", spp, dl)
    mask = spec.diff_vertex_mask()
    _close(dpos.cpu().numpy().astype(np.float64)[mask], ref[mask])
    ds.close()


def test_pixel_boundary_first_call_captured(gpu_ctx):
    """The scratch of a small pixel term is its stream's: a scene's first such
    call may be a captured one."""
    import torch
    W, H, spp = 72, 40, 4
    spec = scenes.box_scene(subdiv=2)
    ds = _capi.DeviceScene(gpu_ctx, spec)
    cam = _capi.make_camera(W, H, **scenes.BOX_CAMERA)
    opt = _capi.make_options(seed=31, max_bounces=2, spp=1, sppe=spp, sppe0=spp)
    dl = torch.from_numpy(np.random.default_rng(2).uniform(0.2, 1.0, (3, W * H)).astype(np.float32)).cuda()
    dpos = torch.zeros(ds.info().num_vertices, 3, device="cuda")
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    film = torch.empty(3, W * H, device="cuda")
    ds.render_fwd(cam, opt, film.data_ptr(), stream=st.cuda_stream)  # the stream's own buffers
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st):
        ds.render_boundary(cam, opt, "pixel", dl.data_ptr(), dpos.data_ptr(), stream=st.cuda_stream)
    eager = torch.zeros_like(dpos)
    ds.render_boundary(cam, opt, "pixel", dl.data_ptr(), eager.data_ptr())
    torch.cuda.synchronize()
    for _ in range(3):
        dpos.zero_()
        g.replay()
        torch.cuda.synchronize()
        _close(dpos.cpu().numpy().astype(np.float64), eager.cpu().numpy().astype(np.float64))
        ds.render_fwd(cam, opt, film.data_ptr())
        torch.cuda.synchronize()
    del g
    ds.close()


# paths in one window of the stream's scratch; samples and paths in several (of
# 2^18 samples, 2^19 paths; the last one is ragged)
@pytest.mark.parametrize("kind,W,H,spp", [("pixel", 301, 220, 16), ("interior", 71, 40, 4), ("interior", 401, 300, 9)])
def test_captured_windows(gpu_ctx, kind, W, H, spp):
    """The windows of the pixel term and of the interior derivative image lie
    in their stream's memory: a scene's first such call may be a captured one,
    of any size, and its graph has no allocation node."""
    import torch
    spec = scenes.box_scene(subdiv=2)
    ds = _capi.DeviceScene(gpu_ctx, spec)
    cam = _capi.make_camera(W, H, **scenes.BOX_CAMERA)
    opt = _capi.make_options(seed=31, max_bounces=2, spp=spp, sppe0=spp)
    dl = torch.from_numpy(np.random.default_rng(2).uniform(0.2, 1.0, (3, W * H)).astype(np.float32)).cuda()
    nv = ds.info().num_vertices
    if kind == "pixel":
        out, eager = torch.zeros(nv, 3, device="cuda"), torch.zeros(nv, 3, device="cuda")

        def call(buf, stream=None):
            ds.render_boundary(cam, opt, "pixel", dl.data_ptr(), buf.data_ptr(), stream=stream)
    else:
        out, eager = torch.zeros(3, W * H, device="cuda"), torch.zeros(3, W * H, device="cuda")
        tpos = torch.zeros(nv, 3, device="cuda")
        tpos[:len(spec.meshes[0].pos)] = torch.tensor([0.3, 0.8, -0.5], device="cuda")

        def call(buf, stream=None):
            ds.render_deriv(cam, opt, "interior", tpos.data_ptr(), None, buf.data_ptr(), stream=stream)
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    film = torch.empty(3, W * H, device="cuda")
    ds.render_fwd(cam, opt, film.data_ptr(), stream=st.cuda_stream)  # the stream's own buffers
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st):
        call(out, st.cuda_stream)
    call(eager)
    torch.cuda.synchronize()
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        _close(out.cpu().numpy().astype(np.float64), eager.cpu().numpy().astype(np.float64))
        ds.render_fwd(cam, opt, film.data_ptr())
        torch.cuda.synchronize()
    del g
    ds.close()


# paths in one window of the replay, and in two of which the second is ragged
@pytest.mark.parametrize("W,H,spp", [(33, 31, 3), (511, 300, 16)])
def test_replay_windows(gpu_ctx, W, H, spp):
    import torch
    spec = scenes.sphere_scene(subdiv=2, smooth=True)
    ds = _capi.DeviceScene(gpu_ctx, spec)
    cam = _capi.make_camera(W, H, **scenes.CAMERA_DEFAULT)
    opt = _capi.make_options(seed=5, max_bounces=2, spp=spp)
    dl = torch.from_numpy(np.random.default_rng(3).uniform(0.2, 1.0, (3, W * H)).astype(np.float32)).cuda()
    nv = ds.info().num_vertices
    nb = ds.checkpoint_bytes(cam, opt)
    ck = torch.empty(nb, dtype=torch.uint8, device="cuda")
    film = torch.empty(3, W * H, device="cuda")
    a, b = torch.zeros(nv, 3, device="cuda"), torch.zeros(nv, 3, device="cuda")
    ds.render_adj(cam, opt, dl.data_ptr(), a.data_ptr())
    ds.render_fwd_ckpt(cam, opt, film.data_ptr(), ck.data_ptr(), nb)
    ds.render_adj_ckpt(cam, opt, ck.data_ptr(), nb, dl.data_ptr(), b.data_ptr())
    torch.cuda.synchronize()
    _close(a.cpu().numpy().astype(np.float64), b.cpu().numpy().astype(np.float64))
    ds.close()


# dL/dI zero in all pixels but one, in whole blocks and halves of the image
@pytest.mark.parametrize("keep", ["pixel", "block", "half", "none"])
def test_replay_of_a_masked_image(gpu_ctx, oracle_mod, keep):
    import torch
    W, H, spp = 50, 37, 3
    spec = scenes.sphere_scene(subdiv=2)
    ds = _capi.DeviceScene(gpu_ctx, spec)
    cam = _capi.make_camera(W, H, **scenes.CAMERA_DEFAULT)
    opt = _capi.make_options(seed=5, max_bounces=2, spp=spp)
    mask = np.zeros((H, W), np.float32)
    y, x = {"pixel": (20, 25), "block": (slice(16, 24), slice(24, 32)), "half": (slice(None), slice(0, 25)),
            "none": (slice(0), slice(0))}[keep]
    mask[y, x] = 1.0
    dl = (np.random.default_rng(3).uniform(0.2, 1.0, (3, W * H)) * mask.reshape(-1)).astype(np.float32)
    dl[1:] *= 0.5 if keep != "pixel" else 0.0  # a pixel counts with any of its channels
    dpos = torch.zeros(ds.info().num_vertices, 3, device="cuda")
    ds.render_adj(cam, opt, torch.from_numpy(dl).cuda().data_ptr(), dpos.data_ptr())
    torch.cuda.synchronize()
    got = dpos.cpu().numpy().astype(np.float64)
    if keep == "none":
        assert not got.any()
    else:
        ref, _ = oracle_mod.Scene(spec).render_adj(scenes.CAMERA_DEFAULT, W, H, 5, 2, spp, dl)
        m = spec.diff_vertex_mask()
        _close(got[m], ref[m])
    ds.close()


# rows: less than a slice of 64, one over, several slices with a remainder
@pytest.mark.parametrize("freq", [1, 2, 3, 8])
def test_solver_slices(gpu_ctx, oracle_mod, freq):
    import torch
    pos, idx = scenes.geodesic_sphere(freq)
    nv, lam = len(pos), 3.0
    M = oracle_mod.laplacian_system(idx, nv, lam).toarray()
    S = gpu_ctx.lsolver(idx, nv, lam)
    b = np.random.default_rng(4).standard_normal((nv, 3)).astype(np.float32)
    db = torch.from_numpy(b).cuda()
    y, x = torch.empty_like(db), torch.zeros_like(db)
    S.apply(db.data_ptr(), y.data_ptr())
    S.solve(db.data_ptr(), x.data_ptr(), max_iter=500, tol=1e-6)
    torch.cuda.synchronize()
    ref = M @ b.astype(np.float64)
    assert np.abs(y.cpu().numpy() - ref).max() <= 1e-5 * np.abs(ref).max()
    xs = np.linalg.solve(M, b.astype(np.float64))
    assert np.abs(x.cpu().numpy() - xs).max() <= 1e-4 * np.abs(xs).max()
    S.close()
