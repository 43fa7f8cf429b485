"""Calls of several threads and captured calls: the memory that a call's
kernels hand their results to one another in is that call's alone.

Films are compared bit for bit with those of calls made one after another,
gradients within the bound of float sums in another order (relative 1e-3 of an
entry plus 1e-5 of the largest one).
"""
import threading

import numpy as np
import pytest

from tensorray_amd import _capi, scenes

pytestmark = pytest.mark.gpu


def _close(got, ref):
    scale = np.abs(ref).max()
    assert scale > 0
    err = np.abs(got - ref) / (1e-3 * np.abs(ref) + 1e-5 * scale)
    assert (err <= 1).all(), err.max()


class _Work:
    """Film, replayed interior gradient and pixel-boundary gradient of one
    scene, on a stream."""

    def __init__(self, ctx, freq, seed, W, H, spp=2):
        import torch
        spec = scenes.sphere_scene(subdiv=0, smooth=False)
        spec.meshes[0].pos, spec.meshes[0].idx = scenes.geodesic_sphere(freq)
        self.ds = _capi.DeviceScene(ctx, spec)
        self.cam = _capi.make_camera(W, H, **scenes.CAMERA_DEFAULT)
        self.opt = _capi.make_options(seed=seed, max_bounces=2, spp=spp, sppe0=4)
        dl = np.random.default_rng(seed).uniform(0.2, 1.0, (3, W * H)).astype(np.float32)
        self.dl = torch.from_numpy(dl).cuda()
        nv = self.ds.info().num_vertices
        self.film = torch.zeros(3, W * H, device="cuda")
        self.adj, self.pixel = torch.zeros(nv, 3, device="cuda"), torch.zeros(nv, 3, device="cuda")

    def clear(self):
        for t in (self.film, self.adj, self.pixel):
            t.zero_()

    def call(self, stream=None):
        self.ds.render_fwd(self.cam, self.opt, self.film.data_ptr(), stream=stream)
        self.ds.render_adj(self.cam, self.opt, self.dl.data_ptr(), self.adj.data_ptr(), stream=stream)
        self.ds.render_boundary(self.cam, self.opt, "pixel", self.dl.data_ptr(), self.pixel.data_ptr(), stream=stream)

    def results(self):
        return [t.cpu().numpy().astype(np.float64) for t in (self.film, self.adj, self.pixel)]

    def check(self, ref, times=1):
        film, adj, pixel = self.results()
        assert np.array_equal(film, ref[0])
        _close(adj, times * ref[1])
        _close(pixel, times * ref[2])


def test_threads_share_a_stream(gpu_ctx):
    """Two threads queue calls of two scenes on the same stream at once."""
    import torch
    works = [_Work(gpu_ctx, 4, 3, 40, 36), _Work(gpu_ctx, 9, 4, 33, 50)]
    refs = []
    for w in works:
        w.call()
        torch.cuda.synchronize()
        refs.append(w.results())
        w.clear()
    torch.cuda.synchronize()
    n = 25
    start = threading.Barrier(2)
    errors = []

    def loop(w):
        try:
            start.wait(30)
            for _ in range(n):
                w.call()
        except Exception as e:  # shown by the main thread
            errors.append(e)

    threads = [threading.Thread(target=loop, args=(w,)) for w in works]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    torch.cuda.synchronize()
    assert not errors, errors
    for w, ref in zip(works, refs):
        w.check(ref, n)
        w.ds.close()
