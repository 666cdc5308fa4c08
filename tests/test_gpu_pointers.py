"""GPU: the entry points that copy to and from the caller's arrays take device
memory and pinned host memory as well as ordinary arrays."""
import ctypes as C

import numpy as np
import pytest
import torch

import zig_ornament_amd as zo
from helpers import zo_params
from zig_ornament_amd import _native as N
from zig_ornament_amd import workloads as W
from zig_ornament_amd.nrc import MLP_PARAMS, RECORD_DTYPE, Nrc

pytestmark = pytest.mark.gpu

KINDS = ["device", "pinned"]


def like(kind, array):
    """A copy of an array in memory of a kind."""
    t = torch.from_numpy(np.ascontiguousarray(array).view(np.uint8).reshape(-1).copy())
    t = t.cuda() if kind == "device" else t.pin_memory()
    torch.cuda.synchronize()
    return t


def bits(t):
    torch.cuda.synchronize()
    return t.cpu().numpy().tobytes()


def ptr(t):
    return C.c_void_p(t.data_ptr())


@pytest.fixture(scope="module")
def scene(device):
    return zo.DeviceScene(device, zo.Bvh(W.build_scene(W.random_spheres(64, 64, 1, 4, grid=range(-4, 4)))))


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("width,height", [(33, 17), (1920, 1080)])  # one part, and more than the kept buffer
def test_images_and_state(scene, kind, width, height):
    print(f"[pointers] {width}x{height} {kind}", flush=True)
    spec = W.random_spheres(width, height, 1, 4, grid=range(-4, 4))
    t = zo.Target(scene, width, height)
    t.render(zo_params(spec), 1)
    n = width * height
    for fn, array in [(N.lib().orn_get_framebuffer, t.framebuffer()), (N.lib().orn_get_accumulation, t.accumulation()),
                      (N.lib().orn_get_rng_state, t.rng_state())]:
        out = like(kind, np.zeros_like(array))
        assert fn(t.handle, ptr(out), n) == 0
        assert bits(out) == array.tobytes()
    rng = np.random.default_rng(1)
    acc, words = rng.random((n, 4), dtype=np.float32), rng.integers(0, 2 ** 32, n, dtype=np.uint32)
    a, w = like(kind, acc), like(kind, words)
    assert N.lib().orn_set_state(t.handle, ptr(a), ptr(w), n) == 0
    assert np.array_equal(t.accumulation(), acc) and np.array_equal(t.rng_state(), words)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n", [300, 5000, 300000])  # traced in host memory, one piece, several
def test_ray_queries(scene, kind, n):
    print(f"[pointers] {n} rays {kind}", flush=True)
    rays = np.random.default_rng(n).uniform(-4, 4, (n, 6)).astype(np.float32)
    want = scene.trace(rays)
    for fn in (N.lib().orn_trace_rays, N.lib().orn_trace_rays_packet):
        for host_rays, host_out in [(False, False), (True, False), (False, True)]:
            r, out = like(kind, rays), like(kind, np.zeros_like(want))
            h = np.zeros_like(want)
            assert fn(scene.handle, C.c_float(0.001), C.c_void_p(rays.ctypes.data) if host_rays else ptr(r), n,
                      C.c_void_p(h.ctypes.data) if host_out else ptr(out)) == 0
            assert (h.tobytes() if host_out else bits(out)) == want.tobytes()


@pytest.mark.parametrize("kind", KINDS)
def test_radiance_cache_arrays(scene, kind):
    print(f"[pointers] radiance cache {kind}", flush=True)
    rng = np.random.default_rng(3)
    nrc, m = Nrc(scene), 1000
    mlp = (0.15 * rng.standard_normal(MLP_PARAMS)).astype(np.float32)
    p = like(kind, mlp)
    assert N.lib().orn_nrc_set_params(nrc.handle, ptr(p), MLP_PARAMS, None, 0) == 0
    out = like(kind, np.zeros_like(mlp))
    assert N.lib().orn_nrc_get_params(nrc.handle, ptr(out), MLP_PARAMS, None, 0) == 0
    assert bits(out) == mlp.tobytes()
    rec = np.zeros(m, RECORD_DTYPE)
    rec["pos"], rec["dir"], rec["normal"] = rng.uniform(-4, 4, (m, 3)), (0, 0, 1), (0, 1, 0)
    rec["albedo"], rec["weight"] = rng.random((m, 3)), rng.random((m, 3))
    want, loss, grad = nrc.query(rec), C.c_float(), np.zeros(MLP_PARAMS, np.float32)
    assert N.lib().orn_nrc_gradients(nrc.handle, C.c_void_p(rec.ctypes.data), m, C.byref(loss),
                                     C.c_void_p(grad.ctypes.data), None, 0) == 0
    r, rgb, g, l2 = like(kind, rec), like(kind, np.zeros((m, 3), np.float32)), like(kind, np.zeros_like(grad)), C.c_float()
    assert N.lib().orn_nrc_query(nrc.handle, ptr(r), m, ptr(rgb), None) == 0
    assert bits(rgb) == np.asarray(want, np.float32).tobytes()
    assert N.lib().orn_nrc_gradients(nrc.handle, ptr(r), m, C.byref(l2), ptr(g), None, 0) == 0
    assert bits(g) == grad.tobytes()
    # the loss is added up by atomics, in any order: 3,000 squares in f32
    assert abs(l2.value - loss.value) <= 3000 * 2.0 ** -24 * loss.value
