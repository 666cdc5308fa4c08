"""GPU: orn_render_noalloc with a tuning that asks for queues by cost, around
the sizes from which it takes the order from its own first samples, against a
target's render in tile order; the scratch it leaves serves the next call."""
import ctypes as C

import numpy as np
import pytest
import torch

import zig_ornament_amd as zo
from helpers import same_bits, zo_params
from zig_ornament_amd import _native as N
from zig_ornament_amd import workloads as W

pytestmark = pytest.mark.gpu


def _noalloc(ds, spec, seed, tuning):
    n = spec.width * spec.height
    acc, fb = torch.zeros((n, 4), device="cuda"), torch.empty((n, 4), device="cuda")
    rng = torch.arange(seed * n, seed * n + n, device="cuda", dtype=torch.int32)
    torch.cuda.synchronize()
    t, p = zo._tuning_struct(**tuning), zo_params(spec)
    assert N.lib().orn_render_noalloc(ds.handle, C.byref(p), spec.spp, C.byref(t), acc.data_ptr(), rng.data_ptr(),
                                      fb.data_ptr(), None) == 0
    torch.cuda.synchronize()
    return acc.cpu().numpy(), rng.cpu().numpy().view(np.uint32), fb.cpu().numpy()


# just below and at 2^17 pixels, 7 and 8 samples; 9,216 and 9,218 tiles; tiles that hold 16 pixels
@pytest.mark.parametrize("split", [0, 50])
@pytest.mark.parametrize("width,height,spp", [(362, 362, 9), (512, 256, 8), (512, 256, 7), (363, 363, 17),
                                              (17, 73728, 8), (17, 73729, 8), (1, 1 << 17, 8), (1 << 17, 1, 8)])
def test_ordered_call_matches_target(device, width, height, spp, split):
    spec = W.random_spheres(width, height, spp, 6, grid=range(-2, 2))
    tuning = dict(regroup_lanes=48, leaf_regroup_lanes=2, node_steps=6, samples_per_job=4, split_percent=split,
                  cost_order=1)
    print(f"[noalloc order] {width}x{height} {spp} spp split {split}", flush=True)
    ds = zo.DeviceScene(device, zo.Bvh(W.build_scene(spec)))
    t = zo.Target(ds, width, height, 1)
    t.set_tuning(**dict(tuning, cost_order=0))
    t.render(zo_params(spec), spp)
    for _ in range(2):
        acc, rng, fb = _noalloc(ds, spec, 1, tuning)
        assert same_bits(acc, t.accumulation())
        assert np.array_equal(rng, t.rng_state())
        assert same_bits(fb, t.framebuffer())
