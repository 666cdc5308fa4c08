"""GPU: images around the pixel counts where a render's waves change from 4 to
8 to 64 working lanes (16,384 and 32,768 pixels on 256 compute units with four
workgroups each), whole and split into jobs, against the oracle."""
import numpy as np
import pytest

import oracle_lib as O
import zig_ornament_amd as zo
from helpers import same_bits, to_oracle_params, zo_params
from zig_ornament_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tuning", [None, dict(regroup_lanes=1, leaf_regroup_lanes=64, split_percent=100,
                                               samples_per_job=1, node_steps=2)])
@pytest.mark.parametrize("width,height", [(1, 1), (3, 5), (128, 128), (145, 113), (182, 180), (331, 99)])
def test_image_matches_oracle(device, width, height, tuning):
    spec = W.random_spheres(width, height, 2, 6, grid=range(-3, 3))
    print(f"[sparse] {width}x{height} {tuning}", flush=True)
    ds = zo.DeviceScene(device, zo.Bvh(W.build_scene(spec)))
    t = zo.Target(ds, width, height)
    if tuning:
        t.set_tuning(**tuning)
    p = zo_params(spec)
    t.render(p, spec.spp)
    n = width * height
    acc, rng = np.zeros((n, 4), np.float32), O.seed_rng(n)
    fb, _ = O.OracleScene(O.build_bvh(spec)).render(to_oracle_params(p), spec.spp, acc, rng)
    assert same_bits(t.accumulation(), acc)
    assert same_bits(t.framebuffer(), fb)
    assert np.array_equal(t.rng_state(), rng)
