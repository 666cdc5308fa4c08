"""GPU: targets and batches whose tuning was never set (the library picks the
launch, with queues by cost from 8 samples per pixel on) against the oracle,
over progressive renders, and what they report about themselves."""
import numpy as np
import pytest

import oracle_lib as O
import zig_ornament_amd as zo
from helpers import same_bits, to_oracle_params, zo_params
from zig_ornament_amd import workloads as W

pytestmark = pytest.mark.gpu

DEFAULTS = dict(regroup_lanes=48, workgroups_per_cu=0, bvh_width=2, leaf_regroup_lanes=16, samples_per_job=16,
                split_percent=0, node_steps=4, workgroup_pool=0, cost_order=0)


@pytest.mark.parametrize("spp", [7, 8, 9])
@pytest.mark.parametrize("width,height", [(33, 47), (240, 200)])
def test_progressive_renders_match_oracle(device, width, height, spp):
    spec = W.cornell(width, height, spp, 6)
    print(f"[untuned] {width}x{height} {spp} spp", flush=True)
    ds = zo.DeviceScene(device, zo.Bvh(W.build_scene(spec)))
    t = zo.Target(ds, width, height)
    oracle = O.OracleScene(O.build_bvh(spec))
    n = width * height
    acc, rng = np.zeros((n, 4), np.float32), O.seed_rng(n)
    for k in range(2):  # the second one queues by the first one's costs
        p = zo_params(spec, current_iteration=float(k * spp))
        t.render(p, spp)
        fb, _ = oracle.render(to_oracle_params(p), spp, acc, rng)
        assert same_bits(t.accumulation(), acc)
        assert same_bits(t.framebuffer(), fb)
    assert t.tuning() == DEFAULTS
    with pytest.raises(zo.OrnamentError):
        t.pixel_costs()  # only those of a render that was asked to record them
    t.set_tuning(cost_order=1)
    with pytest.raises(zo.OrnamentError):
        t.pixel_costs()
    t.render(zo_params(spec, current_iteration=float(2 * spp)), spp)
    assert t.pixel_costs().shape == (n,)


def test_batch_and_its_first_set_tuning(device):
    specs = [W.random_spheres(40, 30, 9, 5, seed=k, grid=range(-2, 2)) for k in range(3)]
    batch = zo.Batch(device, [(zo.Bvh(W.build_scene(s)), s.width, s.height, k) for k, s in enumerate(specs)])
    print("[untuned] batch", flush=True)
    images = []
    for tuning in (None, DEFAULTS, dict(cost_order=1)):
        if tuning:
            batch.set_tuning(**tuning)
        for k, s in enumerate(specs):
            n = s.width * s.height
            batch.set_state(k, np.zeros((n, 4), np.float32), (np.arange(n) + k * n).astype(np.uint32))
        batch.render([zo_params(s) for s in specs], [s.spp for s in specs])
        images.append([batch.accumulation(k) for k in range(len(specs))])
        if tuning is None:
            assert batch.tuning() == DEFAULTS
    for other in images[1:]:
        assert all(same_bits(a, b) for a, b in zip(images[0], other))
    acc, rng = np.zeros((1200, 4), np.float32), O.seed_rng(1200, 1)
    O.OracleScene(O.build_bvh(specs[1])).render(to_oracle_params(zo_params(specs[1])), 9, acc, rng)
    assert same_bits(images[0][1], acc)
