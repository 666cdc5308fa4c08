"""GPU: cost-ordered queues that start with heavy pixels (pixels whose serial
work bounds the launch, run in waves of few lanes) against the oracle: images
whose few costly pixels sit in one band or in all of them, partial tiles, and a
batch with one such image."""
import numpy as np
import pytest

import oracle_lib as O
import zig_ornament_amd as zo
from helpers import same_bits, to_oracle_params, zo_params
from zig_ornament_amd import workloads as W

pytestmark = pytest.mark.gpu


def _spec(width, height, spp, depth):
    # a few spheres on the ground under much sky: most pixels end at once
    return W.random_spheres(width, height, spp, depth, seed=3, grid=range(-2, 2))


def _check(got, oracle, spec, first, acc, rng, *item):
    fb, _ = oracle.render(to_oracle_params(zo_params(spec, current_iteration=float(first))), spec.spp, acc, rng)
    assert same_bits(got.accumulation(*item), acc)
    assert same_bits(got.framebuffer(*item), fb)


# 32,769 pixels and more: full waves; one tile row gives bands of few tiles, or none
@pytest.mark.parametrize("width,height,spp,depth", [(16, 2100, 4, 16), (2100, 17, 3, 16), (201, 170, 5, 24),
                                                    (640, 80, 2, 8)])
def test_ordered_renders_match_oracle(device, width, height, spp, depth):
    spec = _spec(width, height, spp, depth)
    print(f"[heavy] {width}x{height} {spp} spp depth {depth}", flush=True)
    t = zo.Target(zo.DeviceScene(device, zo.Bvh(W.build_scene(spec))), width, height)
    t.set_tuning(cost_order=1)
    oracle = O.OracleScene(O.build_bvh(spec))
    n = width * height
    acc, rng = np.zeros((n, 4), np.float32), O.seed_rng(n)
    for k in range(3):
        t.render(zo_params(spec, current_iteration=float(k * spp)), spp)
        _check(t, oracle, spec, k * spp, acc, rng)


def test_batch_with_one_costly_image(device):
    specs = [_spec(40, 30, 1, 2), _spec(64, 48, 12, 24), _spec(250, 160, 1, 2)]
    batch = zo.Batch(device, [(zo.Bvh(W.build_scene(s)), s.width, s.height, k) for k, s in enumerate(specs)])
    batch.set_tuning(cost_order=1)
    oracles = [O.OracleScene(O.build_bvh(s)) for s in specs]
    print("[heavy] batch", flush=True)
    state = [(np.zeros((s.width * s.height, 4), np.float32), O.seed_rng(s.width * s.height, k))
             for k, s in enumerate(specs)]
    for k in range(3):
        batch.render([zo_params(s, current_iteration=float(k * s.spp)) for s in specs], [s.spp for s in specs])
        for i, s in enumerate(specs):
            _check(batch, oracles[i], s, k * s.spp, *state[i], i)
