"""GPU: targets and batches whose tuning was never set, at the sizes from which
the library queues their pixels by cost (8 samples and 131,072 pixels; a batch
by its pixels alone) and just below: a first render whose first samples record
the costs, and renders queued by those of the one before. The whole state
equals that of a target in tile order, and some pixels' the oracle's."""
import numpy as np
import pytest

import oracle_lib as O
import zig_ornament_amd as zo
from helpers import same_bits, to_oracle_params, zo_params
from zig_ornament_amd import workloads as W

pytestmark = pytest.mark.gpu

TILE_ORDER = dict(samples_per_job=64, split_percent=0, cost_order=0)  # whole pixels


class Checked:
    """The oracle's state of some pixels of an image, over progressive renders."""

    def __init__(self, spec, arrays, seed, count=1500):
        n = spec.width * spec.height
        self.pixels = np.sort(np.random.default_rng(seed).choice(n, count, replace=False)).astype(np.uint32)
        self.acc = np.zeros((count, 4), np.float32)
        self.rng = (self.pixels + np.uint32(seed * n)).astype(np.uint32)
        self.scene = O.OracleScene(arrays)

    def render(self, params, spp, acc, rng):
        self.scene.render_pixels(to_oracle_params(params), spp, self.pixels, self.acc, self.rng)
        assert same_bits(acc[self.pixels], self.acc)
        assert np.array_equal(rng[self.pixels], self.rng)


@pytest.mark.parametrize("spp", [7, 8, 9])
@pytest.mark.parametrize("width,height", [(362, 362), (512, 256), (517, 261)])  # 131,044, 131,072, ragged
def test_targets_around_131072_pixels(device, width, height, spp):
    spec = W.instanced_scene(20000, width, spp, 5)
    spec.height = height
    spec.camera = spec.camera[:3] + (width / height,) + spec.camera[4:]
    arrays = zo.Bvh(W.build_scene(spec))
    scene = zo.DeviceScene(device, arrays)
    untuned, plain = zo.Target(scene, width, height, 2), zo.Target(scene, width, height, 2)
    plain.set_tuning(**TILE_ORDER)
    checked = Checked(spec, arrays, 2)
    for k in range(3):
        print(f"[untuned] {width}x{height} {spp} spp, render {k}", flush=True)
        p = zo_params(spec, current_iteration=float(k * spp))
        for t in (untuned, plain):
            t.render(p, spp)
        assert same_bits(untuned.accumulation(), plain.accumulation())
        assert same_bits(untuned.framebuffer(), plain.framebuffer())
        assert np.array_equal(untuned.rng_state(), plain.rng_state())
        checked.render(p, spp, untuned.accumulation(), untuned.rng_state())
    with pytest.raises(zo.OrnamentError):
        untuned.pixel_costs()  # recorded, but not asked for
    untuned.set_tuning(cost_order=1)
    with pytest.raises(zo.OrnamentError):
        untuned.pixel_costs()
    p = zo_params(spec, current_iteration=float(3 * spp))
    for t in (untuned, plain):
        t.render(p, spp)
    assert same_bits(untuned.accumulation(), plain.accumulation())
    assert untuned.pixel_costs().shape == (width * height,)


@pytest.mark.parametrize("sides", [(256, 255), (256, 256)])  # 130,561 and 131,072 pixels
def test_batches_around_131072_pixels(device, sides):
    specs = [W.instanced_scene(3000 * (k + 1), side, 2 + k, 5, seed=k) for k, side in enumerate(sides)]
    arrays = [zo.Bvh(W.build_scene(s)) for s in specs]
    batch = zo.Batch(device, [(a, s.width, s.height, k) for k, (a, s) in enumerate(zip(arrays, specs))])
    checked = [Checked(s, a, k) for k, (a, s) in enumerate(zip(arrays, specs))]
    plain = [zo.Target(zo.DeviceScene(device, a), s.width, s.height, k) for k, (a, s) in enumerate(zip(arrays, specs))]
    for t in plain:
        t.set_tuning(**TILE_ORDER)
    for r in range(3):
        print(f"[untuned] batch {sides}, replay {r}", flush=True)
        params = [zo_params(s, current_iteration=float(r * s.spp)) for s in specs]
        batch.render(params, [s.spp for s in specs])
        for k, s in enumerate(specs):
            plain[k].render(params[k], s.spp)
            assert same_bits(batch.accumulation(k), plain[k].accumulation())
            assert same_bits(batch.framebuffer(k), plain[k].framebuffer())
            checked[k].render(params[k], s.spp, batch.accumulation(k), batch.rng_state(k))
