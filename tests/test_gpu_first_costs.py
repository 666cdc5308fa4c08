"""GPU: the per-pixel costs after a target's first set_tuning are those of the
render that followed it, whatever the library recorded for itself before."""
import numpy as np
import pytest

import zig_ornament_amd as zo
from helpers import zo_params
from zig_ornament_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("start", [16.0, 16.5])  # 16.5 + n is not split, so it is recorded in one launch
def test_costs_of_untuned_renders_are_dropped(device, start):
    spec = W.cornell(512, 256, 16, 6)
    scene = zo.DeviceScene(device, zo.Bvh(W.build_scene(spec)))
    costs = {}
    for earlier in (0, 16):
        target = zo.Target(scene, spec.width, spec.height, 1)
        if earlier:
            target.render(zo_params(spec), earlier)  # untuned: the library orders its queues and records
        target.set_tuning(cost_order=1)
        with pytest.raises(zo.OrnamentError):
            target.pixel_costs()
        target.render(zo_params(spec, current_iteration=start), 1)
        costs[earlier] = target.pixel_costs().astype(np.float64).sum()
        print(f"[costs] {earlier} spp before: {costs[earlier]:.3g} ticks", flush=True)
    # one sample's time either way; what the earlier render records is some 14 samples'
    assert costs[16] < 3.0 * costs[0]
