"""GPU: a tuning that launches more workgroups than fit on the compute units
renders the same bits in about the time of one that fits."""
import numpy as np
import pytest

import zig_ornament_amd as zo
from helpers import zo_params
from zig_ornament_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cost_order", [0, 1])
@pytest.mark.parametrize("name", ["spheres", "cornell", "meshes"])
def test_more_workgroups_than_fit(device, name, cost_order):
    spec = {"spheres": lambda: W.random_spheres(500, 500, 8, 8), "cornell": lambda: W.cornell(500, 500, 8, 8),
            "meshes": lambda: W.instanced_scene(50000, 500, 8)}[name]()
    scene = zo.DeviceScene(device, zo.Bvh(W.build_scene(spec)))
    p, ms, images = zo_params(spec), {}, {}
    for groups in (0, 32, 64):
        target = zo.Target(scene, spec.width, spec.height, 1)
        target.set_tuning(workgroups_per_cu=groups, cost_order=cost_order)
        times = []
        for k in range(5):
            target.render(p, spec.spp)
            times.append(target.last_render_ms())
            if k == 0:
                images[groups] = np.array(target.framebuffer())
        ms[groups] = min(times)
        print(f"[workgroups] {name} order {cost_order}, {groups} per CU: {ms[groups]:.3f} ms", flush=True)
    assert np.array_equal(images[0], images[32]) and np.array_equal(images[0], images[64])
    # full waves of the same pixels: the launches differ by idle workgroups alone
    assert max(ms[32], ms[64]) < 1.5 * ms[0]
