"""GPU: state and ray arrays of sizes around the pinned buffer's parts (1 MB,
32 MB in all), the limit of queries traced in host memory (4,096 rays), the
rays per launch (131,072) and the kept workspace (64 MB) arrive whole."""
import numpy as np
import pytest

import zig_ornament_amd as zo
from zig_ornament_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def scene(device):
    return zo.DeviceScene(device, zo.Bvh(W.build_scene(W.random_spheres(64, 64, 1, 4, grid=range(-4, 4)))))


@pytest.mark.parametrize("width,height", [(1, 1), (256, 256), (257, 255), (701, 601), (2048, 1024), (2051, 1024)])
def test_state_round_trip(scene, width, height):
    print(f"[copies] {width}x{height}", flush=True)
    rng = np.random.default_rng(width)
    t = zo.Target(scene, width, height)
    acc = rng.random((width * height, 4), dtype=np.float32)
    words = rng.integers(0, 2 ** 32, width * height, dtype=np.uint32)
    t.set_state(acc, words)
    assert np.array_equal(t.accumulation(), acc)
    assert np.array_equal(t.rng_state(), words)


@pytest.mark.parametrize("n", [1, 255, 4096, 4097, 131072, 131073, 1300001])
def test_rays_of_a_long_query_are_each_their_own(scene, n):
    print(f"[copies] {n} rays", flush=True)
    rng = np.random.default_rng(n)
    rays = rng.uniform(-4, 4, (n, 6)).astype(np.float32)
    whole = scene.trace(rays)
    for at in {0, max(0, n - 300), n // 2}:  # by 300, traced in host memory
        part = scene.trace(rays[at:at + 300])
        assert part.tobytes() == whole[at:at + 300].tobytes()
    tail = scene.trace(rays[-300:], packet=True)
    assert tail.tobytes() == whole[-300:].tobytes()
