"""GPU: scenes that keep the reference's search order run other kernels than
scenes of the same size with a search tree, and are tuned apart from them."""
import copy
import json

import numpy as np
import pytest

import zig_ornament_amd as zo
from helpers import zo_params
from zig_ornament_amd import workloads as W

pytestmark = pytest.mark.gpu


def test_search_order_is_part_of_the_tuning_class(device, tmp_path):
    spec = W.random_spheres(48, 32, 1, 3, grid=range(-2, 2))
    arrays = zo.Bvh(W.build_scene(spec))
    shrunk = copy.copy(arrays)
    shrunk.tlas_nodes = np.array(arrays.tlas_nodes)
    inner = np.nonzero(shrunk.tlas_nodes["node_type"] == 0)[0]
    shrunk.tlas_nodes["rmax_or_v3"][inner[::4]] -= np.float32(0.1)  # no longer nested: no search tree
    cache, p = str(tmp_path / "tuning.json"), zo_params(spec)
    for a in (arrays, shrunk):
        print("[tuning] autotune", flush=True)
        zo.Target(zo.DeviceScene(device, a), spec.width, spec.height).autotune(p, spec.spp, cache_path=cache)
    keys = sorted(json.load(open(cache)))
    assert len(keys) == 2 and keys[1] == keys[0] + "|unordered"
    shipped = json.load(open(zo.TUNING_CACHE))
    assert not any(k.endswith("|unordered") for k in shipped)  # its classes are scenes with one
