"""GPU: closest hits where transforms were moved, turned or sheared under kept
boxes, so that boxes no longer hold what is in them. Uploads take such arrays;
the hits are those of the reference's order over the same boxes. Plain queries
(nearest first) against packet queries, which take the reference's order, and
both against the oracle where they differ and on a sample. Bit for bit."""
import copy

import numpy as np
import pytest

import zig_ornament_amd as zo
from test_gpu_grazing_rays import box_mesh, check, mesh_spec, sphere_spec
from zig_ornament_amd import workloads as W

pytestmark = pytest.mark.gpu


def change(arrays, how, seed):
    """New transforms (and their inverses) under the same boxes. A stored matrix
    is its columns, one after the other: as rows of an array it acts from the right."""
    rng = np.random.default_rng(seed)
    m = np.asarray(arrays.transforms, np.float64).reshape(-1, 4, 4).copy()
    for k in range(1, len(m), 2):
        if how == "moved":
            m[k, 3, :3] += rng.uniform(-0.5, 0.5, 3) * np.linalg.norm(m[k, 0, :3])
        elif how == "sheared":
            m[k, :3, :3] = m[k, :3, :3] @ (np.eye(3) + 0.25 * rng.normal(size=(3, 3)))
        else:  # flattened, and turned
            q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
            m[k, :3, :3] = np.diag([1.0, 0.2, 1.5]) @ m[k, :3, :3] @ q
        m[k - 1] = np.linalg.inv(m[k])
    arrays = copy.copy(arrays)
    arrays.transforms = m.astype(np.float32).reshape(np.shape(arrays.transforms))
    return arrays


def rays_through(lo, hi, n, seed):
    rng = np.random.default_rng(seed)
    a = rng.uniform(lo, hi, (n, 3))
    return np.concatenate([a, rng.uniform(lo, hi, (n, 3)) - a], 1).astype(np.float32)


@pytest.mark.parametrize("how", ["moved", "sheared", "flattened"])
@pytest.mark.parametrize("what", ["spheres", "meshes", "both"])
def test_boxes_that_leave_out_what_is_in_them(device, what, how):
    rng = np.random.default_rng(3)
    centres, radii = rng.uniform(-8, 8, (600, 3)), rng.uniform(0.2, 1.0, 600)
    if what == "spheres":
        spec = sphere_spec(centres, radii)
    else:
        spec, _ = mesh_spec(box_mesh(2), 150, 16.0, 4)
        if what == "both":
            spec.spheres = [(tuple(map(float, c)), float(r), 0) for c, r in zip(centres[:200], radii)]
    arrays = change(zo.Bvh(W.build_scene(spec)), how, seed=5)
    rays = rays_through(-9.0, 9.0, 1 << 20, seed=6)
    print(f"[boxes] {what} {how}: {len(rays)} rays", flush=True)
    assert check(device, arrays, arrays, rays) > 0.3


def test_a_sphere_without_an_inverse(device):
    """A flat transform among the spheres: nothing bounds its distances."""
    rng = np.random.default_rng(7)
    spec = sphere_spec(rng.uniform(-4, 4, (40, 3)), rng.uniform(0.2, 1.0, 40))
    arrays = copy.copy(zo.Bvh(W.build_scene(spec)))
    m = np.array(arrays.transforms, np.float32).reshape(-1, 4, 4)
    m[8, :, 2] = 0.0  # an inverse that drops one axis
    arrays.transforms = m.reshape(np.shape(arrays.transforms))
    rays = rays_through(-5.0, 5.0, 1 << 18, seed=8)
    print(f"[boxes] flat: {len(rays)} rays", flush=True)
    assert check(device, arrays, arrays, rays) > 0.1
