"""GPU: the nearest-first search of the SAH tree against the oracle's
traversal in the reference's order, on scenes made to tell them apart: exact
ties, flat axis-aligned boxes, coordinates far from the origin, centres that
cannot be split, one-primitive trees, and arrays whose boxes are not nested
(which keep the reference's order). Hits are equal bit for bit."""
import copy

import numpy as np
import pytest

import oracle_lib as O
import zig_ornament_amd as zo
from helpers import ray_set
from zig_ornament_amd import workloads as W

pytestmark = pytest.mark.gpu

GREY = [("lambertian", (0.5, 0.5, 0.5), None), ("lambertian", (0.2, 0.3, 0.4), None)]


def _spec(name, spheres=(), instances=0, at=(0.0, 0.0, 0.0), span=4.0, eye=8.0):
    at = np.asarray(at, np.float64)
    spec = W.SceneSpec(name, 64, 64, 1, 4, camera=(tuple(at + (0, 1, -eye)), tuple(at), (0, 1, 0), 1.0, 50.0, 0.0,
                                                   eye))
    spec.materials = list(GREY)
    spec.spheres = [(tuple(float(x) for x in at + np.asarray(c)), r, i % 2) for i, (c, r) in enumerate(spheres)]
    if instances:
        verts, vi, normals, ni, uvs, ui = W.icosphere_mesh(2)
        m = W.mat_translation(*at)
        spec.meshes.append(("mesh", verts, vi, normals, ni, uvs, ui, m, 0))
        rng = np.random.default_rng(5)
        for k in range(instances):
            spec.instances.append((0, W.mat_translation(*(at + rng.uniform(-span, span, 3))), k % 2))
    return spec


def _grid(n, step=1.0, r=0.4):
    i = np.arange(n) - n // 2
    return [((float(x) * step, float(y) * step, float(z) * step), r) for x in i for y in i for z in i]


def _triangle():
    spec = _spec("triangle")
    v = np.array([[-1, -1, 0, 1], [1, -1, 0, 1], [0, 1, 0, 1]], np.float32)
    n = np.array([[0, 0, -1, 0]], np.float32)
    uv = np.zeros((1, 2), np.float32)
    z = np.zeros(3, np.uint32)
    spec.meshes = [("mesh", v, np.arange(3, dtype=np.uint32), n, z, uv, z, np.eye(4, dtype=np.float32), 0)]
    return spec


def specs():
    twins = _spec("twins", _grid(3) * 2, instances=6)
    twins.instances += [(m, t, 1 - k) for m, t, k in twins.instances]  # every instance twice, at the same place
    return {
        "twins": twins,                                            # every hit is a tie
        "walls": W.cornell(),                                      # flat boxes: t lies on the box
        "grid": _spec("grid", _grid(6, 1.0, 0.5)),                 # touching spheres, equal centres per axis
        "chain": _spec("chain", [((2.0 ** (i - 12), 0.0, 0.0), 2.0 ** (i - 14)) for i in range(24)], eye=3000.0),
        "concentric": _spec("concentric", [((0.0, 0.0, 0.0), 0.1 + 0.05 * i) for i in range(40)]),  # median splits only
        "far": _spec("far", _grid(4, 1.5, 0.4), instances=12, at=(4096.0, -2048.0, 8192.0)),
        "sphere": _spec("sphere", [((0.0, 0.0, 0.0), 1.0)]),
        "triangle": _triangle(),
        "ground": W.random_spheres(64, 64, 1, 4, grid=range(-3, 3)),
    }


def _rays(spec, arrays, seed):
    rng = np.random.default_rng(seed)
    rays = ray_set(spec, arrays, 6000, seed)
    eye = np.array(spec.camera[0], np.float64)
    at = np.array(spec.camera[1], np.float64)
    targets = np.array([c for c, _, _ in spec.spheres] or [at], np.float64)
    for entry in spec.meshes:
        if entry[0] == "mesh":  # shared vertices and edge midpoints of the base mesh
            v = entry[1][:, :3] + np.asarray(entry[7])[3, :3]
            targets = np.concatenate([targets, v, 0.5 * (v[:-1] + v[1:])])
    aim = targets[rng.integers(0, len(targets), 3000)] + rng.choice([0.0, 0.0, 0.25, 1.0], (3000, 3))
    axis = np.zeros((3000, 3))
    axis[np.arange(3000), rng.integers(0, 3, 3000)] = rng.choice([-1.0, 1.0, 0.01], 3000)
    near = np.concatenate([aim - 7.0 * axis, axis], 1)               # axis-parallel, through centres and vertices
    straight = np.concatenate([np.broadcast_to(eye, aim.shape), aim - eye], 1)
    inside = np.concatenate([aim, rng.normal(size=aim.shape)], 1)    # starting on centres and surfaces
    return np.concatenate([rays, near, straight, inside]).astype(np.float32)


def _compare(device, arrays, oracle_arrays, rays, t_min):
    g = zo.DeviceScene(device, arrays).trace(rays, t_min)
    o = O.OracleScene(oracle_arrays).trace(rays, t_min)
    assert np.array_equal(g["hit"], o["hit"])
    h = o["hit"] == 1
    for f in ["material_index", "node_type", "inverted_transform_id"]:
        assert np.array_equal(g[f][h], o[f][h]), f
    assert np.array_equal(g["t"][h].view(np.uint32), o["t"][h].view(np.uint32))
    m = h & (o["node_type"] == 2)
    assert np.array_equal(g["tri_id"][m], o["tri_id"][m])
    assert np.array_equal(g["uv"][m].view(np.uint32), o["uv"][m].view(np.uint32))
    return h.mean()


@pytest.mark.parametrize("t_min", [0.001, 0.0, -3.0])
@pytest.mark.parametrize("name", sorted(specs()))
def test_closest_hits_are_the_references(device, name, t_min):
    spec = specs()[name]
    arrays = zo.Bvh(W.build_scene(spec))
    rays = _rays(spec, arrays, seed=11)
    print(f"[search] {name} t_min {t_min}: {len(rays)} rays", flush=True)
    assert _compare(device, arrays, O.build_bvh(spec), rays, t_min) > 0.05


@pytest.mark.parametrize("change", ["shrunk", "infinite", "triangle"])
def test_boxes_that_are_not_nested_keep_the_references_order(device, change):
    """A box smaller than what is below it hides primitives from the reference;
    only its own order and boxes give its hits."""
    spec = _spec("nested", _grid(3), instances=8)
    arrays = zo.Bvh(W.build_scene(spec))
    rays = _rays(spec, arrays, seed=3)
    arrays = copy.copy(arrays)
    if change == "triangle":
        inner = np.nonzero(arrays.blas_nodes["node_type"] == 0)[0]
        leaf = [i for i in inner if arrays.blas_nodes["node_type"][arrays.blas_nodes["left_or_custom_id"][i]] == 3]
        arrays.blas_nodes["lmax_or_v1"][leaf[::3]] -= np.float32(0.05)
    else:
        inner = np.nonzero(arrays.tlas_nodes["node_type"] == 0)[0]
        arrays.tlas_nodes["rmax_or_v3"][inner[::4]] += np.float32(-0.3 if change == "shrunk" else np.inf)
    print(f"[search] {change}: {len(rays)} rays", flush=True)
    assert _compare(device, arrays, arrays, rays, 0.001) > 0.05


def test_spheres_with_any_transform_keep_the_whole_matrix(device):
    """One sheared, rotated or mirrored sphere among them sends every sphere
    leaf through its whole matrix."""
    spec = _spec("sheared", _grid(3))
    arrays = zo.Bvh(W.build_scene(spec))
    rays = _rays(spec, arrays, seed=9)
    plain = _compare(device, arrays, arrays, rays, 0.001)
    arrays = copy.copy(arrays)
    arrays.transforms[8, 4] += np.float32(0.25)  # off the diagonal of a leaf's inverse
    arrays.transforms[10, 0] *= np.float32(-1.0)
    print(f"[search] sheared: {len(rays)} rays", flush=True)
    assert plain > 0.05 and _compare(device, arrays, arrays, rays, 0.001) > 0.05
    assert _compare(device, arrays, arrays, rays, 0.0) > 0.05
