"""GPU: closest hits of rays that graze what they hit, where rounding puts a
hit far from its box: rays nearly in the plane of a triangle (the reference
tests no determinant), nearly along a face of a rotated box (its slab distances
are large numbers' differences) and nearly tangent to a sphere. Plain queries
(nearest first) against packet queries, which take the reference's order, over
a million rays of each kind, and both against the oracle on the first ones.
Equal bit for bit."""
import numpy as np
import pytest

import oracle_lib as O
import zig_ornament_amd as zo
from zig_ornament_amd import workloads as W

pytestmark = pytest.mark.gpu

N = 1 << 20


def box_mesh(n):
    """The faces of [-1, 1]^3 in n x n squares of two triangles each."""
    g = np.linspace(-1.0, 1.0, n + 1)
    verts, tris = [], []
    for axis in range(3):
        for side in (-1.0, 1.0):
            first = len(verts)
            for a in g:
                for b in g:
                    p = np.ones(4)
                    p[(axis + 1) % 3], p[(axis + 2) % 3], p[axis] = a, b, side
                    verts.append(p)
            for i in range(n):
                for j in range(n):
                    k = first + i * (n + 1) + j
                    tris += [k, k + 1, k + n + 2, k, k + n + 2, k + n + 1]
    return np.array(verts, np.float32), np.array(tris, np.uint32)


def wall_mesh(n):
    verts, tris = box_mesh(n)
    one = (n + 1) ** 2
    return verts[:one], tris[: 6 * n * n]


def ring_mesh(n, m):
    """A torus: triangle planes of it pass through its middle."""
    a, b = np.meshgrid(2 * np.pi * np.arange(n) / n, 2 * np.pi * np.arange(m) / m, indexing="ij")
    r = 1.0 + 0.4 * np.cos(b)
    verts = np.stack([r * np.cos(a), 0.4 * np.sin(b), r * np.sin(a), np.ones_like(a)], -1).reshape(-1, 4)
    i, j = np.meshgrid(np.arange(n), np.arange(m), indexing="ij")
    k00, k01 = i * m + j, i * m + (j + 1) % m
    k10, k11 = (i + 1) % n * m + j, (i + 1) % n * m + (j + 1) % m
    return verts.astype(np.float32), np.stack([k00, k01, k11, k00, k11, k10], -1).reshape(-1).astype(np.uint32)


def mesh_spec(mesh, count, box, seed):
    """Instances of a mesh, scaled, turned any way and placed in a box."""
    rng = np.random.default_rng(seed)
    verts, vi = mesh
    spec = W.SceneSpec("turned", 64, 64, 1, 4, camera=((0, 1, -9), (0, 0, 0), (0, 1, 0), 1.0, 50.0, 0.0, 9.0))
    spec.materials = [("lambertian", (0.5, 0.5, 0.5), None)]
    mats = []
    for _ in range(count):
        q = rng.normal(size=4)
        k = rng.uniform(0.5, 2.0)
        mats.append(W.mat_mul(W.mat_mul(W.mat_scaling(k, k, k), W.mat_from_quat(q / np.linalg.norm(q))),
                              W.mat_translation(*rng.uniform(-box / 2, box / 2, 3))))
    z = np.zeros(len(vi), np.uint32)
    spec.meshes.append(("mesh", verts, vi, np.array([[0, 0, 1, 0]], np.float32), z, np.zeros((1, 2), np.float32), z,
                        mats[0], 0))
    spec.instances = [(0, m, 0) for m in mats[1:]]
    world = verts[vi].reshape(-1, 3, 4).astype(np.float64)[None] @ np.array(mats, np.float64)[:, None]
    return spec, world.reshape(-1, 3, 4)[:, :, :3]


def mesh_rays(tris, lean, seed):
    """Rays through points of triangles, `lean(rng)` off their plane."""
    rng = np.random.default_rng(seed)
    t = tris[rng.integers(0, len(tris), N)]
    b = rng.random((N, 3))
    b[: N // 4, 0] = 0.0  # on an edge
    p = ((b / b.sum(1, keepdims=True))[:, :, None] * t).sum(1)
    n = np.cross(t[:, 1] - t[:, 0], t[:, 2] - t[:, 0])
    n /= np.linalg.norm(n, axis=1, keepdims=True)
    d = rng.normal(size=(N, 3))
    d -= (d * n).sum(1, keepdims=True) * n
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    d += (lean(rng) * rng.choice([-1.0, 1.0], N))[:, None] * n
    return np.concatenate([p - 10.0 ** rng.uniform(-3, 1, (N, 1)) * d, d], 1).astype(np.float32)


def sphere_spec(centres, radii):
    spec = W.SceneSpec("spheres", 64, 64, 1, 4, camera=((0, 1, -9), (0, 0, 0), (0, 1, 0), 1.0, 50.0, 0.0, 9.0))
    spec.materials = [("lambertian", (0.5, 0.5, 0.5), None)]
    spec.spheres = [(tuple(float(x) for x in c), float(r), 0) for c, r in zip(centres, radii)]
    return spec


def sphere_rays(centres, radii, seed):
    """Rays nearly tangent to spheres, where those touch their boxes and elsewhere."""
    rng = np.random.default_rng(seed)
    i = rng.integers(0, len(radii), N)
    n = rng.normal(size=(N, 3)) * 10.0 ** rng.uniform(-5, 0, (N, 1))
    n[np.arange(N), rng.integers(0, 3, N)] += rng.choice([-1.0, 1.0], N)
    n /= np.linalg.norm(n, axis=1, keepdims=True)
    p = centres[i] + n * (radii[i] * (1.0 + rng.choice([-1.0, 0.0, 1.0], N) * 10.0 ** rng.uniform(-8, -2, N)))[:, None]
    d = rng.normal(size=(N, 3))
    d -= (d * n).sum(1, keepdims=True) * n
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    d += (rng.choice([-1.0, 0.0, 1.0], N) * 10.0 ** rng.uniform(-8, -1, N))[:, None] * n
    far = np.where(rng.random(N) < 0.5, 10.0 ** rng.uniform(-4, 1, N) * radii[i], 10.0 ** rng.uniform(-1, 2, N))
    return np.concatenate([p - far[:, None] * d, d], 1).astype(np.float32)


def differing(a, b):
    """Where two sets of hits are not the same bits."""
    ne = a["hit"] != b["hit"]
    h = b["hit"] == 1
    for f in ["material_index", "node_type", "inverted_transform_id", "t"]:
        ne |= h & (a[f].view(np.uint32) != b[f].view(np.uint32))
    m = h & (b["node_type"] == 2)
    ne |= m & ((a["tri_id"] != b["tri_id"]) | (a["uv"].view(np.uint32) != b["uv"].view(np.uint32)).any(1))
    return ne


def check(device, arrays, oracle_arrays, rays, t_min=0.001):
    scene = zo.DeviceScene(device, arrays)
    near, packet = scene.trace(rays, t_min), scene.trace(rays, t_min, packet=True)
    ne = differing(near, packet)
    few = np.concatenate([np.nonzero(ne)[0][:100], np.arange(3000)])  # disagreements, and a sample
    oracle = O.OracleScene(oracle_arrays).trace(rays[few], t_min)
    assert not differing(packet[few], oracle).any()
    assert not differing(near[few], oracle).any()
    assert not ne.any(), int(ne.sum())
    return packet["hit"].mean()


def in_plane(rng):
    return rng.choice([0.0, 1e-7, 1e-6, 1e-5, 1e-4], N)


def grazing(rng):
    return 10.0 ** rng.uniform(-6, 0, N)


MESHES = {
    "box": lambda: mesh_spec(box_mesh(1), 6, 3.0, 1),           # faces of two triangles
    "boxes": lambda: mesh_spec(box_mesh(1), 2000, 20.0, 2),
    "tiles": lambda: mesh_spec(box_mesh(6), 300, 20.0, 3),      # flat faces of many triangles
    "walls": lambda: mesh_spec(wall_mesh(4), 400, 16.0, 4),     # open: the core lies in front of them
    "ring": lambda: mesh_spec(ring_mesh(24, 12), 3, 3.0, 6),    # no core: searched whole
    "rings": lambda: mesh_spec(ring_mesh(24, 12), 60, 9.0, 7),  # many of them: the reference's order
    "balls": lambda: mesh_spec(W.icosphere_mesh(3)[:2], 200, 12.0, 5),
}


@pytest.mark.parametrize("lean", [grazing, in_plane])
@pytest.mark.parametrize("name", sorted(MESHES))
def test_rays_along_triangles_hit_what_the_reference_hits(device, name, lean):
    spec, tris = MESHES[name]()
    rays = mesh_rays(tris, lean, seed=7)
    print(f"[grazing] {name}, {lean.__name__}: {len(rays)} rays", flush=True)
    assert check(device, zo.Bvh(W.build_scene(spec)), O.build_bvh(spec), rays) > 0.3


def test_rays_along_triangles_beside_spheres(device):
    spec, tris = mesh_spec(box_mesh(2), 200, 16.0, 6)
    rng = np.random.default_rng(8)
    spec.spheres = [(tuple(float(x) for x in rng.uniform(-8, 8, 3)), float(rng.uniform(0.2, 1.0)), 0)
                    for _ in range(200)]
    rays = mesh_rays(tris, grazing, seed=9)
    print(f"[grazing] boxes and spheres: {len(rays)} rays", flush=True)
    assert check(device, zo.Bvh(W.build_scene(spec)), O.build_bvh(spec), rays) > 0.3


@pytest.mark.parametrize("name", ["apart", "touching", "ground", "far"])
def test_rays_along_spheres_hit_what_the_reference_hits(device, name):
    rng = np.random.default_rng(11)
    centres, radii = rng.uniform(-10, 10, (1000, 3)), 10.0 ** rng.uniform(-2, 0, 1000)
    if name == "touching":
        i = np.arange(8.0)
        centres, radii = np.stack(np.meshgrid(i, i, i), -1).reshape(-1, 3), np.full(512, 0.5)
    elif name == "ground":
        centres, radii = np.concatenate([centres, [[0.0, -1000.0, 0.0]]]), np.append(radii, 995.0)
    elif name == "far":
        centres = centres + (4096.0, -2048.0, 8192.0)
    spec = sphere_spec(centres, radii)
    rays = sphere_rays(centres, radii, seed=12)
    print(f"[grazing] spheres {name}: {len(rays)} rays", flush=True)
    assert check(device, zo.Bvh(W.build_scene(spec)), O.build_bvh(spec), rays) > 0.2
