"""The four-lanes-per-ray traversal at the sizes where it can go wrong, ids and
t bit for bit against the oracle (acceleration/sbvh.cpp:478-515): blocks of
four and their remainders, large leaves, ray counts around the pool and the
share sizes, stacks deeper than the part in LDS, rays far from the scene and of
more than unit length (whose boxes are widened), coordinates past the
acceptance shortcut's range."""
import numpy as np
import pytest

import pyoracle as O
from swpathtracer_amd import api, scenes
import swpathtracer_amd._lib as L

pytestmark = pytest.mark.gpu


def _rays(rng, n, lo, hi, length=1.0):
    r = np.zeros((n, 8), np.float32)
    r[:, 0:3] = rng.uniform(lo, hi, (n, 3))
    d = rng.normal(size=(n, 3))
    r[:, 4:7] = length * d / np.linalg.norm(d, axis=1, keepdims=True)
    return r


def _aimed(rng, n, verts, distance, length=1.0):
    """Rays from `distance` away towards points of the primitives."""
    r = _rays(rng, n, -1, 1, 1.0)
    v = verts.reshape(-1, 3, 3)[rng.integers(len(verts), size=n)]
    b = rng.dirichlet([1, 1, 1], n).astype(np.float32)
    p = np.einsum("nk,nkc->nc", b, v)
    r[:, 0:3] = p - distance * r[:, 4:7]
    r[:, 4:7] *= length
    return r


def _check(device, verts, rays, kinds=None):
    device.set_scene(api.Bvh(verts, kinds=kinds))
    t, p = device.trace_host(rays)
    t_c, p_c, _, _ = O.Scene(verts, kinds=kinds).trace(rays)
    assert np.array_equal(p, p_c), f"{np.sum(p != p_c)} of {len(p)} ids differ"
    hit = p_c != L.SPT_MISS
    assert np.array_equal(t[hit].view(np.uint32), t_c[hit].view(np.uint32))
    assert np.all(np.isinf(t[~hit]))
    return hit.mean()


def _soup(rng, n, size, extent=1.0):
    c = rng.uniform(-extent, extent, (n, 1, 3))
    return (c + rng.uniform(-size, size, (n, 3, 3))).reshape(n, 9).astype(np.float32)


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 8, 9, 16, 17, 64, 65, 300])
def test_block_remainders(device, n):
    """n triangles about one centroid (one large leaf) and n spread ones."""
    rng = np.random.default_rng(n)
    nested = (rng.uniform(-1, 1, (n, 3, 3)) * np.linspace(0.2, 1.0, n)[:, None, None])
    nested -= nested.mean(1, keepdims=True)
    assert _check(device, nested.reshape(n, 9).astype(np.float32), _rays(rng, 5000, -1.2, 1.2)) > 0
    _check(device, _soup(rng, n, 0.4), _rays(rng, 5000, -1.2, 1.2))


@pytest.mark.parametrize("n_rays", [1, 2, 3, 4, 5, 31, 32, 33, 63, 64, 65, 127, 129, 4096, 30_001, 262_147])
def test_ray_counts(device, n_rays):
    rng = np.random.default_rng(n_rays)
    m = scenes.displaced_mesh(24, 48)
    r = _rays(rng, n_rays, -1.3, 1.3)
    r[:: 7, 0] = 9.0  # some miss the root box and never enter the pool
    _check(device, m.verts, r)


def test_deep_stacks(device):
    """Large overlapping triangles: a ray meets nearly every box on its way down."""
    rng = np.random.default_rng(5)
    assert _check(device, _soup(rng, 20_000, 1.0), _rays(rng, 300, -1, 1)) > 0.9


@pytest.mark.parametrize("distance,length", [(20.0, 1.0), (300.0, 1.0), (5000.0, 1.0), (2.0, 30.0), (2.0, 0.01),
                                             (40.0, 40.0)])
def test_far_and_scaled_rays(device, distance, length):
    rng = np.random.default_rng(int(distance * 10 + length))
    m = scenes.displaced_mesh(96, 192)
    assert _check(device, m.verts, _aimed(rng, 40_000, m.verts, distance, length)) > 0.5


@pytest.mark.parametrize("scale,offset", [(1.0, 3000.0), (2000.0, 0.0), (0.02, 1.0)])
def test_other_coordinate_ranges(device, scale, offset):
    rng = np.random.default_rng(8)
    v = (scenes.displaced_mesh(48, 96).verts * scale + offset).astype(np.float32)
    assert _check(device, v, _aimed(rng, 40_000, v, 2.0 * scale)) > 0.3


def test_axis_aligned_rays(device):
    """Zero direction components, origins on box planes of the root."""
    rng = np.random.default_rng(9)
    sc = scenes.cornell_icosphere(subdiv=3)
    r = _rays(rng, 30_000, -1, 1)
    axis = rng.integers(3, size=len(r))
    r[:, 4:7] = 0.0
    r[np.arange(len(r)), 4 + axis] = rng.choice([-1.0, 1.0], len(r))
    r[::3, 1] = -1.0
    _check(device, sc.verts, r)


@pytest.mark.parametrize("spheres,triangles", [(1, 0), (2, 0), (4, 0), (1, 3), (0, 4), (2, 3)])
@pytest.mark.parametrize("distance", [3.0, 5000.0])
def test_scenes_of_one_block(device, spheres, triangles, distance):
    """Up to four primitives are tested without a tree (five with one)."""
    rng = np.random.default_rng(10 * spheres + triangles)
    n = spheres + triangles
    v = _soup(rng, n, 0.6)
    kinds = np.zeros(n, np.uint32)
    kinds[:spheres] = L.SPT_PRIM_SPHERE
    v[:spheres, 3:] = 0.0
    v[:spheres, 3] = rng.uniform(0.3, 0.9, spheres)
    for n_rays in (1, 255, 257, 70_001):
        r = _rays(rng, n_rays, -1, 1)
        r[:, 0:3] -= np.float32(distance) * r[:, 4:7]
        r[::9, 0:3] = rng.uniform(-0.3, 0.3, r[::9, 0:3].shape)
        r[::101, 5] = np.nan
        _check(device, v, r, kinds=kinds)


@pytest.mark.parametrize("width, height", [(1, 1), (3, 5), (4, 4), (17, 2), (131, 67)])
def test_count_caster_at_ragged_sizes(device, width, height):
    """Tiles of 4 x 4 pixels and their remainders, stacks in LDS only and beyond
    it, a scene whose root is a leaf. Counts are whole numbers: equal."""
    cam = dict(position=(0.2, 0.3, 2.5), look_at=(0, 0, 0), fov=50.0)
    mesh = scenes.displaced_mesh(rings=48, segments=96)
    rng = np.random.default_rng(width * 1000 + height)
    # long thin overlapping triangles: rays meet most boxes of the tree
    heap = rng.uniform(-1, 1, (600, 3, 3)).astype(np.float32)
    for verts in (mesh.verts, heap, mesh.verts.reshape(-1, 3, 3)[:2]):
        device.set_scene(api.Bvh(verts))
        c = api.pinhole(width, height, **cam)
        assert np.array_equal(device.raycast(c, L.SPT_RAYCAST_COUNT), O.Scene(verts).raycast(c, 2))


@pytest.mark.parametrize("width, height", [(1024, 1024), (1031, 1025)])
def test_count_caster_around_the_pixel_limit(device, width, height):
    """A small tree just below and above the size from which a lane counts a ray."""
    verts = scenes.displaced_mesh(rings=12, segments=24).verts
    device.set_scene(api.Bvh(verts))
    c = api.pinhole(width, height, position=(0.2, 0.3, 2.5), look_at=(0, 0, 0), fov=50.0)
    assert np.array_equal(device.raycast(c, L.SPT_RAYCAST_COUNT), O.Scene(verts).raycast(c, 2))


@pytest.mark.parametrize("n_spheres, n_tris", [(1, 9), (9, 3), (6, 40)])
@pytest.mark.parametrize("length", [0.5, 1.0, 3.0])
def test_spheres_in_large_leaves(device, n_spheres, n_tris, length):
    """With directions that are not of unit length the sphere test accepts hit
    points off the sphere, anywhere in its leaf's box: a leaf's parts that hold
    spheres keep that box. Equal centroids make one leaf of all of them."""
    rng = np.random.default_rng(100 * n_spheres + n_tris)
    verts = np.zeros((n_spheres + n_tris, 9), np.float32)
    kinds = np.zeros(n_spheres + n_tris, np.uint32)
    verts[:n_spheres, 3] = rng.uniform(0.02, 0.3, n_spheres)
    kinds[:n_spheres] = L.SPT_PRIM_SPHERE
    a, b = rng.uniform(-1, 1, (2, n_tris, 3))
    verts[n_spheres:] = np.concatenate([a, b, -a - b], axis=1)
    hit = _check(device, verts, _rays(rng, 20000, -2, 2, length), kinds)
    assert 0.0 < hit < 1.0
    # the same beside a distant group, so that the leaf is not the root
    far = verts.copy()
    far[:n_spheres, 0:3] += 8
    far[n_spheres:] += 8
    rays = _rays(rng, 20000, -2, 2, length)
    rays[::2, 0:3] += 8
    _check(device, np.concatenate([verts, far]), rays, np.concatenate([kinds, kinds]))


@pytest.mark.parametrize("n", [1, 4, 7])
@pytest.mark.parametrize("length", [0.5, 1.0, 3.0])
def test_spheres_in_a_root_leaf(device, n, length):
    """The root's box has no padding: a hit point accepted off the sphere does
    not mean that the ray meets it. Many rays pass close to the box."""
    rng = np.random.default_rng(n)
    verts = np.zeros((n, 9), np.float32)
    verts[:, 3] = rng.uniform(0.2, 0.5, n)
    kinds = np.full(n, L.SPT_PRIM_SPHERE, np.uint32)
    _check(device, verts, _rays(rng, 400000, -1, 1, length), kinds)
