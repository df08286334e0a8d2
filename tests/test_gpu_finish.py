"""Paths run to their end in one launch (small calls, and the last paths of
larger ones) against the bounce-by-bounce launches, which a call that times its
kernels keeps: the same radiance of every path bit for bit, the same number of
rays and bounces. Path counts around a wave's 64 lanes, the launch's 2^18 and
the hand-over after some bounces; a queue smaller than the call; unsorted
shading; roulette and fixed depths; layered and batched scenes; 30 materials,
more than the LDS table holds and more than are sorted."""
import numpy as np
import pytest

from swpathtracer_amd import api, scenes
import swpathtracer_amd._lib as L

pytestmark = pytest.mark.gpu


def _same_bits(a, b):
    return np.array_equal(np.ascontiguousarray(a).view(np.uint32), np.ascontiguousarray(b).view(np.uint32))


@pytest.fixture(autouse=True)
def default_tuning(device):
    device.set_tuning()
    yield
    device.set_tuning()


def _render(device, sc, flags):
    device.set_scene(api.Bvh(sc.verts), sc.normals, sc.mat_ids)
    device.set_materials(sc.materials)
    img, paths = device.render_image(sc.camera, sc.integrator, per_path=True, extra_flags=flags)
    st = device.render_stats()
    return img, paths, (st["paths"], st["rays"], st["bounces"])


def _compare(device, sc, flags=0):
    img, paths, st = _render(device, sc, flags)
    img0, paths0, st0 = _render(device, sc, flags | L.SPT_RENDER_TIME_KERNELS)
    assert _same_bits(paths, paths0), f"{np.sum(np.any(paths != paths0, 1))} paths differ"
    assert st == st0
    np.testing.assert_allclose(img, img0, rtol=1e-5, atol=1e-6)  # film: atomics' order


@pytest.mark.parametrize("width,height,spp", [(1, 1, 1), (9, 7, 1), (64, 1, 1), (13, 5, 1), (97, 61, 1), (512, 512, 1),
                                              (511, 513, 1), (512, 513, 1), (300, 301, 16)])
@pytest.mark.parametrize("depth", [5, -1])
def test_path_counts(device, width, height, spp, depth):
    sc = scenes.cornell_icosphere(width=width, height=height, spp=spp, subdiv=2)
    if depth < 0:
        sc.integrator.termination, sc.integrator.path_length, sc.integrator.max_depth = "russian-roulette", 3, 16
    _compare(device, sc)


@pytest.mark.parametrize("capacity", [1000, 70_000, 1 << 18])
def test_queue_smaller_than_the_call(device, capacity):
    sc = scenes.cornell_icosphere(width=300, height=301, spp=4, subdiv=2)
    img0, paths0, st0 = _render(device, sc, L.SPT_RENDER_TIME_KERNELS)
    device.set_tuning(path_capacity=capacity)
    img, paths, st = _render(device, sc, 0)
    assert _same_bits(paths, paths0)
    assert st[:2] == st0[:2]


@pytest.mark.parametrize("flags", [0, L.SPT_RENDER_NO_SORT])
def test_layered_material(device, flags):
    _compare(device, scenes.mesh_in_box(rings=32, segments=64, width=320, height=240, spp=9), flags)


@pytest.mark.parametrize("n_mats", [30, 60, 1100])
def test_many_materials(device, n_mats):
    sc = scenes.cornell_icosphere(width=300, height=301, spp=4, subdiv=3)
    rng = np.random.default_rng(n_mats)
    kinds = [lambda: api.lambertian(tuple(rng.uniform(0.2, 0.9, 3))), lambda: api.ggx_conductor(float(rng.uniform(0.05, 0.5))),
             lambda: api.smooth_dielectric(float(rng.uniform(1.2, 1.8)))]
    n0 = len(sc.materials)
    sc.materials = sc.materials + [api.material([kinds[k % 3]()]) for k in range(n_mats - n0)]
    ids = np.array(sc.mat_ids)
    some = rng.random(len(ids)) < 0.7
    some[:12] = False  # the walls and the light
    ids[some] = rng.integers(n0, n_mats, size=int(some.sum()))
    sc.mat_ids = ids.astype(sc.mat_ids.dtype)
    _compare(device, sc)


def test_batches(device):
    scs = scenes.batch_scenes(n=5, seed=4, min_tris=500, max_tris=3000, min_side=120, max_side=200, spp_choices=(4, 9),
                              max_depth=8)
    b = api.Batch(device, scs, per_path=True)
    b.render()
    for i, sc in enumerate(scs):
        _, paths0, _ = _render(device, sc, L.SPT_RENDER_TIME_KERNELS)
        assert _same_bits(b.path_radiance(i), paths0)
    b.close()


def test_batch_of_layered_scenes(device):
    scs = [scenes.mesh_in_box(rings=16 + 4 * k, segments=32 + 8 * k, width=500 + 30 * k, height=300, spp=4, seed=k)
           for k in range(3)]
    b = api.Batch(device, scs, per_path=True)
    b.render()
    for i, sc in enumerate(scs):
        _, paths0, _ = _render(device, sc, L.SPT_RENDER_TIME_KERNELS)
        assert _same_bits(b.path_radiance(i), paths0)
    b.close()


def test_layered_materials_outside_the_table(device):
    """60 materials (read from memory, not LDS), all layered, in calls of bounces."""
    sc = scenes.mesh_in_box(rings=24, segments=48, width=400, height=400, spp=9)
    n0 = len(sc.materials)
    rng = np.random.default_rng(3)
    layered = next(m for m in sc.materials if m.n_layers > 1)
    sc.materials = list(sc.materials) + [layered] * (60 - n0)
    ids = np.array(sc.mat_ids)
    k = next(i for i, m in enumerate(sc.materials) if m.n_layers > 1)
    ids[ids == k] = rng.choice([k] + list(range(n0, 60)), size=int((ids == k).sum()))
    ref = scenes.mesh_in_box(rings=24, segments=48, width=400, height=400, spp=9)
    _, want, _ = _render(device, ref, 0)
    sc.mat_ids = ids.astype(sc.mat_ids.dtype)
    for flags in (0, L.SPT_RENDER_TIME_KERNELS):
        _, paths, _ = _render(device, sc, flags)
        assert _same_bits(paths, want)
