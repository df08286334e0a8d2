"""The number of paths up to which one launch runs them all to their end: calls
just below, at and above it, and queues of these sizes in larger calls, where the
last paths are handed over. Radiance bit for bit, rays and bounces as launched
bounce by bounce."""
import os
import re

import pytest

from swpathtracer_amd import scenes
import swpathtracer_amd._lib as L
from test_gpu_finish import _compare, _render, _same_bits, default_tuning  # noqa: F401

pytestmark = pytest.mark.gpu

SOURCE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "swpathtracer_amd", "csrc",
                      "spt_render.hip")
LIMIT = 1 << int(re.search(r"kFinishPaths = 1u << (\d+);", open(SOURCE).read()).group(1))


def _scene(pixels):
    """A scene whose image has exactly that many pixels."""
    h = next(k for k in (512, 256, 128, 64, 32, 16, 8, 7, 6, 5, 4, 3, 2, 1) if pixels % k == 0)
    sc = scenes.cornell_icosphere(width=pixels // h, height=h, spp=1, subdiv=2)
    sc.integrator.termination, sc.integrator.path_length, sc.integrator.max_depth = "russian-roulette", 3, 16
    return sc


@pytest.mark.parametrize("paths", [LIMIT - 1, LIMIT, LIMIT + 1])
def test_calls_around_the_limit(device, paths):
    _compare(device, _scene(paths))


@pytest.mark.parametrize("capacity", [LIMIT - 1, LIMIT, LIMIT + 1])
@pytest.mark.parametrize("use_graph", [1, 2])
def test_queues_around_the_limit(device, capacity, use_graph):
    sc = _scene(LIMIT + LIMIT // 2)
    _, paths0, st0 = _render(device, sc, L.SPT_RENDER_TIME_KERNELS)
    device.set_tuning(path_capacity=capacity, use_graph=use_graph)
    _, paths, st = _render(device, sc, 0)
    assert _same_bits(paths, paths0)
    assert st[:2] == st0[:2]
