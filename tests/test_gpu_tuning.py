"""The wavefronts a call runs, seen from its traversal launches, which calls that
time their kernels count over all wavefronts (one a bounce, and up to four more
by which the host runs ahead): a default call runs one, also once its reported
tuning has been set again."""
import pytest

from swpathtracer_amd import api, scenes
import swpathtracer_amd._lib as L

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def default_tuning(device):
    device.set_tuning()
    yield
    device.set_tuning()


def test_reported_tuning_set_again(device):
    # 6.3M paths: three wavefronts run where three are asked for
    sc = scenes.cornell_icosphere(width=256, height=256, spp=100, subdiv=2)
    sc.integrator.termination, sc.integrator.path_length, sc.integrator.max_depth = "russian-roulette", 3, 16
    device.set_scene(api.Bvh(sc.verts), sc.normals, sc.mat_ids)
    device.set_materials(sc.materials)

    def launches():
        device.render_image(sc.camera, sc.integrator, extra_flags=L.SPT_RENDER_TIME_KERNELS)
        return device.render_stats()["extend_launches"]

    one = launches()
    device.set_tuning(wavefronts=3)
    three = launches()
    assert three > 2 * one
    several = (one + three) / 2
    device.set_tuning(**device.get_tuning())  # three were asked for
    assert launches() > several
    device.set_tuning()
    t = device.get_tuning()
    assert t["wavefronts"] == 3
    device.set_tuning(**t)
    assert launches() < several and device.get_tuning() == t
    device.set_tuning(wavefronts=1)
    device.set_tuning(**{**t, "check_every": 8})
    assert launches() < several
