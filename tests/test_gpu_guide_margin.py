"""The training gradient at record counts that end inside a tile of 128 (1000 =
7 * 128 + 104), with records for which every ReLU's side is certain, against the
oracle. Two factors of a product are bf16, and a different fp32 summation order
can flip the rounding of either (2^-8 of it): a layer's gradient is allowed 2^-7
of its norm. Such a flip moves a pre-activation by at most 2^-8 |input| |weight|,
about 5e-4 here: records with one within 2^-8 of 0 are left out."""
import numpy as np
import pytest

import guide_ref as G
from test_gpu_guide import _encode, _records, _theta, box_scene  # noqa: F401

pytestmark = pytest.mark.gpu


def _certain(theta, rng, n, bmin, bext):
    rec = _records(rng, 40 * n, bmin, bext)
    _, (_, a1, _, a2, _, a3, _) = G.forward(theta, _encode(rec, bmin, bext))
    clear = np.minimum.reduce([np.abs(a).min(1) for a in (a1, a2, a3)]) > 2.0 ** -8
    assert clear.sum() >= n
    return rec[clear][:n]


@pytest.mark.parametrize("n", [104, 999, 1000, 1001])
def test_gradient_of_certain_units(device, box_scene, n):  # noqa: F811
    _, bmin, bext = box_scene
    device.guide_init(seed=5)
    theta = _theta(12, out_scale=3.0)
    device.guide_set_params(theta)
    rec = _certain(theta, np.random.default_rng(n), n, bmin, bext)
    g, loss = device.guide_gradient(rec)
    r = rec.astype(np.float64)
    loss_r, g_r = G.batch_grad(theta, _encode(rec, bmin, bext), r[:, 9:12], r[:, 12], loss_scale=65536.0)
    assert abs(loss - loss_r) <= 2.0 ** -7 * max(abs(loss_r), 1.0)
    gp, gr = G.unpack(g.astype(np.float64)), G.unpack(g_r)
    for name, _ in G.SHAPES:
        a, b = gp[name].ravel(), gr[name].ravel()
        assert np.linalg.norm(a - b) <= 2.0 ** -7 * np.linalg.norm(b) + 1e-12, name
    assert np.all(g[G._pad_mask()] == 0.0)
