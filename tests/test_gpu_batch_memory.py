"""What a batch keeps on the device: the four-wide tree with its triangle
blocks and leaf boxes, and the shading records."""
import pytest

from swpathtracer_amd import api, scenes

pytestmark = pytest.mark.gpu


def test_bytes_per_triangle(device):
    """Per triangle 48 B of shading, 48 B in a block of four (3.5 of its places
    are used on average), about 0.14 nodes of 64 B and half a leaf box of 32 B:
    some 130 B. The binary tree and its triangles, which no kernel of a batch
    reads, would add 48 B and 64 B a binary node."""
    scs = scenes.batch_scenes(n=3, seed=4, min_tris=20_000, max_tris=60_000, min_side=32, max_side=48, spp_choices=(1,),
                              max_depth=3)
    b = api.Batch(device, scs)
    b.render()
    st, _ = b.stats()
    tris = sum(len(sc.verts) for sc in scs)
    assert st["triangles"] == tris
    assert 100 * tris < st["device_bytes"] < 150 * tris
    b.close()
