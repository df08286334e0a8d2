"""The four-wide tree and triangle blocks that the traversal reads
(swpathtracer_amd/csrc/quad_tree.cpp, compiled here for the host): every
primitive lies in one block, every box as the device decodes it holds what a ray
may hit below it, and no ray needs more stack than the tree reports."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from swpathtracer_amd import api, scenes
import swpathtracer_amd._lib as L
from test_host_build import _scenes as host_scenes

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "swpathtracer_amd", "csrc")
REC = np.dtype([("v0", "<f4", 3), ("e1", "<f4", 3), ("e2", "<f4", 3), ("prim", "<u4"), ("mat", "<u4"), ("kind", "<u4")])
NONE, LEAF, SPHERE, EXACT = 0xFFFFFFFF, 0x80000000, 0x80000000, 0x80000000
SOURCE = """
#include <cstring>
#include "quad_tree.h"
static spt::QuadTree tree;
extern "C" {
void q_clear() { tree = spt::QuadTree(); }
unsigned q_append(const spt_node64* n, unsigned nn, const spt_tri48* t, unsigned nt, const float* box, unsigned base) {
    return spt::append_quad_tree(n, nn, t, nt, box, base, tree);
}
void q_sizes(unsigned* s) {
    s[0] = (unsigned)tree.nodes.size();
    s[1] = (unsigned)tree.prims.size();
    s[2] = (unsigned)tree.boxes.size();
}
void q_read(void* n, void* p, void* b) {
    std::memcpy(n, tree.nodes.data(), tree.nodes.size() * sizeof(spt::QuadNode));
    std::memcpy(p, tree.prims.data(), tree.prims.size() * sizeof(spt::QuadPrim));
    std::memcpy(b, tree.boxes.data(), tree.boxes.size() * sizeof(spt::QuadBox));
}
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("quad")
    (d / "q.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-shared", "-fPIC", "-I", CSRC, "-I",
                    os.path.join(ROOT, "include"), str(d / "q.cpp"), os.path.join(CSRC, "quad_tree.cpp"), "-o",
                    str(d / "q.so")], check=True)
    lib = C.CDLL(str(d / "q.so"))
    lib.q_append.argtypes = [C.c_void_p, C.c_uint, C.c_void_p, C.c_uint, C.c_void_p, C.c_uint]
    lib.q_append.restype = C.c_uint
    lib.q_sizes.argtypes = [C.c_void_p]
    lib.q_read.argtypes = [C.c_void_p] * 3
    return lib


def _read(lib):
    n = np.zeros(3, np.uint32)
    lib.q_sizes(n.ctypes.data)
    out = [np.zeros((n[0], 16), np.uint32), np.zeros((n[1] // 4, 4, 12), np.uint32), np.zeros((n[2], 8), np.float32)]
    lib.q_read(*[a.ctypes.data for a in out])
    return out


def _append(lib, nodes, tris, box, base=0):
    """Stack bound of the tree appended, and the arrays of all trees so far."""
    cap = lib.q_append(nodes.ctypes.data if len(nodes) else None, len(nodes), tris.ctypes.data, len(tris),
                       box.ctypes.data, base)
    return cap, _read(lib)


def _decode(node):
    """Child bounds (4, 2, 3) in float64: origin + byte * step, the step of axis a
    the word shifted left by 9 a, read as a float, times 2^-24."""
    org = node[0:3].view(np.float32).astype(np.float64)
    step = [float(np.array([(int(node[3]) << (9 * a)) & 0xFFFFFFFF], np.uint32).view(np.float32)[0]) / 2.0 ** 24
            for a in range(3)]
    out = np.zeros((4, 2, 3))
    for c in range(4):
        xy, z = int(node[4 + 3 * c]), int(node[5 + 3 * c])
        q = [[xy & 255, (xy >> 16) & 255, z & 255], [(xy >> 8) & 255, xy >> 24, (z >> 8) & 255]]
        for side in range(2):
            out[c, side] = org + np.array(q[side]) * step
    return out


def _leaves(nodes, tris, box):
    if len(nodes) == 0:
        return [(0, len(tris), box[:3].astype(np.float64), box[3:].astype(np.float64))]
    return [(int(nd[s + "ref"]), int(nd[s + "cnt"]), nd[s + "min"].astype(np.float64), nd[s + "max"].astype(np.float64))
            for nd in nodes for s in ("l", "r") if nd[s + "cnt"] > 0]


def _extent(tris):
    """Bounds of every primitive and which are spheres."""
    v0, e1, e2 = (tris[f].astype(np.float64) for f in ("v0", "e1", "e2"))
    sphere = tris["kind"] == L.SPT_PRIM_SPHERE
    v = np.stack([v0, v0 + e1, v0 + e2])
    r = np.abs(e1[:, 0:1])
    return np.where(sphere[:, None], v0 - r, v.min(0)), np.where(sphere[:, None], v0 + r, v.max(0)), sphere


def _check(lib, nodes, tris, box, base=0, first_node=0, first_block=0):
    cap, (qn, qp, qb) = _append(lib, nodes, tris, box, base)
    lo, hi, sphere = _extent(tris)
    # what the traversal has to reach: a leaf's box cut to each triangle and its padding; all of it, and
    # the 1e-3 that its acceptance allows, where it holds spheres or less than its primitives
    d = box[3:].astype(np.float64) - box[:3]
    reach = 1.5 * np.sqrt((d * d).sum())
    least = 2e-6 * (np.abs(box).max() + reach)
    e1, e2 = (np.linalg.norm(tris[f].astype(np.float64), axis=1) for f in ("e1", "e2"))
    pad = np.minimum(1e-3, np.maximum(0.5 * reach * e1 * e2, least)) * (1 - 1e-5)
    need_lo, need_hi = np.zeros_like(lo), np.zeros_like(hi)
    leaf_of = np.full(len(tris), -1)
    exact = np.zeros(len(tris), bool)
    leaves = _leaves(nodes, tris, box)
    for k, (first, cnt, mn, mx) in enumerate(leaves):
        s = slice(first, first + cnt)
        assert np.all(leaf_of[s] == -1)
        leaf_of[s] = k
        clips = not (np.all(lo[s] >= mn - 1e-4) and np.all(hi[s] <= mx + 1e-4))
        exact[s] = clips or max(np.abs(lo[s]).max(), np.abs(hi[s]).max()) > 1024
        if clips or sphere[s].any():
            need_lo[s], need_hi[s] = mn - 1e-3, mx + 1e-3
        else:
            m = (mn - 1e-3, mx + 1e-3) if len(nodes) == 0 else (mn, mx)
            need_lo[s], need_hi[s] = np.maximum(m[0], lo[s] - pad[s, None]), np.minimum(m[1], hi[s] + pad[s, None])
    seen_node, seen_block, seen = set(), set(), np.zeros(len(tris), int)

    def block(b):
        assert b not in seen_block and b >= first_block
        seen_block.add(b)
        used = [p for p in qp[b] if p[9] != NONE]
        assert used or len(tris) == 0
        assert all(p[9] == NONE for p in qp[b][len(used):])  # unused places come last
        ids = [int(p[9]) - base for p in used]
        for p, i in zip(used, ids):
            seen[i] += 1
            assert np.array_equal(p[0:9], np.concatenate([tris[f][i] for f in ("v0", "e1", "e2")]).view(np.uint32))
            assert p[11] == (int(tris["mat"][i]) | (SPHERE if sphere[i] else 0))
            assert bool(p[10] & EXACT) == bool(exact[i])
            first, cnt, mn, mx = leaves[leaf_of[i]]
            assert np.array_equal(qb[p[10] & ~np.uint32(EXACT)][[0, 1, 2, 4, 5, 6]],
                                  np.concatenate([mn, mx]).astype(np.float32))
        return need_lo[ids].min(0), need_hi[ids].max(0), 0

    def visit(i):
        """What lies below a node, and the stack entries a ray may need there."""
        assert i not in seen_node and i >= first_node
        seen_node.add(i)
        dec, parts = _decode(qn[i]), []
        refs = [int(qn[i][6 + 3 * c]) for c in range(4)]
        for c, ref in enumerate(refs):
            if ref == NONE:
                assert all(r == NONE for r in refs[c:])
                break
            part = block(ref & 0x7FFFFFFF) if ref & LEAF else visit(ref)
            assert np.all(dec[c, 0] <= part[0]) and np.all(dec[c, 1] >= part[1]), (i, c, dec[c], part)
            parts.append(part)
        return (np.min([p[0] for p in parts], 0), np.max([p[1] for p in parts], 0),
                len(parts) - 1 + max(max(p[2] for p in parts), 1))

    entries = visit(first_node)[2]
    assert len(seen_node) == len(qn) - first_node and len(seen_block) == len(qp) - first_block
    assert np.all(seen == 1)
    assert 0 < entries <= cap
    return cap, len(qn), len(qp)


def _export(verts, kinds=None):
    nodes, tris, _, box = api.Bvh(verts, kinds=kinds).export()
    rec = tris.view(np.uint32).reshape(len(tris), 12).copy().view(REC).reshape(-1)
    rec["mat"] = np.arange(len(rec)) % 7
    return nodes, rec, box


def _verts(name):
    rng = np.random.default_rng(3)
    if name == "far_and_small":  # grid steps near float spacing
        return (rng.uniform(-1e-2, 1e-2, (2000, 9)) + np.array([3e4, -7e3, 1e5] * 3)).astype(np.float32)
    if name == "large_leaf":  # one centroid: no split
        t = rng.uniform(-1, 1, (300, 3, 3)) * np.linspace(0.2, 1.0, 300)[:, None, None]
        return (t - t.mean(1, keepdims=True)).astype(np.float32).reshape(-1, 9)
    return host_scenes()[name]


NAMES = ["one", "two", "duplicates", "coplanar_grid", "random_soup", "cornell", "displaced", "far_and_small", "large_leaf"]


@pytest.mark.parametrize("name", NAMES)
def test_tree_of_triangles(lib, name):
    lib.q_clear()
    _check(lib, *_export(_verts(name)))


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 16, 17, 65, 257])
def test_remainders_of_blocks(lib, n):
    lib.q_clear()
    _check(lib, *_export(_verts("large_leaf")[:n]))
    lib.q_clear()
    _check(lib, *_export(_verts("random_soup")[:n]))


def test_spheres_among_triangles(lib):
    rng = np.random.default_rng(1)
    v, kinds = np.zeros((200, 9), np.float32), np.zeros(200, np.uint32)
    v[:] = (rng.uniform(-2, 2, (200, 1, 3)) + rng.uniform(-0.3, 0.3, (200, 3, 3))).reshape(200, 9)
    kinds[::3] = L.SPT_PRIM_SPHERE
    v[::3, 3:] = 0
    v[::3, 3] = rng.uniform(0.05, 0.4, len(v[::3]))
    v[100:140, 0:3] = 0.25  # spheres of one centre, in a leaf with the triangles between them
    lib.q_clear()
    _check(lib, *_export(v, kinds))


@pytest.mark.parametrize("name", ["random_soup", "large_leaf", "one"])
def test_boxes_that_clip(lib, name):
    nodes, tris, box = _export(_verts(name))
    rng = np.random.default_rng(2)
    for s in ("l", "r"):
        leaf = (nodes[s + "cnt"] > 0) & (rng.random(len(nodes)) < 0.5)
        nodes[s + "max"][leaf] = 0.5 * (nodes[s + "min"][leaf] + nodes[s + "max"][leaf])
    if len(nodes) == 0:
        box[3:] = 0.5 * (box[:3] + box[3:])
    lib.q_clear()
    _check(lib, nodes, tris, box)


def test_leaves_in_another_order(lib):
    """An uploaded tree may keep its leaves' primitives in any order: a block never
    takes primitives that are not those of its leaves."""
    nodes, tris, box = _export(_verts("random_soup"))
    leaves = _leaves(nodes, tris, box)
    order = np.random.default_rng(4).permutation(len(leaves))
    new, at, moved = np.zeros_like(tris), 0, {}
    for k in order:
        first, cnt = leaves[k][:2]
        new[at:at + cnt] = tris[first:first + cnt]
        moved[first] = at
        at += cnt
    for s in ("l", "r"):
        for nd in nodes:
            if nd[s + "cnt"] > 0:
                nd[s + "ref"] = moved[int(nd[s + "ref"])]
    lib.q_clear()
    _check(lib, nodes, new, box)


def test_trees_of_several_scenes(lib):
    """Appended trees: indices rebased, earlier trees untouched."""
    lib.q_clear()
    base = first_node = first_block = 0
    before = None
    for name in ("cornell", "one", "large_leaf", "random_soup"):
        nodes, tris, box = _export(_verts(name))
        _, first_node, first_block = _check(lib, nodes, tris, box, base, first_node, first_block)
        base += len(tris)
        now = _read(lib)
        if before is not None:
            assert np.array_equal(now[0][:len(before[0])], before[0]) and np.array_equal(now[1][:len(before[1])], before[1])
        before = now
