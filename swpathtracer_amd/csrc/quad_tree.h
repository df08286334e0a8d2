// quad_tree.h - the tree and triangle blocks the quad traversal reads
// (spt_quad.h), built on the host from the binary tree. Plain C++ (no HIP).
#pragma once

#include <stdint.h>

#include <vector>

#include "spt.h"

namespace spt {

// Four-wide node, 64 B: a header that the four lanes of a quad read together
// and one 12-B record per child that one lane reads.
//   grid: origin x y z and the word `steps`, whose bits, read as a float after
//   a shift by 0, 9 and 18, are the grid step of x, y and z times 2^24 (the
//   bits below an axis's exponent are its mantissa; the builder accounts for
//   them). A child bound is origin + byte * step, lo rounded down, hi up.
//   child: lo.x hi.x lo.y hi.y | lo.z hi.z 0 0 | reference: node index, or
//   kQuadLeaf | block index, or kQuadNone.
// The bytes are unpacked two at a time to 16-bit halves with a zero high
// byte, i.e. as half-float denormals byte * 2^-24, which the device's mixed
// FMA takes as an operand (hence the 2^24 in the steps).
struct QuadNode {
    float ox, oy, oz;
    uint32_t steps;
    struct Child {
        uint32_t xy, z, ref;
    } child[4];
};
static_assert(sizeof(QuadNode) == 64, "QuadNode layout");

constexpr uint32_t kQuadLeaf = 0x80000000u;
constexpr uint32_t kQuadNone = 0xFFFFFFFFu;
constexpr uint32_t kQuadSphere = 0x80000000u;  // QuadPrim::kind_mat: sphere flag beside the material
// QuadPrim::box: every hit is compared with the leaf's box, which does not hold
// its primitives, or a coordinate of them exceeds 1024 (a float ulp, 6e-5 below
// it, is far inside the 5e-4 margin of the traversal's acceptance shortcut)
constexpr uint32_t kQuadExact = 0x80000000u;

// One primitive of a block of four (192 B, a lane each): the geometry of
// spt_tri48, its index in leaf order (kQuadNone: unused slot, a degenerate
// triangle nothing hits), the exact box of its leaf and its material.
struct QuadPrim {
    float v0[3], e1[3], e2[3];
    uint32_t index, box, kind_mat;
};
static_assert(sizeof(QuadPrim) == 48, "QuadPrim layout");

// Exact padded box of one leaf of the binary tree.
struct QuadBox {
    float mn[3], pad0, mx[3], pad1;
};
static_assert(sizeof(QuadBox) == 32, "QuadBox layout");

struct QuadTree {
    std::vector<QuadNode> nodes;
    std::vector<QuadPrim> prims;  // blocks of four
    std::vector<QuadBox> boxes;
    // whether nodes and blocks can be addressed with 32-bit byte offsets
    bool small() const {
        return nodes.size() * sizeof(QuadNode) < (1ull << 32) && prims.size() * sizeof(QuadPrim) < (1ull << 32);
    }
};

// Appends the tree of one scene: pair nodes (pre-order; none: the root is one
// leaf of all primitives), primitives in leaf order with their materials,
// root box. Primitive indices are rebased by prim_base. Returns the stack
// entries a traversal of it can need, 0 when an index does not fit its field.
uint32_t append_quad_tree(const spt_node64* nodes, uint32_t n_nodes, const spt_tri48* tris, uint32_t n_tris,
                          const float* root_box, uint32_t prim_base, QuadTree& out);

}  // namespace spt
