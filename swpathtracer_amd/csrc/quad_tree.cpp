// quad_tree.cpp - collapses the binary SAH tree into the four-wide tree with
// four-triangle blocks of the quad traversal.
//
// A node visit costs about the same whatever its children hold and a block
// tests four triangles at once, so the collapse minimises the surface-area
// cost over all ways of choosing up to four descendants per node and of
// merging subtrees of at most four triangles into one block, by dynamic
// programming from the leaves up (the method of Ylitie, Karras and Laine,
// "Efficient Incoherent Ray Traversal on GPUs Through Compressed Wide BVHs",
// 2017, sec. 3). On the 1M-triangle mesh in the box that leaves 124,933 nodes
// instead of the 236,620 of opening the largest child until there are four
// (41% of those held only two), and a path tracer's ray visits 6.7 nodes and
// 2.0 blocks instead of 7.1 and 2.1.
//
// The reference pads every child box by 1e-3 around its primitives. That is
// more than small triangles need: the traversal only has to reach every
// candidate the reference would accept, and such a candidate lies on its
// triangle up to the rounding of the triangle test. So the boxes here are the
// given ones cut to the triangles' bounds plus a padding of their own
// (prim_pad). Not so a leaf with spheres, or whose box does not hold its
// primitives (an uploaded tree may clip them): there hits are accepted off the
// primitive, or outside the box, so such leaves and the nodes above them get the
// leaf's box and the 1e-3 around it that its acceptance allows. The mesh in the box goes from
// 10.3 to 8.3 steps for rays off its surfaces, the longest of a million of them
// from 1036 to 651 (near the poles of the displaced sphere hundreds of slivers
// are thinner than 1e-3).
#include "quad_tree.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <limits>

namespace spt {

namespace {

constexpr uint32_t kBlockPrims = 4;
constexpr float kNodeCost = 1.0f, kBlockCost = 2.0f;  // a block test runs about twice a node's instructions

struct Item {  // one child of a binary node
    float lo[3], hi[3];
    uint32_t ref, cnt;  // cnt > 0: leaf [ref, ref + cnt)
};

void load_item(const spt_node64& nd, int s, Item& e) {
    const float* lo = s == 0 ? nd.lmin : nd.rmin;
    const float* hi = s == 0 ? nd.lmax : nd.rmax;
    for (int k = 0; k < 3; ++k) {
        e.lo[k] = lo[k];
        e.hi[k] = hi[k];
    }
    e.ref = s == 0 ? nd.lref : nd.rref;
    e.cnt = s == 0 ? nd.lcnt : nd.rcnt;
}

float area(const Item& e) {
    const float dx = e.hi[0] - e.lo[0], dy = e.hi[1] - e.lo[1], dz = e.hi[2] - e.lo[2];
    return dx * dy + dy * dz + dz * dx;
}

// Best costs of a binary node's subtree as a forest of at most 1, 2 or 3
// roots, and the choices that give them.
struct Plan {
    float cost[4];      // [j]: at most j roots
    uint8_t split[5];   // [j]: roots given to the left child when j are used (2..4)
    uint8_t used[4];    // [j]: how many roots the best forest of at most j uses
    bool block;         // one root: the subtree is a block
    uint32_t first, count;  // its primitives, when they are one range of at most four (count 0: not so)
};

struct Box {
    float lo[3], hi[3];
};

// Padding of a triangle's box: how far the point where a ray crosses the
// plane can be from the point (u, v, t) of a float triangle test that accepts
// it. In units of 2^-24 |o - v0| |e1| |e2| / |det| the two are at most 2.7
// apart in the plane and 5.3 along the ray (9 million accepted tests, grazing
// to the limit |det| = 1e-6, against double); 8 of those units at that
// smallest det and at the largest distance the paddings cover (1.5 diagonals
// of the root box: ray origins within one diagonal of its centre, unit
// directions; the traversal widens the boxes for other rays) are
// 0.5 * reach * |e1| |e2|. At least the rounding of the box tests themselves,
// at most the reference's 1e-3.
float prim_pad(const spt_tri48& t, float reach, float least) {
    auto len = [](const float* e) { return std::sqrt(e[0] * e[0] + e[1] * e[1] + e[2] * e[2]); };
    const float p = std::max(0.5f * reach * len(t.e1) * len(t.e2), least);
    return p < 1e-3f ? p : 1e-3f;
}

class Builder {
public:
    Builder(const spt_node64* nodes, uint32_t n_nodes, const spt_tri48* tris, const float* root_box,
            uint32_t prim_base, QuadTree& out)
        : nodes_(nodes), n_(n_nodes), tris_(tris), base_(prim_base), out_(out) {
        float d2 = 0.0f, mag = 0.0f;
        for (int k = 0; k < 3; ++k) {
            const float e = root_box[3 + k] - root_box[k];
            d2 += e * e;
            mag = std::max(mag, std::max(std::fabs(root_box[k]), std::fabs(root_box[3 + k])));
        }
        reach_ = 1.5f * std::sqrt(d2);
        least_ = 2e-6f * (mag + reach_);
        if (!(least_ < 1e-3f)) least_ = 1e-3f;  // large (or NaN) coordinates: the reference's padding
        if (!(reach_ >= 0.0f)) reach_ = std::numeric_limits<float>::infinity();
    }

    uint32_t run(uint32_t n_tris, const float* root_box) {
        std::vector<Work> work;
        const uint32_t root = (uint32_t)out_.nodes.size();
        out_.nodes.emplace_back();
        if (n_ == 0) {  // the root is a leaf: its box is the (unpadded) root box
            Part p;
            p.kind = Part::kRange;
            for (int k = 0; k < 3; ++k) {
                p.box.lo[k] = root_box[k];
                p.box.hi[k] = root_box[3 + k];
            }
            p.first = 0;
            p.count = n_tris;
            p.loose = loose(p.box, 0, n_tris);
            p.leaf_box = add_box(p.box, 0, n_tris);
            widen(p.box);
            work.push_back({root, 1, 0, true, p});
        } else {
            plan();
            work.push_back({root, 1, 0, false, Part{}});
        }
        uint32_t depth = 1;
        while (!work.empty()) {
            const Work w = work.back();
            work.pop_back();
            depth = std::max(depth, w.depth);
            std::vector<Part> parts;
            if (w.chunk) {
                split_range(w.part, parts);
            } else {
                const uint8_t k = plan_[w.bin].split[4];
                gather(w.bin, 0, k, parts);
                gather(w.bin, 1, 4 - k, parts);
            }
            QuadNode q = quantise(parts);
            for (size_t i = 0; i < parts.size(); ++i) {
                Part& p = parts[i];
                if (p.kind == Part::kInner || p.count > kBlockPrims) {
                    q.child[i].ref = (uint32_t)out_.nodes.size();
                    out_.nodes.emplace_back();
                    work.push_back({q.child[i].ref, w.depth + 1, p.bin, p.kind != Part::kInner, p});
                } else {
                    q.child[i].ref = kQuadLeaf | emit_block(p);
                }
            }
            out_.nodes[w.slot] = q;
        }
        if (out_.nodes.size() >= kQuadLeaf || out_.prims.size() / kBlockPrims >= kQuadLeaf - 1u) return 0;
        return 3 * depth + 1;
    }

private:
    // One child of a four-wide node being made.
    struct Part {
        enum Kind { kInner, kRange, kMerged } kind = kInner;
        Item box{};
        uint32_t bin = 0;              // kInner, kMerged: binary node
        uint32_t first = 0, count = 0; // kRange (part of one leaf), kMerged (a subtree of several)
        uint32_t leaf_box = 0;         // kRange
        bool loose = false;            // kRange: parts of it keep its box
    };
    struct Work {
        uint32_t slot, depth, bin;
        bool chunk;  // the node splits one large leaf range
        Part part;
    };

    // A triangle's bounds and padding (in double, rounded outward).
    void prim_box(uint32_t tri, Box& b) const {
        const spt_tri48& t = tris_[tri];
        const double pad = prim_pad(t, reach_, least_);
        for (int k = 0; k < 3; ++k) {
            const double v0 = t.v0[k], v1 = v0 + t.e1[k], v2 = v0 + t.e2[k];
            const double lo = std::min(v0, std::min(v1, v2)), hi = std::max(v0, std::max(v1, v2));
            b.lo[k] = std::nextafter((float)(lo - pad), -std::numeric_limits<float>::infinity());
            b.hi[k] = std::nextafter((float)(hi + pad), std::numeric_limits<float>::infinity());
        }
    }

    // Whether the box of a leaf reaches as far as its primitives (to 1e-4, which
    // the rounding of v0 + e1 and the acceptance shortcut leave room for).
    bool holds(const Item& e, uint32_t first, uint32_t count) const {
        for (uint32_t i = first; i < first + count; ++i) {
            const spt_tri48& t = tris_[i];
            for (int k = 0; k < 3; ++k) {
                double lo = t.v0[k], hi = lo;
                if (t.pad[1] == SPT_PRIM_SPHERE) {
                    lo -= std::fabs((double)t.e1[0]);
                    hi += std::fabs((double)t.e1[0]);
                } else {
                    const double v1 = lo + t.e1[k], v2 = lo + t.e2[k];
                    lo = std::min(lo, std::min(v1, v2));
                    hi = std::max(hi, std::max(v1, v2));
                }
                if (!(lo >= (double)e.lo[k] - 1e-4 && hi <= (double)e.hi[k] + 1e-4)) return false;
            }
        }
        return true;
    }
    bool small_coords(uint32_t first, uint32_t count) const {
        for (uint32_t i = first; i < first + count; ++i) {
            const spt_tri48& t = tris_[i];
            for (int k = 0; k < 3; ++k)
                if (!(std::fabs(t.v0[k]) <= 1024.0f && std::fabs(t.v0[k] + t.e1[k]) <= 1024.0f &&
                      std::fabs(t.v0[k] + t.e2[k]) <= 1024.0f))
                    return false;
        }
        return true;
    }
    // Whether hits in a leaf are not accepted at its primitives alone: a sphere's
    // test accepts hit points off it when the direction is not of unit length.
    bool loose(const Item& e, uint32_t first, uint32_t count) const {
        for (uint32_t i = first; i < first + count; ++i)
            if (tris_[i].pad[1] == SPT_PRIM_SPHERE) return true;
        return !holds(e, first, count);
    }
    // Hit points are accepted up to 1e-3 outside their leaf's box.
    template <typename E>
    static void widen(E& e) {
        for (int k = 0; k < 3; ++k) {
            e.lo[k] = std::nextafter(e.lo[k] - 2e-3f, -std::numeric_limits<float>::infinity());
            e.hi[k] = std::nextafter(e.hi[k] + 2e-3f, std::numeric_limits<float>::infinity());
        }
    }

    // Bounds of triangles [first, first + count).
    Box range_box(uint32_t first, uint32_t count) const {
        Box u;
        prim_box(first, u);
        for (uint32_t i = 1; i < count; ++i) {
            Box b;
            prim_box(first + i, b);
            join(u, b);
        }
        return u;
    }
    static void join(Box& a, const Box& b) {
        for (int k = 0; k < 3; ++k) {
            a.lo[k] = std::min(a.lo[k], b.lo[k]);
            a.hi[k] = std::max(a.hi[k], b.hi[k]);
        }
    }
    // The given box cut to what it holds (a NaN bound of either stays out of the way).
    template <typename E>
    static void cut(E& e, const Box& b) {
        for (int k = 0; k < 3; ++k) {
            if (e.lo[k] < b.lo[k]) e.lo[k] = b.lo[k];
            if (e.hi[k] > b.hi[k]) e.hi[k] = b.hi[k];
        }
    }

    // A child of a binary node with the box the traversal gets (after plan()).
    void item(uint32_t bin, int s, Item& e) const {
        load_item(nodes_[bin], s, e);
        settle(bin, s, e);
    }
    void settle(uint32_t bin, int s, Item& e) const {
        const Box& u = boxes_[2 * (size_t)bin + s];
        if (loose_[2 * (size_t)bin + s])
            for (int k = 0; k < 3; ++k) {
                e.lo[k] = u.lo[k];
                e.hi[k] = u.hi[k];
            }
        else
            cut(e, u);
    }

    float leaf_cost(float a, uint32_t cnt) const {
        if (cnt <= kBlockPrims) return a * kBlockCost;
        return a * (kBlockCost * (float)((cnt + kBlockPrims - 1) / kBlockPrims) + kNodeCost);
    }
    float item_cost(const Item& e, int j) const { return e.cnt ? leaf_cost(area(e), e.cnt) : plan_[e.ref].cost[j]; }

    void plan() {
        plan_.resize(n_);
        boxes_.resize(2 * (size_t)n_);
        loose_.resize(2 * (size_t)n_);
        for (uint32_t i = n_; i-- > 0;) {  // children come after their parent
            Plan& p = plan_[i];
            Item l, r, b;
            for (int s = 0; s < 2; ++s) {
                Item& e = s == 0 ? l : r;
                load_item(nodes_[i], s, e);
                Box& u = boxes_[2 * (size_t)i + s];
                if (e.cnt && loose(e, e.ref, e.cnt)) {
                    loose_[2 * (size_t)i + s] = true;
                    for (int k = 0; k < 3; ++k) {
                        u.lo[k] = e.lo[k];
                        u.hi[k] = e.hi[k];
                    }
                    widen(u);
                } else if (e.cnt) {
                    u = range_box(e.ref, e.cnt);
                } else {
                    loose_[2 * (size_t)i + s] = loose_[2 * (size_t)e.ref] || loose_[2 * (size_t)e.ref + 1];
                    Item cl, cr;
                    item(e.ref, 0, cl);
                    item(e.ref, 1, cr);
                    for (int k = 0; k < 3; ++k) {
                        u.lo[k] = std::min(cl.lo[k], cr.lo[k]);
                        u.hi[k] = std::max(cl.hi[k], cr.hi[k]);
                    }
                }
                settle(i, s, e);
            }
            for (int k = 0; k < 3; ++k) {
                b.lo[k] = std::min(l.lo[k], r.lo[k]);
                b.hi[k] = std::max(l.hi[k], r.hi[k]);
            }
            const float a = area(b);
            const uint32_t lf = l.cnt ? l.ref : plan_[l.ref].first, lc = l.cnt ? l.cnt : plan_[l.ref].count;
            const uint32_t rf = r.cnt ? r.ref : plan_[r.ref].first, rc = r.cnt ? r.cnt : plan_[r.ref].count;
            p.first = lf;
            // uploaded trees may order their leaves freely: only one run of primitives is merged
            p.count = (lc && rc && lc <= kBlockPrims && rc <= kBlockPrims && lc + rc <= kBlockPrims && lf + lc == rf)
                          ? lc + rc
                          : 0u;
            float forest[5];
            for (int j = 2; j <= 4; ++j) {
                forest[j] = std::numeric_limits<float>::infinity();
                p.split[j] = 1;
                for (int k = std::max(1, j - 3); k <= std::min(3, j - 1); ++k) {
                    const float c = item_cost(l, k) + item_cost(r, j - k);
                    if (c < forest[j]) {
                        forest[j] = c;
                        p.split[j] = (uint8_t)k;
                    }
                }
            }
            const float inner = forest[4] + a * kNodeCost;
            const float merged = p.count ? leaf_cost(a, p.count) : std::numeric_limits<float>::infinity();
            p.block = p.count && !(inner < merged);
            p.cost[1] = p.block ? merged : inner;
            p.used[1] = 1;
            for (int j = 2; j <= 3; ++j) {
                const bool fewer = p.cost[j - 1] <= forest[j];
                p.cost[j] = fewer ? p.cost[j - 1] : forest[j];
                p.used[j] = fewer ? p.used[j - 1] : (uint8_t)j;
            }
        }
    }

    // The forest of at most j roots under child s of a binary node, appended to parts.
    void gather(uint32_t bin, int s, int j, std::vector<Part>& parts) {
        Item e, given;
        load_item(nodes_[bin], s, given);
        item(bin, s, e);
        Part p;
        p.box = e;
        if (e.cnt) {
            p.kind = Part::kRange;
            p.first = e.ref;
            p.count = e.cnt;
            p.loose = loose_[2 * (size_t)bin + s];
            p.leaf_box = add_box(given, e.ref, e.cnt);
            parts.push_back(p);
            return;
        }
        const Plan& pl = plan_[e.ref];
        j = pl.used[j];
        if (j == 1) {
            p.kind = pl.block ? Part::kMerged : Part::kInner;
            p.bin = e.ref;
            p.first = pl.first;
            p.count = pl.block ? pl.count : 0u;
            parts.push_back(p);
            return;
        }
        gather(e.ref, 0, pl.split[j], parts);
        gather(e.ref, 1, j - pl.split[j], parts);
    }

    // A leaf of more than four primitives: up to four parts of a power of
    // four of blocks each.
    void split_range(const Part& p, std::vector<Part>& parts) {
        uint64_t step = kBlockPrims;
        while (step * 4 < p.count) step *= 4;
        for (uint64_t at = 0; at < p.count; at += step) {
            Part q = p;
            q.first = p.first + (uint32_t)at;
            q.count = (uint32_t)std::min<uint64_t>(step, p.count - at);
            if (!p.loose) cut(q.box, range_box(q.first, q.count));
            parts.push_back(q);
        }
    }

    // Index of the box of leaf [first, first + count), as the primitives keep it.
    uint32_t add_box(const Item& e, uint32_t first, uint32_t count) {
        QuadBox b{};
        std::memcpy(b.mn, e.lo, sizeof(b.mn));
        std::memcpy(b.mx, e.hi, sizeof(b.mx));
        out_.boxes.push_back(b);
        const bool near = holds(e, first, count) && small_coords(first, count);
        return ((uint32_t)out_.boxes.size() - 1) | (near ? 0u : kQuadExact);
    }

    void put(QuadPrim* dst, uint32_t tri, uint32_t box) {
        const spt_tri48& t = tris_[tri];
        std::memcpy(dst->v0, t.v0, sizeof(t.v0));
        std::memcpy(dst->e1, t.e1, sizeof(t.e1));
        std::memcpy(dst->e2, t.e2, sizeof(t.e2));
        dst->index = base_ + tri;
        dst->box = box;
        dst->kind_mat = (t.pad[0] & ~kQuadSphere) | (t.pad[1] == SPT_PRIM_SPHERE ? kQuadSphere : 0u);
    }

    void emit_leaves(uint32_t bin, QuadPrim*& at) {
        for (int s = 0; s < 2; ++s) {
            Item e;
            load_item(nodes_[bin], s, e);
            if (e.cnt) {
                const uint32_t box = add_box(e, e.ref, e.cnt);
                for (uint32_t k = 0; k < e.cnt; ++k) put(at++, e.ref + k, box);
            } else {
                emit_leaves(e.ref, at);
            }
        }
    }

    uint32_t emit_block(const Part& p) {
        const size_t first = out_.prims.size();
        QuadPrim none{};
        none.index = kQuadNone;
        out_.prims.resize(first + kBlockPrims, none);
        QuadPrim* at = &out_.prims[first];
        if (p.kind == Part::kMerged) {
            emit_leaves(p.bin, at);
        } else {
            for (uint32_t k = 0; k < p.count; ++k) put(at++, p.first + k, p.leaf_box);
        }
        return (uint32_t)(first / kBlockPrims);
    }

    static float bits_float(uint32_t u) {
        float f;
        std::memcpy(&f, &u, 4);
        return f;
    }

    // The node's grid and its children's bytes. The step of z is a power of
    // two; those of y and x carry the fields below them as mantissa bits, so
    // each exponent is the smallest whose step, so decoded, spans the axis.
    static QuadNode quantise(const std::vector<Part>& parts) {
        QuadNode q{};
        float* origin[3] = {&q.ox, &q.oy, &q.oz};
        double step[3];
        uint32_t steps = 0;
        for (int a = 2; a >= 0; --a) {
            float mn = std::numeric_limits<float>::infinity(), mx = -mn;
            for (const Part& p : parts) {
                mn = std::min(mn, p.box.lo[a]);
                mx = std::max(mx, p.box.hi[a]);
            }
            if (!(mn <= mx) || !std::isfinite(mn)) mn = std::isfinite(mx) ? std::min(mn, mx) : 0.0f;
            if (!std::isfinite(mn)) mn = 0.0f;
            *origin[a] = mn;
            const int shift = 5 + 9 * (2 - a);  // exponent field of the axis
            const double ext = std::isfinite(mx) ? (double)mx - mn : std::numeric_limits<double>::max();
            uint32_t e = 1;
            const double want = ext / 255.0 * 16777216.0;
            if (want > 0.0) e = (uint32_t)std::min(254.0, std::max(1.0, std::floor(std::log2(want)) + 126.0));
            auto decoded = [&](uint32_t f) {
                return (double)bits_float((steps | (f << shift)) << (9 * a)) / 16777216.0;
            };
            while (e < 254 && decoded(e) * 255.0 < ext) ++e;
            step[a] = decoded(e);
            steps |= e << shift;
        }
        q.steps = steps;
        for (size_t i = 0; i < 4; ++i) {
            if (i >= parts.size()) {
                q.child[i].ref = kQuadNone;
                continue;
            }
            uint32_t lo[3], hi[3];
            for (int a = 0; a < 3; ++a) {
                const double o = *origin[a];
                const double fl = std::floor(((double)parts[i].box.lo[a] - o) / step[a]);
                const double fh = std::ceil(((double)parts[i].box.hi[a] - o) / step[a]);
                lo[a] = fl > 0.0 ? (uint32_t)std::min(fl, 255.0) : 0u;  // NaN bounds span the grid
                hi[a] = fh < 255.0 ? (uint32_t)std::max(fh, 0.0) : 255u;
                while (lo[a] > 0 && o + lo[a] * step[a] > parts[i].box.lo[a]) --lo[a];
                while (hi[a] < 255 && o + hi[a] * step[a] < parts[i].box.hi[a]) ++hi[a];
            }
            q.child[i].xy = lo[0] | (hi[0] << 8) | (lo[1] << 16) | (hi[1] << 24);
            q.child[i].z = lo[2] | (hi[2] << 8);
        }
        return q;
    }

    const spt_node64* nodes_;
    uint32_t n_;
    const spt_tri48* tris_;
    uint32_t base_;
    QuadTree& out_;
    float reach_ = 0.0f, least_ = 0.0f;  // prim_pad
    std::vector<Plan> plan_;
    std::vector<Box> boxes_;  // [2 i + s]: what child s of binary node i holds
    std::vector<bool> loose_;  // [2 i + s]: that child is its box, whatever the node gives it
};

}  // namespace

uint32_t append_quad_tree(const spt_node64* nodes, uint32_t n_nodes, const spt_tri48* tris, uint32_t n_tris,
                          const float* root_box, uint32_t prim_base, QuadTree& out) {
    return Builder(nodes, n_nodes, tris, root_box, prim_base, out).run(n_tris, root_box);
}

}  // namespace spt
