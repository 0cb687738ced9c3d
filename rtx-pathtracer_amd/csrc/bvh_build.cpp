// Host BVH builder: binned surface-area heuristic (Wald, "On fast
// construction of SAH-based bounding volume hierarchies", 2007) for a
// binary tree, collapsed into four-wide nodes (bvh_wide.cpp packs those into
// the nodes the traversal kernels read).  It replaces the driver's BLAS/TLAS build (src/SceneLoader.cpp:1101-1193), whose source
// is not available.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <limits>
#include <stdexcept>

#include "bvh.h"

namespace rtx {

namespace {

struct Box {
    float lo[3], hi[3];
    void reset() {
        for (int a = 0; a < 3; ++a) {
            lo[a] = std::numeric_limits<float>::infinity();
            hi[a] = -std::numeric_limits<float>::infinity();
        }
    }
    void grow(const Box &b) {
        for (int a = 0; a < 3; ++a) {
            lo[a] = std::min(lo[a], b.lo[a]);
            hi[a] = std::max(hi[a], b.hi[a]);
        }
    }
    void grow(const float p[3]) {
        for (int a = 0; a < 3; ++a) {
            lo[a] = std::min(lo[a], p[a]);
            hi[a] = std::max(hi[a], p[a]);
        }
    }
    float area() const {
        float dx = hi[0] - lo[0], dy = hi[1] - lo[1], dz = hi[2] - lo[2];
        if (dx < 0 || dy < 0 || dz < 0) return 0.0f;
        return 2.0f * (dx * dy + dy * dz + dz * dx);
    }
};

// 64 SAH bins, and the SAH cost (not a size threshold) deciding every split
// above one primitive: on the 262144-triangle room 64 bins against 32 visit
// 2% fewer nodes, and SAH-sized leaves cut the triangle tests per ray from
// 8.8 to 3.6 for 1% more node visits (traversal time per step -4.9%).
constexpr int kBins = 64;
constexpr int kSahDepthLimit = 32; // deeper subtrees use object-median splits
constexpr int kLeafTarget = 1;
constexpr uint32_t kSmallCount = 24; // subtrees searched primitive by primitive

struct Builder {
    std::vector<Box> primBox;
    std::vector<float> centroid; // 3 per prim
    std::vector<uint32_t> order;
    std::vector<BvhNode> nodes;
    uint32_t maxDepth = 0;

    // The binned search on axis a for a few primitives: sorted by bin, only
    // the bins that hold one are visited.  An empty bin's cut costs what the
    // cut before it does and is never taken, so the choice is the full
    // search's; resetting and sweeping 64 bins for the many small subtrees
    // was most of the build.
    void sweepSmall(uint32_t start, uint32_t count, int a, float lo, float scale, float &bestCost, int &bestAxis,
                    int &bestBin) const {
        int bin[kSmallCount];
        uint32_t prim[kSmallCount];
        for (uint32_t i = 0; i < count; ++i) {
            const uint32_t p = order[start + i];
            int b = (int)((centroid[3 * (size_t)p + a] - lo) * scale);
            b = std::min(std::max(b, 0), kBins - 1);
            uint32_t k = i;
            for (; k > 0 && bin[k - 1] > b; --k) {
                bin[k] = bin[k - 1];
                prim[k] = prim[k - 1];
            }
            bin[k] = b;
            prim[k] = p;
        }
        float right[kSmallCount]; // area of primitives k.. on
        Box acc;
        acc.reset();
        for (uint32_t k = count; k-- > 1;) {
            acc.grow(primBox[prim[k]]);
            right[k] = acc.area();
        }
        acc.reset();
        for (uint32_t k = 0; k + 1 < count; ++k) {
            acc.grow(primBox[prim[k]]);
            if (bin[k] == bin[k + 1]) continue;
            const float cost = acc.area() * (k + 1) + right[k + 1] * (count - k - 1);
            if (cost < bestCost) {
                bestCost = cost;
                bestAxis = a;
                bestBin = bin[k];
            }
        }
    }

    // Returns the link for the subtree over order[start, start+count).
    int32_t build(uint32_t start, uint32_t count, uint32_t depth, Box &outBox) {
        outBox.reset();
        Box cbox;
        cbox.reset();
        for (uint32_t i = start; i < start + count; ++i) {
            outBox.grow(primBox[order[i]]);
            cbox.grow(&centroid[3 * (size_t)order[i]]);
        }
        maxDepth = std::max(maxDepth, depth);
        if (count <= (uint32_t)kLeafTarget && depth + 1 < (uint32_t)kMaxBvhDepth)
            return makeLeaf(start, count);
        if (depth + 1 >= (uint32_t)kMaxBvhDepth) {
            if (count > (uint32_t)kLeafMaxPrims) throw std::runtime_error("BVH depth limit exceeded");
            return makeLeaf(start, count);
        }
        uint32_t mid = start;
        bool found = false;
        int axis = 0;
        for (int a = 1; a < 3; ++a)
            if (cbox.hi[a] - cbox.lo[a] > cbox.hi[axis] - cbox.lo[axis]) axis = a;
        if (depth < (uint32_t)kSahDepthLimit) {
            float bestCost = std::numeric_limits<float>::infinity();
            int bestAxis = -1, bestBin = -1;
            for (int a = 0; a < 3; ++a) {
                float ext = cbox.hi[a] - cbox.lo[a];
                if (!(ext > 0.0f)) continue;
                if (count <= kSmallCount) {
                    sweepSmall(start, count, a, cbox.lo[a], kBins / ext, bestCost, bestAxis, bestBin);
                    continue;
                }
                Box bb[kBins];
                uint32_t bc[kBins] = {0};
                for (auto &b : bb) b.reset();
                float scale = kBins / ext;
                for (uint32_t i = start; i < start + count; ++i) {
                    uint32_t p = order[i];
                    int bin = (int)((centroid[3 * (size_t)p + a] - cbox.lo[a]) * scale);
                    bin = std::min(std::max(bin, 0), kBins - 1);
                    bb[bin].grow(primBox[p]);
                    bc[bin]++;
                }
                Box right[kBins];
                uint32_t rc[kBins];
                Box acc;
                acc.reset();
                uint32_t n = 0;
                for (int b = kBins - 1; b > 0; --b) {
                    acc.grow(bb[b]);
                    n += bc[b];
                    right[b] = acc;
                    rc[b] = n;
                }
                acc.reset();
                n = 0;
                for (int b = 0; b < kBins - 1; ++b) {
                    acc.grow(bb[b]);
                    n += bc[b];
                    if (n == 0 || rc[b + 1] == 0) continue;
                    float cost = acc.area() * n + right[b + 1].area() * rc[b + 1];
                    if (cost < bestCost) {
                        bestCost = cost;
                        bestAxis = a;
                        bestBin = b;
                    }
                }
            }
            float leafCost = outBox.area() * count;
            // cost model: traversal step = 1, triangle test = 1 (relative)
            if (bestAxis >= 0 && (count > (uint32_t)kLeafMaxPrims || bestCost + outBox.area() < leafCost)) {
                float ext = cbox.hi[bestAxis] - cbox.lo[bestAxis];
                float scale = kBins / ext;
                auto it = std::partition(order.begin() + start, order.begin() + start + count, [&](uint32_t p) {
                    int bin = (int)((centroid[3 * (size_t)p + bestAxis] - cbox.lo[bestAxis]) * scale);
                    bin = std::min(std::max(bin, 0), kBins - 1);
                    return bin <= bestBin;
                });
                mid = (uint32_t)(it - order.begin());
                found = mid > start && mid < start + count;
            } else if (bestAxis >= 0 || count <= (uint32_t)kLeafMaxPrims) {
                if (count <= (uint32_t)kLeafMaxPrims) return makeLeaf(start, count);
            }
        }
        if (!found) { // object median on the widest centroid axis (or by index if degenerate)
            mid = start + count / 2;
            std::nth_element(order.begin() + start, order.begin() + mid, order.begin() + start + count,
                             [&](uint32_t x, uint32_t y) {
                                 float cx = centroid[3 * (size_t)x + axis], cy = centroid[3 * (size_t)y + axis];
                                 return cx < cy || (cx == cy && x < y);
                             });
        }
        uint32_t id = (uint32_t)nodes.size();
        nodes.emplace_back();
        Box lb, rb;
        int32_t l = build(start, mid - start, depth + 1, lb);
        int32_t r = build(mid, start + count - mid, depth + 1, rb);
        setNode(nodes[id], lb, rb, l, r);
        return (int32_t)id;
    }

    static void setNode(BvhNode &n, const Box &l, const Box &r, int32_t ll, int32_t rl) {
        n.a[0] = l.lo[0]; n.a[1] = l.lo[1]; n.a[2] = l.lo[2]; n.a[3] = l.hi[0];
        n.b[0] = l.hi[1]; n.b[1] = l.hi[2]; n.b[2] = r.lo[0]; n.b[3] = r.lo[1];
        n.c[0] = r.lo[2]; n.c[1] = r.hi[0]; n.c[2] = r.hi[1]; n.c[3] = r.hi[2];
        n.d[0] = ll;
        n.d[1] = rl;
        n.d[2] = 0;
        n.d[3] = 0;
    }
};

// Collapse of the binary tree into four-wide nodes: a node's children start
// as the binary node's two; the internal child with the largest surface
// area is replaced by its two children until there are four or only leaves
// remain.  Nodes are emitted parent first (depth-first), children in the
// binary tree's left-to-right order.
struct Collapser {
    const std::vector<BvhNode> &in;
    std::vector<Bvh4Node> out;
    uint32_t maxDepth;

    struct Child {
        Box box;
        int32_t link;
    };
    static Child childOf(const BvhNode &n, int k) {
        Child c;
        if (k == 0) {
            c.box.lo[0] = n.a[0]; c.box.lo[1] = n.a[1]; c.box.lo[2] = n.a[2];
            c.box.hi[0] = n.a[3]; c.box.hi[1] = n.b[0]; c.box.hi[2] = n.b[1];
        } else {
            c.box.lo[0] = n.b[2]; c.box.lo[1] = n.b[3]; c.box.lo[2] = n.c[0];
            c.box.hi[0] = n.c[1]; c.box.hi[1] = n.c[2]; c.box.hi[2] = n.c[3];
        }
        c.link = n.d[k];
        return c;
    }
    // Emits the four-wide node for binary node `id`; returns its index.
    int32_t collapse(int32_t id, uint32_t depth) {
        maxDepth = std::max(maxDepth, depth);
        Child ch[4];
        int n = 2;
        ch[0] = childOf(in[id], 0);
        ch[1] = childOf(in[id], 1);
        while (n < 4) {
            int best = -1;
            float bestArea = -1.0f;
            for (int k = 0; k < n; ++k)
                if (ch[k].link >= 0 && ch[k].box.area() > bestArea) {
                    bestArea = ch[k].box.area();
                    best = k;
                }
            if (best < 0) break;
            const BvhNode &bn = in[ch[best].link];
            for (int k = n; k > best + 1; --k) ch[k] = ch[k - 1];
            ch[best] = childOf(bn, 0);
            ch[best + 1] = childOf(bn, 1);
            n++;
        }
        int32_t self = (int32_t)out.size();
        out.emplace_back();
        int32_t links[4];
        for (int k = 0; k < 4; ++k) links[k] = makeLeaf(0, 1);
        for (int k = 0; k < n; ++k) links[k] = ch[k].link >= 0 ? collapse(ch[k].link, depth + 1) : ch[k].link;
        Bvh4Node &o = out[self];
        std::memset(&o, 0, sizeof(o));
        for (int k = 0; k < 4; ++k) {
            Box bx;
            if (k < n) {
                bx = ch[k].box;
            } else {
                for (int a = 0; a < 3; ++a) bx.lo[a] = bx.hi[a] = 1e30f; // unused slot
            }
            o.f[0][k] = bx.lo[0];
            o.f[1][k] = bx.hi[0];
            o.f[2][k] = bx.lo[1];
            o.f[3][k] = bx.hi[1];
            o.f[4][k] = bx.lo[2];
            o.f[5][k] = bx.hi[2];
            o.link[k] = links[k];
        }
        return self;
    }
};

// Pad a coordinate bound outwards by (|x| + S) 2^-20, S the scene's largest
// coordinate magnitude (at least 1): the FP32 hits that the watertight test
// accepts just outside an edge.  packWide pads as much again for the box
// test's rounding (kExitSlack, bvh.h).
inline float padLo(float x, float S) { return x - (std::fabs(x) + S) * 9.5367431640625e-07f; }
inline float padHi(float x, float S) { return x + (std::fabs(x) + S) * 9.5367431640625e-07f; }

} // namespace

void buildBvh(const float *tv, uint32_t numTris, BvhBuildResult &out) {
    auto t0 = std::chrono::steady_clock::now();
    Builder b;
    b.primBox.resize(numTris);
    b.centroid.resize(3 * (size_t)numTris);
    b.order.resize(numTris);
    float S = 1.0f;
    for (size_t k = 0; k < 9 * (size_t)numTris; ++k) S = std::max(S, std::fabs(tv[k]));
    for (uint32_t i = 0; i < numTris; ++i) {
        Box &bx = b.primBox[i];
        bx.reset();
        for (int k = 0; k < 3; ++k) bx.grow(&tv[9 * (size_t)i + 3 * k]);
        for (int a = 0; a < 3; ++a) {
            bx.lo[a] = padLo(bx.lo[a], S);
            bx.hi[a] = padHi(bx.hi[a], S);
            b.centroid[3 * (size_t)i + a] = 0.5f * (bx.lo[a] + bx.hi[a]);
        }
        b.order[i] = i;
    }
    Box all;
    all.reset();
    int32_t root = numTris > 0 ? b.build(0, numTris, 0, all) : makeLeaf(0, 1);
    if (root < 0) {
        // a single leaf (or nothing): wrap it in an internal root whose
        // second child has an empty box and is never entered
        Box empty; // a point far outside any ray's [tmin, tmax]: never entered
        for (int a = 0; a < 3; ++a) empty.lo[a] = empty.hi[a] = 1e30f;
        if (numTris == 0) all = empty;
        b.nodes.emplace_back();
        Builder::setNode(b.nodes.back(), all, empty, root, makeLeaf(0, 1));
        b.maxDepth = 0;
    }
    out.scale = S;
    out.binaryDepth = b.maxDepth + 1;
    Collapser c{b.nodes, {}, 0};
    c.collapse(0, 1);
    out.nodes = std::move(c.out);
    out.primOrder = std::move(b.order);
    out.maxDepth = c.maxDepth;
    auto t1 = std::chrono::steady_clock::now();
    out.buildMs = std::chrono::duration<double, std::milli>(t1 - t0).count();
}

} // namespace rtx
