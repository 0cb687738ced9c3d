// Eight-wide, quantised nodes for the traversal kernels, packed from the
// builder's four-wide tree (bvh_build.cpp).
//
// The traversal is bound by the address processing of its node loads (one
// cache access per lane and 16-byte load) and by the number of dependent
// visits a ray makes, not by bytes: so a node holds as many children as fit
// in few 16-byte loads.  Eight children with boxes on an 8-bit grid take 80
// bytes, five loads; four children in FP32 took seven.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <limits>
#include <stdexcept>

#include "bvh.h"

namespace rtx {

namespace {

// Bounds are clamped to this before they are quantised (a vertex that is not
// finite is never hit, so only its neighbours need their boxes), so that an
// extent stays finite.
constexpr float kFar = 1.7e38f;

// 2^e and the exponent of a positive normal double
inline double powerOf2(int e) {
    const uint64_t bits = (uint64_t)(e + 1023) << 52;
    double d;
    std::memcpy(&d, &bits, sizeof(d));
    return d;
}
inline int exponentOf(double d) {
    uint64_t bits;
    std::memcpy(&bits, &d, sizeof(d));
    return (int)(bits >> 52) - 1023;
}

struct Bounds {
    float lo[3], hi[3];
    void grow(const Bounds &b) {
        for (int a = 0; a < 3; ++a) {
            lo[a] = std::min(lo[a], b.lo[a]);
            hi[a] = std::max(hi[a], b.hi[a]);
        }
    }
    float area() const {
        const float dx = hi[0] - lo[0], dy = hi[1] - lo[1], dz = hi[2] - lo[2];
        return std::min(2.0f * (dx * dy + dy * dz + dz * dx), 1e30f); // finite costs whatever the box
    }
};

// The four-wide tree as a binary one: an inner node's children, or a leaf's
// triangles [first, first + count).
struct Bin {
    Bounds box;
    int32_t left = -1, right = -1;
    uint32_t first = 0, count = 0;
    bool leaf() const { return left < 0; }
};

struct Packer {
    const std::vector<Bvh4Node> &in;
    const std::vector<uint32_t> &order;
    float pad; // S 2^-20, the absolute part of the extra padding
    WideBvh &out;
    std::vector<Bin> bins;

    static int childCount(const Bvh4Node &n) {
        int c = 4;
        while (c > 0 && n.f[0][c - 1] == 1e30f && n.f[1][c - 1] == 1e30f) c--;
        return c;
    }
    static Bounds childBox(const Bvh4Node &n, int k) {
        Bounds b;
        for (int a = 0; a < 3; ++a) {
            float lo = n.f[2 * a][k], hi = n.f[2 * a + 1][k];
            if (!(lo <= hi)) { // no finite vertex on this axis: nothing in it is ever hit
                lo = -kFar;
                hi = kFar;
            }
            b.lo[a] = std::min(std::max(lo, -kFar), kFar);
            b.hi[a] = std::min(std::max(hi, -kFar), kFar);
        }
        return b;
    }

    // ------------------------------------------------------ binary tree
    int32_t makeInner(int32_t left, int32_t right) {
        Bin b;
        b.left = left;
        b.right = right;
        b.box = bins[left].box;
        b.box.grow(bins[right].box);
        bins.push_back(b);
        return (int32_t)bins.size() - 1;
    }
    int32_t makeTris(const Bounds &box, uint32_t first, uint32_t count) {
        if (count > kWideLeafMax) { // more than a leaf child holds
            const int32_t l = makeTris(box, first, count / 2), r = makeTris(box, first + count / 2, count - count / 2);
            return makeInner(l, r);
        }
        Bin b;
        b.box = box;
        b.first = first;
        b.count = count;
        bins.push_back(b);
        return (int32_t)bins.size() - 1;
    }
    int32_t fromChild(int32_t node, int k) {
        const int32_t l = in[node].link[k];
        if (l >= 0) return fromRange(l, 0, childCount(in[l]));
        const uint32_t code = ~(uint32_t)l;
        return makeTris(childBox(in[node], k), code >> 4, (code & 15u) + 1u);
    }
    // The children [a, b) of a four-wide node: they are in the binary build's
    // left-to-right order, and the cheapest of the at most three cuts stands
    // for the binary split.
    int32_t fromRange(int32_t node, int a, int b) {
        if (b - a == 1) return fromChild(node, a);
        Bounds below[4], above[4];
        below[a] = childBox(in[node], a);
        for (int k = a + 1; k < b; ++k) (below[k] = below[k - 1]).grow(childBox(in[node], k));
        above[b - 1] = childBox(in[node], b - 1);
        for (int k = b - 2; k >= a; --k) (above[k] = above[k + 1]).grow(childBox(in[node], k));
        int cut = a + 1;
        float best = std::numeric_limits<float>::infinity();
        for (int c = a + 1; c < b; ++c) {
            const float cost = below[c - 1].area() + above[c].area();
            if (cost < best) {
                best = cost;
                cut = c;
            }
        }
        const int32_t l = fromRange(node, a, cut), r = fromRange(node, cut, b);
        return makeInner(l, r);
    }

    // Writes node `self` over subtree `id` and, after it, the nodes below;
    // its inner children get consecutive nodes, its leaves consecutive
    // triangles, both in slot order.
    void pack(int32_t id, uint32_t self, uint32_t depth) {
        out.maxDepth = std::max(out.maxDepth, depth);
        // The largest inner child is opened until the node is full.  (The
        // collapse of least expected cost, by dynamic programming over the
        // slots, fills 7.4 slots a node instead of 4.5 and makes rays visit 2%
        // fewer nodes, but it merges and lifts leaves: 6 to 9% more triangle
        // tests, and the 1080p images took 1% longer.)
        int32_t kids[8] = {id};
        int n = 1;
        while (n < 8) {
            int best = -1;
            float bestArea = -1.0f;
            for (int k = 0; k < n; ++k)
                if (!bins[kids[k]].leaf() && bins[kids[k]].box.area() > bestArea) {
                    bestArea = bins[kids[k]].box.area();
                    best = k;
                }
            if (best < 0) break;
            const Bin &o = bins[kids[best]];
            kids[best] = o.left;
            kids[n++] = o.right;
        }
        const Bin *ch[8] = {};
        for (int k = 0; k < n; ++k) ch[k] = &bins[kids[k]];
        Bounds all = ch[0]->box;
        for (int k = 1; k < n; ++k) all.grow(ch[k]->box);
        // Slots by direction: bit a of a slot says on which side of the node
        // its child lies along axis a, so that visiting slots in the order of
        // (slot ^ the ray's sign bits) goes roughly front to back.  Greedy:
        // the child and slot that agree most first.
        int slotOf[8], at[8];
        float toward[8][8];
        for (int k = 0; k < n; ++k) {
            float c[3];
            for (int a = 0; a < 3; ++a)
                c[a] = (0.5f * ch[k]->box.lo[a] + 0.5f * ch[k]->box.hi[a]) - (0.5f * all.lo[a] + 0.5f * all.hi[a]);
            for (int s = 0; s < 8; ++s)
                toward[k][s] = (s & 1 ? c[0] : -c[0]) + (s & 2 ? c[1] : -c[1]) + (s & 4 ? c[2] : -c[2]);
        }
        for (int s = 0; s < 8; ++s) at[s] = -1;
        uint32_t open = (1u << n) - 1u;
        for (int done = 0; done < n; ++done) {
            int bk = -1, bs = -1;
            for (int k = 0; k < n; ++k) {
                if (!((open >> k) & 1u)) continue;
                for (int s = 0; s < 8; ++s)
                    if (at[s] < 0 && (bk < 0 || toward[k][s] > toward[bk][bs])) bk = k, bs = s;
            }
            open &= ~(1u << bk);
            slotOf[bk] = bs;
            at[bs] = bk;
        }
        // the grid: origin and a power of two per axis, boxes rounded outwards
        Bvh8Node node;
        std::memset(&node, 0, sizeof(node));
        for (int a = 0; a < 3; ++a) {
            double lo[8], hi[8], least = std::numeric_limits<double>::infinity(), most = -least;
            for (int k = 0; k < n; ++k) {
                const double l = ch[k]->box.lo[a], h = ch[k]->box.hi[a];
                lo[k] = l - (std::fabs(l) * 0x1p-20 + pad);
                hi[k] = h + (std::fabs(h) * 0x1p-20 + pad);
                least = std::min(least, lo[k]);
                most = std::max(most, hi[k]);
            }
            float p = (float)least;
            if ((double)p > least) p = std::nextafter(p, -std::numeric_limits<float>::infinity());
            const double ext = most - (double)p;
            int e = ext > 0.0 ? std::max(exponentOf(ext * (1.0 / 255.0)), -126) : -126;
            while (powerOf2(e) * 255.0 < ext) e++;
            node.p[a] = p;
            node.e[a] = (uint8_t)(e + 127);
            const double inv = powerOf2(-e);
            for (int k = 0; k < n; ++k) {
                // both at least 0 and, by the choice of e, at most 255; truncation is the floor
                const double l = std::max((lo[k] - (double)p) * inv, 0.0), h = std::min((hi[k] - (double)p) * inv, 255.0);
                const int qh = (int)h;
                node.q[2 * a][slotOf[k]] = (uint8_t)(int)std::min(l, 255.0);
                node.q[2 * a + 1][slotOf[k]] = (uint8_t)(qh + ((double)qh < h ? 1 : 0));
            }
        }
        uint32_t inner = 0;
        const uint32_t firstTri = (uint32_t)out.triOrder.size();
        for (int s = 0; s < 8; ++s) {
            if (at[s] < 0) continue;
            const Bin &c = *ch[at[s]];
            node.valid |= (uint8_t)(1u << s);
            if (!c.leaf()) {
                node.imask |= (uint8_t)(1u << s);
                inner++;
            } else {
                node.counts |= c.count << (4 * s);
                for (uint32_t t = c.first; t < c.first + c.count; ++t) out.triOrder.push_back(order[t]);
            }
        }
        const uint32_t base = (uint32_t)out.nodes.size();
        if ((uint64_t)base + inner > kWideNodeMax) throw std::runtime_error("BVH has too many nodes");
        node.childBase = base * kWideNodeSlots;
        node.triBase = firstTri * 3u;
        out.nodes.resize(out.nodes.size() + inner);
        out.nodes[self] = node;
        uint32_t next = base;
        for (int s = 0; s < 8; ++s)
            if (at[s] >= 0 && !ch[at[s]]->leaf()) pack(kids[at[s]], next++, depth + 1);
    }
};

} // namespace

void packWide(const BvhBuildResult &tree, WideBvh &out) {
    out = WideBvh{};
    out.triOrder.reserve(tree.primOrder.size());
    if (tree.primOrder.empty()) { // one node without children
        out.nodes.resize(1);
        std::memset(&out.nodes[0], 0, sizeof(Bvh8Node));
        out.maxDepth = 1;
        return;
    }
    Packer p{tree.nodes, tree.primOrder, std::min(tree.scale, kFar) * 0x1p-20f, out, {}};
    p.bins.reserve(8 * tree.nodes.size());
    const int32_t root = p.fromRange(0, 0, Packer::childCount(tree.nodes[0]));
    out.nodes.resize(1);
    p.pack(root, 0, 1);
    if (out.maxDepth > (uint32_t)kStackCapacity) throw std::runtime_error("BVH too deep for the traversal stack");
}

} // namespace rtx
