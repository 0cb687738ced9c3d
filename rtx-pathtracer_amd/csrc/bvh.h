// Bounding-volume hierarchy layout and host builder (pure C++).
#pragma once

#include <cstdint>
#include <vector>

namespace rtx {

// ----------------------------------------------------------------- BVH
// The builder makes a binary SAH tree (64-byte two-box nodes) and collapses
// it into four-wide nodes in FP32:
//   f[0] = lo.x of children 0-3   f[1] = hi.x
//   f[2] = lo.y                   f[3] = hi.y
//   f[4] = lo.z                   f[5] = hi.z
//   link[0..3], pad
// link >= 0: internal node index; link < 0: leaf, ~link = start << 4 | (count - 1).
// An unused child slot has a point box at 1e30 that no ray reaches.
struct BvhNode {
    float a[4], b[4], c[4];
    int32_t d[4];
};
static_assert(sizeof(BvhNode) == 64, "BvhNode must be 64 bytes");

struct Bvh4Node {
    float f[6][4];
    int32_t link[4];
    int32_t pad[4];
};
static_assert(sizeof(Bvh4Node) == 128, "Bvh4Node must be 128 bytes");

// The eight-wide nodes the kernels read, packed from the four-wide tree: 80 B,
// five 16-byte loads.  A child's box on axis a is p[a] + 2^(e[a] - 127) *
// [q[2a][slot], q[2a + 1][slot]], rounded outwards from the four-wide box
// grown by a further (|x| + S) 2^-20.  valid and imask have a bit per slot:
// used, and an inner node (the others are leaves).  The inner children are
// the nodes after childBase and the leaves' triangles those after triBase,
// both in slot order; a leaf's triangle count (1 to 15) is its nibble of counts.
// childBase and triBase are in 16-byte units from the start of their arrays.
struct Bvh8Node {
    float p[3];
    uint8_t e[3];
    uint8_t imask;
    uint32_t childBase, triBase, counts;
    uint8_t valid;
    uint8_t pad[3];
    uint8_t q[6][8];
};
static_assert(sizeof(Bvh8Node) == 80, "Bvh8Node must be 80 bytes");
constexpr uint32_t kWideNodeSlots = 5;       // 16-byte loads per node
constexpr uint32_t kWideLeafMax = 15;        // triangles of one leaf child
constexpr uint64_t kWideNodeMax = 0xFFFFFFFFull / kWideNodeSlots;
constexpr uint32_t kWideNodeBytes = 80;

// ------------------------------------------------- rays against the boxes
// The arithmetic of the traversal's box test (nodeStep, dev_traverse.h), for the
// kernels and for the CPU check of it.
#ifdef __HIP__
#define RTX_BOX __attribute__((host, device)) inline
#else
#define RTX_BOX inline
#endif
// Plane q of an axis is at ray parameter
// fma(q, 2^(e - 127) * inv, planeOrigin(p, inv, o * inv)).

// A zero direction component gets a tiny stand-in, so that its planes come out
// as far away on one side or the other instead of 0 * inf.
RTX_BOX float slabDirection(float d) { return d != 0.0f ? d : __builtin_copysignf(1e-30f, d); }

// The parameter of the plane through p.  Where it overflows (a component near
// zero and a plane far away) every plane of the node would be at the same
// infinity, and a box that the ray is in would be culled, so it is made NaN:
// the axis' planes are NaN then, which the minima and maxima pass over, and the
// axis constrains nothing.  (x * 0 is NaN for an infinite x.  A step
// 2^(e - 127) inv that overflows by itself has the next plane 1e31 away.)
// One FMA an axis and visit: the 1080p room 61.9 ms (62.3 without), its cache
// frames 304.0 (303.7), the 256x256 preview 1.17 (1.16).  Bounding 1 / d by the
// scene's extent where a ray is set up costs the visits nothing, but the
// shading kernels, which set rays up in a rare branch, spilled more: cache
// frames 308 ms beside 304.
RTX_BOX float planeOrigin(float p, float inv, float oinv) {
    const float x = __builtin_fmaf(p, inv, -oinv);
    return __builtin_fmaf(x, 0.0f, x);
}

// Entry and exit are each off by less than a factor 1 + gamma_4, gamma_4 =
// 4 u / (1 - 4 u) with u = 2^-24 (Ize, "Robust BVH ray traversal", JCGT 2013):
// u from 1 / d, u from the last FMA of a plane at l, and less than 2 u from
// o inv and the origin plane's FMA, whose errors add up to (2 |o| + |p|) u in
// units of |inv|.  The padding that packWide adds, 16 u (|l| + S), holds those
// for |o| up to 7.5 S (o on the plane's axis); from farther away what is left
// of them is below 2 u |l - o|.  So 1 + 10 u, which is above (1 + gamma_4) /
// (1 - gamma_4), never culls a box that the exact ray touches, from any origin.
constexpr float kExitSlack = 1.0000006f;
// The box is entered unless this is negative (a NaN, of two infinities, counts
// as entered).
RTX_BOX float entryMargin(float tnear, float tfar) { return __builtin_fmaf(tfar, kExitSlack, -tnear); }

constexpr int kLeafMaxPrims = 16;
constexpr int kMaxBvhDepth = 48;   // depth limit of the binary build
constexpr int kStackCapacity = 64; // traversal stack entries, at most one a level of eight-wide nodes

inline int32_t makeLeaf(uint32_t start, uint32_t count) {
    return ~(int32_t)((start << 4) | (count - 1));
}

struct BvhBuildResult {
    std::vector<Bvh4Node> nodes;
    std::vector<uint32_t> primOrder; // triangle ids in leaf order
    uint32_t maxDepth = 0;   // of the four-wide tree (levels of nodes)
    uint32_t binaryDepth = 0;
    double buildMs = 0;
    float scale = 1.0f; // largest coordinate magnitude, at least 1 (the padding's S)
};

struct WideBvh {
    std::vector<Bvh8Node> nodes;    // root at 0
    std::vector<uint32_t> triOrder; // triangle ids in the leaves' order
    uint32_t maxDepth = 0;
};

// Binned-SAH build over triangles given as 9 floats each (world space).
void buildBvh(const float *triVerts, uint32_t numTris, BvhBuildResult &out);

// The eight-wide nodes of a built tree (bvh_wide.cpp).
void packWide(const BvhBuildResult &tree, WideBvh &out);

} // namespace rtx
