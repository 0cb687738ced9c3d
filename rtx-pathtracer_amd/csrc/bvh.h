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
