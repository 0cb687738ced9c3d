// Structural check of the eight-wide nodes (rtx::packWide, csrc/bvh_wide.cpp)
// over the triangle sets of bvh_check.cpp: every triangle is reached once from
// the root, inner children and leaf triangles lie inside their arrays, no
// tree is deeper than the traversal's stack, and every finite vertex of a
// leaf's triangles lies inside the decoded box of that leaf and of all its
// ancestors, with the padding the traversal's rounding needs.
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>
#include "bvh.h"
using namespace rtx;
static int fails = 0;
struct Range { double lo[3], hi[3]; };
struct Entry { uint32_t node; std::vector<Range> boxes; };
static void check(const std::vector<float> &v, const char *name) {
    const uint32_t n = (uint32_t)(v.size() / 9);
    BvhBuildResult r;
    WideBvh w;
    try {
        buildBvh(v.data(), n, r);
        packWide(r, w);
    } catch (std::exception &e) { printf("%s: threw %s\n", name, e.what()); ++fails; return; }
    std::vector<int> cover(n, 0);
    std::vector<bool> reached(w.nodes.size(), false);
    if (w.triOrder.size() != n || w.maxDepth > (uint32_t)kStackCapacity) { printf("%s: %zu triangles, depth %u\n", name, w.triOrder.size(), w.maxDepth); ++fails; return; }
    const double S = std::isfinite(r.scale) ? r.scale : 0.0;
    double children = 0;
    std::vector<Entry> st{{0, {}}};
    while (!st.empty()) {
        Entry en = st.back();
        st.pop_back();
        if (en.node >= w.nodes.size() || reached[en.node]) { printf("%s: node %u\n", name, en.node); ++fails; return; }
        reached[en.node] = true;
        const Bvh8Node &nd = w.nodes[en.node];
        if ((nd.imask & ~nd.valid) || nd.childBase % kWideNodeSlots || nd.triBase % 3) { printf("%s: masks\n", name); ++fails; return; }
        uint32_t inner = nd.childBase / kWideNodeSlots, tri = nd.triBase / 3;
        for (int s = 0; s < 8; ++s) {
            const uint32_t count = (nd.counts >> (4 * s)) & 15u;
            if (!((nd.valid >> s) & 1)) { if (count) { printf("%s: unused slot with triangles\n", name); ++fails; return; } continue; }
            children++;
            Range b;
            for (int a = 0; a < 3; ++a) {
                b.lo[a] = nd.p[a] + std::ldexp((double)nd.q[2 * a][s], nd.e[a] - 127);
                b.hi[a] = nd.p[a] + std::ldexp((double)nd.q[2 * a + 1][s], nd.e[a] - 127);
            }
            std::vector<Range> boxes = en.boxes;
            boxes.push_back(b);
            if ((nd.imask >> s) & 1) {
                if (count) { printf("%s: inner child with triangles\n", name); ++fails; return; }
                st.push_back({inner++, boxes});
                continue;
            }
            if (count == 0 || count > kWideLeafMax) { printf("%s: leaf of %u\n", name, count); ++fails; return; }
            for (uint32_t k = 0; k < count; ++k, ++tri) {
                if (tri >= n || w.triOrder[tri] >= n) { printf("%s: leaf past the triangles\n", name); ++fails; return; }
                cover[w.triOrder[tri]]++;
                const float *t = &v[9 * (size_t)w.triOrder[tri]];
                for (const Range &x : boxes)
                    for (int q = 0; q < 3; ++q)
                        for (int a = 0; a < 3; ++a) {
                            const double c = t[3 * q + a], pad = (std::fabs(c) + S) * 0x1p-19 * 0.99;
                            if (!std::isfinite(c) || std::fabs(c) > 1e38) continue;
                            if (c - pad < x.lo[a] || c + pad > x.hi[a]) { printf("%s: vertex %.9g of %u outside [%.9g, %.9g]\n", name, c, w.triOrder[tri], x.lo[a], x.hi[a]); ++fails; return; }
                        }
            }
        }
    }
    for (uint32_t i = 0; i < n; ++i) if (cover[i] != 1) { printf("%s: triangle %u covered %d times\n", name, i, cover[i]); ++fails; break; }
    for (size_t i = 0; i < reached.size(); ++i) if (!reached[i]) { printf("%s: node %zu not reached\n", name, i); ++fails; break; }
    printf("%s: %u triangles, %zu nodes, %.2f children a node, depth %u\n", name, n, w.nodes.size(), children / w.nodes.size(), w.maxDepth);
}
int main() {
    std::mt19937 g(1);
    std::uniform_real_distribution<float> u(-1, 1);
    auto rnd = [&](uint32_t n, float s) { std::vector<float> v(9 * (size_t)n); for (auto &x : v) x = u(g) * s; return v; };
    check({}, "empty");
    for (uint32_t n : {1u, 2u, 7u, 8u, 9u, 15u, 16u, 17u, 64u, 65u}) check(rnd(n, 1), ("random" + std::to_string(n)).c_str());
    check(rnd(100000, 10), "random100k");
    { auto v = rnd(20000, 1e-3f); for (size_t i = 0; i < v.size(); ++i) v[i] += 1000.0f; check(v, "far20k"); }
    for (uint32_t k : {15u, 16u, 17u, 5000u}) { auto v = rnd(1, 1); std::vector<float> w; for (uint32_t i = 0; i < k; ++i) w.insert(w.end(), v.begin(), v.end()); check(w, ("identical" + std::to_string(k)).c_str()); }
    { std::vector<float> w(9 * 3000, 0.5f); check(w, "points3000"); }
    { std::vector<float> w; for (int i = 0; i < 4000; ++i) { float x = i * 1e-3f; float t[9] = {x, 0, 0, x, 1, 0, x, 0, 1}; w.insert(w.end(), t, t + 9); } check(w, "planes4000"); }
    { auto v = rnd(2000, 1); for (size_t i = 0; i < v.size(); i += 97) v[i] = NAN; check(v, "nan"); }
    { auto v = rnd(2000, 1); for (size_t i = 0; i < 900; ++i) v[i] = NAN; check(v, "nan_triangles"); }
    { auto v = rnd(2000, 1); for (size_t i = 0; i < v.size(); i += 89) v[i] = INFINITY; check(v, "inf"); }
    { auto v = rnd(3000, 1); for (size_t i = 0; i < v.size(); i += 3) v[i] *= 1e30f; check(v, "huge"); }
    { auto v = rnd(3000, 1); for (size_t i = 0; i < v.size(); i += 3) v[i] *= 1e-38f; check(v, "flat"); }
    { std::vector<float> w; for (int i = 0; i < 60000; ++i) { float x = std::ldexp(1.0f, -(i % 120)); float t[9] = {x, x, x, x * 2, x, x, x, x * 2, x}; w.insert(w.end(), t, t + 9); } check(w, "geometric60000"); }
    { std::vector<float> w; for (int i = 0; i < 60000; ++i) { const float x = std::pow(4.0f, -(float)(i % 60)) * ((i / 60) % 2 ? -1.0f : 1.0f); float t[9] = {x, x, x, x * 2, x, x, x, x * 2, x}; w.insert(w.end(), t, t + 9); } check(w, "nested60000"); } // a four-wide tree of more than 21 levels
    printf("fails %d\n", fails);
    return fails != 0;
}
