// The traversal's box test (csrc/bvh.h) over the nodes of rtx::packWide: a ray
// walks the tree as nodeStep does (csrc/dev_traverse.h; order and stack apart),
// and every triangle whose bounding box the exact ray touches, in 80-bit
// arithmetic, must lie in a leaf that the walk reaches.  Rays that run along
// an axis, exactly and nearly, random ones, from inside and from far outside,
// over scenes whose extent is 1 to 1e30.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <limits>
#include <random>
#include <string>
#include <vector>
#include "bvh.h"
using namespace rtx;
static int fails = 0;
struct Ray { float o[3], d[3]; };

// max and min that pass over a NaN, as the device's do
static float above(float a, float b) { return std::isnan(a) ? b : std::isnan(b) ? a : a > b ? a : b; }
static float below(float a, float b) { return std::isnan(a) ? b : std::isnan(b) ? a : a < b ? a : b; }

static void walk(const WideBvh &w, const Ray &r, float tmin, float tmax, std::vector<bool> &reached) {
    float inv[3], oinv[3];
    for (int a = 0; a < 3; ++a) {
        inv[a] = 1.0f / slabDirection(r.d[a]);
        oinv[a] = r.o[a] * inv[a];
    }
    std::vector<uint32_t> st{0};
    while (!st.empty()) {
        const Bvh8Node &n = w.nodes[st.back()];
        st.pop_back();
        uint32_t inner = n.childBase / kWideNodeSlots, tri = n.triBase / 3;
        for (int s = 0; s < 8; ++s) {
            if (!((n.valid >> s) & 1)) continue;
            float tn = 0.0f, tf = 0.0f;
            for (int a = 0; a < 3; ++a) {
                const uint32_t e = (uint32_t)n.e[a] << 23;
                float scale;
                std::memcpy(&scale, &e, 4);
                scale *= inv[a];
                const float org = planeOrigin(n.p[a], inv[a], oinv[a]);
                const bool neg = inv[a] < 0.0f;
                const float en = std::fma((float)n.q[2 * a + (neg ? 1 : 0)][s], scale, org);
                const float ex = std::fma((float)n.q[2 * a + (neg ? 0 : 1)][s], scale, org);
                tn = a ? above(tn, en) : en;
                tf = a ? below(tf, ex) : ex;
            }
            const float m = entryMargin(above(tn, tmin), below(tf, tmax));
            const bool enter = std::isnan(m) || !std::signbit(m);
            const uint32_t count = (n.counts >> (4 * s)) & 15u;
            if ((n.imask >> s) & 1) {
                if (enter) st.push_back(inner);
                ++inner;
            } else {
                for (uint32_t k = 0; k < count; ++k, ++tri)
                    if (enter) reached[w.triOrder[tri]] = true;
            }
        }
    }
}

// Whether the exact ray touches the bounding box of triangle t in [tmin, tmax].
static bool touches(const float *t, const Ray &r, long double tmin, long double tmax) {
    long double n = tmin, f = tmax;
    for (int a = 0; a < 3; ++a) {
        const long double lo = std::fmin(t[a], std::fmin(t[3 + a], t[6 + a])), hi = std::fmax(t[a], std::fmax(t[3 + a], t[6 + a]));
        const long double o = r.o[a], d = r.d[a];
        if (d == 0) {
            if (o < lo || o > hi) return false;
            continue;
        }
        const long double x = (lo - o) / d, y = (hi - o) / d;
        n = std::fmax(n, std::fmin(x, y));
        f = std::fmin(f, std::fmax(x, y));
    }
    return n <= f;
}

static void check(const std::vector<float> &v, const std::vector<Ray> &rays, const std::string &name) {
    const uint32_t n = (uint32_t)(v.size() / 9);
    BvhBuildResult b;
    WideBvh w;
    buildBvh(v.data(), n, b);
    packWide(b, w);
    size_t touched = 0, lost = 0;
    for (const Ray &r : rays) {
        std::vector<bool> reached(n, false);
        walk(w, r, 0.0f, std::numeric_limits<float>::max(), reached);
        for (uint32_t i = 0; i < n; ++i) {
            if (!touches(&v[9 * (size_t)i], r, 0.0L, std::numeric_limits<float>::max())) continue;
            ++touched;
            if (reached[i]) continue;
            if (lost++ == 0)
                printf("%s: triangle %u not reached from (%g, %g, %g) along (%g, %g, %g)\n", name.c_str(), i, r.o[0],
                       r.o[1], r.o[2], r.d[0], r.d[1], r.d[2]);
        }
    }
    if (touched < rays.size() / 4) { printf("%s: only %zu triangles touched\n", name.c_str(), touched); ++fails; }
    if (lost) ++fails;
    printf("%s: %zu rays, %zu triangles touched, %zu not reached\n", name.c_str(), rays.size(), touched, lost);
}

int main() {
    std::mt19937 g(3);
    std::uniform_real_distribution<float> u(-1, 1);
    const float tiny[] = {0.0f, -0.0f, 1e-10f, -1e-20f, 1e-30f, -1e-33f, 1e-36f, -1e-37f, 1e-40f, -1e-44f};
    for (float ext : {1.0f, 100.0f, 1e3f, 1e6f, 4e8f, 1e9f, 1e15f, 1e20f, 1e25f, 1e30f}) {
        // a ground over the whole extent and boxes of all sizes on it
        std::vector<float> v{-ext, -ext, 0, ext, -ext, 0, ext, ext, 0, -ext, -ext, 0, ext, ext, 0, -ext, ext, 0};
        for (int i = 0; i < 400; ++i) {
            float c[3];
            for (float &x : c) x = u(g) * ext;
            const float size = ext * std::ldexp(1.0f, -(i % 20));
            for (int k = 0; k < 9; ++k) v.push_back(c[k % 3] + u(g) * size);
        }
        std::vector<Ray> rays;
        auto aim = [&](Ray &r, float far) { // at a point of a triangle, from far extents away
            const size_t t = (size_t)((u(g) * 0.5f + 0.5f) * 0.999f * (v.size() / 9));
            float d[3], len = 0;
            for (float &x : d) x = u(g), len += x * x;
            for (int a = 0; a < 3; ++a) {
                r.d[a] = d[a] / std::sqrt(len);
                r.o[a] = (v[9 * t + a] + v[9 * t + 3 + a] + v[9 * t + 6 + a]) / 3.0f - r.d[a] * (far * ext);
            }
        };
        for (float s : tiny)
            for (float s2 : tiny)
                for (int axis = 0; axis < 3; ++axis)
                    for (int k = 0; k < 4; ++k) {
                        Ray r;
                        aim(r, 0.0f);
                        r.d[axis] = k & 1 ? 1.0f : -1.0f;
                        r.d[(axis + 1) % 3] = s;
                        r.d[(axis + 2) % 3] = s2;
                        r.o[axis] -= r.d[axis] * (k & 2 ? 3.0f : 0.5f) * ext;
                        rays.push_back(r);
                    }
        for (float far : {0.0f, 0.5f, 3.0f, 10.0f, 30.0f, 100.0f, 1e3f, 1e4f, 1e5f})
            for (int k = 0; k < 300; ++k) {
                Ray r;
                aim(r, far);
                rays.push_back(r);
            }
        char name[32];
        snprintf(name, sizeof(name), "extent %g", ext);
        check(v, rays, name);
    }
    printf("fails %d\n", fails);
    return fails != 0;
}
