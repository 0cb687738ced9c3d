// BVH traversal on the device.  Replaces the RT-core traversal behind the
// reference's traceRayEXT calls (closest hit: shaders/raytrace.rgen:1011-1022;
// shadow any-hit with TerminateOnFirstHit: raytrace.rgen:622-638) and the
// sphere intersection shader (raytrace.sphere.rint:11-29).
//
// Stack-based traversal (Aila & Laine 2009) over eight-wide quantised nodes
// (csrc/bvh.h).  The stack's first LDS_DEPTH entries live in LDS (one column
// per thread, so consecutive lanes hit consecutive banks), deeper entries in
// a private array; an entry is one node's children still to visit, so the
// stack holds at most one a level (kStackCapacity).
#pragma once

#include "dev_math.h"
#include "dev_texture.h"
#include "internal.h"

namespace rtx {

struct TravRay {
    V3 o, d, inv;
    V3 oinv; // o * inv: a plane at l is fma(l, inv, -oinv) away
    // the slots a node's children are looked at in first, by the ray's signs:
    // of each half, quarter and pair (WideBvh's slot order)
    uint32_t near4, near2, near1;
    int kx, ky, kz;
    float Sx, Sy, Sz;
};

RTX_DI TravRay makeTravRay(V3 o, V3 d) {
    TravRay r;
    r.o = o;
    r.d = d;
    r.inv = v3(1.0f / slabDirection(d.x), 1.0f / slabDirection(d.y), 1.0f / slabDirection(d.z));
    r.oinv = v3(o.x * r.inv.x, o.y * r.inv.y, o.z * r.inv.z);
    r.near1 = r.inv.x < 0.0f ? 0xAAu : 0x55u;
    r.near2 = r.inv.y < 0.0f ? 0xCCu : 0x33u;
    r.near4 = r.inv.z < 0.0f ? 0xF0u : 0x0Fu;
    // watertight test set-up (Woop, Benthin, Wald, JCGT 2013)
    float ax = fabsf(d.x), ay = fabsf(d.y), az = fabsf(d.z);
    int kz = (ax > ay) ? (ax > az ? 0 : 2) : (ay > az ? 1 : 2);
    int kx = kz == 2 ? 0 : kz + 1;
    int ky = kx == 2 ? 0 : kx + 1;
    if (sel(d, kz) < 0.0f) {
        int t = kx;
        kx = ky;
        ky = t;
    }
    r.kx = kx;
    r.ky = ky;
    r.kz = kz;
    float dkz = sel(d, kz);
    r.Sx = sel(d, kx) / dkz;
    r.Sy = sel(d, ky) / dkz;
    r.Sz = 1.0f / dkz;
    return r;
}

// Watertight ray/triangle test.  Products are not contracted into FMAs so
// that the edge functions of a shared edge are exact negatives.  Returns
// the hit distance and the barycentrics of vertices 1 and 2 (the
// reference's hit attributes, raytrace.rchit:28).
RTX_DI bool isectTri(const TravRay &r, float4 a, float4 b, float4 c, float tmin, float tmax, float &t, float &u,
                     float &v) {
#pragma clang fp contract(off)
    V3 A = v3(a) - r.o, B = v3(b) - r.o, C = v3(c) - r.o;
    float Az0 = sel(A, r.kz), Bz0 = sel(B, r.kz), Cz0 = sel(C, r.kz);
    float Ax = sel(A, r.kx) - r.Sx * Az0, Ay = sel(A, r.ky) - r.Sy * Az0;
    float Bx = sel(B, r.kx) - r.Sx * Bz0, By = sel(B, r.ky) - r.Sy * Bz0;
    float Cx = sel(C, r.kx) - r.Sx * Cz0, Cy = sel(C, r.ky) - r.Sy * Cz0;
    float U = Cx * By - Cy * Bx;
    float V = Ax * Cy - Ay * Cx;
    float W = Bx * Ay - By * Ax;
    if (U == 0.0f || V == 0.0f || W == 0.0f) {
        U = (float)((double)Cx * (double)By - (double)Cy * (double)Bx);
        V = (float)((double)Ax * (double)Cy - (double)Ay * (double)Cx);
        W = (float)((double)Bx * (double)Ay - (double)By * (double)Ax);
    }
    if ((U < 0.0f || V < 0.0f || W < 0.0f) && (U > 0.0f || V > 0.0f || W > 0.0f)) return false;
    float det = U + V + W;
    if (det == 0.0f) return false;
    float Az = r.Sz * Az0, Bz = r.Sz * Bz0, Cz = r.Sz * Cz0;
    float T = U * Az + V * Bz + W * Cz;
    float tt = T / det;
    if (!(tt >= tmin && tt <= tmax)) return false;
    t = tt;
    u = V / det;
    v = W / det;
    return true;
}

// raytrace.sphere.rint:11-29: both roots reported, nearest in [tmin, tmax] kept
RTX_DI bool isectSphere(const rtx_sphere &s, V3 o, V3 d, float tmin, float tmax, float &t) {
    V3 oc = o - v3(s.center);
    float dotDOC = dot(d, oc);
    float rootTerm = dotDOC * dotDOC - dot(oc, oc) + s.radius * s.radius;
    if (rootTerm < 0.0f) return false;
    float root = sqrtf(rootTerm);
    float t1 = -dotDOC + root, t2 = -dotDOC - root;
    bool hit = false;
    float best = tmax;
    if (t1 >= tmin && t1 <= best) {
        best = t1;
        hit = true;
    }
    if (t2 >= tmin && t2 <= best) {
        best = t2;
        hit = true;
    }
    t = best;
    return hit;
}

// Stack with LDS_DEPTH entries in LDS (column per thread, stride BLOCK)
// and the remainder in a private array of kStackCapacity - LDS_DEPTH
// entries.  The private array is a separate local of the caller, not a
// member: a dynamically indexed array inside the struct keeps the whole
// struct in scratch, sp included, and every push and pop then waits on a
// scratch load of sp.
// The two pointers carry their address spaces (3: LDS, 5: private), so that
// a pop, which reads one or the other, compiles to ds_read and scratch_load
// rather than to a flat load of a selected pointer.
typedef uint32_t U32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) U32x2 LdsEntry;
typedef __attribute__((address_space(5))) U32x2 PrivEntry;

template <int BLOCK, int LDS_DEPTH> struct HybridStack {
    static constexpr int kSpill = kStackCapacity - LDS_DEPTH;
    LdsEntry *lds;
    PrivEntry *priv;
    int sp;
    // ldsColumn: this thread's column of the block's LDS stack (stride BLOCK);
    // spill: kSpill private entries.
    RTX_DI void bind(U32x2 *ldsColumn, U32x2 *spill) {
        lds = (LdsEntry *)ldsColumn;
        priv = (PrivEntry *)spill;
    }
    RTX_DI void push(U32x2 x) {
        if (sp < LDS_DEPTH) lds[sp * BLOCK] = x;
        else priv[sp - LDS_DEPTH] = x;
        sp++;
    }
    RTX_DI U32x2 pop() {
        sp--;
        return sp < LDS_DEPTH ? lds[sp * BLOCK] : priv[sp - LDS_DEPTH];
    }
};

// Whole stack in a private array (kStackCapacity entries, the caller's).
struct PrivateStack {
    PrivEntry *priv;
    int sp;
    RTX_DI PrivateStack(U32x2 *spill) : priv((PrivEntry *)spill), sp(0) {}
    RTX_DI void push(U32x2 x) { priv[sp++] = x; }
    RTX_DI U32x2 pop() { return priv[--sp]; }
};

struct VisitCount {
    uint32_t nodes = 0, prims = 0;
};

// Where a ray is in the tree: the inner children of one node still to visit
// (group.x their node's childBase, group.y the slots to visit in bits 0-7 and
// the node's imask in bits 8-15; no bit set: no more nodes), and the leaves of
// the last node still to test (slots in leaves, the node's triBase and counts)
// after the triLeft triangles from tri on of the leaf under way.
struct TravPos {
    U32x2 group;
    uint32_t leaves, triBase, counts;
    uint32_t tri, triLeft;
    RTX_DI bool atNode() const { return (group.y & 0xFFu) != 0u; }
    RTX_DI bool atLeaf() const { return (leaves | triLeft) != 0u; }
};
// The root, as the only child of a node that is not there.
RTX_DI void startPos(TravPos &p) {
    p.group = U32x2{0u, 0x101u};
    p.leaves = p.triLeft = 0u;
}
RTX_DI void endPos(TravPos &p) {
    p.group.y = 0u;
    p.leaves = p.triLeft = 0u;
}

RTX_DI float ubyte(uint32_t w, int k) { return (float)((w >> (8 * k)) & 0xFFu); }

// Of a set of slots, the one the ray comes to first.
RTX_DI int nearSlot(const TravRay &r, uint32_t set) {
    uint32_t h = set & r.near4;
    set = h ? h : set;
    h = set & r.near2;
    set = h ? h : set;
    h = set & r.near1;
    set = h ? h : set;
    return __ffs(set) - 1;
}

// The four-wide FP32 nodes before these took seven 16-byte loads and 28
// visits a ray in the 262,144-triangle room, and the loads' address
// processing bounded the launch (TA busy 95%, 0.70 cache accesses a cycle and
// CU).  These take five loads and 19 visits (TA busy 81%, 0.81 accesses); the
// launch is bound by vector instructions, 0.30 a SIMD and cycle with half the
// lanes active, 48 conversions and 48 FMAs of a visit's 180 first (v_perm pairs
// into v_fma_mix instead of conversions measured the same): 1.49 -> 0.97 ms for
// 2 x 1080p paths (1.85 before the rays went out in chunks), 0.90 in the
// present build.
// One node visit: the next of the group's children in the ray's order is
// taken (the rest pushed), its children's boxes are tested against
// [tmin, tmax], and the entered ones become the group and the leaves to test.
// With no inner child entered the next stack entry becomes the group.
//
// A box plane is one FMA, fma(q, 2^e inv, planeOrigin).  Its rounding is covered
// by the boxes' padding and by the slack on the exit distance (kExitSlack,
// bvh.h), so a box the exact ray touches is never culled, and the hits do not
// depend on the tree.  A NaN plane (an overflow, planeOrigin; 0 * inf) constrains
// nothing: min and max return their other operand.
template <class SceneT, class Stack>
RTX_DI void nodeStep(const SceneT &S, const TravRay &r, float tmin, float tmax, TravPos &pos, Stack &st) {
    const int slot = nearSlot(r, pos.group.y & 0xFFu);
    const uint32_t rank = __popc((pos.group.y >> 8) & ((1u << slot) - 1u));
    const float4 *np = S.nodes + (size_t)(pos.group.x + rank * kWideNodeSlots);
    const uint4 n0 = *reinterpret_cast<const uint4 *>(np), n1 = *reinterpret_cast<const uint4 *>(np + 1);
    const uint4 bx = *reinterpret_cast<const uint4 *>(np + 2), by = *reinterpret_cast<const uint4 *>(np + 3),
                bz = *reinterpret_cast<const uint4 *>(np + 4);
    pos.group.y &= ~(1u << slot);
    if (pos.atNode()) st.push(pos.group);
    const float sx = __uint_as_float((n0.w & 0xFFu) << 23) * r.inv.x;
    const float sy = __uint_as_float(((n0.w >> 8) & 0xFFu) << 23) * r.inv.y;
    const float sz = __uint_as_float(((n0.w >> 16) & 0xFFu) << 23) * r.inv.z;
    const float ox = planeOrigin(__uint_as_float(n0.x), r.inv.x, r.oinv.x);
    const float oy = planeOrigin(__uint_as_float(n0.y), r.inv.y, r.oinv.y);
    const float oz = planeOrigin(__uint_as_float(n0.z), r.inv.z, r.oinv.z);
    const bool negx = r.near1 == 0xAAu, negy = r.near2 == 0xCCu, negz = r.near4 == 0xF0u;
    uint32_t miss = 0; // bit 7 - slot
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        const uint32_t lx = half ? bx.y : bx.x, hx = half ? bx.w : bx.z, ly = half ? by.y : by.x,
                       hy = half ? by.w : by.z, lz = half ? bz.y : bz.x, hz = half ? bz.w : bz.z;
        const uint32_t nx = negx ? hx : lx, fx = negx ? lx : hx, ny = negy ? hy : ly, fy = negy ? ly : hy,
                       nz = negz ? hz : lz, fz = negz ? lz : hz;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float tn = fmaxf(fmaxf(fmaxf(fmaf(ubyte(nx, k), sx, ox), fmaf(ubyte(ny, k), sy, oy)),
                                         fmaf(ubyte(nz, k), sz, oz)),
                                   tmin);
            const float tf = fminf(fminf(fminf(fmaf(ubyte(fx, k), sx, ox), fmaf(ubyte(fy, k), sy, oy)),
                                         fmaf(ubyte(fz, k), sz, oz)),
                                   tmax);
            // the sign of exit - entry, shifted into the slots' misses
            miss = __builtin_amdgcn_alignbit(miss, __float_as_uint(entryMargin(tn, tf)), 31);
        }
    }
    const uint32_t imask = n0.w >> 24;
    const uint32_t hits = (__brev(~miss) >> 24) & (n1.w & 0xFFu);
    pos.leaves = hits & ~imask;
    pos.triBase = n1.y;
    pos.counts = n1.z;
    pos.group = U32x2{n1.x, (hits & imask) | (imask << 8)};
    if (!pos.atNode() && st.sp != 0) pos.group = st.pop();
}

// The next triangle to test (in 16-byte units), at a leaf.
RTX_DI uint32_t nextTri(TravPos &pos) {
    if (pos.triLeft == 0u) {
        const int shift = 4 * (__ffs(pos.leaves) - 1);
        pos.leaves &= pos.leaves - 1u;
        const uint32_t below = pos.counts & ((1u << shift) - 1u);
        // the nibbles' sum: at most 7 x 15
        const uint32_t sum = (((below & 0x0F0F0F0Fu) + ((below >> 4) & 0x0F0F0F0Fu)) * 0x01010101u) >> 24;
        pos.tri = pos.triBase + 3u * sum;
        pos.triLeft = (pos.counts >> shift) & 15u;
    }
    const uint32_t t = pos.tri;
    pos.tri += 3u;
    pos.triLeft--;
    return t;
}

// Closest hit (ANY = false) or first hit (ANY = true) in [tmin, tmax].
// Returns the primitive id (triangles 0..numTris-1, then spheres) or -1.
// Closest-hit ties in t go to the smaller primitive id.  Triangles marked
// with kAlphaBit pass the any-hit alpha test first (randomUInt: the frame's).
template <bool ANY, bool COUNT, class Stack>
RTX_DI int traverse(const DevScene &S, const TravRay &r, float tmin, float &tmax, float &bu, float &bv,
                    Stack &st, VisitCount &vc, uint32_t randomUInt = 0) {
    int best = -1;
    for (uint32_t i = 0; i < S.numSpheres; ++i) {
        float t;
        if (isectSphere(S.spheres[i], r.o, r.d, tmin, tmax, t)) {
            int id = (int)(S.numTris + i);
            if (ANY) return id;
            if (best < 0 || t < tmax || id < best) {
                tmax = t;
                best = id;
                bu = bv = 0.0f;
            }
        }
    }
    st.sp = 0;
    TravPos pos;
    startPos(pos);
    while (pos.atNode()) {
        if (COUNT) vc.nodes++;
        nodeStep(S, r, tmin, tmax, pos, st);
        while (pos.atLeaf()) {
            const float4 *tp = S.tris + (size_t)nextTri(pos);
            if (COUNT) vc.prims++;
            float t, u, v;
            if (isectTri(r, tp[0], tp[1], tp[2], tmin, tmax, t, u, v)) {
                int id = __float_as_int(tp[0].w);
                if (id & kAlphaBit) {
                    id &= ~kAlphaBit;
                    if (!alphaAccept(S, id, r.o.x, t, u, v, randomUInt)) continue;
                }
                if (ANY) return id;
                if (best < 0 || t < tmax || id < best) {
                    tmax = t;
                    best = id;
                    bu = u;
                    bv = v;
                }
            }
        }
    }
    return best;
}

// The part of a scene that traversal reads, per lane: launches that trace
// rays of several scenes (jobs of the serving pool) point each lane at its
// ray's scene when the ray is fetched.
struct LaneScene {
    const float4 *nodes;
    const float4 *tris;
    const rtx_sphere *spheres;
    uint32_t numTris, numSpheres;
    const DevScene *full; // for the any-hit alpha test
};
RTX_DI void pointAt(LaneScene &ls, const DevScene &S, const DevScene *full) {
    ls.nodes = S.nodes;
    ls.tris = S.tris;
    ls.spheres = S.spheres;
    ls.numTris = S.numTris;
    ls.numSpheres = S.numSpheres;
    ls.full = full;
}
RTX_DI bool alphaAccept(const LaneScene &S, int prim, float ox, float t, float bu, float bv, uint32_t randomUInt) {
    return alphaAccept(*S.full, prim, ox, t, bu, bv, randomUInt);
}

// ------------------------------------------------------------------
// Persistent traversal with lane refill (Aila & Laine 2009, sections 4-5):
// each wave loops until the queue is drained; lanes whose ray finished
// fetch a new ray, and node visits and leaf tests alternate: a lane that
// enters leaves waits until enough of the wave's lanes do, then those
// intersect a leaf each together.
struct LaneRay {
    TravRay r;
    float tmin, tmax, bu, bv;
    int best;
    TravPos pos;
    uint32_t idx;
    uint32_t randomUInt; // the frame's, for the any-hit alpha test
    bool any;            // kHitLane: this lane's ray wants any hit
};

// How a persistent launch ends its rays: at the closest hit, at the first
// hit, or per lane (LaneRay::any), so that one launch traces occlusion and
// closest-hit rays side by side.
constexpr int kHitClosest = 0, kHitAny = 1, kHitLane = 2;

// Intersects the lane's next triangle; returns true when an any-hit ray is
// done.
template <int HIT, bool COUNT, bool ALPHA, class SceneT>
RTX_DI bool triStep(const SceneT &S, LaneRay &L, VisitCount &vc) {
    const bool ANY = HIT == kHitAny || (HIT == kHitLane && L.any);
    const float4 *tp = S.tris + (size_t)nextTri(L.pos);
    const float4 v0 = tp[0], v1 = tp[1], v2 = tp[2];
    if (COUNT) vc.prims++;
    float t, u, v;
    if (!isectTri(L.r, v0, v1, v2, L.tmin, L.tmax, t, u, v)) return false;
    int id = __float_as_int(v0.w);
    if (ALPHA && (id & kAlphaBit)) {
        id &= ~kAlphaBit;
        if (!alphaAccept(S, id, L.r.o.x, t, u, v, L.randomUInt)) return false;
    }
    if (ANY) {
        L.best = id;
        return true;
    }
    if (L.best < 0 || t < L.tmax || id < L.best) {
        L.tmax = t;
        L.best = id;
        L.bu = u;
        L.bv = v;
    }
    return false;
}

// Starts a ray: spheres are tested up front (all workloads have few).
template <int HIT, class SceneT> RTX_DI void beginRay(const SceneT &S, LaneRay &L) {
    const bool ANY = HIT == kHitAny || (HIT == kHitLane && L.any);
    L.best = -1;
    L.bu = L.bv = 0.0f;
    startPos(L.pos);
    for (uint32_t i = 0; i < S.numSpheres; ++i) {
        float t;
        if (isectSphere(S.spheres[i], L.r.o, L.r.d, L.tmin, L.tmax, t)) {
            int id = (int)(S.numTris + i);
            if (L.best < 0 || t < L.tmax || id < L.best) {
                L.tmax = t;
                L.best = id;
            }
            if (ANY) {
                endPos(L.pos);
                return;
            }
        }
    }
}

// Drives the persistent loop.  load(idx, L) fills L.r/L.tmin/L.tmax (and
// L.any under kHitLane); S is the scene (a DevScene for launches over one
// scene, or a per-lane LaneScene that load() points at the ray's scene);
// store(L) consumes a finished ray.  `fetch` must be zero at launch.  Each
// wave first takes its own slice of up to 64 rays of the grid's static span
// without an atomic, so a launch over a short or empty queue costs no
// contention; the rays past the static span go out in chunks, one atomic a
// chunk, and the wave refills its idle lanes from the chunk it holds whenever
// at least kRefillLanes of them are idle (or all are).
//
// A short queue is bound by the latency of its longest rays, and every node
// or leaf step of a lane's neighbours lengthens its own chain: so a queue that
// would not fill the waves is spread over 1 / kSpread of them, a few rays
// each.  Closest hits through the host call, 2047 rays in the 262,144-triangle
// room: 134 us with 64 rays a wave, 105 us spread (8191: 158 and 129); 1080p
// cache frames, whose last bounces are short, 452 and 442 ms for 44 frames.
// Over all the waves, 30,000 and more rays in a small scene lost up to 30%
// (three times the wave steps); over a quarter or an eighth of them the large
// scene's 8191 rays lost 7 to 11%.
//
// The work counter is one word that every XCD updates, so its atomics are
// served one after another, a few nanoseconds each: with one a refill (about
// 20 rays) they bounded a 4.1 M-ray launch at 1.85 ms.  A chunk is a
// kChunksPerWave-th of a wave's share of the rest, so that the waves end
// together, at least a whole wave's worth and at most kChunkMax: 8 chunks of
// at most 512 rays took that launch to 1.49 ms (32 of at most 256, or 4 of at
// most 1024, within 0.5% of it).
// Once the queue is drained the wave stops fetching, so `fetch` ends below
// n + kChunkMax * waves.
constexpr int kRefillLanes = 24;          // 16 to 32: within 0.3% of each other; 8: 1% slower
constexpr uint32_t kChunksPerWave = 8, kChunkMax = 512;
constexpr uint32_t kSpread = 2;
// Inner nodes are visited while at least kNodeNum / kNodeDen of the active
// lanes have one to visit; then every lane at a leaf intersects that leaf.
// A ray visits some four inner nodes a leaf, so waiting until every lane is at
// a leaf left two thirds of the lanes idle.  2/3 measured the same, 1/2 and
// 7/8 1-2% slower; so did one triangle a lane and pass instead of one leaf.
constexpr int kNodeNum = 3, kNodeDen = 4;

template <int HIT, bool COUNT, bool ALPHA, class SceneT, class Stack, class Load, class Store>
RTX_DI void persistentTrace(const SceneT &S, uint32_t n, uint32_t *fetch, Stack &st, VisitCount &vc, Load load,
                            Store store) {
    LaneRay L;
    endPos(L.pos);
    L.idx = 0;
    L.any = HIT == kHitAny;
    bool active = false;
    bool first = true, last = false, drained = false; // wave-uniform: no chunk yet, none after this one, none left
    const uint32_t waves = gridDim.x * (blockDim.x >> 6); // blockDim.x is a multiple of 64
    const uint32_t spread = max(waves / kSpread, 1u);
    const uint32_t slice = min(n / spread + (n % spread != 0u ? 1u : 0u), 64u);
    const uint32_t staticSpan = waves * slice;
    const uint32_t waveBase = (blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * slice;
    uint32_t cur = 0, end = 0; // wave-uniform: the chunk of rays the wave still holds
    const uint32_t chunk =
        n <= staticSpan ? 64u : min(max((n - staticSpan) / (waves * kChunksPerWave), 64u), kChunkMax);
    for (;;) {
        // refill idle lanes (the whole wave is converged here)
        const bool idle = !active;
        const uint64_t m = __ballot(idle);
        const int nIdle = __popcll(m);
        const bool anyActive = nIdle < 64; // gfx950 waves are 64 wide; blocks are whole waves
        if (!drained && (nIdle >= kRefillLanes || !anyActive)) {
            const int lane = (int)__lane_id();
            if (cur == end) { // the wave's chunk is used up
                if (first) { // every lane idle: the wave's static slice
                    first = false;
                    cur = waveBase;
                    end = waveBase + slice;
                    last = staticSpan >= n;
                } else {
                    uint32_t base = 0;
                    if (lane == 0) base = atomicAdd(fetch, chunk);
                    cur = staticSpan + __builtin_amdgcn_readfirstlane(base);
                    end = cur + chunk;
                    last = end >= n;
                }
                end = min(end, n);
                cur = min(cur, end);
            }
            const uint32_t base = cur;
            const uint32_t take = min((uint32_t)nIdle, end - cur);
            cur += take;
            drained = last && cur == end;
            if (idle) {
                const uint64_t below = lane == 0 ? 0ull : (m & ((~0ull) >> (64 - lane)));
                const uint32_t rank = (uint32_t)__popcll(below), idx = base + rank;
                if (rank < take) {
                    L.idx = idx;
                    load(idx, L);
                    st.sp = 0;
                    beginRay<HIT>(S, L);
                    active = true;
                }
            }
        }
        const int nActive = __popcll(__ballot(active));
        if (nActive == 0) break;
        // inner nodes while most of the active lanes have one to visit
        int nNode;
        do {
            if (!L.pos.atLeaf() && L.pos.atNode()) {
                if (COUNT) vc.nodes++;
                nodeStep(S, L.r, L.tmin, L.tmax, L.pos, st);
            }
            nNode = __popcll(__ballot(!L.pos.atLeaf() && L.pos.atNode()));
        } while (nNode * kNodeDen >= nActive * kNodeNum && nNode > 0);
        // the next leaf of every lane at one
        if (L.pos.atLeaf()) {
            do {
                if (triStep<HIT, COUNT, ALPHA>(S, L, vc)) endPos(L.pos);
            } while (L.pos.triLeft != 0u);
        }
        if (active && !L.pos.atLeaf() && !L.pos.atNode()) {
            store(L);
            active = false;
        }
    }
}

} // namespace rtx
