// Irradiance-cache lookup on the device.  Replaces the reference's cache
// acceleration structure (a refitted AABB BLAS, src/IrradianceCache.cpp:19-44,
// 81-104) and its point query through the intersection and any-hit shaders
// (shaders/raytrace.rgen:748-773, raytrace.irradiance.rint:11-21,
// raytrace.irradiance.rahit:18-51).
//
// Index: a multi-level hashed grid.  A record of radius r lives at the
// level L whose cells (c0 * 2^L) are a little wider than r grown by a
// rounding margin m, in every cell of that level its sphere's box (half-width
// m) touches: at most 3 per axis.  Cells between r and 2r wide keep the
// records a lookup tests but does not accept few (the cell's neighbourhood
// of reach r spans 3r-4r per axis against 4r-6r for cells of 2r-4r).
// Each occupied level has its own range of buckets, and a record files at
// most one item per bucket, so a lookup needs no cell key: it visits one
// bucket per occupied level and weighs the records in it whose sphere
// contains the point, in (level, record id) order.  A record that contains
// the point is filed in the point's cell at its level, so it is in the
// bucket visited there, once; items of other cells that share the bucket
// either do not contain the point or are that same record.
#pragma once

#include "dev_math.h"
#include "dev_shading.h"
#include "internal.h"

namespace rtx {

constexpr int kIcMaxLevel = 24;
constexpr int kIcAxisBits = 19;
constexpr int32_t kIcAxisHalf = 1 << (kIcAxisBits - 1);

RTX_DI float icCellSize(float c0, int level) { return ldexpf(c0, level); }

RTX_DI int32_t icCellCoord(float v, float cs) {
    float q = floorf(v / cs);
    q = fminf(fmaxf(q, -(float)kIcAxisHalf), (float)(kIcAxisHalf - 1));
    return (int32_t)q;
}

RTX_DI uint64_t icKey(int level, int32_t ix, int32_t iy, int32_t iz) {
    const uint64_t m = (1ull << kIcAxisBits) - 1;
    return ((uint64_t)level << (3 * kIcAxisBits)) | (((uint64_t)(ix + kIcAxisHalf) & m) << (2 * kIcAxisBits)) |
           (((uint64_t)(iy + kIcAxisHalf) & m) << kIcAxisBits) | ((uint64_t)(iz + kIcAxisHalf) & m);
}

// The bucket of a cell key at `level`: the nb buckets are split into
// 2^ceil(log2(occupied levels)) equal ranges, one per occupied level in
// ascending order (levelMask: the occupied levels), and the key hashed
// into its level's range.
RTX_DI uint32_t icBucket(uint64_t key, uint32_t nb, uint32_t levelMask, int level) {
    // splitmix64 finaliser
    key ^= key >> 30;
    key *= 0xbf58476d1ce4e5b9ull;
    key ^= key >> 27;
    key *= 0x94d049bb133111ebull;
    key ^= key >> 31;
    const uint32_t nl = (uint32_t)__popc(levelMask);
    const int partBits = nl <= 1u ? 0 : 32 - __clz((int)(nl - 1u));
    const uint32_t per = nb >> partBits;
    const uint32_t rank = (uint32_t)__popc(levelMask & ((1u << level) - 1u));
    return rank * per + ((uint32_t)key & (per - 1u));
}

// The level a sphere of grown radius m is filed under: the first whose cells
// are at least 1.001 m wide, so that its box (2m wide) spans at most 3 cells
// per axis whatever the rounding of its bounds.
RTX_DI int icLevel(float c0, float m) {
    int level = 0;
    float cs = c0;
    while (cs < 1.001f * m && level < kIcMaxLevel) {
        cs *= 2.0f;
        ++level;
    }
    return level;
}

// The jobs [j0, jEnd) of an IcJobRange other than kIcJobsHost.
RTX_DI void icJobRange(const IcBuffers &ic, int range, uint32_t firstJob, uint32_t &j0, uint32_t &jEnd) {
    switch (range) {
    case kIcJobsUpdates: j0 = 0, jEnd = ic.frame[3]; break;
    case kIcJobsCreations: j0 = ic.frame[3], jEnd = ic.frame[4]; break;
    default: j0 = firstJob, jEnd = ic.frame[4]; break;
    }
}

// raytrace.rgen:806-813
RTX_DI bool isICCapable(int type, bool onGlossy) {
    if (type == RTX_MAT_DIFFUSE || type == RTX_MAT_LIGHT) return true;
    return onGlossy && !hasDiscreteDirection(type);
}

// raytrace.rgen:815-828
RTX_DI V3 approxDiffuse(const Mat &m, V3 normal, V3 wi) {
    switch (m.type) {
    case RTX_MAT_DIFFUSE:
    case RTX_MAT_LIGHT:
    case RTX_MAT_PHONG: return m.kd * (1.0f / kPi);
    case RTX_MAT_ROUGH_CONDUCTOR: return v3(fresnelConductor(dot(wi, normal), m.eta, m.k) * (1.0f / kPi));
    default: return v3(-1.0f);
    }
}

struct IcQueryParams {
    float invA;          // 1 / irradianceA
    bool gradients;      // useIrradianceGradients
    bool visibility;     // irradianceCachePerformVisibilityCheck
};

// The bucket of x's cell at one level of the index.
RTX_DI uint32_t icLevelBucket(const DevIC &ic, float c0, uint32_t levelMask, int level, V3 x) {
    const float cs = icCellSize(c0, level);
    const uint64_t key = icKey(level, icCellCoord(x.x, cs), icCellCoord(x.y, cs), icCellCoord(x.z, cs));
    return icBucket(key, ic.nb, levelMask, level);
}

// The fields of a record a lookup weighs with (gradients only when used).
struct IcRec {
    V3 normal, color, rotGrad, transGrad;
    float harmonicR;
};

// From the item's second and third 16 bytes, and the entry's gradients.
RTX_DI IcRec icLoadRec(const DevIC &ic, const IcItem *item, bool gradients) {
    const float4 a = reinterpret_cast<const float4 *>(item)[1], b = reinterpret_cast<const float4 *>(item)[2];
    IcRec r;
    r.normal = v3(a);
    r.harmonicR = a.w;
    r.color = v3(b);
    if (gradients) {
        const rtx_cache_data &e = ic.entries[__float_as_uint(b.w)];
        r.rotGrad = v3(e.rotGrad);
        r.transGrad = v3(e.transGrad);
    } else {
        r.rotGrad = r.transGrad = v3(0.0f);
    }
    return r;
}

// One record's term of the weighted mean (raytrace.irradiance.rint:17-20,
// raytrace.irradiance.rahit:18-51) for a point x inside its sphere
// (oc = x - centre): its weight and colour, false when it does not count.
RTX_DI bool icWeigh(const IcQueryParams &qp, V3 n, V3 oc, const IcRec &e, float &w, V3 &col) {
    const V3 ni = e.normal;
    w = 1.0f / (length(oc) / e.harmonicR + sqrtf(1.0f - dot(n, ni)));
    if (isnan(w) || isinf(w)) w = 1000000.0f;
    if (w <= qp.invA) return false;
    if (qp.visibility && !(-0.001f <= dot(oc, (n + ni) / 2.0f))) return false;
    col = e.color;
    if (qp.gradients) {
        float E = length(col);
        V3 cn = E != 0.0f ? normalize(col) : v3(0.0f);
        col = cn * (E + dot(cross(ni, n), e.rotGrad) + dot(oc, e.transGrad));
    }
    return true;
}

// A lookup's work is uneven: a point's buckets hold anything from no item to
// over a hundred (32 on average in the 262K-triangle room's 10,000 records, a
// fifth of them containing the point), and half a wave's lanes have no lookup
// at all.  With a walk per lane 80% of the lanes were idle while the wave
// waited for its longest, and every step of it paid for a record's whole term
// (two square roots and three divisions) as soon as one lane needed it.  Here
// the wave shares the items of all its lookups.  (lookup, item) pairs are
// numbered by lookup, then level, then bucket order; each step tests kIcChunk
// pairs per lane against a bound of the containment test and puts the pairs
// that may pass in a list in LDS, in order; whenever the list fills the wave,
// each lane weighs one of them, and the first lane of each lookup's run adds
// the run's terms in order, which is the order of a lane's own walk.
// A launch's share of it is bound by the dependent steps (tests, then terms)
// of single waves where a frame has few paths, else by their instructions.
// The 256x192 split-and-roulette frames: 108,000 cycles a wave with a walk per
// lane, 122,000 with the lanes sharing the items but weighing them where they
// are tested, 61,000 so (their shading launches 88 -> 50 us); 44 1080p cache
// frames of that room: 277 -> 236 ms of shading.
constexpr int kIcChunk = 4;  // pairs a lane tests per step
constexpr int kIcLevels = 8; // levels whose buckets are read together

struct IcWave { // one wave's part of a block's LDS
    float4 qa[64];                  // per lookup: point, normal.x
    float2 qb[64];                  // normal.yz
    float4 sum[64];                 // weight total, weighted colour
    uint32_t first[64 * kIcLevels]; // per (lookup, level): its first item - its first pair
    uint32_t seg[64 * kIcChunk];    // per pair of a step: 1 + the (lookup, level) that starts there
    uint2 list[64 * (kIcChunk + 1)]; // pairs to weigh: item, lookup
    float4 acc[64];                 // a lane's term: weight, colour
};

RTX_DI void icWaveSync() { // LDS written by other lanes of the wave is visible
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// The terms of list[h .. h + m), one a lane (rank: the lane's place among the
// executing ones), added to their lookups' sums.
RTX_DI void icWeighList(const DevIC &ic, const IcQueryParams &qp, IcWave &ws, uint32_t h, uint32_t m, uint32_t rank,
                        uint32_t lane) {
    bool ok = false, head = false;
    uint32_t lookup = 0;
    if (rank < m) {
        const uint2 e = ws.list[h + rank];
        lookup = e.y;
        head = rank == 0 || ws.list[h + rank - 1].y != lookup;
        const IcItem *item = &ic.items[e.x];
        const float4 c = *reinterpret_cast<const float4 *>(item);
        const IcRec rec = icLoadRec(ic, item, qp.gradients);
        const float4 qa = ws.qa[lookup];
        const float2 qb = ws.qb[lookup];
        const V3 oc = v3(qa) - v3(c);
        if (length(oc) <= c.w) {
            float w;
            V3 col;
            ok = icWeigh(qp, V3{qa.w, qb.x, qb.y}, oc, rec, w, col);
            if (ok) ws.acc[lane] = make_float4(w, col.x, col.y, col.z);
        }
    }
    icWaveSync();
    const uint64_t accepted = __ballot(ok), heads = __ballot(head);
    if (head) {
        const uint64_t above = heads & (~1ull << lane);
        uint64_t run = accepted & (~0ull << lane); // up to the next lookup's first lane
        if (above != 0) run &= (above & (0ull - above)) - 1ull;
        if (run != 0) {
            const float4 s = ws.sum[lookup];
            float total = s.x;
            V3 sum = V3{s.y, s.z, s.w};
            do {
                const float4 a = ws.acc[__ffsll((unsigned long long)run) - 1];
                run &= run - 1ull;
                sum = sum + a.x * V3{a.y, a.z, a.w};
                total += a.x;
            } while (run != 0);
            ws.sum[lookup] = make_float4(total, sum.x, sum.y, sum.z);
        }
    }
    icWaveSync();
}

// Weighted cache colour at x (normal n) for the lanes that want it, from the
// whole wave: called by converged lanes, all of which work.  False when no
// record accepts x.  Records are weighed in (level, bucket order) order.
RTX_DI bool icQueryWave(const DevIC &ic, const IcQueryParams &qp, IcWave &ws, bool want, V3 x, V3 n, V3 &color) {
    const uint64_t wanting = __ballot(want);
    if (wanting == 0) return false;
    const uint32_t mask = (uint32_t)__builtin_amdgcn_readfirstlane((int)ic.meta[0]);
    if (mask == 0) return false;
    const float c0 = __uint_as_float(ic.meta[2]);
    const uint32_t lane = __lane_id();
    const uint64_t below = (1ull << lane) - 1ull, exec = __ballot(true);
    const uint32_t workers = (uint32_t)__popcll(exec), rank = (uint32_t)__popcll(exec & below);
    const int topLane = 63 - __clzll((long long)exec);
    const uint32_t q = (uint32_t)__popcll(wanting & below);
    icWaveSync(); // the previous lookups' readers are done
    if (want) {
        ws.qa[q] = f4(x, n.x);
        ws.qb[q] = make_float2(n.y, n.z);
        ws.sum[q] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    for (uint32_t lm = mask; lm != 0;) {
        uint32_t start[kIcLevels], pre[kIcLevels], mine = 0;
#pragma unroll
        for (int k = 0; k < kIcLevels; ++k) {
            start[k] = pre[k] = 0;
            if (lm != 0) {
                if (want) {
                    const uint32_t b = icLevelBucket(ic, c0, mask, __ffs(lm) - 1, x);
                    start[k] = ic.bucketStart[b];
                    pre[k] = ic.bucketStart[b + 1];
                }
                lm &= lm - 1;
            }
        }
#pragma unroll
        for (int k = 0; k < kIcLevels; ++k) {
            pre[k] -= start[k];
            mine += pre[k];
        }
        // this lane's first pair and the wave's number of pairs, bit by bit
        uint32_t off = 0, pairs = 0;
        for (int bit = 0; bit < 32 && __ballot((mine >> bit) != 0) != 0; ++bit) {
            const uint64_t m = __ballot((mine >> bit) & 1u);
            off += (uint32_t)__popcll(m & below) << bit;
            pairs += (uint32_t)__popcll(m) << bit;
        }
#pragma unroll
        for (int k = 0; k < kIcLevels; ++k) {
            const uint32_t count = pre[k];
            if (want && count != 0) ws.first[q * kIcLevels + k] = start[k] - off;
            pre[k] = count != 0 ? off : 0xFFFFFFFFu;
            off += count;
        }
        uint32_t listed = 0, carry = 0; // carry: seg of the last pair of the step before
        for (uint32_t base = 0; base < pairs; base += workers * kIcChunk) {
            // which (lookup, level) each pair is of: written where one starts,
            // and carried on to the pairs that follow
            uint4 &mySeg = *reinterpret_cast<uint4 *>(&ws.seg[kIcChunk * rank]);
            mySeg = make_uint4(0u, 0u, 0u, 0u);
            icWaveSync();
#pragma unroll
            for (int k = 0; k < kIcLevels; ++k)
                if (pre[k] - base < workers * kIcChunk) ws.seg[pre[k] - base] = 1u + q * kIcLevels + k;
            icWaveSync();
            const uint4 s4 = mySeg;
            uint32_t seg[kIcChunk] = {s4.x, s4.y, s4.z, s4.w};
#pragma unroll
            for (int u = 1; u < kIcChunk; ++u) seg[u] = seg[u] != 0 ? seg[u] : seg[u - 1];
            const uint64_t started = __ballot(seg[kIcChunk - 1] != 0) & below;
            const uint32_t from = (uint32_t)__shfl((int)seg[kIcChunk - 1], started != 0 ? 63 - __clzll((long long)started) : (int)lane);
            const uint32_t before = started != 0 ? from : carry;
#pragma unroll
            for (int u = 0; u < kIcChunk; ++u) seg[u] = seg[u] != 0 ? seg[u] : before;
            carry = (uint32_t)__builtin_amdgcn_readlane((int)seg[kIcChunk - 1], topLane);
            uint32_t item[kIcChunk];
            float4 c[kIcChunk];
            bool in[kIcChunk];
#pragma unroll
            for (int u = 0; u < kIcChunk; ++u) {
                const uint32_t p = base + kIcChunk * rank + u;
                in[u] = p < pairs;
                item[u] = in[u] ? ws.first[seg[u] - 1u] + p : 0u;
                if (in[u]) c[u] = *reinterpret_cast<const float4 *>(&ic.items[item[u]]);
            }
            // a bound of |x - centre| <= radius without its square root (the
            // rounding of either side is below 1e-6)
            uint32_t found = 0;
#pragma unroll
            for (int u = 0; u < kIcChunk; ++u) {
                if (in[u]) {
                    const V3 oc = v3(ws.qa[(seg[u] - 1u) / kIcLevels]) - v3(c[u]);
                    in[u] = dot(oc, oc) <= fmaf(c[u].w * c[u].w, 1.00001f, 1e-37f);
                }
                found += in[u] ? 1u : 0u;
            }
            const uint64_t f0 = __ballot(found & 1u), f1 = __ballot(found & 2u), f2 = __ballot(found & 4u);
            uint32_t at = listed + (uint32_t)__popcll(f0 & below) + 2u * (uint32_t)__popcll(f1 & below) +
                          4u * (uint32_t)__popcll(f2 & below);
            listed += (uint32_t)__popcll(f0) + 2u * (uint32_t)__popcll(f1) + 4u * (uint32_t)__popcll(f2);
#pragma unroll
            for (int u = 0; u < kIcChunk; ++u)
                if (in[u]) ws.list[at++] = make_uint2(item[u], (seg[u] - 1u) / kIcLevels);
            icWaveSync();
            if (listed < workers) continue;
            uint32_t h = 0;
            for (; listed - h >= workers; h += workers) icWeighList(ic, qp, ws, h, workers, rank, lane);
            const uint2 rest = h + rank < listed ? ws.list[h + rank] : make_uint2(0u, 0u);
            icWaveSync();
            if (h + rank < listed) ws.list[rank] = rest;
            listed -= h;
            icWaveSync();
        }
        if (listed != 0) icWeighList(ic, qp, ws, 0, listed, rank, lane);
    }
    icWaveSync();
    if (!want) return false;
    const float4 s = ws.sum[q];
    if (s.x > 0.0f) {
        color = V3{s.y, s.z, s.w} / s.x;
        return true;
    }
    return false;
}

} // namespace rtx
