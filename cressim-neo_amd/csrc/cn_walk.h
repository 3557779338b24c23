// cn_walk.h -- the reference's 27-cell candidate walk over the run table of the sorted cell keys.
#pragma once

#include "cn_device.h"

namespace cn {

// The run table of one substep: runs of equal keys in sorted order, a bucket index over the top
// key bits, and the cell coordinates (w: the scene's key prefix) of every slot.
struct RunTable {
    const uint32_t *run_key;
    const uint32_t *run_start;
    const int4 *run_info;   // (cx, cy, cz, kRunPure | run_class or 0)
    const uint32_t *bucket;
    uint32_t bucket_shift;
    const int4 *cellc;
};

// run_info.w: bit 0 the run holds a single cell; above it the particle class of every member plus
// one, or 0 when they differ (or the substep has no use for it).
constexpr int kRunPure = 1;
__device__ __forceinline__ int run_class_word(uint32_t cls) { return (int)((cls + 1u) << 1); }
__device__ __forceinline__ uint32_t run_class(int w) { return ((uint32_t)w >> 1) - 1u; }  // kInvalid: differ

// The record of run r from its members: (cx, cy, cz, w).  Pure runs hold a single cell; mixed runs
// (hash collisions or wrapped Morton coordinates) are filtered per particle like the reference
// (:94-98).  cls: the slots' classes when the contact candidates want each run's one class (null
// otherwise).  The members are read four at a time, so a run of a few particles costs one round trip.
__device__ __forceinline__ int4 run_record(uint32_t s, uint32_t e, const int4 *__restrict__ cellc,
                                           const uint32_t *__restrict__ cls)
{
    const int4 c0 = cellc[s];
    const uint32_t k0 = cls ? cls[s] : 0u;
    bool pure = true, one = cls != nullptr;
    for (uint32_t q = s + 1; q < e && (pure || one); q += 4) {
        int4 cq[4];
        uint32_t kq[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const uint32_t i = min(q + u, e - 1u);
            cq[u] = cellc[i];
            kq[u] = cls ? cls[i] : 0u;
        }
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            pure &= cq[u].x == c0.x && cq[u].y == c0.y && cq[u].z == c0.z;
            one &= kq[u] == k0;
        }
    }
    return make_int4(c0.x, c0.y, c0.z, (pure ? kRunPure : 0) | (one ? run_class_word(k0) : 0));
}

// The run of a key: a binary search of its bucket's runs.  A bucket is a range of keys, so where a
// scene fills a corner of its key range (a pool whose key holds the scene, a small body in a large
// box) one bucket holds hundreds of runs: the linear scan it replaces made the 48-scene pool's halo
// lookups 312 us a substep.
__device__ __forceinline__ int find_run(uint32_t key, const RunTable &t)
{
    const uint32_t b = key >> t.bucket_shift;
    uint32_t lo = t.bucket[b];
    const uint32_t e = t.bucket[b + 1];
    uint32_t hi = e;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (t.run_key[mid] < key) lo = mid + 1u;
        else hi = mid;
    }
    return (lo < e && t.run_key[lo] == key) ? (int)lo : -1;
}

// f(slot) for the particles of the 27 cells around cell ci in dz, dy, dx order, each cell's
// particles in ascending particle index (its slots), until f returns false.  A cell whose hash
// equals the empty-table marker is never found (physics_fluid_build_neighbors.cs.hlsl:81-85 with
// FindParticleCellRange); a run shared by several cells (hash collision, Morton wrap) is filtered
// by cell coordinates (:94-98).
template <class F>
__device__ __forceinline__ void walk_runs(int4 ci, const RunTable &t, const SubstepConsts &c, F &&f)
{
    for (int dz = -1; dz <= 1; ++dz)
        for (int dy = -1; dy <= 1; ++dy)
            for (int dx = -1; dx <= 1; ++dx) {
                const int tx = ci.x + dx, ty = ci.y + dy, tz = ci.z + dz;
                if (cell_hash(tx, ty, tz) == kInvalid) continue;
                const int r = find_run(cell_key(tx, ty, tz, (uint32_t)ci.w, c.key_mode, c.morton_bits), t);
                if (r < 0) continue;
                const int4 info = t.run_info[r];
                const bool pure = (info.w & kRunPure) != 0;
                if (pure && (info.x != tx || info.y != ty || info.z != tz)) continue;
                const uint32_t qe = t.run_start[r + 1];
                for (uint32_t q = t.run_start[r]; q < qe; ++q) {
                    if (!pure) {
                        const int4 cq = t.cellc[q];
                        if (cq.x != tx || cq.y != ty || cq.z != tz) continue;
                    }
                    if (!f(q)) return;
                }
            }
}

}  // namespace cn
