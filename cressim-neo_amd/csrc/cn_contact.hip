// cn_contact.hip -- particle-particle contacts on gfx950.
//
// Reference passes: buildParticleParticleCandidatePairs (physics_pass_dispatcher.cpp:1102-1197,
// physics_particle_{count,emit}_particle_particle_candidates.cs.hlsl with
// IsValidParticleParticleCandidate, physics_particle_broad_phase_query.hlsli:65-117) once per
// substep from the predicted positions; per contact iteration
// physics_particle_generate_explicit_contacts.cs.hlsl:80-189, the compaction of active contacts,
// physics_particle_solve_explicit_contacts.cs.hlsl:25-246 and
// physics_particle_apply_position_corrections.cs.hlsl:8-30; after the velocity update
// physics_particle_solve_contact_velocities.cs.hlsl:26-170 and
// physics_particle_apply_contact_velocities.cs.hlsl per velocity iteration.
//
// The reference emits each pair once (lower particle index first) and accumulates both sides'
// corrections with float CAS atomics, in no fixed order.  Here every particle keeps its candidate
// partners in its own 27-cell walk order, evaluates each pair's contact itself (the arithmetic of
// the pair is the same from either side: lower index first) and sums its side's corrections in
// that order, so results are deterministic and equal to the oracle's.  Contacts are Jacobi: a
// solve pass writes every particle's summed correction, an apply pass adds them.  Particle-
// particle contacts are those of free particles (no rigid proxies, no suturing).  Solids of one
// phase group pair up only when the group collides with itself, minus constraint-adjacent pairs.
//
// Particle-rigid contacts: solid particles against the scene's static colliders, every collider a
// static body of its own (buildParticleRigidCandidatePairs with
// physics_particle_count_particle_rigid_candidates.cs.hlsl:112-151; per contact iteration
// physics_particle_rigid_generate_contacts.cs.hlsl:30-190 and
// physics_particle_rigid_solve_contacts.cs.hlsl:26-140 into the same correction, after the
// particle-particle terms; after the particle-particle velocity iterations
// physics_particle_rigid_solve_contact_velocities.cs.hlsl:27-130 with its apply per iteration).
// The candidates are the particle's collider bitmask of the reorder pass, in LBVH visit order.  A
// static body has zero inverse mass and inertia and does not move: its effective mass is zero and
// its contact point's displacement and velocity are exactly zero.  The velocity pass regenerates
// each contact from the position of the last contact iteration, which is kept per particle.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "cn_rigid.h"
#include "cn_walk.h"

namespace cn {

struct ContactArgs {
    float4 *pos;              // slot order
    float4 *vel;
    const float4 *prev;
    float4 *cur;              // fluid solver positions x* + delta (free particles: w = 0)
    float4 *dacc;             // current fluid delta; w: the contacts' path of the substep
    const uint32_t *cls;
    const uint32_t *id;
    const ParticleClass *classes;
    const float4 *part_mats;
    const uint32_t *active;   // per scene
    const SceneInfo *scenes;
    RunTable rt;
    const uint32_t *blk_first_run;
    const uint32_t *nblk;
    const uint32_t *blk_halo;
    uint32_t *plist;          // partner slots, k-major: plist[k * n + t]
    uint32_t *pcount;
    float4 *crec;             // contact of each partner: (normal, penetration), k-major
    uint32_t *cbits;          // bit k: partner k's contact is active
    float4 *corr;             // summed correction of the pass
    uint32_t *meta;
    const uint32_t *adj_off;  // constraint adjacency by particle index (null: none)
    const uint32_t *adj_cnt;
    const uint32_t *adj_idx;
    const Collider *col;      // static colliders in visit order (SceneInfo.col0 per scene)
    const uint32_t *bnd;      // per slot: candidate colliders (a solid's rigid candidates)
    const uint16_t *bndl;     // their lists (scenes of many colliders)
    float4 *rgen;             // per slot: position of the last contact generation
    uint32_t n, pcap;
};

__device__ __forceinline__ const ParticleClass &pclass(const ContactArgs &a, uint32_t slot)
{
    return a.classes[a.cls[slot]];
}

// IsAdjacentParticle, physics_particle_broad_phase_query.hlsli:50-62: particle index `other` among
// the adjacency list of particle index `self`.
__device__ __forceinline__ bool adjacent(const ContactArgs &a, uint32_t self, uint32_t other)
{
    if (!a.adj_off) return false;
    const uint32_t off = a.adj_off[self], cnt = a.adj_cnt[self];
    for (uint32_t k = 0; k < cnt; ++k)
        if (a.adj_idx[off + k] == other) return true;
    return false;
}

// The class part of IsValidParticleParticleCandidate (symmetric in the pair).  same_group: the pair
// also needs its particles not to share a constraint.
__device__ __forceinline__ bool classes_pair(const ParticleClass &A, const ParticleClass &B, bool &same_group)
{
    same_group = false;
    if (A.env != B.env) return false;
    if ((A.mask & B.layer) == 0u || (B.mask & A.layer) == 0u) return false;
    if (A.kind == CN_PARTICLE_KIND_FLUID && B.kind == CN_PARTICLE_KIND_FLUID) return false;
    // one phase group: only when both have self collision on and they share no constraint
    if (A.kind == CN_PARTICLE_KIND_SOLID && B.kind == CN_PARTICLE_KIND_SOLID &&
        (A.phase & kPhaseGroupMask) == (B.phase & kPhaseGroupMask)) {
        same_group = true;
        return (A.phase & kPhaseSelfCollide) && (B.phase & kPhaseSelfCollide);
    }
    return true;
}

__device__ __forceinline__ void order_pair(const ContactArgs &a, uint32_t t, uint32_t q, uint32_t &lo, uint32_t &hi,
                                           bool &t_is_hi)
{
    t_is_hi = a.id[q] < a.id[t];
    lo = t_is_hi ? q : t;
    hi = t_is_hi ? t : q;
}

// CombineContactMaterial, physics_rigid_solver_shared.hlsli:37-43: (friction, restitution, static)
__device__ __forceinline__ float3 combine_material(const ContactArgs &a, uint32_t lo, uint32_t hi)
{
    const float4 ma = a.part_mats[pclass(a, lo).part_mat], mb = a.part_mats[pclass(a, hi).part_mat];
    return make_float3(fsqrt(fmaxd(0.0f, ma.x) * fmaxd(0.0f, mb.x)), fmaxd(fmaxd(0.0f, ma.y), fmaxd(0.0f, mb.y)),
                       fsqrt(fmaxd(0.0f, ma.w) * fmaxd(0.0f, mb.w)));
}

// ---------------------------------------------------------------------------------------------
// candidates
// ---------------------------------------------------------------------------------------------
// One particle's candidate partners, taken in walk order.
struct Partners {
    const ContactArgs &a;
    uint32_t t;
    float4 p;
    ParticleClass pc;
    uint32_t cnt = 0;
    // IsValidParticleParticleCandidate with slot q: the distance (the same from either side: the
    // differences only change sign), the classes, and the adjacency from the lower particle index
    __device__ __forceinline__ void test(uint32_t q)
    {
        const float4 pq = a.pos[q];
        const ParticleClass &B = a.classes[a.cls[q]];
        const float dx = pq.x - p.x, dy = pq.y - p.y, dz = pq.z - p.z;
        const float cr = pc.radius + B.radius;
        if (!(dot3(dx, dy, dz, dx, dy, dz) <= cr * cr) || q == t) return;
        bool same_group;
        if (!classes_pair(pc, B, same_group)) return;
        if (same_group) {
            uint32_t lo, hi;
            bool t_hi;
            order_pair(a, t, q, lo, hi, t_hi);
            if (adjacent(a, a.id[lo], a.id[hi])) return;
        }
        if (cnt < a.pcap) a.plist[(size_t)cnt * a.n + t] = q;
        ++cnt;
    }
    __device__ __forceinline__ void store()
    {
        if (cnt > a.pcap) atomicAdd(&a.meta[4], 1u);
        a.pcount[t] = min(cnt, a.pcap);
    }
};

// Walk of the run table: hash keys, and cell blocks without a halo descriptor.
__device__ __forceinline__ void partners_walk(const ContactArgs &a, const SubstepConsts &c, uint32_t t)
{
    Partners w{a, t, a.pos[t], pclass(a, t)};
    if (!a.active[w.pc.scene]) return;
    if (a.scenes[w.pc.scene].pairs)
        walk_runs(a.rt.cellc[t], a.rt, c, [&](uint32_t q) {
            w.test(q);
            return true;
        });
    w.store();
}

__global__ __launch_bounds__(kBlock) void k_contact_partners_walk(ContactArgs a, SubstepConsts c)
{
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    if (t < a.n) partners_walk(a, c, t);
}

// A workgroup per 4x4x4-cell block, its halo's cell ranges in LDS.  In most blocks no pair can
// exist (only fluid, or one body without self collision, within reach: kHdPairs) and nothing is
// walked; the others read the 27 cells' slots without looking their runs up.  What remains is the
// latency of the candidates' positions and classes, two independent loads each.  On the 360,448
// particles of the mixed scene the walk of every particle through the run table took 568 us a
// substep.
__global__ __launch_bounds__(kBlock) void k_contact_partners(ContactArgs a, SubstepConsts c)
{
    __shared__ uint32_t hoff[kHalo + 1];
    __shared__ uint32_t hstart[kHalo];
    const uint32_t nb = a.nblk[0], tid = threadIdx.x;
    for (uint32_t b = blockIdx.x; b < nb; b += gridDim.x) {
        if (b >= c.blk_cap) {
            const uint32_t p0 = a.rt.run_start[a.blk_first_run[b]], p1 = a.rt.run_start[a.blk_first_run[b + 1]];
            for (uint32_t t = p0 + tid; t < p1; t += kBlock) partners_walk(a, c, t);
            continue;
        }
        const uint32_t *hd = a.blk_halo + (size_t)b * kHaloStride;
        const uint32_t p0 = hd[kHdP0], p1 = hd[kHdP1], flags = hd[kHdFlags];
        if (!a.active[hd[kHdScene]]) continue;
        if (flags == kHdNoFluid || (flags == 1u && !hd[kHdPairs])) {
            for (uint32_t t = p0 + tid; t < p1; t += kBlock) a.pcount[t] = 0u;
            continue;
        }
        if (flags == 0u || !a.scenes[hd[kHdScene]].pairs) {
            for (uint32_t t = p0 + tid; t < p1; t += kBlock) partners_walk(a, c, t);
            continue;
        }
        __syncthreads();  // the last block's walks are done with the tables
        for (uint32_t k = tid; k <= kHalo; k += kBlock) {
            hoff[k] = hd[kHdOff + k];
            if (k < kHalo) hstart[k] = hd[kHdStart + k];
        }
        const int bx = (int)hd[kHdBase], by = (int)hd[kHdBase + 1], bz = (int)hd[kHdBase + 2];
        __syncthreads();
        for (uint32_t t = p0 + tid; t < p1; t += kBlock) {
            const int4 ci = a.rt.cellc[t];
            const int hc = (ci.x - bx + 1) + 6 * (ci.y - by + 1) + 36 * (ci.z - bz + 1);
            Partners w{a, t, a.pos[t], pclass(a, t)};
            for (int r = 0; r < 27; ++r) {
                const int h = hc + (r % 3 - 1) + 6 * ((r / 3) % 3 - 1) + 36 * (r / 9 - 1);
                const uint32_t q0 = hstart[h], q1 = q0 + (hoff[h + 1] - hoff[h]);
                for (uint32_t q = q0; q < q1; ++q) w.test(q);
            }
            w.store();
        }
    }
}

// ---------------------------------------------------------------------------------------------
// position iteration: generate + solve (sum in partner order), then apply
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_contact_solve(ContactArgs a, SubstepConsts c)
{
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= a.n) return;
    const ParticleClass &pc = pclass(a, t);
    if (!a.active[pc.scene]) return;
    const SceneInfo sc = a.scenes[pc.scene];
    if (!(sc.pairs | sc.rigid)) return;
    const uint32_t cnt = a.pcount[t];
    float sx = 0.0f, sy = 0.0f, sz = 0.0f;
    uint32_t bits = 0;
    const float relax = c.cfg[kCfgSoftContactRelax];
    for (uint32_t k = 0; k < cnt; ++k) {
        const uint32_t q = a.plist[(size_t)k * a.n + t];
        uint32_t lo, hi;
        bool t_hi;
        order_pair(a, t, q, lo, hi, t_hi);
        // generate_explicit_contacts :140-188
        const float4 pa = a.pos[lo], pb = a.pos[hi];
        const float dx = pb.x - pa.x, dy = pb.y - pa.y, dz = pb.z - pa.z;
        const float d2 = dot3(dx, dy, dz, dx, dy, dz);
        const float cr = pclass(a, lo).radius + pclass(a, hi).radius;
        float nx = 0.0f, ny = 0.0f, nz = 0.0f, pen = 0.0f;
        bool on = false;
        if (d2 <= kEps) {
            on = true;
            ny = 1.0f;
            pen = cr;
        } else {
            const float dist = fsqrt(d2);
            const float p0 = cr - dist;
            if (p0 > 0.0f) {
                on = true;
                nx = fdiv(dx, dist);
                ny = fdiv(dy, dist);
                nz = fdiv(dz, dist);
                pen = p0;
            }
        }
        a.crec[(size_t)k * a.n + t] = make_float4(nx, ny, nz, pen);
        if (!on) continue;
        bits |= 1u << k;
        // solve_explicit_contacts :103-246 for a pair of free particles
        const float wa = pa.w, wb = pb.w;
        if (wa <= kEps && wb <= kEps) continue;
        const float pn = fmind(fmaxd(pen - c.cfg[kCfgContactSlop], 0.0f), c.cfg[kCfgSoftMaxCorrection]);
        if (pn <= 0.0f) continue;
        const float3 nr = safe_normalize(nx, ny, nz);
        const float4 va = a.prev[lo], vb = a.prev[hi];
        const float rx = (pb.x - vb.x) - (pa.x - va.x);
        const float ry = (pb.y - vb.y) - (pa.y - va.y);
        const float rz = (pb.z - vb.z) - (pa.z - va.z);
        const float denom = wa + wb;
        if (denom <= kEps) continue;
        const float lambda = fdiv(pn, denom) * relax;
        float cax = -nr.x * (wa * lambda), cay = -nr.y * (wa * lambda), caz = -nr.z * (wa * lambda);
        float cbx = nr.x * (wb * lambda), cby = nr.y * (wb * lambda), cbz = nr.z * (wb * lambda);
        const float rn = dot3(rx, ry, rz, nr.x, nr.y, nr.z);
        const float3 mat = combine_material(a, lo, hi);
        const float3 fd = friction_delta(c.cfg, rx - nr.x * rn, ry - nr.y * rn, rz - nr.z * rn, pn, mat.x, mat.z);
        const float fdist = len3(fd.x, fd.y, fd.z);
        if (fdist > 0.0f) {
            const float tden = wa + wb;
            if (tden > kEps) {
                const float tl = fdiv(fdist, tden) * relax;
                const float tx = fdiv(fd.x, fdist), ty = fdiv(fd.y, fdist), tz = fdiv(fd.z, fdist);
                cax = cax + tx * (wa * tl);
                cay = cay + ty * (wa * tl);
                caz = caz + tz * (wa * tl);
                cbx = cbx - tx * (wb * tl);
                cby = cby - ty * (wb * tl);
                cbz = cbz - tz * (wb * tl);
            }
        }
        if (t_hi) {
            if (wb > kEps) {
                sx = sx + cbx;
                sy = sy + cby;
                sz = sz + cbz;
            }
        } else if (wa > kEps) {
            sx = sx + cax;
            sy = sy + cay;
            sz = sz + caz;
        }
    }
    a.cbits[t] = bits;
    // particle-rigid contacts of a solid particle (rigid solve_contacts :45-140 with a static body)
    const uint32_t rm = pc.kind == CN_PARTICLE_KIND_SOLID ? a.bnd[t] : 0u;
    if (rm) {
        const float4 p = a.pos[t];
        a.rgen[t] = p;
        const float4 pv = a.prev[t];
        const float4 pm = a.part_mats[pc.part_mat];
        each_candidate(rm, a.bndl, t, [&](uint32_t k) {
            const Collider &cc = a.col[sc.col0 + k];
            float4 rec;
            float3 d;
            if (!rigid_contact(cc, p.x, p.y, p.z, pc.radius, rec)) return;
            if (!rigid_position(p, pv, rec, pm, cc, c, d)) return;
            sx = sx + d.x;
            sy = sy + d.y;
            sz = sz + d.z;
        });
    }
    a.corr[t] = make_float4(sx, sy, sz, 0.0f);
}

// apply_position_corrections :8-30 (every free particle; those without contacts add zero); a fluid
// particle's solver position follows its new x*
__global__ __launch_bounds__(kBlock) void k_contact_apply(ContactArgs a)
{
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= a.n) return;
    const ParticleClass &pc = pclass(a, t);
    if (!a.active[pc.scene]) return;
    const SceneInfo &sc = a.scenes[pc.scene];
    if (!(sc.pairs | sc.rigid)) return;
    float4 p = a.pos[t];
    if (p.w <= kEps) return;
    const float4 d = a.corr[t];
    p.x = p.x + d.x;
    p.y = p.y + d.y;
    p.z = p.z + d.z;
    a.pos[t] = p;
    if (pc.kind == CN_PARTICLE_KIND_FLUID) {
        // The displacement bound of the candidate lists goes on from the delta pass's: its w keeps
        // the length of the contacts' path so far, rounded up with the slack of the new position.  (Without
        // it scenes with contacts walked in every iteration: 83 us against 52 over 262,144 fluid particles.)
        float4 dl = a.dacc[t];
        const float qx = p.x + dl.x, qy = p.y + dl.y, qz = p.z + dl.z;
        const float slack = (fmaxd(fmaxd(fabsf(p.x), fabsf(p.y)), fabsf(p.z)) +
                             fmaxd(fmaxd(fabsf(qx), fabsf(qy)), fabsf(qz))) * 4.76837158e-7f + 1.0e-30f;
        if (d.x != 0.0f || d.y != 0.0f || d.z != 0.0f) {
            dl.w = (dl.w + len3(d.x, d.y, d.z)) * 1.000001f + slack;
            a.dacc[t].w = dl.w;
        }
        a.cur[t] = make_float4(qx, qy, qz, len3(dl.x, dl.y, dl.z) + slack + dl.w);
    }
}

// ---------------------------------------------------------------------------------------------
// velocity iteration over the last generated contacts
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_contact_velocity(ContactArgs a, SubstepConsts c)
{
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= a.n) return;
    const uint32_t scene = pclass(a, t).scene;
    if (!a.active[scene] || !a.scenes[scene].pairs) return;
    const uint32_t cnt = a.pcount[t], bits = a.cbits[t];
    float sx = 0.0f, sy = 0.0f, sz = 0.0f;
    for (uint32_t k = 0; k < cnt; ++k) {
        if (!((bits >> k) & 1u)) continue;
        const uint32_t q = a.plist[(size_t)k * a.n + t];
        uint32_t lo, hi;
        bool t_hi;
        order_pair(a, t, q, lo, hi, t_hi);
        const float wa = a.pos[lo].w, wb = a.pos[hi].w;
        if (wa <= kEps && wb <= kEps) continue;
        const float4 rec = a.crec[(size_t)k * a.n + t];
        const float3 nr = safe_normalize(rec.x, rec.y, rec.z);
        const float4 va = a.vel[lo], vb = a.vel[hi];
        const float nv = dot3(vb.x - va.x, vb.y - va.y, vb.z - va.z, nr.x, nr.y, nr.z);
        if (nv >= 0.0f) continue;
        const float denom = wa + wb;
        if (denom <= kEps) continue;
        const bool rest_on = (-nv > c.cfg[kCfgRestitutionVelocity]) &&
                             (rec.w <= c.cfg[kCfgRestitutionPenetration] * c.cfg[kCfgContactSlop]);
        const float restitution = rest_on ? fsat(combine_material(a, lo, hi).y) : 0.0f;
        const float desired = rest_on ? (-restitution * nv) : 0.0f;
        const float imp = fmaxd(0.0f, fdiv(desired - nv, denom));
        const float tx = nr.x * imp, ty = nr.y * imp, tz = nr.z * imp;
        if (t_hi) {
            if (wb > kEps) {
                sx = sx + tx * wb;
                sy = sy + ty * wb;
                sz = sz + tz * wb;
            }
        } else if (wa > kEps) {
            sx = sx + -tx * wa;
            sy = sy + -ty * wa;
            sz = sz + -tz * wa;
        }
    }
    a.corr[t] = make_float4(sx, sy, sz, 0.0f);
}

// apply_contact_velocities: v += correction for free particles
__global__ __launch_bounds__(kBlock) void k_contact_velocity_apply(ContactArgs a)
{
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= a.n) return;
    const uint32_t scene = pclass(a, t).scene;
    if (!a.active[scene] || !a.scenes[scene].pairs) return;
    if (a.pos[t].w <= kEps) return;
    float4 v = a.vel[t];
    const float4 d = a.corr[t];
    v.x = v.x + d.x;
    v.y = v.y + d.y;
    v.z = v.z + d.z;
    a.vel[t] = v;
}

// The particle-rigid velocity iterations (rigid solve_contact_velocities :44-128 with a static
// body, each followed by apply_contact_velocities): a particle's correction reads only its own
// velocity and the static colliders, so all iterations of a particle run in one thread, each
// adding its summed correction (zero without contacts) to a free particle's velocity.
__global__ __launch_bounds__(kBlock) void k_rigid_velocity(ContactArgs a, SubstepConsts c, uint32_t iters)
{
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= a.n) return;
    const ParticleClass &pc = pclass(a, t);
    if (!a.active[pc.scene]) return;
    const SceneInfo sc = a.scenes[pc.scene];
    if (!(sc.rigid | sc.rigid_pid)) return;
    const float w = a.pos[t].w;
    if (w <= kEps) return;
    const uint32_t rm = pc.kind == CN_PARTICLE_KIND_SOLID ? a.bnd[t] : 0u;
    const float4 g = rm ? a.rgen[t] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const float4 pm = a.part_mats[pc.part_mat];
    float4 v = a.vel[t];
    for (uint32_t it = 0; it < iters; ++it) {
        float sx = 0.0f, sy = 0.0f, sz = 0.0f;
        each_candidate(rm, a.bndl, t, [&](uint32_t k) {
            const Collider &cc = a.col[sc.col0 + k];
            float4 rec;
            if (!rigid_contact(cc, g.x, g.y, g.z, pc.radius, rec)) return;
            const float3 nr = safe_normalize(rec.x, rec.y, rec.z);
            // the contact point's velocity is +0, so the relative velocity is v - 0 = v
            const float nv = dot3(v.x, v.y, v.z, nr.x, nr.y, nr.z);
            if (nv >= 0.0f) return;
            const float denom = w + 0.0f;
            if (denom <= kEps) return;
            const bool rest_on = (-nv > c.cfg[kCfgRestitutionVelocity]) &&
                                 (rec.w <= c.cfg[kCfgRestitutionPenetration] * c.cfg[kCfgContactSlop]);
            const float restitution = rest_on ? fsat(rigid_material(pm, cc.material).y) : 0.0f;
            const float desired = rest_on ? (-restitution * nv) : 0.0f;
            const float imp = fmaxd(0.0f, fdiv(desired - nv, denom));
            sx = sx + (nr.x * imp) * w;
            sy = sy + (nr.y * imp) * w;
            sz = sz + (nr.z * imp) * w;
        });
        v.x = v.x + sx;
        v.y = v.y + sy;
        v.z = v.z + sz;
    }
    a.vel[t] = v;
}

__global__ __launch_bounds__(kBlock) void k_rigid_pick(RigidPidArgs a, SubstepConsts c)
{
    const uint32_t j = xcd_tile(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
    if (j >= a.nsoft) return;
    const uint32_t pid = a.soft_ids[j];
    const uint32_t scene = a.pid_scene[pid];
    uint32_t v = kPickSkip;
    if (a.active[scene] && a.scenes[scene].rigid_pid) {
        const uint32_t t = a.slot_of[min(pid, a.npid - 1u)];
        const ParticleClass &pc = a.classes[c.uniform_class ? 0u : a.cls[t]];
        v = pc.kind == CN_PARTICLE_KIND_SOLID && a.bnd[t] != 0u ? t : kPickNone;
    }
    a.pick[pid] = v;
}

__global__ __launch_bounds__(kBlock) void k_rigid_pid(RigidPidArgs a, SubstepConsts c)
{
    const uint32_t j = xcd_tile(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
    if (j >= a.nsoft) return;
    const uint32_t pid = a.soft_ids[j], v = a.pick[pid];
    if (v == kPickSkip) return;
    const SceneInfo &sc = a.scenes[a.pid_scene[pid]];
    float4 *posi = a.posi + ((a.solved * __popc(sc.soft_stages)) & 1u ? (size_t)a.npid : 0);
    const float4 p = posi[pid];
    if (p.w > kEps) posi[pid] = rigid_pid_particle(a, c, sc.col0, v, p);
}

static ContactArgs contact_args(const SceneBuffers &s, const SubstepConsts &c, int din)
{
    ContactArgs a;
    const int cur = s.cur;
    a.pos = s.pos[cur];
    a.vel = s.vel[cur];
    a.prev = s.prev[cur];
    a.cur = s.curpos;
    a.dacc = s.dacc[din];
    a.cls = s.cls[cur];
    a.id = s.id[cur];
    a.classes = s.classes;
    a.part_mats = s.part_mats;
    a.active = s.scene_active;
    a.scenes = s.scenes;
    a.rt = RunTable{s.run_key, s.run_start, s.run_info, s.bucket, c.bucket_shift, s.cellc};
    a.blk_first_run = s.blk_first_run;
    a.nblk = s.nblk;
    a.blk_halo = s.blk_halo;
    a.plist = s.ct_list;
    a.pcount = s.ct_count;
    a.crec = s.ct_rec;
    a.cbits = s.ct_bits;
    a.corr = s.ct_corr;
    a.meta = s.meta;
    a.adj_off = s.adj_off;
    a.adj_cnt = s.adj_cnt;
    a.adj_idx = s.adj_idx;
    a.col = s.colliders;
    a.bnd = s.bnd;
    a.bndl = s.bndl;
    a.rgen = s.ct_gen;
    a.n = c.n;
    a.pcap = kContactPartners;
    return a;
}

static uint32_t grid_c(uint32_t n) { return (n + kBlock - 1) / kBlock; }

void launch_contact_partners(const SceneBuffers &s, const SubstepConsts &c, hipStream_t st)
{
    const ContactArgs a = contact_args(s, c, 0);
    // pair candidates (with hash keys there are no cell blocks); without them the pass writes zero counts
    if (c.key_mode == CN_KEY_MORTON && c.pairs)
        hipLaunchKernelGGL(k_contact_partners, dim3(std::min(grid_c(c.n), 4096u)), dim3(kBlock), 0, st, a, c);
    else
        hipLaunchKernelGGL(k_contact_partners_walk, dim3(grid_c(c.n)), dim3(kBlock), 0, st, a, c);
}

void launch_contact_iteration(const SceneBuffers &s, const SubstepConsts &c, int din, hipStream_t st)
{
    const ContactArgs a = contact_args(s, c, din);
    hipLaunchKernelGGL(k_contact_solve, dim3(grid_c(c.n)), dim3(kBlock), 0, st, a, c);
    hipLaunchKernelGGL(k_contact_apply, dim3(grid_c(c.n)), dim3(kBlock), 0, st, a);
}

void launch_contact_velocity(const SceneBuffers &s, const SubstepConsts &c, hipStream_t st)
{
    const ContactArgs a = contact_args(s, c, 0);
    hipLaunchKernelGGL(k_contact_velocity, dim3(grid_c(c.n)), dim3(kBlock), 0, st, a, c);
    hipLaunchKernelGGL(k_contact_velocity_apply, dim3(grid_c(c.n)), dim3(kBlock), 0, st, a);
}

RigidPidArgs rigid_pid_args(const SceneBuffers &s, uint32_t solved)
{
    RigidPidArgs a;
    a.posi = s.posi;
    a.soft_ids = s.soft_ids;
    a.nsoft = s.nsoft;
    a.slot_of = s.slot_of;
    a.pid_scene = s.pid_scene;
    a.active = s.scene_active;
    a.scenes = s.scenes;
    a.col = s.colliders;
    a.bnd = s.bnd;
    a.bndl = s.bndl;
    a.prev = s.prev[s.cur];
    a.cls = s.cls[s.cur];
    a.classes = s.classes;
    a.part_mats = s.part_mats;
    a.rgen = s.ct_gen;
    a.pick = s.rigid_pick;
    a.npid = s.npid;
    a.solved = solved;
    return a;
}

void launch_rigid_pick(const SceneBuffers &s, const SubstepConsts &c, hipStream_t st)
{
    if (!s.nsoft) return;
    hipLaunchKernelGGL(k_rigid_pick, dim3(grid_c(s.nsoft)), dim3(kBlock), 0, st, rigid_pid_args(s, 0), c);
}

void launch_rigid_pid(const SceneBuffers &s, const SubstepConsts &c, uint32_t solved, hipStream_t st)
{
    if (!s.nsoft) return;
    hipLaunchKernelGGL(k_rigid_pid, dim3(grid_c(s.nsoft)), dim3(kBlock), 0, st, rigid_pid_args(s, solved), c);
}

void launch_rigid_velocity(const SceneBuffers &s, const SubstepConsts &c, uint32_t iters, hipStream_t st)
{
    const ContactArgs a = contact_args(s, c, 0);
    hipLaunchKernelGGL(k_rigid_velocity, dim3(grid_c(c.n)), dim3(kBlock), 0, st, a, c, iters);
}

}  // namespace cn
