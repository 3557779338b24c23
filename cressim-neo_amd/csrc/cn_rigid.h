#ifndef CN_RIGID_H
#define CN_RIGID_H
// cn_rigid.h -- particle-rigid contacts of one particle against static colliders, and the form of them
// that the soft passes solve in particle-index order (cn_contact.hip holds the passes and the
// reference's file names).
#include "cn_internal.h"

namespace cn {

constexpr int kCfgSoftContactRelax = 2;
constexpr int kCfgSoftMaxCorrection = 3;
constexpr int kCfgRestitutionVelocity = 4;
constexpr int kCfgRestitutionPenetration = 5;

// SafeNormalize, physics_math.hlsli:6-12, with rsqrt as 1 / sqrt
__device__ __forceinline__ float3 safe_normalize(float x, float y, float z)
{
    const float l2 = dot3(x, y, z, x, y, z);
    if (l2 <= kEps) return make_float3(0.0f, 1.0f, 0.0f);
    const float r = fdiv(1.0f, fsqrt(l2));
    return make_float3(x * r, y * r, z * r);
}

// ComputePositionFrictionDelta, physics_rigid_solver_shared.hlsli:50-67
__device__ __forceinline__ float3 friction_delta(const float *cfg, float ex, float ey, float ez, float pen, float kin,
                                                 float stat)
{
    const float td = len3(ex, ey, ez);
    if (td <= cfg[kCfgPosFrictionMin] || pen <= kEps) return make_float3(0.0f, 0.0f, 0.0f);
    const float sl = fsat(stat) * pen;
    if (td <= sl) return make_float3(ex, ey, ez);
    const float ks = fmind(fdiv(fsat(kin) * pen, td), 1.0f);
    return make_float3(ex * ks, ey * ks, ez * ks);
}

// physics_particle_rigid_generate_contacts.cs.hlsl:82-176 for one static collider: the position
// in the collider frame, the shape's signed distance and local normal, penetration = radius -
// distance.  Returns true with (world normal, penetration) when the penetration is positive; the
// world normal is SafeNormalize of the rotated local normal.
__device__ __forceinline__ bool rigid_contact(const Collider &c, float px, float py, float pz, float radius,
                                              float4 &rec)
{
    if (!c.enabled) return false;
    float ux, uy, uz;
    quat_rotate(-c.q[0], -c.q[1], -c.q[2], c.q[3], __fsub_rn(px, c.c[0]), __fsub_rn(py, c.c[1]),
                __fsub_rn(pz, c.c[2]), ux, uy, uz);  // QuaternionInverseRotate
    float nx = 0.0f, ny = 1.0f, nz = 0.0f, sd = 0.0f;
    if (c.shape == CN_SHAPE_SPHERE) {
        const float len = len3(ux, uy, uz);
        if (len > kEps) {
            nx = fdiv(ux, len); ny = fdiv(uy, len); nz = fdiv(uz, len);
        }
        sd = __fsub_rn(len, c.he[0]);
    } else if (c.shape == CN_SHAPE_BOX) {
        box_local_contact(c.he, ux, uy, uz, sd, nx, ny, nz);
    } else {
        // capsule: the closest point of the world segment; the world normal (fallback +x) is taken
        // into the collider frame
        const float gx = __fsub_rn(c.sb[0], c.sa[0]), gy = __fsub_rn(c.sb[1], c.sa[1]), gz = __fsub_rn(c.sb[2], c.sa[2]);
        const float lsq = dot3(gx, gy, gz, gx, gy, gz);
        float t = 0.0f;
        if (lsq > kEps) {
            const float wx = __fsub_rn(px, c.sa[0]), wy = __fsub_rn(py, c.sa[1]), wz = __fsub_rn(pz, c.sa[2]);
            t = fsat(fdiv(dot3(wx, wy, wz, gx, gy, gz), lsq));
        }
        const float ex = __fsub_rn(px, __fadd_rn(c.sa[0], __fmul_rn(t, gx)));
        const float ey = __fsub_rn(py, __fadd_rn(c.sa[1], __fmul_rn(t, gy)));
        const float ez = __fsub_rn(pz, __fadd_rn(c.sa[2], __fmul_rn(t, gz)));
        const float len = len3(ex, ey, ez);
        float wx = 1.0f, wy = 0.0f, wz = 0.0f;
        if (len > kEps) {
            wx = fdiv(ex, len); wy = fdiv(ey, len); wz = fdiv(ez, len);
        }
        sd = __fsub_rn(len, c.he[0]);
        quat_rotate(-c.q[0], -c.q[1], -c.q[2], c.q[3], wx, wy, wz, nx, ny, nz);
    }
    const float pen = __fsub_rn(radius, sd);
    if (!(pen > 0.0f)) return false;
    float wx, wy, wz;
    quat_rotate(c.q[0], c.q[1], c.q[2], c.q[3], nx, ny, nz, wx, wy, wz);
    const float3 n = safe_normalize(wx, wy, wz);
    rec = make_float4(n.x, n.y, n.z, pen);
    return true;
}

// CombineContactMaterial of a particle material and a collider's
__device__ __forceinline__ float3 rigid_material(const float4 pm, const float *cm)
{
    return make_float3(fsqrt(fmaxd(0.0f, pm.x) * fmaxd(0.0f, cm[0])), fmaxd(fmaxd(0.0f, pm.y), fmaxd(0.0f, cm[1])),
                       fsqrt(fmaxd(0.0f, pm.w) * fmaxd(0.0f, cm[3])));
}

// rigid solve_contacts :45-140 against a static body: the position correction of a particle at p
// (inverse mass p.w; pv its position at the start of the substep) with contact rec = (normal,
// penetration) against collider cc; false when the contact adds nothing.  The displacement of a
// static body's contact point is +0, its effective mass 0.
__device__ __forceinline__ bool rigid_position(const float4 p, const float4 pv, const float4 rec, const float4 pm,
                                               const Collider &cc, const SubstepConsts &c, float3 &d)
{
    const float w = p.w;
    if (w <= kEps) return false;
    const float pn = fmind(fmaxd(rec.w - c.cfg[kCfgContactSlop], 0.0f), c.cfg[kCfgSoftMaxCorrection]);
    if (pn <= 0.0f) return false;
    const float3 nr = safe_normalize(rec.x, rec.y, rec.z);
    const float3 mat = rigid_material(pm, cc.material);
    const float denom = w + 0.0f;
    if (denom <= kEps) return false;
    const float relax = c.cfg[kCfgSoftContactRelax];
    const float lambda = fdiv(pn, denom) * relax;
    float cx = nr.x * (w * lambda), cy = nr.y * (w * lambda), cz = nr.z * (w * lambda);
    // relative displacement = (contact point - its previous position) - (x - x_prev), the first
    // term +0 for a static body
    const float rx = 0.0f - (p.x - pv.x), ry = 0.0f - (p.y - pv.y), rz = 0.0f - (p.z - pv.z);
    const float rn = dot3(rx, ry, rz, nr.x, nr.y, nr.z);
    const float3 fd = friction_delta(c.cfg, rx - nr.x * rn, ry - nr.y * rn, rz - nr.z * rn, pn, mat.x, mat.z);
    const float fdist = len3(fd.x, fd.y, fd.z);
    if (fdist > 0.0f) {
        const float tden = w + 0.0f;
        if (tden > kEps) {
            const float tl = fdiv(fdist, tden);
            const float k = (tl * w) * relax;
            cx = cx + fdiv(fd.x, fdist) * k;
            cy = cy + fdiv(fd.y, fdist) * k;
            cz = cz + fdiv(fd.z, fdist) * k;
        }
    }
    d = make_float3(cx, cy, cz);
    return true;
}

// The particle-rigid contacts of a scene whose every particle is constrained and which holds no
// particle-particle pair, in particle-index order on the soft phase's positions right after its
// last apply of the iteration (the reference's contact pass of the iteration, for such a scene):
// each candidate's contact at the current position, the static-body solve, their sum (zero without
// contacts) added to a free particle.  The scene then needs no slot-order contact pass, and its
// constrained positions stay in particle-index order across the iteration.
struct RigidPidArgs {
    float4 *posi;
    const uint32_t *soft_ids;
    uint32_t nsoft;
    const uint32_t *slot_of;
    const uint32_t *pid_scene;
    const uint32_t *active;
    const SceneInfo *scenes;
    const Collider *col;
    const uint32_t *bnd;      // slot order
    const uint16_t *bndl;
    const float4 *prev;       // slot order
    const uint32_t *cls;      // slot order
    const ParticleClass *classes;
    const float4 *part_mats;
    float4 *rgen;             // slot order
    uint32_t *pick;           // per constrained particle, by its index: kPickSkip, kPickNone or its slot
    uint32_t npid;
    uint32_t solved;          // soft iterations since the gather, in the tiled passes' two position buffers
};

// What the iterations of a substep do for a constrained particle, fixed for the substep (slot,
// class, collider candidates): nothing (its scene is not stepped or not solved here), add a zero
// sum (no candidates), or solve the candidates of its slot.
constexpr uint32_t kPickSkip = 0xffffffffu, kPickNone = 0xfffffffeu;

// One such particle's contacts at p (free); v: its pick, not kPickSkip.
__device__ __forceinline__ float4 rigid_pid_particle(const RigidPidArgs &a, const SubstepConsts &c, uint32_t col0,
                                                     uint32_t v, float4 p)
{
    float sx = 0.0f, sy = 0.0f, sz = 0.0f;
    if (v != kPickNone) {
        const uint32_t t = v, rm = a.bnd[t];
        const ParticleClass &pc = a.classes[c.uniform_class ? 0u : a.cls[t]];
        a.rgen[t] = p;
        const float4 pv = a.prev[t];
        const float4 pm = a.part_mats[pc.part_mat];
        each_candidate(rm, a.bndl, t, [&](uint32_t k) {
            const Collider &cc = a.col[col0 + k];
            float4 rec;
            float3 d;
            if (!rigid_contact(cc, p.x, p.y, p.z, pc.radius, rec)) return;
            if (!rigid_position(p, pv, rec, pm, cc, c, d)) return;
            sx = sx + d.x;
            sy = sy + d.y;
            sz = sz + d.z;
        });
    }
    p.x = p.x + sx;
    p.y = p.y + sy;
    p.z = p.z + sz;
    return p;
}

}  // namespace cn

#endif
