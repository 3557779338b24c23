// cn_soft.hip -- XPBD soft-body and cloth constraints on gfx950.
//
// Reference passes (assets/shaders/physics/soft/solver/): physics_soft_solve_edge_constraints.cs.hlsl
// :10-74, physics_soft_solve_bend_constraints.cs.hlsl:20-86,
// physics_cloth_solve_dihedral_constraints.cs.hlsl:20-95, physics_soft_solve_tet_constraints.cs.hlsl
// :15-87, physics_soft_apply_{edge,bend,tet}_corrections.cs.hlsl and
// physics_clear_soft_constraint_state.cs.hlsl:14-54.  Each solve is Jacobi over its constraint type:
// every constraint reads the current positions, updates its lambda and gives one correction record
// per vertex; then, per particle, the records of its incident constraints are summed in ascending
// constraint order (the incidence lists of physics_scene_gpu_state.cpp:3273-3360) and the sum added to
// the position: in one launch per group over tiles of particles, or in passes over the whole pool.  Constraints refer to
// particle indices; positions live in slot order, reached through slot_of[particle index].
#include <hip/hip_runtime.h>

#include <utility>

#include "cn_rigid.h"

namespace cn {

// Workgroup size of the soft passes.  They run beside the persistent fluid workgroups (eight waves
// each); measured on a pool of fluid, tet and cloth scenes, 512 threads step it in 49.3 ms against
// 50.6 at 256, 51.5 at 128 and 55.7 at 1024.
constexpr uint32_t kSoftBlock = 512;

static inline uint32_t grid_n(uint32_t n) { return (n + kSoftBlock - 1) / kSoftBlock; }

// A constraint's correction records, written where its vertices' incidence lists read them.
struct RecOut {
    CorrRec *rec;
    const uint32_t *map;
    __device__ CorrRec &operator[](uint32_t k) const { return rec[map[k]]; }
};

__device__ __forceinline__ CorrRec rec3(float x, float y, float z) { return CorrRec{x, y, z}; }

__device__ __forceinline__ float4 ldp(const SoftArgs &a, uint32_t particle) { return a.posi[particle]; }

// Constraints and particles of scenes that this step leaves untouched are skipped (records kept);
// a step of every scene skips the two dependent loads of the check.
__device__ __forceinline__ bool live(const SoftArgs &a, uint32_t particle)
{
    return a.all_live || a.active[a.pid_scene[particle]] != 0u;
}

__device__ __forceinline__ void cross3d(float ax, float ay, float az, float bx, float by, float bz, float &ox, float &oy,
                                        float &oz)
{
    ox = ay * bz - az * by;
    oy = az * bx - ax * bz;
    oz = ax * by - ay * bx;
}

// The solves of one constraint: the correction record of each vertex and the new lambda from the
// vertices' positions (inverse mass in w).  False: a degenerate constraint, whose records are zero (a
// tet's keep their previous values) and whose lambda stays.
__device__ __forceinline__ bool solve_edge(const float4 pa, const float4 pb, float rest, float compliance,
                                           const SoftArgs &a, float lambda, float &lam, CorrRec (&r)[2])
{
    if (compliance != compliance) return false;  // disabled
    const float wa = pa.w, wb = pb.w, wsum = wa + wb;
    if (wsum <= kEps) return false;
    const float dx = pb.x - pa.x, dy = pb.y - pa.y, dz = pb.z - pa.z;
    const float l2 = dot3(dx, dy, dz, dx, dy, dz);
    if (l2 <= kEps) return false;
    const float len = fsqrt(l2);
    const float gax = fdiv(-dx, len), gay = fdiv(-dy, len), gaz = fdiv(-dz, len);
    const float gbx = -gax, gby = -gay, gbz = -gaz;
    const float alpha = fdiv(compliance, fmaxd(a.dt * a.dt, kEps));
    const float C = len - rest;
    const float den = wsum + alpha;
    if (den <= kEps) return false;
    const float dl = fdiv(-(C + alpha * lambda), den);
    lam = lambda + dl;
    const float fa = wa * dl, fb = wb * dl;
    r[0] = rec3(fa * gax * a.relax, fa * gay * a.relax, fa * gaz * a.relax);
    r[1] = rec3(fb * gbx * a.relax, fb * gby * a.relax, fb * gbz * a.relax);
    return true;
}

__device__ __forceinline__ bool solve_bend(const float4 p0, const float4 p1, const float4 p2, float rest,
                                           float compliance, const SoftArgs &a, float lambda, float &lam,
                                           CorrRec (&r)[4])
{
    const float w0 = p0.w, w1 = p1.w, w2 = p2.w;
    if (w0 + w1 + w2 <= kEps) return false;
    const float e0x = p0.x - p1.x, e0y = p0.y - p1.y, e0z = p0.z - p1.z;
    const float e1x = p2.x - p1.x, e1y = p2.y - p1.y, e1z = p2.z - p1.z;
    const float l0s = dot3(e0x, e0y, e0z, e0x, e0y, e0z), l1s = dot3(e1x, e1y, e1z, e1x, e1y, e1z);
    if (l0s <= kEps || l1s <= kEps) return false;
    const float l0 = fsqrt(l0s), l1 = fsqrt(l1s);
    const float d0x = fdiv(e0x, l0), d0y = fdiv(e0y, l0), d0z = fdiv(e0z, l0);
    const float d1x = fdiv(e1x, l1), d1y = fdiv(e1y, l1), d1z = fdiv(e1z, l1);
    const float ct = fclamp(dot3(d0x, d0y, d0z, d1x, d1y, d1z), -1.0f + 1.0e-4f, 1.0f - 1.0e-4f);
    const float st = fsqrt(fmaxd(1.0f - ct * ct, 1.0e-8f));
    const float theta = cephes_acosf(ct);
    const float q0 = fmaxd(l0 * st, kEps), q2 = fmaxd(l1 * st, kEps);
    const float g0x = fdiv(-(d1x - ct * d0x), q0);
    const float g0y = fdiv(-(d1y - ct * d0y), q0);
    const float g0z = fdiv(-(d1z - ct * d0z), q0);
    const float g2x = fdiv(-(d0x - ct * d1x), q2);
    const float g2y = fdiv(-(d0y - ct * d1y), q2);
    const float g2z = fdiv(-(d0z - ct * d1z), q2);
    const float g1x = -(g0x + g2x);
    const float g1y = -(g0y + g2y);
    const float g1z = -(g0z + g2z);
    const float den = w0 * dot3(g0x, g0y, g0z, g0x, g0y, g0z) + w1 * dot3(g1x, g1y, g1z, g1x, g1y, g1z) +
                      w2 * dot3(g2x, g2y, g2z, g2x, g2y, g2z);
    const float alpha = fdiv(compliance, fmaxd(a.dt * a.dt, kEps));
    if (den + alpha <= kEps) return false;
    const float C = theta - rest;
    const float dl = fdiv(-(C + alpha * lambda), den + alpha);
    lam = lambda + dl;
    const float f0 = w0 * dl, f1 = w1 * dl, f2 = w2 * dl, x = a.relax;
    r[0] = rec3(f0 * g0x * x, f0 * g0y * x, f0 * g0z * x);
    r[1] = rec3(f1 * g1x * x, f1 * g1y * x, f1 * g1z * x);
    r[2] = rec3(f2 * g2x * x, f2 * g2y * x, f2 * g2z * x);
    r[3] = rec3(0.0f, 0.0f, 0.0f);
    return true;
}

__device__ __forceinline__ bool solve_dihedral(const float4 e0m, const float4 e1m, const float4 o0m, const float4 o1m,
                                               float rest, float compliance, const SoftArgs &a, float lambda,
                                               float &lam, CorrRec (&r)[4])
{
    // p0, p1 opposite vertices; p2, p3 edge vertices
    const float ex = e1m.x - e0m.x, ey = e1m.y - e0m.y, ez = e1m.z - e0m.z;
    const float el2 = dot3(ex, ey, ez, ex, ey, ez);
    float n0x, n0y, n0z, n1x, n1y, n1z;
    cross3d(e0m.x - o0m.x, e0m.y - o0m.y, e0m.z - o0m.z, e1m.x - o0m.x, e1m.y - o0m.y, e1m.z - o0m.z, n0x, n0y, n0z);
    cross3d(e1m.x - o1m.x, e1m.y - o1m.y, e1m.z - o1m.z, e0m.x - o1m.x, e0m.y - o1m.y, e0m.z - o1m.z, n1x, n1y, n1z);
    const float n0s = dot3(n0x, n0y, n0z, n0x, n0y, n0z), n1s = dot3(n1x, n1y, n1z, n1x, n1y, n1z);
    if (el2 <= kEps || n0s <= kEps || n1s <= kEps) {
        return false;
    }
    const float el = fsqrt(el2);
    const float iel = fdiv(1.0f, el);
    const float s0x = fdiv(n0x, n0s), s0y = fdiv(n0y, n0s), s0z = fdiv(n0z, n0s);
    const float s1x = fdiv(n1x, n1s), s1y = fdiv(n1y, n1s), s1z = fdiv(n1z, n1s);
    const float f00 = dot3(o0m.x - e1m.x, o0m.y - e1m.y, o0m.z - e1m.z, ex, ey, ez) * iel;
    const float f01 = dot3(o1m.x - e1m.x, o1m.y - e1m.y, o1m.z - e1m.z, ex, ey, ez) * iel;
    const float f10 = dot3(e0m.x - o0m.x, e0m.y - o0m.y, e0m.z - o0m.z, ex, ey, ez) * iel;
    const float f11 = dot3(e0m.x - o1m.x, e0m.y - o1m.y, e0m.z - o1m.z, ex, ey, ez) * iel;
    const float g0x = -(f00 * s0x + f01 * s1x), g0y = -(f00 * s0y + f01 * s1y), g0z = -(f00 * s0z + f01 * s1z);
    const float g1x = -(f10 * s0x + f11 * s1x), g1y = -(f10 * s0y + f11 * s1y), g1z = -(f10 * s0z + f11 * s1z);
    const float g2x = -(el * s0x), g2y = -(el * s0y), g2z = -(el * s0z);
    const float g3x = -(el * s1x), g3y = -(el * s1y), g3z = -(el * s1z);
    const float r0 = fsqrt(n0s), r1 = fsqrt(n1s);
    const float u0x = fdiv(n0x, r0), u0y = fdiv(n0y, r0), u0z = fdiv(n0z, r0);
    const float u1x = fdiv(n1x, r1), u1y = fdiv(n1y, r1), u1z = fdiv(n1z, r1);
    float cx, cy, cz;
    cross3d(u0x, u0y, u0z, u1x, u1y, u1z, cx, cy, cz);
    const float theta = cephes_atan2f(dot3(ex * iel, ey * iel, ez * iel, cx, cy, cz),
                                      fclamp(dot3(u0x, u0y, u0z, u1x, u1y, u1z), -1.0f, 1.0f));
    const float two_pi = 6.283185307179586f, pi = 3.141592653589793f;
    float C = theta - rest;
    C = C - two_pi * floorf(fdiv(C + pi, two_pi));
    const float w0 = e0m.w, w1 = e1m.w, w2 = o0m.w, w3 = o1m.w;
    const float den = w0 * dot3(g0x, g0y, g0z, g0x, g0y, g0z) + w1 * dot3(g1x, g1y, g1z, g1x, g1y, g1z) +
                      w2 * dot3(g2x, g2y, g2z, g2x, g2y, g2z) + w3 * dot3(g3x, g3y, g3z, g3x, g3y, g3z);
    const float alpha = fdiv(compliance, fmaxd(a.dt * a.dt, kEps));
    if (den + alpha <= kEps) {
        return false;
    }
    const float dl = fdiv(-(C + alpha * lambda), den + alpha);
    lam = lambda + dl;
    const float f0 = w0 * dl, f1 = w1 * dl, f2 = w2 * dl, f3 = w3 * dl, x = a.relax;
    r[0] = rec3(f0 * g0x * x, f0 * g0y * x, f0 * g0z * x);
    r[1] = rec3(f1 * g1x * x, f1 * g1y * x, f1 * g1z * x);
    r[2] = rec3(f2 * g2x * x, f2 * g2y * x, f2 * g2z * x);
    r[3] = rec3(f3 * g3x * x, f3 * g3y * x, f3 * g3z * x);
    return true;
}

__device__ __forceinline__ bool solve_tet(const float4 p0, const float4 p1, const float4 p2, const float4 p3,
                                          float rest, float compliance, const SoftArgs &a, float lambda, float &lam,
                                          CorrRec (&r)[4])
{
    const float w0 = p0.w, w1 = p1.w, w2 = p2.w, w3 = p3.w;
    if ((w0 + w1 + w2 + w3) <= kEps) return false;
    float cx, cy, cz;
    cross3d(p1.x - p0.x, p1.y - p0.y, p1.z - p0.z, p2.x - p0.x, p2.y - p0.y, p2.z - p0.z, cx, cy, cz);
    const float sv = fdiv(dot3(cx, cy, cz, p3.x - p0.x, p3.y - p0.y, p3.z - p0.z), 6.0f);
    const float sgn = sv >= 0.0f ? 1.0f : -1.0f;
    const float C = fabsf(sv) - rest;
    const float f = fdiv(sgn, 6.0f);
    float g0x, g0y, g0z, g1x, g1y, g1z, g2x, g2y, g2z, g3x, g3y, g3z;
    cross3d(p3.x - p1.x, p3.y - p1.y, p3.z - p1.z, p2.x - p1.x, p2.y - p1.y, p2.z - p1.z, g0x, g0y, g0z);
    cross3d(p2.x - p0.x, p2.y - p0.y, p2.z - p0.z, p3.x - p0.x, p3.y - p0.y, p3.z - p0.z, g1x, g1y, g1z);
    cross3d(p3.x - p0.x, p3.y - p0.y, p3.z - p0.z, p1.x - p0.x, p1.y - p0.y, p1.z - p0.z, g2x, g2y, g2z);
    cross3d(p1.x - p0.x, p1.y - p0.y, p1.z - p0.z, p2.x - p0.x, p2.y - p0.y, p2.z - p0.z, g3x, g3y, g3z);
    g0x = g0x * f; g0y = g0y * f; g0z = g0z * f;
    g1x = g1x * f; g1y = g1y * f; g1z = g1z * f;
    g2x = g2x * f; g2y = g2y * f; g2z = g2z * f;
    g3x = g3x * f; g3y = g3y * f; g3z = g3z * f;
    const float sg = w0 * dot3(g0x, g0y, g0z, g0x, g0y, g0z) + w1 * dot3(g1x, g1y, g1z, g1x, g1y, g1z) +
                     w2 * dot3(g2x, g2y, g2z, g2x, g2y, g2z) + w3 * dot3(g3x, g3y, g3z, g3x, g3y, g3z);
    const float alpha = fdiv(compliance, fmaxd(a.dt * a.dt, kEps));
    const float den = sg + alpha;
    if (den <= kEps) return false;
    const float dl = fdiv(-(C + alpha * lambda), den);
    lam = lambda + dl;
    const float f0 = w0 * dl, f1 = w1 * dl, f2 = w2 * dl, f3 = w3 * dl, x = a.relax;
    r[0] = rec3(f0 * g0x * x, f0 * g0y * x, f0 * g0z * x);
    r[1] = rec3(f1 * g1x * x, f1 * g1y * x, f1 * g1z * x);
    r[2] = rec3(f2 * g2x * x, f2 * g2y * x, f2 * g2z * x);
    r[3] = rec3(f3 * g3x * x, f3 * g3y * x, f3 * g3z * x);
    return true;
}

// ---------------------------------------------------------------------------------------------
// tiled passes: a constraint group's solve and apply in one launch
// ---------------------------------------------------------------------------------------------
// A workgroup takes one tile (SoftTile): positions of its particles and of those its constraints reach
// into LDS, every constraint that touches one of its particles solved (a constraint on the border of
// tiles by each of them), the records of its own particles summed in ascending constraint order from
// LDS, the new positions written.  Positions and lambdas alternate between two buffers, so a tile
// reads what every tile started from whatever has finished.  Against the passes over the whole pool
// (a solve that writes every vertex's record to memory, an apply that reads them back) a tet moves
// some 45 bytes instead of 144 and an edge 35 instead of 80, for 1.3 to 1.5 times the solves, and an
// iteration takes half the launches: 48 mixed scenes 6,033 -> 4,955 us a step, a 256 x 256 cloth
// 996 -> 829 us (both of 4 substeps and 4 iterations; 2 x 2 launches an iteration before, 2 now).
// What bounds it: the latency of a tile's three phases (load, solve, sum), 500 tiles of 128 to 64,000
// particles being two a CU.
constexpr int kTileThreads = 512;
// RIGID: a scene's last group also solves the iteration's particle-rigid contacts of its particles (a
// launch of their own took 5 us an iteration: a 256 x 256 cloth's step 829 us against 766, a 32^3 tet
// block's 863 against 780).
template <int G, bool RIGID>
__global__ __launch_bounds__(kTileThreads) void k_soft_tile(SoftArgs a, RigidPidArgs ra, SubstepConsts c)
{
    extern __shared__ float4 lp[];
    constexpr uint32_t A = G == 0 ? 2u : 4u;  // vertices per constraint
    const uint32_t tid = threadIdx.x;
    const SoftTile T = a.tiles[(G > 0 ? a.ntiles[0] : 0u) + (G > 1 ? a.ntiles[1] : 0u) + xcd_tile(blockIdx.x, gridDim.x)];
    if (!a.all_live && !a.active[T.scene]) return;
    const uint32_t stages = a.scenes[T.scene].soft_stages;
    const uint32_t step = a.solved * __popc(stages) + __popc(stages & ((1u << G) - 1u));
    const float4 *__restrict__ pin = a.posi + (step & 1u ? (size_t)a.n : 0);
    float4 *__restrict__ pout = a.posi + (step & 1u ? 0 : (size_t)a.n);
    CorrRec *rec = reinterpret_cast<CorrRec *>(lp + T.nown + T.nhalo);
    for (uint32_t k = tid; k < T.nown + T.nhalo; k += kTileThreads)
        lp[k] = pin[k < T.nown ? a.own[T.own0 + k] : a.halo[T.halo0 + (k - T.nown)]];
    __syncthreads();
    for (uint32_t k = tid; k < T.nent; k += kTileThreads) {
        const uint32_t e = T.ent0 + k, cw = a.con[G][e], con = cw & ~kTileOwner;
        uint32_t v[A], s[A];
#pragma unroll
        for (uint32_t u = 0; u < A; u += 2) {
            const uint32_t vw = a.verts[G][(size_t)e * (A / 2) + u / 2], sw = a.slots[G][(size_t)e * (A / 2) + u / 2];
            v[u] = vw & 0xffffu;
            v[u + 1] = vw >> 16;
            s[u] = sw & 0xffffu;
            s[u + 1] = sw >> 16;
        }
        const float2 prm = a.prm[G][con];
        const float lambda = a.first ? 0.0f : a.lam_in[G][con];
        float lam = lambda;
        CorrRec r[A];
#pragma unroll
        for (uint32_t u = 0; u < A; ++u) r[u] = rec3(0.0f, 0.0f, 0.0f);
        if constexpr (G == 0) {
            solve_edge(lp[v[0]], lp[v[1]], prm.x, prm.y, a, lambda, lam, r);
        } else if constexpr (G == 1) {
            if (con < a.nb) solve_bend(lp[v[0]], lp[v[1]], lp[v[2]], prm.x, prm.y, a, lambda, lam, r);
            else solve_dihedral(lp[v[0]], lp[v[1]], lp[v[2]], lp[v[3]], prm.x, prm.y, a, lambda, lam, r);
        } else {
            // A degenerate tet keeps its records, which therefore have a place in memory too.  Where the
            // compliance term alone exceeds the threshold and no inverse mass is negative none can
            // become degenerate within the step: they are written by its last iteration only (every
            // iteration: a pool of fluid, tet and cloth scenes 5,314 us a step against 4,912).
            CorrRec *kept = a.corr_t + 4 * (size_t)con;
            const float4 p0 = lp[v[0]], p1 = lp[v[1]], p2 = lp[v[2]], p3 = lp[v[3]];
            const bool sure = fdiv(prm.y, fmaxd(a.dt * a.dt, kEps)) > kEps && p0.w >= 0.0f && p1.w >= 0.0f &&
                              p2.w >= 0.0f && p3.w >= 0.0f;
            const bool on = solve_tet(p0, p1, p2, p3, prm.x, prm.y, a, lambda, lam, r);
            if (!on) {
#pragma unroll
                for (uint32_t u = 0; u < A; ++u) r[u] = kept[u];
            } else if ((cw & kTileOwner) && (!sure || a.keep_tets)) {
#pragma unroll
                for (uint32_t u = 0; u < A; ++u) kept[u] = r[u];
            }
        }
        if (cw & kTileOwner) a.lam_out[G][con] = lam;
#pragma unroll
        for (uint32_t u = 0; u < A; ++u)
            if (s[u] != kTileNoRec) rec[s[u]] = r[u];
    }
    __syncthreads();
    const SceneInfo &sc = a.scenes[T.scene];
    const bool contacts = RIGID && (stages >> (G + 1)) == 0u && sc.rigid_pid;
    for (uint32_t k = tid; k < T.nown; k += kTileThreads) {
        float4 p = lp[k];
        const uint32_t pid = a.own[T.own0 + k];
        const uint32_t k0 = a.starts[T.start0 + k], k1 = a.starts[T.start0 + k + 1];
        if (k0 != k1 && !(p.w <= kEps)) {
            float tx = 0.0f, ty = 0.0f, tz = 0.0f;
            for (uint32_t q = k0; q < k1; ++q) {
                tx = tx + rec[q].x;
                ty = ty + rec[q].y;
                tz = tz + rec[q].z;
            }
            p.x = p.x + tx;
            p.y = p.y + ty;
            p.z = p.z + tz;
        }
        if (RIGID && contacts && p.w > kEps) p = rigid_pid_particle(ra, c, sc.col0, ra.pick[pid], p);
        pout[pid] = p;
    }
}

// ---------------------------------------------------------------------------------------------
// passes over the whole pool, where a particle has more constraints than a tile's LDS holds records
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(kSoftBlock) void k_solve_edges(SoftArgs a)
{
    const uint32_t e = xcd_tile(blockIdx.x, gridDim.x) * kSoftBlock + threadIdx.x;
    if (e >= a.ne) return;
    const EdgeDev E = a.edges[e];
    if (!live(a, E.a)) return;
    const RecOut out{a.corr_e, a.map_e + 2 * (size_t)e};
    CorrRec r[2] = {rec3(0.0f, 0.0f, 0.0f), rec3(0.0f, 0.0f, 0.0f)};
    const float lambda = a.first ? 0.0f : a.lam_e[e];
    float lam = lambda;
    const bool on = solve_edge(ldp(a, E.a), ldp(a, E.b), E.rest_length, E.compliance, a, lambda, lam, r);
    if (on || a.first) a.lam_e[e] = lam;
    out[0] = r[0];
    out[1] = r[1];
}

__global__ __launch_bounds__(kSoftBlock) void k_solve_bends(SoftArgs a)
{
    const uint32_t b = xcd_tile(blockIdx.x, gridDim.x) * kSoftBlock + threadIdx.x;
    if (b >= a.nb) return;
    const BendDev B = a.bends[b];
    if (!live(a, B.p0)) return;
    const RecOut out{a.corr_b, a.map_b + 4 * (size_t)b};
    const CorrRec z = rec3(0.0f, 0.0f, 0.0f);
    CorrRec r[4] = {z, z, z, z};
    const float lambda = a.first ? 0.0f : a.lam_b[b];
    float lam = lambda;
    const bool on = solve_bend(ldp(a, B.p0), ldp(a, B.p1), ldp(a, B.p2), B.rest_angle, B.compliance, a, lambda, lam, r);
    if (on || a.first) a.lam_b[b] = lam;
#pragma unroll
    for (int k = 0; k < 4; ++k) out[k] = r[k];
}

__global__ __launch_bounds__(kSoftBlock) void k_solve_dihedrals(SoftArgs a)
{
    const uint32_t d = xcd_tile(blockIdx.x, gridDim.x) * kSoftBlock + threadIdx.x;
    if (d >= a.nd) return;
    const uint32_t ci = a.nb + d;
    const DihedralDev D = a.dih[d];
    if (!live(a, D.e0)) return;
    const RecOut out{a.corr_b, a.map_b + 4 * (size_t)ci};
    const CorrRec z = rec3(0.0f, 0.0f, 0.0f);
    CorrRec r[4] = {z, z, z, z};
    const float lambda = a.first ? 0.0f : a.lam_b[ci];
    float lam = lambda;
    const bool on = solve_dihedral(ldp(a, D.e0), ldp(a, D.e1), ldp(a, D.o0), ldp(a, D.o1), D.rest_angle, D.compliance, a,
                                   lambda, lam, r);
    if (on || a.first) a.lam_b[ci] = lam;
#pragma unroll
    for (int k = 0; k < 4; ++k) out[k] = r[k];
}

__global__ __launch_bounds__(kSoftBlock) void k_solve_tets(SoftArgs a)
{
    const uint32_t t = xcd_tile(blockIdx.x, gridDim.x) * kSoftBlock + threadIdx.x;
    if (t >= a.nt) return;
    const TetDev T = a.tets[t];
    if (!live(a, T.p[0])) return;
    CorrRec r[4];
    const float lambda = a.first ? 0.0f : a.lam_t[t];
    float lam = lambda;
    const bool on = solve_tet(ldp(a, T.p[0]), ldp(a, T.p[1]), ldp(a, T.p[2]), ldp(a, T.p[3]), T.rest_volume, T.compliance,
                              a, lambda, lam, r);
    if (on || a.first) a.lam_t[t] = lam;
    if (!on) return;  // the records keep their previous values
    const RecOut out{a.corr_t, a.map_t + 4 * (size_t)t};
#pragma unroll
    for (int k = 0; k < 4; ++k) out[k] = r[k];
}

// Per constrained particle, in particle-index order: its incident records, stored contiguously in incidence
// order, summed in that order, then added to its position.
__global__ __launch_bounds__(kSoftBlock) void k_apply_corrections(SoftArgs a, const uint32_t *__restrict__ start,
                                                              const CorrRec *__restrict__ rec)
{
    const uint32_t j = xcd_tile(blockIdx.x, gridDim.x) * kSoftBlock + threadIdx.x;
    if (j >= a.nsoft) return;
    const uint32_t pid = a.soft_ids[j];
    const uint32_t k0 = start[pid], k1 = start[pid + 1];
    if (k0 == k1 || !live(a, pid)) return;
    float4 p = a.posi[pid];
    if (p.w <= kEps) return;
    float tx = 0.0f, ty = 0.0f, tz = 0.0f;
    for (uint32_t k = k0; k < k1; k += 4) {
        CorrRec cr[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) cr[u] = rec[min(k + u, k1 - 1)];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u)
            if (k + u < k1) {
                tx = tx + cr[u].x;
                ty = ty + cr[u].y;
                tz = tz + cr[u].z;
            }
    }
    p.x = p.x + tx;
    p.y = p.y + ty;
    p.z = p.z + tz;
    a.posi[pid] = p;
}

// The soft phase works on the constrained particles in particle-index order, where the
// constraints' vertices are neighbors in memory: gathered from slot order before it, put back after.
__global__ __launch_bounds__(kSoftBlock) void k_soft_gather(SoftArgs a)
{
    const uint32_t j = xcd_tile(blockIdx.x, gridDim.x) * kSoftBlock + threadIdx.x;
    if (j >= a.nsoft) return;
    const uint32_t pid = a.soft_ids[j];
    if (!live(a, pid)) return;  // a scene left out of the step may not be in the slots stepped
    a.posi[pid] = a.pos[a.slot_of[pid]];
}

__global__ __launch_bounds__(kSoftBlock) void k_soft_scatter(SoftArgs a)
{
    const uint32_t j = xcd_tile(blockIdx.x, gridDim.x) * kSoftBlock + threadIdx.x;
    if (j >= a.nsoft) return;
    const uint32_t pid = a.soft_ids[j];
    if (!live(a, pid)) return;
    const uint32_t steps = a.tiles ? a.solved * __popc(a.scenes[a.pid_scene[pid]].soft_stages) : 0u;
    a.pos[a.slot_of[pid]] = a.posi[(steps & 1u ? (size_t)a.n : 0) + pid];
}

// The launch of a group's tiles.
template <int G>
static void launch_tile(const SoftArgs &a, const RigidPidArgs &ra, const SubstepConsts &c, bool rigid, hipStream_t st)
{
    if (!a.ntiles[G]) return;
    hipLaunchKernelGGL((rigid ? k_soft_tile<G, true> : k_soft_tile<G, false>), dim3(a.ntiles[G]), dim3(kTileThreads),
                       a.lds[G], st, a, ra, c);
}

// rigid: with the iteration's particle-rigid contacts in particle-index order, after the last group.
void launch_soft_iteration(SoftArgs &a, const SceneBuffers &s, const SubstepConsts &c, bool rigid, bool gather, bool scatter,
                           bool solve, hipStream_t st)
{
    // physics_solver.cpp:915-1019: edges solve/apply, bends + dihedrals solve/apply, tets solve/apply
    if (gather) a.solved = 0;
    if (a.nsoft && gather) hipLaunchKernelGGL(k_soft_gather, dim3(grid_n(a.nsoft)), dim3(kSoftBlock), 0, st, a);
    const uint32_t g = grid_n(a.nsoft);
    if (solve && a.tiles) {
        const RigidPidArgs ra = rigid_pid_args(s, 0);
        launch_tile<0>(a, ra, c, rigid, st);
        launch_tile<1>(a, ra, c, rigid, st);
        launch_tile<2>(a, ra, c, rigid, st);
        ++a.solved;
        for (int k = 0; k < 3; ++k) std::swap(a.lam_in[k], a.lam_out[k]);
    } else if (solve) {
        // the applies run over the constrained particles; a group without constraints has nothing to apply
        if (a.ne) {
            hipLaunchKernelGGL(k_solve_edges, dim3(grid_n(a.ne)), dim3(kSoftBlock), 0, st, a);
            hipLaunchKernelGGL(k_apply_corrections, dim3(g), dim3(kSoftBlock), 0, st, a, a.inc_e_start, a.corr_e);
        }
        if (a.nb) hipLaunchKernelGGL(k_solve_bends, dim3(grid_n(a.nb)), dim3(kSoftBlock), 0, st, a);
        if (a.nd) hipLaunchKernelGGL(k_solve_dihedrals, dim3(grid_n(a.nd)), dim3(kSoftBlock), 0, st, a);
        if (a.nb + a.nd)
            hipLaunchKernelGGL(k_apply_corrections, dim3(g), dim3(kSoftBlock), 0, st, a, a.inc_b_start, a.corr_b);
        if (a.nt) {
            hipLaunchKernelGGL(k_solve_tets, dim3(grid_n(a.nt)), dim3(kSoftBlock), 0, st, a);
            hipLaunchKernelGGL(k_apply_corrections, dim3(g), dim3(kSoftBlock), 0, st, a, a.inc_t_start, a.corr_t);
        }
    }
    if (rigid && !(solve && a.tiles)) launch_rigid_pid(s, c, a.tiles ? a.solved : 0u, st);
    if (a.nsoft && scatter) hipLaunchKernelGGL(k_soft_scatter, dim3(g), dim3(kSoftBlock), 0, st, a);
}

}  // namespace cn
