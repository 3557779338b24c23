// cn_fluid.hip -- PBF fluid iterations on gfx950: the density-constraint pass and the
// delta + apply + clamp pass, both tiled over aligned 4x4x4-cell Morton blocks whose 6x6x6-cell
// halo is staged in LDS, and the exact neighbor-list pass of the per-pass entry.
//
// Reference passes (assets/shaders/physics/fluid/solver/): physics_fluid_build_neighbors.cs.hlsl
// :21-147, physics_fluid_compute_density_lambda.cs.hlsl:26-115,
// physics_fluid_compute_delta_positions.cs.hlsl:27-157, physics_fluid_apply_delta_positions.cs.hlsl
// :11-31, physics_fluid_clamp_boundary.cs.hlsl:23-80.  Every iteration the reference builds each
// fluid particle's neighbor list -- the fluid particles within h of its current position x* + delta,
// found by walking the 27 cells around its broadphase cell in dz, dy, dx order, each cell's
// particles in ascending slot, keeping the first max_fluid_neighbors -- and its density and delta
// passes iterate that list.
//
// Here a workgroup takes one aligned 4x4x4-cell block and stages its 6x6x6-cell halo in LDS, laid
// out cell by cell with x fastest, so the three dx cells of one (dz, dy) row are one contiguous LDS
// range and the 27-cell walk is nine range loops.  The density pass walks them with a loop body
// that only tests and compacts: the list it writes holds 16-bit halo offsets, not slots.  The sums
// then run over the compacted list, where every lane of a wave has work, and so does the delta
// pass, which stages the density records of the same halo and reads the list in the same offsets.
// The in-radius test sqrt(d2) < h is evaluated as d2 < T(h), T being the smallest float whose
// correctly rounded square root is >= h (the rounded square root is monotone), so the root is taken
// for listed neighbors only.  Blocks that cannot be staged (impure cells, a halo over the LDS
// capacity) and hash-key scenes walk the run table and sum in the walk.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "cn_internal.h"
#include "cn_walk.h"

namespace cn {

// Record position of particles that no neighbor walk may list (non-fluid or zero inverse mass):
// every squared distance to it is +inf, which fails d2 < T.
constexpr float kFarAway = __builtin_huge_valf();

struct FluidArgs {
    const float4 *pos;        // x* (slot order)
    const uint32_t *cls;
    const int4 *cellc;
    const uint32_t *bnd;
    const uint16_t *bndl;
    const float4 *din;        // accumulated delta of the previous iteration
    float4 *dout;
    float4 *cur;              // (x* + delta, D) at the start of the iteration (kNoMass: no neighbor)
    float4 *cs;               // density-pass records: (x* + delta, C)
    float4 *nc;               // surface normal * tension, C
    uint32_t *nbr;
    uint32_t *nbr_cnt;
    uint16_t *list;           // listed neighbors as halo offsets in slot groups (list_words)
    uint32_t *lcnt;           // what the delta pass walks (list_word)
    uint16_t *slist;          // iteration-0 candidates as halo offsets in slot groups, LDS blocks
    uint32_t *scnt;           // the same for the candidate list
    const uint32_t *run_key;
    const uint32_t *run_start;
    const int4 *run_info;
    int4 *run_info_out;
    const uint32_t *run_count;
    const uint32_t *bucket;
    uint32_t bucket_shift;
    const uint32_t *blk_first_run;
    const uint32_t *nblk;
    uint32_t *blk_halo;
    uint32_t *wide_blk;
    uint32_t *iter_state;
    const ParticleClass *classes;
    const cn_fluid_material *fm;
    const FluidConst *fc;     // per fluid material: what follows from its radius
    const Collider *col;
    const SceneInfo *scenes;
    const uint32_t *active;   // per scene: stepped this cn_step
    uint32_t *meta;
    uint32_t it;
    uint32_t tile;            // halo particles this launch can stage in LDS
    uint32_t wide_only;       // the delta pass takes the listed wide blocks only
};

__device__ __forceinline__ RunTable run_table(const FluidArgs &a)
{
    return RunTable{a.run_key, a.run_start, a.run_info, a.bucket, a.bucket_shift, a.cellc};
}

// ShouldProcessFluidNeighbor, physics_fluid_neighbor_build.hlsli:48-70 (the index test is the caller's)
__device__ __forceinline__ bool neighbor_ok(const ParticleClass &self, const ParticleClass &o)
{
    return o.kind == CN_PARTICLE_KIND_FLUID && o.env == self.env && (self.mask & o.layer) != 0u &&
           (o.mask & self.layer) != 0u;
}

__device__ __forceinline__ uint32_t wave_max(uint32_t v)
{
    for (int off = 32; off > 0; off >>= 1) {
        const uint32_t o = __shfl_xor(v, off);
        v = o > v ? o : v;
    }
    return v;
}
__device__ __forceinline__ uint32_t wave_sum(uint32_t v)
{
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// ---------------------------------------------------------------------------------------------
// candidate walks, in the reference's order: f(k) per candidate until f returns false
// ---------------------------------------------------------------------------------------------

// The same walk over a staged halo (hc = the particle's halo cell): nine LDS ranges.
template <class F>
__device__ __forceinline__ void walk_rows(const uint32_t *hoff, int hc, F &&f)
{
    for (int dz = -1; dz <= 1; ++dz)
        for (int dy = -1; dy <= 1; ++dy) {
            const int h0 = hc - 1 + 6 * dy + 36 * dz;
            const uint32_t f1 = hoff[h0 + 3];
            for (uint32_t k = hoff[h0]; k < f1; ++k)
                if (!f(k)) return;
        }
}

// Block queue: the blocks are split into kXcds contiguous chunks, one per die, so neighboring
// blocks (which share halo cells) run under the same L2; a workgroup drains its die's chunk, then
// helps the others.  Each workgroup's first block is its rank among its die's workgroups, without a
// counter; the counters hand out what is left, and none is touched when a chunk has no more blocks
// than workgroups with a fixed first one.  (A counter's atomic is a round trip to the memory side of
// about a microsecond: taking the first block and finding eight drained chunks by atomics cost a
// launch over the 64,000-particle dam break some 10 us of its 40.)  Run by one thread, when the block
// before is done: a block taken while the one before was still worked on waited for it where the others
// had none left (4,096 particles spread among 262 colliders, 6.6 ms a step against 4.3; a random fill of
// 1,048,573, 5.86 against 5.69).
// Workgroups of a die with a fixed first block: those of the density pass that are resident in a large
// scene.  (64, what the delta pass keeps resident, left a third of the density pass's without work: a step
// of 4,194,304 particles 17.3 ms against 16.3, of 1,048,573 5.6 against 5.7.)
constexpr uint32_t kFixedPerDie = 96;
struct BlockQueue {
    uint32_t die, open;  // open: bit d set while chunk d may have blocks
    bool helping;
    __device__ explicit BlockQueue(uint32_t wg) : die(wg % kXcds), open((1u << kXcds) - 1u), helping(false) {}
    __device__ static uint32_t begin(uint32_t nblk, uint32_t d) { return (uint32_t)(((uint64_t)nblk * d) / kXcds); }
    __device__ static uint32_t fixed(uint32_t d) { return min((gridDim.x - d + kXcds - 1u) / kXcds, kFixedPerDie); }
    // the fixed first block of workgroup wg, or kInvalid (the same for every thread)
    __device__ static uint32_t first(uint32_t wg, uint32_t nblk)
    {
        const uint32_t d = wg % kXcds, r = wg / kXcds, b0 = begin(nblk, d);
        return r < kFixedPerDie && r < begin(nblk, d + 1) - b0 ? b0 + r : kInvalid;
    }
    __device__ uint32_t next(uint32_t *q, uint32_t nblk)
    {
        while (open) {
            if (open & (1u << die)) {
                const uint32_t b0 = begin(nblk, die), cnt = begin(nblk, die + 1) - b0, fx = fixed(die);
                if (cnt > fx) {
                    const uint32_t t = fx + atomicAdd(q + die * kQueueStride, 1u);
                    if (t < cnt) return b0 + t;
                }
                open &= ~(1u << die);
                if (!helping) {
                    // its own chunk is drained: one look at all counters tells which others are not
                    helping = true;
#pragma unroll
                    for (uint32_t d = 0; d < kXcds; ++d) {
                        const uint32_t c = begin(nblk, d + 1) - begin(nblk, d), f = fixed(d);
                        if (c <= f || f + __hip_atomic_load(q + d * kQueueStride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= c)
                            open &= ~(1u << d);
                    }
                }
            }
            die = (die + 1) % kXcds;
        }
        return kInvalid;
    }
};

struct MetaAcc {
    uint32_t req = 0, trunc = 0, listed = 0, lds = 0, runs = 0, reuse = 0;
};

__device__ __forceinline__ void flush_meta(const MetaAcc &ma, const FluidArgs &a)
{
    const uint32_t wmax = wave_max(ma.req);
    const uint32_t wtr = wave_sum(ma.trunc);
    const uint32_t wls = wave_sum(ma.listed);
    const uint32_t wru = wave_sum(ma.reuse);
    if ((threadIdx.x & 63u) == 0) {
        if (wmax) atomicMax(&a.meta[0], wmax);
        if (wtr) atomicAdd(&a.meta[1], wtr);
        if (wru) atomicAdd(&a.meta[9], wru);
        if (a.it == 0 && wls) atomicAdd((unsigned long long *)&a.meta[2], (unsigned long long)wls);
    }
    if (threadIdx.x == 0) {
        if (ma.lds) atomicAdd(&a.meta[5], ma.lds);
        if (ma.runs) atomicAdd(&a.meta[6], ma.runs);
    }
}

// The persistent tiled passes gather one block's counters at a time into workgroup totals in LDS
// (so no per-lane accumulator lives across blocks) and flush those once at the end.
constexpr uint32_t kWgMetaWords = 6;  // largest request, truncations, listed, reuses, LDS blocks, run blocks

__device__ __forceinline__ void meta_to_wg(const MetaAcc &ma, uint32_t *s_meta)
{
    const uint32_t wmax = wave_max(ma.req);
    const uint32_t wtr = wave_sum(ma.trunc);
    const uint32_t wls = wave_sum(ma.listed);
    const uint32_t wru = wave_sum(ma.reuse);
    if ((threadIdx.x & 63u) == 0) {
        if (wmax) atomicMax(&s_meta[0], wmax);
        if (wtr) atomicAdd(&s_meta[1], wtr);
        if (wls) atomicAdd(&s_meta[2], wls);
        if (wru) atomicAdd(&s_meta[3], wru);
    }
    if (threadIdx.x == 0) {
        s_meta[4] += ma.lds;
        s_meta[5] += ma.runs;
    }
}

__device__ __forceinline__ void flush_wg_meta(const uint32_t *s_meta, const FluidArgs &a)
{
    if (threadIdx.x != 0) return;
    if (s_meta[0]) atomicMax(&a.meta[0], s_meta[0]);
    if (s_meta[1]) atomicAdd(&a.meta[1], s_meta[1]);
    if (s_meta[3]) atomicAdd(&a.meta[9], s_meta[3]);
    if (a.it == 0 && s_meta[2]) atomicAdd((unsigned long long *)&a.meta[2], (unsigned long long)s_meta[2]);
    if (s_meta[4]) atomicAdd(&a.meta[5], s_meta[4]);
    if (s_meta[5]) atomicAdd(&a.meta[6], s_meta[5]);
}

// ---------------------------------------------------------------------------------------------
// density pass: physics_fluid_build_neighbors.cs.hlsl:88-131 (the list filter) with
// physics_fluid_compute_density_lambda.cs.hlsl:26-115 (density, surface normal, constraint)
// ---------------------------------------------------------------------------------------------
struct DensitySum {
    float density = 0.0f, snx = 0.0f, sny = 0.0f, snz = 0.0f;
    uint32_t inr = 0, req = 0;
};

// Quotients of one neighbor pair, held negated where that saves the final negation of
// fdiv_rcp_neg: nn = -(dx, dy, dz) / dist, nq = -(dist / h), omq = 1 - dist / h (as 1 + nq) and the spiky
// derivative der = (-2 k (1 - q)) / h (FluidSpikyKernelDerivative, physics_fluid_common.hlsli:31-42;
// 0 unless eps < dist < h), computed as -((2 k omq) / h).  The consumers take -(a b) = (-a) b and
// x - (-y) = x + y, which are exact, so every result has the bits of the plain forms.  FAST divides
// through reciprocals (fdiv_rcp_neg: 1 / dist once per pair, 1 / h once per particle); quot_fast_ok
// says when that is exact, and the other particles take the IEEE divisions.
struct PairQuot {
    float nnx, nny, nnz, nq, omq, der;  // nq = -(dist / h)
};

// fdiv_rcp_neg is exact for every quotient of pair_quot when h <= 1024 and each coordinate of the
// particle has magnitude >= 2^-62: a nonzero coordinate difference is then >= 2^-86 (both values
// are multiples of 2^-86, or the difference exceeds half the larger one), the live distances lie
// in (eps, h), and with h in [1e-4, 1024] the spiky numerator 2 k (1 - q) lies in
// [2^-51, 2^43] (k = 15 / (pi h^3), 1 - q >= 2^-24 when nonzero), so every dividend is 0 or
// >= 2^-96 and every quotient lies in [2^-100, 2^100).
__device__ __forceinline__ bool quot_fast_ok(float h, float sx, float sy, float sz)
{
    return h <= 1024.0f && fminf(fminf(fabsf(sx), fabsf(sy)), fabsf(sz)) >= 0x1p-62f;
}

// LIVE: the caller adds the pair's terms only for eps < dist < h (a listed neighbor that is not
// coincident), so the zero the derivative takes outside that range is never read.
// y = 1 / dist, correctly rounded (FAST); k2 = 2 k.
template <bool FAST, bool LIVE = false>
__device__ __forceinline__ void pair_quot_y(PairQuot &p, float dx, float dy, float dz, float dist, float h, float ih,
                                            float k2, float y)
{
    float &nq = p.nq;
    if (FAST) {
        p.nnx = fdiv_rcp_neg(dx, dist, y);
        p.nny = fdiv_rcp_neg(dy, dist, y);
        p.nnz = fdiv_rcp_neg(dz, dist, y);
        nq = fdiv_rcp_neg(dist, h, ih);
    } else {
        p.nnx = fdiv(-dx, dist);
        p.nny = fdiv(-dy, dist);
        p.nnz = fdiv(-dz, dist);
        nq = -fdiv(dist, h);
    }
    p.omq = __fadd_rn(1.0f, nq);
    const float num = __fmul_rn(k2, p.omq);
    const float der = FAST ? fdiv_rcp_neg(num, h, ih) : -fdiv(num, h);
    p.der = LIVE ? der : ((dist <= kEps || dist >= h) ? 0.0f : der);
}

// y0: the estimate of 1 / dist that its square root gave (fsqrt_rsq)
template <bool FAST, bool LIVE = false>
__device__ __forceinline__ void pair_quot(PairQuot &p, float dx, float dy, float dz, float dist, float h, float ih,
                                          float k, float y0)
{
    pair_quot_y<FAST, LIVE>(p, dx, dy, dz, dist, h, ih, __fmul_rn(2.0f, k), FAST ? frcp_exact(dist, y0) : 0.0f);
}

struct DensitySelf {
    ParticleClass pc;
    float4 s;
    float h, t2, kw, ih;  // ih = 1 / h
    bool tension;
    bool fd;          // the neighbor quotients may use fdiv_rcp_neg (pair_quot)
};

// Returns false (and writes the unreachable record) for particles that take no part in the solve.
__device__ __forceinline__ bool density_begin(DensitySelf &x, uint32_t i, const float4 s, uint32_t ic,
                                              const FluidArgs &a)
{
    x.pc = a.classes[ic];
    x.s = s;
    if (x.pc.kind != CN_PARTICLE_KIND_FLUID || s.w < 0.0f) {
        a.cs[i] = make_float4(kFarAway, kFarAway, kFarAway, 0.0f);
        return false;
    }
    const FluidConst fc = a.fc[x.pc.fluid_mat];
    x.h = fc.h;
    x.t2 = fc.t2;
    x.kw = fc.kw;
    x.ih = fc.ih;
    x.fd = quot_fast_ok(x.h, s.x, s.y, s.z);
    x.tension = fmaxd(a.fm[x.pc.fluid_mat].surface_tension, 0.0f) > kEps;
    return true;
}

__device__ __forceinline__ bool density_walks(const DensitySelf &x, bool uniform, const SubstepConsts &c)
{
    return c.cap > 0 && (!uniform || neighbor_ok(x.pc, x.pc));
}

// The list filter: candidate pj (class qcls) is a neighbor.
template <bool UNIFORM>
__device__ __forceinline__ bool density_test(const DensitySelf &x, const float4 pj, uint32_t qcls, const FluidArgs &a)
{
    if (!UNIFORM && !neighbor_ok(x.pc, a.classes[qcls])) return false;
    if (pj.w < 0.0f) return false;
    const float dx = x.s.x - pj.x, dy = x.s.y - pj.y, dz = x.s.z - pj.z;
    return dot3(dx, dy, dz, dx, dy, dz) < x.t2;
}

// Density and (negated) surface-normal terms of one listed neighbor, and its squared distance.
struct DensityTerm {
    float w, ngx, ngy, ngz, d2;
};

// TENSION = false: the particle's material has no surface tension (x.tension false), so the normal
// terms are left out at compile time.  FAST: quotients through reciprocals (x.fd holds).
template <bool TENSION, bool FAST>
__device__ __forceinline__ DensityTerm density_term(const DensitySelf &x, const float4 pj)
{
    DensityTerm t;
    const float dx = x.s.x - pj.x, dy = x.s.y - pj.y, dz = x.s.z - pj.z;
    t.d2 = dot3(dx, dy, dz, dx, dy, dz);
    float y0;
    const float dist = fsqrt_nearzero_free(t.d2, y0);
    const float omq = FAST ? __fadd_rn(1.0f, fdiv_rcp_neg(dist, x.h, x.ih)) : __fsub_rn(1.0f, fdiv(dist, x.h));
    // every term the callers add is a neighbor's (dist < h): the kernel's range test is left out
    t.w = spiky_w_om_in(omq, x.kw);
    t.ngx = t.ngy = t.ngz = 0.0f;
    if (TENSION && x.tension && !(dist <= kEps || dist >= x.h)) {
        // FluidSpikyKernelGradient, physics_fluid_common.hlsli:44-53, negated: der * -(d / dist)
        PairQuot p;
        pair_quot<FAST>(p, dx, dy, dz, dist, x.h, x.ih, x.kw, y0);
        t.ngx = p.der * p.nnx;
        t.ngy = p.der * p.nny;
        t.ngz = p.der * p.nnz;
    }
    return t;
}

template <bool TENSION = true>
__device__ __forceinline__ void density_add(DensitySum &d, const DensitySelf &x, const DensityTerm &t)
{
    d.density = d.density + t.w;
    if (TENSION && x.tension) {
        d.snx = d.snx - t.ngx;
        d.sny = d.sny - t.ngy;
        d.snz = d.snz - t.ngz;
    }
}

// Calls f(collider) for every candidate collider of a slot in visit order; col0 is the first collider of
// the lane's scene, and a wave may hold particles of several (the launches of a thread per slot).
// Candidates held as a bitmask are taken collider by collider over the wave's particles of a scene, so
// each is read once through the scalar cache (the tables are constant during a launch); candidates held
// as a list, which differ from lane to lane, lane by lane.  A step of 64,000 fluid particles among 24 pegs
// takes 2.5 ms (masks lane by lane: 3.9), among 768 pegs 4.7 ms (lists taken collider by collider over the
// wave, each pass for the lanes whose next one it is: 19.4).
__device__ __forceinline__ Collider const_collider(const Collider *col)
{
    typedef const __attribute__((address_space(4))) uint32_t *ConstWords;
    const ConstWords w = (ConstWords)(uintptr_t)col;
    union {
        uint32_t u[sizeof(Collider) / 4];
        Collider c;
    } v;
#pragma unroll
    for (uint32_t k = 0; k < sizeof(Collider) / 4; ++k) v.u[k] = w[k];
    return v.c;
}
template <class F>
__device__ __forceinline__ void each_collider(uint32_t word, const FluidArgs &a, uint32_t i, uint32_t col0, F &&f)
{
    const bool listed = (word & kBndList) != 0u;
    uint32_t mask = listed ? 0u : word;
    for (uint64_t left = __ballot(mask != 0u); left; left = __ballot(mask != 0u)) {
        // the first scene that has some: the candidates of any of its lanes, then each for the lanes it is one of
        const uint32_t c0 = (uint32_t)__builtin_amdgcn_readlane((int)col0, (int)__builtin_ctzll(left));
        const uint32_t mine = col0 == c0 ? mask : 0u;
        uint32_t all = 0;
        for (uint64_t more = __ballot(mine != 0u); more; more = __ballot((mine & ~all) != 0u))
            all |= (uint32_t)__builtin_amdgcn_readlane((int)mine, (int)__builtin_ctzll(more));
        for (; all; all &= all - 1u) {
            const uint32_t k = (uint32_t)__builtin_ctz(all);
            const Collider cc = const_collider(a.col + c0 + k);
            if ((mine >> k) & 1u) f(cc);
        }
        mask &= ~mine;
    }
    if (listed) {
        const uint16_t *l = a.bndl + (size_t)i * kBndListCap;
        const uint32_t n = min(word & 0xffu, kBndListCap);
        for (uint32_t q = 0; q < n; ++q) {
            const Collider cc = a.col[col0 + l[q]];  // whole, so that its loads go out together
            f(cc);
        }
    }
}

// Boundary ghost density (physics_fluid_boundary_common.hlsli:112-138), the constraint and the record.
__device__ __forceinline__ void density_end(uint32_t i, uint32_t bw, const DensitySum &d, const DensitySelf &x,
                                            MetaAcc &ma, const FluidArgs &a, const SubstepConsts &c)
{
    float density = d.density;
    const float bscale = c.cfg[kCfgFluidBndDensity];
    const uint32_t col0 = a.scenes[x.pc.scene].col0;
    each_collider(bw, a, i, col0, [&](const Collider &cc) {
        float gx, gy, gz;
        if (!ghost_delta(cc, x.s.x, x.s.y, x.s.z, x.h, gx, gy, gz)) return;
        float ux, uy, uz;
        const float gd = len3_dir(gx, gy, gz, ux, uy, uz);
        if (gd >= x.h) return;
        density = density + spiky_w_k(gd, x.h, x.kw) * bscale;
    });
    // the material is read again here rather than held in registers across the walk
    const cn_fluid_material &m = a.fm[x.pc.fluid_mat];
    const float rho0 = fmaxd(m.rest_density, 1.0f);
    const float C =
        fmaxd(density - rho0, -rho0 * fmaxd(c.cfg[kCfgFluidMaxUnder], 0.0f)) * m.density_constraint_scale;
    a.cs[i] = make_float4(x.s.x, x.s.y, x.s.z, C);
    if (x.tension) {
        const float st = fmaxd(m.surface_tension, 0.0f);
        a.nc[i] = make_float4(d.snx * st, d.sny * st, d.snz * st, C);
    }
    ma.req = max(ma.req, d.req);
    ma.trunc += d.req > c.cap ? 1u : 0u;
    ma.listed += d.inr;
}

// Run-table walk with the sums taken in the walk.
// UNIFORM: every particle the walk meets has class ucls.
template <bool UNIFORM>
__device__ __forceinline__ void density_global(uint32_t i, MetaAcc &ma, const FluidArgs &a, const SubstepConsts &c,
                                               uint32_t ucls = 0u)
{
    if (!a.active[a.classes[UNIFORM ? ucls : a.cls[i]].scene]) return;
    DensitySelf x;
    if (!density_begin(x, i, a.cur[i], UNIFORM ? ucls : a.cls[i], a)) return;
    DensitySum d;
    if (density_walks(x, UNIFORM, c))
        walk_runs(a.cellc[i], run_table(a), c, [&](uint32_t q) {
            if (q == i) return true;
            const float4 pj = a.cur[q];
            if (!density_test<UNIFORM>(x, pj, UNIFORM ? 0u : a.cls[q], a)) return true;
            ++d.req;
            if (d.inr < c.cap) {
                ++d.inr;
                density_add(d, x, density_term<true, false>(x, pj));
            }
            return true;
        });
    density_end(i, a.bnd[i], d, x, ma, a, c);
}

// ---------------------------------------------------------------------------------------------
// delta pass: physics_fluid_compute_delta_positions.cs.hlsl:27-157, then
// physics_fluid_apply_delta_positions.cs.hlsl:11-31 and physics_fluid_clamp_boundary.cs.hlsl:23-80
// on the same particle.
// ---------------------------------------------------------------------------------------------
// relDelta = delta_i - delta_j is zero on the first iteration, and the CFL term can only act when
// |relDelta| >= cfl, i.e. never while 2 max|delta| < cfl (max|delta| of the previous iteration).
__device__ __forceinline__ bool cfl_term_on(const cn_fluid_material &m, const FluidArgs &a, const SubstepConsts &c)
{
    const float cfl = fmaxd(m.cfl_radius, 0.0f);
    if (!(a.it > 0 && cfl > kEps)) return false;
    const float md2 = a.it - 1 < kIterStateWords ? __uint_as_float(a.iter_state[kStateMaxDisp + a.it - 1]) : 3.4e38f;
    return !(4.0f * md2 * c.cfl_guard < cfl * cfl);
}
__device__ __forceinline__ bool visc_term_on(const cn_fluid_material &m, const FluidArgs &a, const SubstepConsts &c)
{
    return a.it > 0 && c.dt * fmaxd(m.viscosity, 0.0f) > kEps;
}

struct DeltaSelf {
    ParticleClass pc;
    float4 di, nci;
    float sx, sy, sz, Ci, h, t2, kw, ih, cohesion, viscosity, cfl, dt;
    bool tension, visc_on, cfl_on, need_rel, fd;
    bool plain;  // no cohesion, viscosity, CFL or tension term: the pressure term alone (delta_plain)
};

struct DeltaTerm {
    float x, y, z;
    bool live;  // a neighbor (dist < h) that is not coincident (dist > eps): it adds a term and a weight
};

// One listed neighbor's term (physics_fluid_compute_delta_positions.cs.hlsl:60-140).
template <bool UNIFORM>
__device__ __forceinline__ DeltaTerm delta_term(const DeltaSelf &x, const float4 cq, const float4 dq, const float4 ncq,
                                                uint32_t qcls, const FluidArgs &a)
{
    DeltaTerm t;
    const float ddx = x.sx - cq.x, ddy = x.sy - cq.y, ddz = x.sz - cq.z;
    const float d2 = dot3(ddx, ddy, ddz, ddx, ddy, ddz);
    float y0;
    const float dist = fsqrt_rsq(d2, y0);
    t.live = d2 < x.t2 && dist > kEps;
    PairQuot p;
    // a listed neighbor (dist < h) whose term counts only when live (dist > eps)
    pair_quot<true, true>(p, ddx, ddy, ddz, dist, x.h, x.ih, x.kw, y0);
    if (!x.fd) pair_quot<false, true>(p, ddx, ddy, ddz, dist, x.h, x.ih, x.kw, y0);
    // sc * n with sc = -0.5 (Ci + Cj) der, as (0.5 (Ci + Cj) der) * -n
    const float msc = 0.5f * (x.Ci + cq.w) * p.der;
    float pdx = msc * p.nnx, pdy = msc * p.nny, pdz = msc * p.nnz;
    const bool same = UNIFORM || x.pc.fluid_mat == a.classes[qcls].fluid_mat;
    if (same) {
        float rx = 0.0f, ry = 0.0f, rz = 0.0f;
        if (x.need_rel) {
            rx = x.di.x - dq.x;
            ry = x.di.y - dq.y;
            rz = x.di.z - dq.z;
        }
        if (x.cohesion > kEps) {
            // the cohesion coefficients are read here (a rare path) rather than held across the loop
            const cn_fluid_material &m = a.fm[x.pc.fluid_mat];
            const float ck = x.cohesion * cohesion_q(dist, x.h, -p.nq, m.cohesion1, m.cohesion2);
            pdx = pdx + p.nnx * ck;
            pdy = pdy + p.nny * ck;
            pdz = pdz + p.nnz * ck;
        }
        if (x.visc_on) {
            const float vs = 1.0f - frcp_exact_ge1(1.0f + x.viscosity * spiky_w_om_in(p.omq, x.kw));
            pdx = pdx - vs * rx;
            pdy = pdy - vs * ry;
            pdz = pdz - vs * rz;
        }
        if (x.cfl_on) {
            // proj = r . n = -(r . nn); proj < -cfl, pcf = proj + cfl = cfl - (r . nn)
            const float nproj = dot3(rx, ry, rz, p.nnx, p.nny, p.nnz);
            if (nproj > x.cfl) {
                const float pcf = x.cfl - nproj;
                pdx = pdx + p.nnx * pcf * 0.5f;
                pdy = pdy + p.nny * pcf * 0.5f;
                pdz = pdz + p.nnz * pcf * 0.5f;
            }
        }
        if (x.tension) {
            pdx = pdx - x.dt * (x.nci.x - ncq.x);
            pdy = pdy - x.dt * (x.nci.y - ncq.y);
            pdz = pdz - x.dt * (x.nci.z - ncq.z);
        }
    }
    t.x = pdx;
    t.y = pdy;
    t.z = pdz;
    return t;
}

struct DeltaSum {
    float x = 0.0f, y = 0.0f, z = 0.0f, w = 0.0f;
};

__device__ __forceinline__ void delta_add(DeltaSum &d, const DeltaTerm &t)
{
    if (!t.live) return;
    d.x = d.x + t.x;
    d.y = d.y + t.y;
    d.z = d.z + t.z;
    d.w = d.w + 1.0f;
}

// A particle's own inputs of the delta pass, loaded together at the top of its loop iteration so
// their round trips to memory overlap (rather than one after another as the code reaches them).
struct DeltaPre {
    float4 p, di;
    uint32_t cls, bnd;
};

template <bool UNIFORM>
__device__ __forceinline__ DeltaPre delta_pre(uint32_t i, const FluidArgs &a, uint32_t ucls = 0u)
{
    DeltaPre r;
    r.p = a.pos[i];
    r.di = a.it > 0 ? a.din[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    r.cls = UNIFORM ? ucls : a.cls[i];
    r.bnd = a.bnd[i];
    return r;
}

// sum(x, d) adds the neighbor terms in list order; own(nc) is the particle's record, or its surface
// normal's.  Returns (|delta| + slack)^2 of the particle.
template <bool UNIFORM, class Sum, class Own>
__device__ __forceinline__ float delta_particle(uint32_t i, const DeltaPre &pre, Sum &&sum, Own &&own,
                                                const FluidArgs &a, const SubstepConsts &c)
{
    const ParticleClass pc = a.classes[pre.cls];
    if (pc.kind != CN_PARTICLE_KIND_FLUID) {
        a.dout[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        return 0.0f;
    }
    const float4 p = pre.p;
    const float4 di = pre.di;
    float ox = 0.0f, oy = 0.0f, oz = 0.0f, ow = 0.0f;
    if (p.w > kEps) {
        DeltaSelf x;
        x.pc = pc;
        x.di = di;
        const float4 csi = own(false);
        x.sx = csi.x;
        x.sy = csi.y;
        x.sz = csi.z;
        x.Ci = csi.w;
        const cn_fluid_material &m = a.fm[pc.fluid_mat];
        const FluidConst fc = a.fc[pc.fluid_mat];
        x.h = fc.h;
        x.t2 = fc.t2;
        x.kw = fc.kw;
        x.ih = fc.ih;
        x.fd = quot_fast_ok(x.h, x.sx, x.sy, x.sz);
        x.dt = c.dt;
        x.cohesion = c.dt * fmaxd(m.cohesion, 0.0f);
        x.viscosity = c.dt * fmaxd(m.viscosity, 0.0f);
        x.cfl = fmaxd(m.cfl_radius, 0.0f);
        x.tension = fmaxd(m.surface_tension, 0.0f) > kEps;
        x.cfl_on = cfl_term_on(m, a, c);
        x.visc_on = visc_term_on(m, a, c);
        x.need_rel = x.cfl_on || x.visc_on;
        x.plain = !(x.need_rel || x.tension || x.cohesion > kEps);
        x.nci = x.tension ? own(true) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        DeltaSum d;
        if (c.cap > 0 && (!UNIFORM || neighbor_ok(pc, pc))) sum(x, d);
        // ComputeFluidBoundaryDeltaFromCandidates, physics_fluid_boundary_common.hlsli:140-167
        float bx = 0.0f, by = 0.0f, bz = 0.0f;
        const float scn = fmaxd(x.Ci, 0.0f);
        const uint32_t col0 = a.scenes[pc.scene].col0;
        each_collider(pre.bnd, a, i, col0, [&](const Collider &cc) {
            float gx, gy, gz;
            if (!ghost_delta(cc, x.sx, x.sy, x.sz, x.h, gx, gy, gz)) return;
            float ux, uy, uz;
            const float gd = len3_dir(gx, gy, gz, ux, uy, uz);
            if (gd <= kEps || gd >= x.h) return;
            const float f = -scn * spiky_dw_k(gd, x.h, x.kw);
            bx = bx + f * ux;
            by = by + f * uy;
            bz = bz + f * uz;
        });
        const float solve = c.cfg[kCfgFluidSolve], bdel = c.cfg[kCfgFluidBndDelta];
        ox = d.x * solve + bx * bdel;
        oy = d.y * solve + by * bdel;
        oz = d.z * solve + bz * bdel;
        ow = d.w;
    }
    // apply
    const float wgt = fmaxd(ow * c.cfg[kCfgFluidRelax], 1.0f);
    const float ax = di.x + fdiv(ox, wgt), ay = di.y + fdiv(oy, wgt), az = di.z + fdiv(oz, wgt);
    // clamp
    const float r = fmaxd(pc.radius, 0.0f);
    float cx = p.x + ax, cy = p.y + ay, cz = p.z + az;
    const uint32_t bw = pre.bnd;
    const uint32_t bcol0 = a.scenes[pc.scene].col0;
    for (int sweep = 0; sweep < 2; ++sweep) {
        bool changed = false;
        each_collider(bw, a, i, bcol0, [&](const Collider &cc) {
            float sd, nx, ny, nz;
            if (!collider_contact(cc, cx, cy, cz, sd, nx, ny, nz)) return;
            if (sd >= r) return;
            const float push = r - sd;
            cx = cx + nx * push;
            cy = cy + ny * push;
            cz = cz + nz * push;
            changed = true;
        });
        if (!changed) break;
    }
    const float ex = cx - p.x, ey = cy - p.y, ez = cz - p.z;
    // w: how far contacts have moved x* in the substep (k_contact_apply)
    const float moved = a.it > 0 ? di.w : 0.0f;
    a.dout[i] = make_float4(ex, ey, ez, moved);
    const float nx = p.x + ex, ny = p.y + ey, nz = p.z + ez;
    // |delta| plus a few ulps of the position: D, the bound on the displacement since iteration 0
    // that the candidate lists go by; it also bounds the next iteration's relDelta for the CFL skip
    const float slack = fmaxd(fmaxd(fabsf(nx), fabsf(ny)), fabsf(nz)) * 4.76837158e-7f + 1.0e-30f;
    const float dl = len3(ex, ey, ez) + slack;
    a.cur[i] = make_float4(nx, ny, nz, p.w > kEps ? dl + moved : kNoMass);
    return dl * dl;
}

// The terms over the run table: the list filter and the cap applied in the walk.
template <bool UNIFORM>
__device__ __forceinline__ void delta_walk(uint32_t i, const DeltaSelf &x, DeltaSum &d, const FluidArgs &a,
                                           const SubstepConsts &c)
{
    const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    uint32_t inr = 0;
    walk_runs(a.cellc[i], run_table(a), c, [&](uint32_t q) {
        if (q == i) return true;
        const uint32_t qc = UNIFORM ? 0u : a.cls[q];
        if (!UNIFORM && !neighbor_ok(x.pc, a.classes[qc])) return true;
        const float4 cq = a.cs[q];
        const float ddx = x.sx - cq.x, ddy = x.sy - cq.y, ddz = x.sz - cq.z;
        if (!(dot3(ddx, ddy, ddz, ddx, ddy, ddz) < x.t2)) return true;
        if (inr >= c.cap) return false;
        ++inr;
        delta_add(d, delta_term<UNIFORM>(x, cq, x.need_rel ? a.din[q] : zero, x.tension ? a.nc[q] : zero, qc, a));
        return true;
    });
}

template <bool UNIFORM>
__device__ __forceinline__ float delta_global(uint32_t i, const FluidArgs &a, const SubstepConsts &c)
{
    if (!a.active[a.classes[UNIFORM ? 0u : a.cls[i]].scene]) return 0.0f;
    return delta_particle<UNIFORM>(
        i, delta_pre<UNIFORM>(i, a), [&](const DeltaSelf &x, DeltaSum &d) { delta_walk<UNIFORM>(i, x, d, a, c); },
        [&](bool nc) { return nc ? a.nc[i] : a.cs[i]; }, a, c);
}

__device__ __forceinline__ void flush_disp(float d2, const FluidArgs &a)
{
    if (a.it >= kIterStateWords) return;
    const uint32_t wm = wave_max(__float_as_uint(d2));
    if ((threadIdx.x & 63u) == 0 && wm) {
        atomicMax(a.iter_state + kStateMaxDisp + a.it, wm);
        atomicMax(&a.meta[7], wm);
    }
}

// ---------------------------------------------------------------------------------------------
// per-block halo descriptors, once per substep
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_blk_halo(FluidArgs a, SubstepConsts c)
{
    __shared__ uint32_t scan[kBlock / 64];
    __shared__ uint32_t s_kinds, s_gmin, s_gmax;  // what the halo holds: kHas* bits, solid phase groups
    constexpr uint32_t kHasFluid = 1, kHasSolid = 2, kHasOther = 4;
    // blocks of scenes with fluid are a prefix; contact pairs can exist in any scene
    const uint32_t nb = min(a.nblk[c.pairs ? 0 : 1], c.blk_cap);
    const uint32_t tid = threadIdx.x;
    // some particle lies outside its scene's window: wrapped cells may share runs, so every run's
    // record is taken from its members, here and (for the later walks) in run_info
    const bool wrapped = a.run_count[1] != 0u;
    const uint32_t *rcls = c.pairs ? a.cls : nullptr;
    if (wrapped)
        for (uint32_t r = blockIdx.x * kBlock + tid; r < a.run_count[0]; r += gridDim.x * kBlock)
            a.run_info_out[r] = run_record(a.run_start[r], a.run_start[r + 1], a.cellc, rcls);
    for (uint32_t b = blockIdx.x; b < nb; b += gridDim.x) {
        const uint32_t p0 = a.run_start[a.blk_first_run[b]], p1 = a.run_start[a.blk_first_run[b + 1]];
        const uint32_t scene = a.classes[a.cls[p0]].scene;
        uint32_t *hd = a.blk_halo + (size_t)b * kHaloStride;
        const bool fluid = a.scenes[scene].has_fluid != 0u, pairs = a.scenes[scene].pairs != 0u;
        if (!fluid && !pairs) {  // no fluid pass visits the block and no contact pair exists in it
            if (tid == 0) {
                hd[kHdFlags] = kHdNoFluid;
                hd[kHdPairs] = 0u;
                hd[kHdP0] = p0;
                hd[kHdP1] = p1;
                hd[kHdScene] = scene;
            }
            continue;
        }
        if (tid == 0) {
            s_kinds = 0u;
            s_gmin = kInvalid;
            s_gmax = 0u;
        }
        __syncthreads();
        const int4 c0 = a.cellc[p0];
        const int bx = c0.x & ~3, by = c0.y & ~3, bz = c0.z & ~3;
        // particles of a wrapped Morton block that lie outside the aligned block, particles whose own
        // cell hashes to the empty-table marker (their cell has no halo range), or halo cells shared
        // with other cells leave the block to the run-table walk
        bool bad = false;
        for (uint32_t i = p0 + tid; i < p1; i += kBlock) {
            const int4 ci = a.cellc[i];
            bad |= (uint32_t)(ci.x - bx) > 3u || (uint32_t)(ci.y - by) > 3u || (uint32_t)(ci.z - bz) > 3u;
            bad |= cell_hash(ci.x, ci.y, ci.z) == kInvalid;
        }
        uint32_t cnt = 0, st = 0;
        if (tid < kHalo) {
            const int tx = bx - 1 + (int)(tid % 6u), ty = by - 1 + (int)((tid / 6u) % 6u), tz = bz - 1 + (int)(tid / 36u);
            if (cell_hash(tx, ty, tz) != kInvalid) {
                const int r = find_run(cell_key(tx, ty, tz, (uint32_t)c0.w, c.key_mode, c.morton_bits), run_table(a));
                if (r >= 0) {
                    const int4 info = wrapped ? run_record(a.run_start[r], a.run_start[r + 1], a.cellc, rcls) : a.run_info[r];
                    if (!(info.w & kRunPure)) bad = true;
                    else if (info.x == tx && info.y == ty && info.z == tz) {
                        st = a.run_start[r];
                        cnt = a.run_start[r + 1] - st;
                        if (pairs) {
                            // what the cell holds; a cell of several classes may hold anything, and
                            // so may a self-colliding group
                            const uint32_t k = run_class(info.w);
                            uint32_t has = kHasOther;
                            if (k != kInvalid) {
                                const ParticleClass pc = a.classes[k];
                                if (pc.kind == CN_PARTICLE_KIND_FLUID) {
                                    has = kHasFluid;
                                } else if (pc.kind == CN_PARTICLE_KIND_SOLID && !(pc.phase & kPhaseSelfCollide)) {
                                    has = kHasSolid;
                                    atomicMin(&s_gmin, pc.phase & kPhaseGroupMask);
                                    atomicMax(&s_gmax, pc.phase & kPhaseGroupMask);
                                }
                            }
                            atomicOr(&s_kinds, has);
                        }
                    }
                }
            }
        }
        const int any_bad = __syncthreads_or(bad ? 1 : 0);
        uint32_t total;
        const uint32_t off = block_exclusive_scan(cnt, scan, total);
        if (tid < kHalo) {
            hd[kHdStart + tid] = st;
            hd[kHdOff + tid] = off;
        }
        if (tid == 0) {
            // blocks the delta pass stages only in the wide tile get their own launch
            if (fluid && !any_bad && total > c.tile_delta && total <= c.tile_wide)
                a.wide_blk[atomicAdd(a.iter_state + kStateWideCount, 1u)] = b;
            hd[kHdOff + kHalo] = total;
            hd[kHdFlags] = any_bad ? 0u : 1u;
            hd[kHdFluidOnly] = a.scenes[scene].fluid_only;
            hd[kHdSuper] = 1u;  // the building density pass clears it where a candidate list overflows
            hd[kHdPairs] = (s_kinds & kHasOther) || (s_kinds & (kHasFluid | kHasSolid)) == (kHasFluid | kHasSolid) ||
                                   ((s_kinds & kHasSolid) && s_gmin != s_gmax)
                               ? 1u
                               : 0u;
            hd[kHdP0] = p0;
            hd[kHdP1] = p1;
            hd[kHdBase] = (uint32_t)bx;
            hd[kHdBase + 1] = (uint32_t)by;
            hd[kHdBase + 2] = (uint32_t)bz;
            hd[kHdScene] = scene;
        }
    }
}

constexpr int kTileBlock = 512;  // threads of a tiled fluid workgroup: one pass over a block's particles
// Waves per SIMD the tiled passes are compiled for.  The density pass fits 80 VGPRs with a few values
// spilled between blocks: three 8-wave workgroups per CU, each a third of its LDS.  The delta pass
// holds more across its term loops (its spills there cost three times the time: 1,320 us at six
// waves with the terms unrolled by four) and runs two workgroups with half the LDS each, which also
// stages larger halos.
constexpr int kDensityWaves = 6, kDeltaWaves = 4;
constexpr uint32_t kTilePad = 4;   // spare entries after each staged density array (walk loads past a range)

// Head of a tiled pass's block: decide LDS or run table, load the halo table (visible after the
// caller's barrier).  skip_to is a halo size above the LDS capacity up to which a block is left to
// the wide launch (0: none).  b is the same for the whole workgroup.
struct TileState {
    uint32_t blk;
    uint32_t p0, p1;
    bool lds, skip;
    bool fluid_only;  // the block's scene
    bool complete;    // every particle of the block has a complete candidate list
    int bx, by, bz;
};

__device__ __forceinline__ void tile_load(TileState &ts, uint32_t b, uint32_t *hoff, uint32_t *hstart,
                                          uint32_t skip_to, const FluidArgs &a, const SubstepConsts &c)
{
    const uint32_t tid = threadIdx.x;
    b = __builtin_amdgcn_readfirstlane(b);
    ts.blk = b;
    ts.lds = false;
    ts.skip = false;
    if (b < c.blk_cap) {
        const uint32_t *hd = a.blk_halo + (size_t)b * kHaloStride;
        // the tables are loaded beside the header, whatever it says
        for (uint32_t t = tid; t <= kHalo; t += blockDim.x) {
            hoff[t] = hd[kHdOff + t];
            if (t < kHalo) hstart[t] = hd[kHdStart + t];
        }
        ts.p0 = hd[kHdP0];
        ts.p1 = hd[kHdP1];
        ts.bx = (int)hd[kHdBase];
        ts.by = (int)hd[kHdBase + 1];
        ts.bz = (int)hd[kHdBase + 2];
        const uint32_t total = hd[kHdOff + kHalo], flags = hd[kHdFlags];
        const uint32_t scene = hd[kHdScene];
        ts.fluid_only = hd[kHdFluidOnly] != 0u;
        ts.complete = hd[kHdSuper] != 0u;
        ts.skip = flags == kHdNoFluid || (!c.all_active && !a.active[scene]);  // no fluid, or untouched this step
        const bool pure = flags != 0u;
        ts.lds = !ts.skip && pure && total <= a.tile;
        ts.skip |= pure && !ts.lds && total <= skip_to;
    } else {
        ts.p0 = a.run_start[a.blk_first_run[b]];
        ts.p1 = a.run_start[a.blk_first_run[b + 1]];
        const uint32_t scene = a.classes[a.cls[ts.p0]].scene;
        ts.skip = !a.active[scene] || !a.scenes[scene].has_fluid;
        ts.fluid_only = ts.complete = false;
    }
}

// Stages the halo: eight lanes per cell, so a cell's records are read as one 128-byte line and each
// thread knows its cells without a search; load(u, slot) issues the loads of four cells' records
// before put(u, staged index, slot) stores any.  (A thread per staged record found its cell by an
// eight-step binary search of LDS per record, about 1 us of a block's latency.)
constexpr uint32_t kStageCells = 4;
template <class Load, class Put>
__device__ __forceinline__ void stage_halo(const uint32_t *hoff, const uint32_t *hstart, Load &&load, Put &&put)
{
    const uint32_t ln = threadIdx.x & 7u, grp = threadIdx.x >> 3, ngrp = blockDim.x >> 3;
    for (uint32_t c0 = grp; c0 < kHalo; c0 += kStageCells * ngrp) {
        uint32_t o[kStageCells], n[kStageCells], s[kStageCells], most = 0;
#pragma unroll
        for (uint32_t u = 0; u < kStageCells; ++u) {
            const uint32_t hc = c0 + u * ngrp, h = min(hc, kHalo - 1u);
            o[u] = hoff[h];
            n[u] = hc < kHalo ? hoff[h + 1] - o[u] : 0u;
            s[u] = hstart[h];
            most = max(most, n[u]);
        }
        for (uint32_t k = ln; k < most; k += 8) {
            // past a cell's end its last record is loaded (of an empty cell slot 0), and not stored
#pragma unroll
            for (uint32_t u = 0; u < kStageCells; ++u) load(u, s[u] + min(k, n[u] - min(n[u], 1u)));
#pragma unroll
            for (uint32_t u = 0; u < kStageCells; ++u)
                if (k < n[u]) put(u, o[u] + k, s[u] + k);
        }
    }
}

__device__ __forceinline__ int halo_cell(const TileState &ts, const int4 ci)
{
    return (ci.x - ts.bx + 1) + 6 * (ci.y - ts.by + 1) + 36 * (ci.z - ts.bz + 1);
}

// ---------------------------------------------------------------------------------------------
// LDS-path loops
// ---------------------------------------------------------------------------------------------

// The density walk over the staged halo: tests every candidate in walk order and compacts those
// within the radius (squared distance below thr2: the neighbor threshold t2, or ts2 for the
// candidate list of a substep) as halo offsets into a list.  Staged particles with zero inverse mass
// carry an unreachable position, so the distance test also rejects them.
//
// Cells that no candidate inside can reach are left out of the walk (the order of the others is
// unchanged): a candidate's position at the substep start lies in its cell and has moved by at most
// the largest displacement since, so when the particle's distance to the cell's box exceeds the
// search radius plus that displacement (in cell units, with slack for the rounding of the cell
// assignment), none of the cell's particles can be within the radius.
struct RowCull {
    float ux, uy, uz;  // the particle's current position in cell units
    int cx, cy, cz;    // its cell
    float lim2;        // squared limit in cell units; +inf walks every cell
};

__device__ __forceinline__ RowCull row_cull(const float4 s, const int4 ci, float inv, float radius, float dmax)
{
    RowCull rc;
    rc.ux = s.x * inv;
    rc.uy = s.y * inv;
    rc.uz = s.z * inv;
    rc.cx = ci.x;
    rc.cy = ci.y;
    rc.cz = ci.z;
    const float slack = 1.0e-4f + 1.0e-6f * fmaxd(fmaxd(fabsf(rc.ux), fabsf(rc.uy)), fabsf(rc.uz));
    const float lim = (radius + dmax) * inv * 1.00001f + slack;
    rc.lim2 = dmax < 3.0e38f && lim < 1.0e18f ? lim * lim : __builtin_huge_valf();
    return rc;
}

__device__ __forceinline__ float gap_below(float u, int c) { return fmaxd(u - (float)c, 0.0f); }
__device__ __forceinline__ float gap_above(float u, int c) { return fmaxd((float)(c + 1) - u, 0.0f); }

// A particle's list in a grouped list buffer: words of four entries, word w kWordStride words after
// word 0, so a wave reads or writes 512 consecutive bytes per word.  (Single 16-bit entries took
// four loads per step of the term loops; their stores, one per push, made every wait for a load a
// wait for the stores before it too.)
constexpr uint32_t kWordStride = kListGroup;
__device__ __forceinline__ uint2 *list_words(uint16_t *buf, uint32_t i, uint32_t rows)
{
    return reinterpret_cast<uint2 *>(reinterpret_cast<char *>(buf) + list_word_base(i, rows));
}

// What a pass keeps per particle about its list: the staged entry of the particle itself, where the
// entries are (kInList: the neighbor list, else the candidate list), and the words (kSuperNone: the
// candidates did not fit).
constexpr uint32_t kInList = 0x8000u, kSuperNone = 0x7fffu, kWordsMask = 0x7fffu;
__device__ __forceinline__ uint32_t list_word(uint32_t entry, uint32_t words) { return (entry << 16) | words; }

// List entries are byte offsets into a staged array of 16-byte records (halo index x 16; the tile
// holds at most kTileMost halo particles, so they fit 16 bits), so the LDS address of a listed
// neighbor's record needs no scaling; staged arrays of 4-byte items take the entry / 4.  A list's
// last word is filled up with the entry after the halo's last particle, which holds a record no
// particle is within any radius of: a word's four entries need no test against the list's length.
constexpr uint32_t kEntryScale = 16;
static_assert(kTileMost * kEntryScale <= 65535u, "the filling entry of the largest tile fits 16 bits");
template <class T>
__device__ __forceinline__ const T &at16(const T *base, uint32_t e)
{
    static_assert(sizeof(T) == 16, "16-byte records");
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + e);
}
__device__ __forceinline__ uint32_t at4(const uint32_t *base, uint32_t e)
{
    return *reinterpret_cast<const uint32_t *>(reinterpret_cast<const char *>(base) + (e >> 2));
}

// Appends halo offsets to a particle's list, keeping the first cap: four are collected in a register
// pair, which is stored when full.  n counts all.
struct ListOut {
    uint2 *p;
    uint32_t cap, n, lo, hi;
    __device__ __forceinline__ ListOut(uint2 *words, uint32_t cap_) : p(words), cap(cap_), n(0), lo(0), hi(0) {}
    __device__ __forceinline__ void shift_in(uint32_t e)
    {
        lo = __builtin_amdgcn_alignbit(hi, lo, 16);
        hi = __builtin_amdgcn_alignbit(e, hi, 16);
    }
    __device__ __forceinline__ void push(uint32_t e)
    {
        if (n < cap) {
            shift_in(e);
            if ((n & 3u) == 3u) {
                *p = make_uint2(lo, hi);
                p += kWordStride;
            }
        }
        ++n;
    }
    // fills the last word; returns the words
    __device__ __forceinline__ uint32_t finish(uint32_t fill)
    {
        const uint32_t m = min(n, cap), r = m & 3u;
        if (r) {
            for (uint32_t u = r; u < 4u; ++u) shift_in(fill);
            *p = make_uint2(lo, hi);
        }
        return (m + 3u) >> 2;
    }
};

// f(word) for each of a list's words (>= 1), two words ahead of use.  Past the end it reads up to
// two words that belong to the slot group's next rows or to the buffer's spare rows.
template <class F>
__device__ __forceinline__ void each_word(const uint2 *p, uint32_t words, F &&f)
{
    uint2 w0 = p[0], w1 = p[kWordStride];
    for (; words; --words) {
        const uint2 e = w0;
        w0 = w1;
        w1 = p[2 * kWordStride];
        p += kWordStride;
        f(e);
    }
}
__device__ __forceinline__ void word_entries(uint2 w, uint32_t (&e)[4])
{
    e[0] = w.x & 0xffffu;
    e[1] = w.x >> 16;
    e[2] = w.y & 0xffffu;
    e[3] = w.y >> 16;
}

// Up to 32 candidates [k, f1) of a walked row: first every candidate's squared distance is tested and
// the outcome shifted into a bit mask, without a branch (four candidates per step; the loads may run
// up to three entries past f1, for which the staged arrays carry kTilePad spare entries), then the
// few that passed are pushed in order.  skip is the staged index of a candidate to leave out (the
// particle itself; any index outside the range leaves none out).  (Testing and pushing candidate by
// candidate spent some 40 cycles of a lone wave's latency on each of the three branches of a push,
// whether or not it happened: 21 us of a 34 us launch over the dam break's 64,000 particles.)
template <bool UNIFORM>
__device__ __forceinline__ void scan_range(uint32_t k, uint32_t f1, uint32_t skip, const float4 *lpos,
                                           const uint32_t *lcls, const DensitySelf &x, float thr2, const FluidArgs &a,
                                           ListOut &lo)
{
    const float4 *pp = lpos + k;
    const uint32_t n = f1 - k;  // 1 .. 32
    uint32_t mask = 0, done = 0;
    for (; done < n; done += 4, pp += 4) {
        float4 pj[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) pj[u] = pp[u];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const float dx = x.s.x - pj[u].x, dy = x.s.y - pj[u].y, dz = x.s.z - pj[u].z;
            mask = (mask << 1) | (dot3(dx, dy, dz, dx, dy, dz) < thr2 ? 1u : 0u);
        }
    }
    mask <<= 32u - done;           // bit 31: the first candidate
    mask &= 0xffffffffu << (32u - n);
    if (skip - k < n) mask &= ~(0x80000000u >> (skip - k));
    while (mask) {
        const uint32_t j = (uint32_t)__builtin_clz(mask);
        mask &= ~(0x80000000u >> j);
        if (!UNIFORM && !neighbor_ok(x.pc, a.classes[lcls[k + j]])) continue;
        lo.push((k + j) * kEntryScale);
    }
}

template <bool UNIFORM>
__device__ __forceinline__ void scan_rows(const uint32_t *hoff, int hc, uint32_t fs, const float4 *lpos,
                                          const uint32_t *lcls, const DensitySelf &x, float thr2,
                                          ListOut &lo, const FluidArgs &a, const RowCull &rc)
{
    const float gxl = gap_below(rc.ux, rc.cx), gxr = gap_above(rc.ux, rc.cx);
    // rows of three cells along x, z outer, y inner
#pragma unroll 1
    for (int r = 0; r < 9; ++r) {
        const int ry = r % 3 - 1, rz = r / 3 - 1;
        const float gy = ry < 0 ? gap_below(rc.uy, rc.cy) : (ry > 0 ? gap_above(rc.uy, rc.cy) : 0.0f);
        const float gz = rz < 0 ? gap_below(rc.uz, rc.cz) : (rz > 0 ? gap_above(rc.uz, rc.cz) : 0.0f);
        const float perp = gy * gy + gz * gz;
        if (!(perp < rc.lim2)) continue;
        const int h0 = hc - 1 + 6 * ry + 36 * rz;
        const uint32_t f1 = hoff[h0 + (gxr * gxr + perp < rc.lim2 ? 3 : 2)];
        for (uint32_t k = hoff[h0 + (gxl * gxl + perp < rc.lim2 ? 0 : 1)]; k < f1; k += 32u)
            scan_range<UNIFORM>(k, min(f1, k + 32u), fs, lpos, lcls, x, thr2, a, lo);
    }
}

// The density terms of the listed particles within the neighbor radius at the current positions, in
// list order; every lane evaluates each term before the test decides whether it is added.  d.req
// counts the neighbors.
template <bool TENSION, bool FAST>
__device__ __forceinline__ void density_words(const uint2 *p, uint32_t words, const float4 *lpos, const DensitySelf &x,
                                              DensitySum &d)
{
    if (!words) return;
    each_word(p, words, [&](uint2 w) {
        uint32_t e[4];
        word_entries(w, e);
        float4 pj[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) pj[u] = at16(lpos, e[u]);
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const DensityTerm t = density_term<TENSION, FAST>(x, pj[u]);
            if (t.d2 < x.t2) {
                ++d.req;
                density_add<TENSION>(d, x, t);
            }
        }
    });
}

__device__ __forceinline__ void density_sums(const uint2 *p, uint32_t words, const float4 *lpos, const DensitySelf &x,
                                             DensitySum &d)
{
    // one vote per particle instead of a test per term
    const bool fast = __all(x.fd);
    if (x.tension) {
        if (fast) density_words<true, true>(p, words, lpos, x, d);
        else density_words<true, false>(p, words, lpos, x, d);
    } else {
        if (fast) density_words<false, true>(p, words, lpos, x, d);
        else density_words<false, false>(p, words, lpos, x, d);
    }
}

// The same over a candidate list that holds more neighbors than the cap: the first cap are summed
// and written to the neighbor list.
__device__ __forceinline__ uint32_t density_capped(const uint2 *p, uint32_t words, const float4 *lpos,
                                                   const DensitySelf &x, uint2 *li, uint32_t cap, uint32_t fill,
                                                   DensitySum &d)
{
    d = DensitySum{};
    ListOut lo(li, cap);
    each_word(p, words, [&](uint2 w) {
        uint32_t e[4];
        word_entries(w, e);
        for (uint32_t u = 0; u < 4; ++u) {
            const DensityTerm t = density_term<true, false>(x, at16(lpos, e[u]));
            if (t.d2 < x.t2) {
                if (lo.n < cap) density_add<true>(d, x, t);
                lo.push(e[u]);
            }
        }
    });
    d.req = lo.n;
    return lo.finish(fill);
}

// The delta terms of a particle without cohesion, viscosity, CFL and tension terms: the pressure
// term of every listed particle within the neighbor radius (delta_term's, restated for the one
// term), in list order.
template <bool FAST>
__device__ __forceinline__ void delta_plain(const uint2 *p, uint32_t words, const float4 *lcs, const DeltaSelf &x,
                                            DeltaSum &d)
{
    const float k2 = __fmul_rn(2.0f, x.kw);
    each_word(p, words, [&](uint2 w) {
        uint32_t e[4];
        word_entries(w, e);
        // two at a time: four hold more registers than the pass has without spilling
#pragma unroll
        for (uint32_t v = 0; v < 4; v += 2) {
            float4 q[2];
            float d2[2], dist[2], y[2];
#pragma unroll
            for (uint32_t u = 0; u < 2; ++u) q[u] = at16(lcs, e[v + u]);
            uint32_t sig = 0;
#pragma unroll
            for (uint32_t u = 0; u < 2; ++u) {
                q[u].x = x.sx - q[u].x;
                q[u].y = x.sy - q[u].y;
                q[u].z = x.sz - q[u].z;
                d2[u] = dot3(q[u].x, q[u].y, q[u].z, q[u].x, q[u].y, q[u].z);
                float y0;
                dist[u] = fsqrt_rsq(d2[u], y0);
                if (FAST) {
                    y[u] = frcp_step(dist[u], y0);
                    sig = max(sig, __float_as_uint(dist[u]) & 0x7fffffu);
                }
            }
            // one test for the two: the significand that the Newton step does not reach
            if (FAST && sig == 0x7fffffu) {
                __asm__ volatile("");
#pragma unroll
                for (uint32_t u = 0; u < 2; ++u) y[u] = frcp_last_significand(dist[u], y[u]);
            }
#pragma unroll
            for (uint32_t u = 0; u < 2; ++u) {
                PairQuot pq;
                pair_quot_y<FAST, true>(pq, q[u].x, q[u].y, q[u].z, dist[u], x.h, x.ih, k2, y[u]);
                const float msc = 0.5f * (x.Ci + q[u].w) * pq.der;
                if (d2[u] < x.t2 && dist[u] > kEps) {
                    d.x = d.x + msc * pq.nnx;
                    d.y = d.y + msc * pq.nny;
                    d.z = d.z + msc * pq.nnz;
                    d.w = d.w + 1.0f;
                }
            }
        }
    });
}

// ---------------------------------------------------------------------------------------------
// kernels
// ---------------------------------------------------------------------------------------------
// MODE: kDensPlain walks every iteration; with candidate lists, kDensBuild (a substep's first
// iteration) walks the wider radius into the candidate lists and takes the neighbors from them,
// and kDensReuse (a later iteration) takes them from the candidate lists in every block whose
// particles' displacements allow it and walks the other blocks.
constexpr int kDensPlain = 0, kDensBuild = 1, kDensReuse = 2;
// UCLS: the particle classes of a tiled fluid launch -- kClsMixed per particle, kClsOne every
// particle class 0, kClsBlock one class per scene with fluid, read from the block's first particle.
constexpr int kClsMixed = 0, kClsOne = 1, kClsBlock = 2;
template <int UCLS, int MODE>
__global__ __launch_bounds__(kTileBlock) __attribute__((amdgpu_waves_per_eu(kDensityWaves))) void k_fluid_density_tiled(
    FluidArgs a, SubstepConsts c)
{
    constexpr bool UNIFORM = UCLS != kClsMixed;
    extern __shared__ float4 dyn[];
    __shared__ uint32_t hoff[kHalo + 1];
    __shared__ uint32_t hstart[kHalo];
    __shared__ uint32_t s_blk;
    __shared__ uint32_t s_meta[kWgMetaWords];
    __shared__ uint32_t s_hmax;  // largest displacement bound in the staged halo (float bits)
    __shared__ uint32_t s_omax;  // the same over the block's own particles with mass (one class)
    constexpr bool BUILD = MODE == kDensBuild, REUSE = MODE == kDensReuse;
    float4 *lpos = dyn;
    uint32_t *lcls = reinterpret_cast<uint32_t *>(dyn + a.tile + kTilePad);
    const uint32_t tid = threadIdx.x;
    // largest |delta|^2 of the previous iteration: bounds how far any fluid particle has moved
    // from its iteration-0 position
    const float md2 = a.it == 0 ? 0.0f : __uint_as_float(a.iter_state[kStateMaxDisp + a.it - 1]);
    // the density launch resets the displacement word its delta pass raises
    if (blockIdx.x == 0 && tid == 0) a.iter_state[kStateMaxDisp + a.it] = 0u;
    const uint32_t nblk = a.nblk[1];  // the blocks of scenes with fluid
    uint32_t *queue = a.iter_state + kStateDensity + a.it * kXcds * kQueueStride;
    if (tid < kWgMetaWords) s_meta[tid] = 0u;  // ordered before any use by the first block's barrier
    if (tid == 0) s_hmax = s_omax = 0u;
    BlockQueue bq(blockIdx.x);
    TileState ts;
    uint32_t after;
    for (uint32_t blk = BlockQueue::first(blockIdx.x, nblk); blk != kInvalid; blk = after) {
        tile_load(ts, blk, hoff, hstart, 0u, a, c);
        __syncthreads();
        if (ts.skip) {
            if (tid == 0) s_blk = bq.next(queue, nblk);
            __syncthreads();
            after = s_blk;
            continue;
        }
        MetaAcc ma;
        // the block's class (wave-uniform: the class and what derives from it sit in scalar
        // registers)
        const uint32_t bcls = UCLS == kClsBlock ? __builtin_amdgcn_readfirstlane(a.cls[ts.p0]) : 0u;
        if (ts.lds) {
            const uint32_t total = hoff[kHalo], fill = total * kEntryScale;
            // a halo of one particle class (the common case in a pool of single-material scenes)
            // takes the class filter out of the walk, as a pool of one class does
            const uint32_t ref = UNIFORM ? bcls : a.cls[ts.p0];
            bool mixed = false;
            uint32_t dmb = 0, dmo = 0;  // displacement bounds are non-negative floats: their bits order them
            float4 lv[kStageCells];
            uint32_t lq[kStageCells];
            stage_halo(
                hoff, hstart,
                [&](uint32_t u, uint32_t q) {
                    lv[u] = a.cur[q];
                    if (!UNIFORM) lq[u] = a.cls[q];
                },
                [&](uint32_t u, uint32_t f, uint32_t q) {
                    float4 v = lv[u];
                    if (v.w < 0.0f) {
                        v.x = v.y = v.z = kFarAway;
                    } else if (REUSE) {
                        dmb = max(dmb, __float_as_uint(v.w));
                        // one class: the block's own particles' part of the reuse check rides along
                        if (UNIFORM && q >= ts.p0 && q < ts.p1) dmo = max(dmo, __float_as_uint(v.w));
                    }
                    lpos[f] = v;
                    if (!UNIFORM) {
                        lcls[f] = lq[u];
                        mixed |= lq[u] != ref;
                    }
                });
            if (tid == 0) lpos[total] = make_float4(kFarAway, kFarAway, kFarAway, kNoMass);
            if (REUSE) {
                dmb = wave_max(dmb);
                if ((tid & 63u) == 0u) atomicMax(&s_hmax, dmb);
                if (UNIFORM) {
                    dmo = wave_max(dmo);
                    if ((tid & 63u) == 0u) atomicMax(&s_omax, dmo);
                }
            }
            const int any_mixed = __syncthreads_or(mixed ? 1 : 0);  // also the barrier after staging
            const bool bu = UNIFORM || !any_mixed;
            // the fluid passes and the contacts record every displacement of a fluid particle
            const bool sup = BUILD || REUSE;
            // The candidates of iteration 0 (within h + skin of x*) hold particle i's list while
            // D_i + D_j < skin for every j in its 27 cells: a pair within h now was within
            // h + D_i + D_j then (D: displacement since iteration 0, x* to x* + delta).  D_j is
            // bounded by the halo's largest; the margins in FluidConst cover the rounding of the
            // squared distances (a few ulps) and of the recorded displacements.  A block where some
            // particle fails, or has no complete candidate list, is walked whole (one decision per
            // block keeps the walk out of the waves of the others).
            bool reuse = false;
            if (REUSE && sup && ts.complete) {
                const float hmax = __uint_as_float(s_hmax);
                if (UNIFORM) {
                    // D_i + hmax < allow holds for every particle with mass exactly when it holds for
                    // their largest D_i (rounded addition is monotone)
                    const ParticleClass pc = a.classes[bcls];
                    reuse = pc.kind != CN_PARTICLE_KIND_FLUID ||
                            __uint_as_float(s_omax) + hmax < a.fc[pc.fluid_mat].allow;
                } else {
                    bool bad = false;
                    for (uint32_t i = ts.p0 + tid; i < ts.p1; i += kTileBlock) {
                        const uint32_t e = a.scnt[i] >> 16;
                        const ParticleClass pc = a.classes[at4(lcls, e)];
                        const float D = at16(lpos, e).w;
                        if (pc.kind == CN_PARTICLE_KIND_FLUID && D >= 0.0f) bad |= !(D + hmax < a.fc[pc.fluid_mat].allow);
                    }
                    reuse = !__syncthreads_or(bad ? 1 : 0);
                }
            }
            // the walk at the neighbor radius (thr2 = t2, radius h) or the candidate radius (ts2)
            auto scan = [&](auto bu_tag, const DensitySelf &x, int4 ci, int hc, uint32_t fs, float thr2,
                            float radius, ListOut &lo) {
                constexpr bool BU = decltype(bu_tag)::value;
                const float inv = c.inv_cell > 0.0f ? c.inv_cell : a.scenes[x.pc.scene].inv_cell;
                // displacement since the cells were assigned: none at iteration 0; later the largest
                // |delta| of the previous iteration, where only the fluid passes move fluid particles
                const float dmax = a.it == 0 ? 0.0f : (ts.fluid_only ? fsqrt(md2) : 3.4e38f);
                const RowCull rc = row_cull(x.s, ci, inv, radius, dmax);
                scan_rows<BU>(hoff, hc, fs, lpos, lcls, x, thr2, lo, a, rc);
            };
            // BLK: the block's halo holds one particle class (bref, wave-uniform), so the class and
            // everything the particle derives from it (material, radius, thresholds) load into
            // scalar registers; a pool of single-material scenes takes this path in its general
            // instantiation
            const uint32_t bref = __builtin_amdgcn_readfirstlane(ref);
            auto particles = [&](auto blk_tag) {
                constexpr bool BLK = decltype(blk_tag)::value;
                for (uint32_t i = ts.p0 + tid; i < ts.p1; i += kTileBlock) {
                    const uint32_t bw = a.bnd[i];  // loaded first, long before its use
                    int4 ci = make_int4(0, 0, 0, 0);
                    int hc = 0;
                    uint32_t entry, words = 0;
                    if (REUSE && reuse) {
                        const uint32_t sw = a.scnt[i];
                        entry = sw >> 16;
                        words = sw & kWordsMask;
                    } else {
                        ci = a.cellc[i];
                        hc = halo_cell(ts, ci);
                        entry = (hoff[hc] + (i - hstart[hc])) * kEntryScale;
                    }
                    DensitySelf x;
                    uint32_t lw = 0, sw = 0;
                    if (density_begin(x, i, at16(lpos, entry),
                                      UNIFORM ? bcls : (BLK ? bref : at4(lcls, entry)), a)) {
                        DensitySum d;
                        if (density_walks(x, BLK || bu, c)) {
                            uint2 *li = list_words(a.list, i, list_rows(c.cap));
                            uint2 *ls = list_words(a.slist, i, kSuperSlots);
                            bool done = REUSE && reuse;
                            if (REUSE && reuse) ++ma.reuse;
                            if (BUILD && sup) {
                                // the candidates within h + skin, then the neighbors among them; a
                                // particle with more candidates than the list holds walks for its
                                // neighbors (and its block never reuses)
                                const FluidConst fc = a.fc[x.pc.fluid_mat];
                                ListOut lo(ls, kSuperSlots);
                                if (BLK || bu) scan(std::true_type{}, x, ci, hc, entry / kEntryScale, fc.ts2, fc.rs, lo);
                                else scan(std::false_type{}, x, ci, hc, entry / kEntryScale, fc.ts2, fc.rs, lo);
                                done = lo.n <= kSuperSlots;
                                words = lo.finish(fill);
                                sw = done ? words : kSuperNone;
                                if (!done) a.blk_halo[(size_t)ts.blk * kHaloStride + kHdSuper] = 0u;
                            }
                            if (done) {
                                density_sums(ls, words, lpos, x, d);
                                lw = words;
                                if (d.req > c.cap)
                                    lw = kInList | density_capped(ls, words, lpos, x, li, c.cap, fill, d);
                            } else {
                                ListOut lo(li, c.cap);
                                if (BLK || bu) scan(std::true_type{}, x, ci, hc, entry / kEntryScale, x.t2, x.h, lo);
                                else scan(std::false_type{}, x, ci, hc, entry / kEntryScale, x.t2, x.h, lo);
                                const uint32_t req = lo.n;
                                words = lo.finish(fill);
                                density_sums(li, words, lpos, x, d);
                                d.req = req;
                                lw = kInList | words;
                            }
                            d.inr = min(d.req, c.cap);
                        }
                        density_end(i, bw, d, x, ma, a, c);
                    }
                    a.lcnt[i] = list_word(entry, lw);
                    if (BUILD && sup) a.scnt[i] = list_word(entry, sw);
                }
            };
            if (!UNIFORM && bu)
                particles(std::true_type{});
            else
                particles(std::false_type{});
            if (tid == 0) ++ma.lds;
        } else {
            for (uint32_t i = ts.p0 + tid; i < ts.p1; i += kTileBlock)
                density_global<UNIFORM>(i, ma, a, c, bcls);
            if (tid == 0) ++ma.runs;
        }
        meta_to_wg(ma, s_meta);
        if (tid == 0) s_blk = bq.next(queue, nblk);  // not before the block is done: see BlockQueue
        __syncthreads();
        after = s_blk;
        if (tid == 0) s_hmax = s_omax = 0u;  // read again only after the next block's staging barrier
    }
    flush_wg_meta(s_meta, a);
}

// WIDE = false: every block, the previous delta staged in LDS beside the records; blocks whose halo
// only fits without it are skipped and left to the WIDE = true launch, which takes the listed wide
// blocks and reads the previous delta from HBM through a staged slot map.
template <int UCLS, bool WIDE>
__global__ __launch_bounds__(kTileBlock) __attribute__((amdgpu_waves_per_eu(kDeltaWaves))) void k_fluid_delta_tiled(
    FluidArgs a, SubstepConsts c)
{
    const bool listed = WIDE && a.wide_only;  // the listed wide blocks, else every block
    constexpr bool UNIFORM = UCLS != kClsMixed;
    extern __shared__ float4 dyn[];
    __shared__ uint32_t hoff[kHalo + 1];
    __shared__ uint32_t hstart[kHalo];
    __shared__ uint32_t s_blk;
    const bool use_d = a.it > 0;
    const bool tension = c.tension != 0u;
    const uint32_t room = a.tile + 1u;  // the halo and the filling entry's record
    float4 *lcs = dyn;
    float4 *ldin = lcs + room;
    float4 *lnc = ldin + (use_d && !WIDE ? room : 0u);
    uint32_t *lcls = reinterpret_cast<uint32_t *>(lnc + (tension ? room : 0u));
    uint32_t *lslot = lcls + (UNIFORM ? 0u : room);
    const uint32_t tid = threadIdx.x;
    const uint32_t nblk = a.nblk[1];
    uint32_t *queue = a.iter_state + kStateDelta + a.it * kXcds * kQueueStride;
    uint32_t *wqueue = a.iter_state + kStateWideQueue + a.it;
    const uint32_t nwide = listed ? a.iter_state[kStateWideCount] : 0u;
    BlockQueue bq(blockIdx.x);
    TileState ts;
    float d2max = 0.0f;
    bool rel_one = false;  // one class in the launch: see rel
    if (UCLS == kClsOne && use_d) {
        const ParticleClass pc0 = a.classes[0];
        rel_one = pc0.kind == CN_PARTICLE_KIND_FLUID &&
                  (cfl_term_on(a.fm[pc0.fluid_mat], a, c) || visc_term_on(a.fm[pc0.fluid_mat], a, c));
    }
    auto next = [&]() -> uint32_t {
        if (!listed) return bq.next(queue, nblk);
        if (nwide <= gridDim.x) return kInvalid;
        const uint32_t t = gridDim.x + atomicAdd(wqueue, 1u);
        return t < nwide ? a.wide_blk[t] : kInvalid;
    };
    const uint32_t first = !listed ? BlockQueue::first(blockIdx.x, nblk)
                                   : (blockIdx.x < nwide ? a.wide_blk[blockIdx.x] : kInvalid);
    uint32_t after;
    for (uint32_t blk = first; blk != kInvalid; blk = after) {
        tile_load(ts, blk, hoff, hstart, WIDE || !use_d ? 0u : c.tile_wide, a, c);
        __syncthreads();
        if (ts.skip) {
            if (tid == 0) s_blk = next();
            __syncthreads();
            after = s_blk;
            continue;
        }
        // the block's class
        const uint32_t bcls = UCLS == kClsBlock ? __builtin_amdgcn_readfirstlane(a.cls[ts.p0]) : 0u;
        const uint32_t ref = UNIFORM ? bcls : a.cls[ts.p0];
        bool bu = UNIFORM;  // one particle class in the halo: every listed neighbor has the particle's material
        if (ts.lds) {
            bool mixed = false;
            float4 lv[kStageCells];
            uint32_t lq[kStageCells];
            stage_halo(
                hoff, hstart,
                [&](uint32_t u, uint32_t q) {
                    lv[u] = a.cs[q];
                    if (!UNIFORM) lq[u] = a.cls[q];
                },
                [&](uint32_t u, uint32_t f, uint32_t q) {
                    lcs[f] = make_float4(lv[u].x, lv[u].y, lv[u].z, lv[u].w);
                    if (!UNIFORM) {
                        lcls[f] = lq[u];
                        mixed |= lq[u] != ref;
                    }
                });
            // the neighbors' previous deltas are read only by the viscosity and CFL terms: staged
            // (the wide layout: their slots) only when one of the block's fluid particles has one on
            bool rel = rel_one;
            if (use_d && UCLS != kClsOne) {
                if (UNIFORM) {
                    const ParticleClass pc0 = a.classes[bcls];
                    rel = pc0.kind == CN_PARTICLE_KIND_FLUID &&
                          (cfl_term_on(a.fm[pc0.fluid_mat], a, c) || visc_term_on(a.fm[pc0.fluid_mat], a, c));
                } else {
                    bool mine = false;
                    for (uint32_t i = ts.p0 + tid; i < ts.p1; i += kTileBlock) {
                        const ParticleClass pc = a.classes[a.cls[i]];
                        mine |= pc.kind == CN_PARTICLE_KIND_FLUID &&
                                (cfl_term_on(a.fm[pc.fluid_mat], a, c) || visc_term_on(a.fm[pc.fluid_mat], a, c));
                    }
                    rel = __syncthreads_or(mine ? 1 : 0) != 0;
                }
            }
            if (WIDE && rel)
                stage_halo(
                    hoff, hstart, [&](uint32_t, uint32_t) {}, [&](uint32_t, uint32_t f, uint32_t q) { lslot[f] = q; });
            if (!WIDE && rel) {
                float4 dv[kStageCells];
                stage_halo(
                    hoff, hstart, [&](uint32_t u, uint32_t q) { dv[u] = a.din[q]; },
                    [&](uint32_t u, uint32_t f, uint32_t) { ldin[f] = make_float4(dv[u].x, dv[u].y, dv[u].z, 0.0f); });
            }
            if (tension) {
                float4 nv[kStageCells];
                stage_halo(
                    hoff, hstart, [&](uint32_t u, uint32_t q) { nv[u] = a.nc[q]; },
                    [&](uint32_t u, uint32_t f, uint32_t) { lnc[f] = make_float4(nv[u].x, nv[u].y, nv[u].z, nv[u].w); });
            }
            if (tid == 0) {  // what the filling entry names
                const uint32_t total = hoff[kHalo];
                lcs[total] = make_float4(kFarAway, kFarAway, kFarAway, 0.0f);
                if (!WIDE && rel) ldin[total] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                if (tension) lnc[total] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                if (!UNIFORM) lcls[total] = ref;
                if (WIDE && rel) lslot[total] = ts.p0;
            }
            const int any_mixed = __syncthreads_or(mixed ? 1 : 0);  // also the barrier after staging
            bu = UNIFORM || !any_mixed;
        }
        // BLK: one particle class in the halo (bref, wave-uniform): the class-derived values of
        // each particle load into scalar registers (the general instantiation in a pool of
        // single-material scenes)
        const uint32_t bref = __builtin_amdgcn_readfirstlane(ref);
        auto particles = [&](auto blk_tag) {
            constexpr bool BLK = decltype(blk_tag)::value;
            for (uint32_t i = ts.p0 + tid; i < ts.p1; i += kTileBlock) {
                // a block that is not staged walks the run table
                const uint32_t lw = ts.lds ? a.lcnt[i] : 0u;
                const DeltaPre pre = delta_pre<UNIFORM || BLK>(i, a, UNIFORM ? bcls : bref);
                const uint2 *p = lw & kInList ? list_words(a.list, i, list_rows(c.cap))
                                              : list_words(a.slist, i, kSuperSlots);
                const float d2 = delta_particle<UNIFORM>(
                    i, pre,
                    [&](const DeltaSelf &x, DeltaSum &d) {
                        if (!ts.lds) {
                            delta_walk<UNIFORM || BLK>(i, x, d, a, c);
                            return;
                        }
                        const uint32_t words = lw & kWordsMask;
                        if (!words) return;
                        const bool fast = __all(x.fd);
                        if (x.plain) {
                            if (fast) delta_plain<true>(p, words, lcs, x, d);
                            else delta_plain<false>(p, words, lcs, x, d);
                            return;
                        }
                        // the general terms, two listed particles at a time
                        each_word(p, words, [&](uint2 w) {
#pragma unroll 2
                            for (uint32_t u = 0; u < 4; ++u) {
                                const uint32_t e = (u & 2u ? w.y : w.x) >> ((u & 1u) * 16u) & 0xffffu;
                                const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                                const float4 dq = !x.need_rel ? zero : (WIDE ? a.din[at4(lslot, e)] : at16(ldin, e));
                                const float4 ncq = x.tension ? at16(lnc, e) : zero;
                                delta_add(d, BLK || bu ? delta_term<true>(x, at16(lcs, e), dq, ncq, 0u, a)
                                                       : delta_term<false>(x, at16(lcs, e), dq, ncq, at4(lcls, e), a));
                            }
                        });
                    },
                    [&](bool nc) {
                        float4 r;
                        if (ts.lds) {
                            const float4 &v = at16(nc ? lnc : lcs, lw >> 16);
                            r = make_float4(v.x, v.y, v.z, v.w);
                        } else {
                            const float4 &v = (nc ? a.nc : a.cs)[i];
                            r = make_float4(v.x, v.y, v.z, v.w);
                        }
                        return r;
                    },
                    a, c);
                d2max = fmaxd(d2max, d2);
            }
        };
        if (!UNIFORM && bu)
            particles(std::true_type{});
        else
            particles(std::false_type{});
        if (tid == 0) s_blk = next();
        __syncthreads();
        after = s_blk;
    }
    flush_disp(d2max, a);
}

// Thread per particle through the run table: hash keys, and iterations past the tracked ones.
template <bool UNIFORM>
__global__ __launch_bounds__(kBlock) void k_fluid_density_global(FluidArgs a, SubstepConsts c)
{
    if (blockIdx.x == 0 && threadIdx.x == 0 && a.it < kIterStateWords) a.iter_state[kStateMaxDisp + a.it] = 0u;
    MetaAcc ma;
    const uint32_t i = xcd_tile(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
    if (i < c.n) density_global<UNIFORM>(i, ma, a, c);
    flush_meta(ma, a);
}

template <bool UNIFORM>
__global__ __launch_bounds__(kBlock) void k_fluid_delta_global(FluidArgs a, SubstepConsts c)
{
    const uint32_t i = xcd_tile(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
    float d2 = 0.0f;
    if (i < c.n) d2 = delta_global<UNIFORM>(i, a, c);
    flush_disp(d2, a);
}

// Exact neighbor lists of iteration 0 (the per-pass entry): the first cap in-radius neighbors in
// walk order, k-major, and their count.
template <bool UNIFORM>
__global__ __launch_bounds__(kBlock) void k_fluid_lists(FluidArgs a, SubstepConsts c)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= c.n) return;
    const ParticleClass pc = a.classes[UNIFORM ? 0u : a.cls[i]];
    const float4 s = a.cur[i];
    uint32_t cnt = 0;
    if (pc.kind == CN_PARTICLE_KIND_FLUID && s.w >= 0.0f && c.cap > 0 && (!UNIFORM || neighbor_ok(pc, pc))) {
        const float t2 = a.fc[pc.fluid_mat].t2;
        walk_runs(a.cellc[i], run_table(a), c, [&](uint32_t q) {
            if (q == i) return true;
            if (!UNIFORM && !neighbor_ok(pc, a.classes[a.cls[q]])) return true;
            const float4 pj = a.cur[q];
            if (pj.w < 0.0f) return true;
            const float dx = s.x - pj.x, dy = s.y - pj.y, dz = s.z - pj.z;
            if (!(dot3(dx, dy, dz, dx, dy, dz) < t2)) return true;
            a.nbr[(size_t)cnt * c.n + i] = q;
            return ++cnt < c.cap;
        });
    }
    a.nbr_cnt[i] = cnt;
}

// Vorticity confinement after the velocity update: physics_fluid_compute_vorticity.cs.hlsl:16-81
// (APPLY = false: vort[i] = (curl, |curl|), zero for particles that do not confine) and
// physics_fluid_apply_vorticity_confinement.cs.hlsl:16-94 (APPLY = true).  Both walk the
// post-update neighbor list (physics_solver.cpp:1262): the first cap in-radius neighbors in walk
// order on the final positions, of which the same-material ones contribute.  Inactive scenes are
// skipped whole (their neighbors are their own).  each(s, t2, self, term) calls term(same material, dx,
// dy, dz, the neighbor's velocity or (APPLY) curl) for every listed neighbor.
template <bool APPLY, class Each>
__device__ __forceinline__ void vorticity_particle(uint32_t i, const ParticleClass &pc, const FluidArgs &a,
                                                   const SubstepConsts &c, float4 *vel, float4 *vort, Each &&each)
{
    const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const cn_fluid_material &m = a.fm[pc.fluid_mat];
    const float conf = fmaxd(m.vorticity_confinement, 0.0f);
    const float4 s = a.pos[i];
    if (conf <= kEps || s.w <= kEps) {
        if (!APPLY) vort[i] = zero;
        return;
    }
    const float4 self = APPLY ? vort[i] : vel[i];
    if (APPLY && self.w <= kEps) return;
    const float h = fmaxd(m.smoothing_radius, 1.0e-4f);
    float ax = 0.0f, ay = 0.0f, az = 0.0f;
    // one listed neighbor's term (same material, inside the kernel's support)
    each(s, a.fc[pc.fluid_mat].t2, [&](bool same, float dx, float dy, float dz, const float4 &o) {
        const float dist = len3(dx, dy, dz);
        // every term is evaluated before the test decides whether it is added (no branch per neighbor)
        const bool add = same && !(dist <= kEps || dist >= h);
        // FluidSpikyKernelGradient, physics_fluid_common.hlsli:45-54
        const float dw = spiky_dw(dist, h);
        const float gx = dw * fdiv(dx, dist), gy = dw * fdiv(dy, dist), gz = dw * fdiv(dz, dist);
        float tx, ty, tz;
        if (APPLY) {
            tx = o.w * gx;
            ty = o.w * gy;
            tz = o.w * gz;
        } else {
            const float wx = o.x - self.x, wy = o.y - self.y, wz = o.z - self.z;
            tx = wy * gz - wz * gy;
            ty = wz * gx - wx * gz;
            tz = wx * gy - wy * gx;
        }
        ax = add ? ax + tx : ax;
        ay = add ? ay + ty : ay;
        az = add ? az + tz : az;
    });
    if (!APPLY) {
        vort[i] = make_float4(ax, ay, az, len3(ax, ay, az));
        return;
    }
    const float gl = len3(ax, ay, az);
    if (gl <= kEps) return;
    const float nx = fdiv(ax, gl), ny = fdiv(ay, gl), nz = fdiv(az, gl);
    const float fx = conf * (ny * self.z - nz * self.y);
    const float fy = conf * (nz * self.x - nx * self.z);
    const float fz = conf * (nx * self.y - ny * self.x);
    const float4 v = vel[i];
    vel[i] = make_float4(v.x + c.dt * fx, v.y + c.dt * fy, v.z + c.dt * fz, 0.0f);
}

// The same over the run table.  The curl pass stores the list where a list buffer is given (nbr,
// neighbor-major); the confinement pass then reads it instead of walking again.
template <bool UNIFORM, bool APPLY>
__device__ __forceinline__ void vorticity_global(uint32_t i, const FluidArgs &a, const SubstepConsts &c, float4 *vel,
                                                 float4 *vort)
{
    const ParticleClass pc = a.classes[UNIFORM ? 0u : a.cls[i]];
    if (!a.active[pc.scene]) return;
    if (pc.kind != CN_PARTICLE_KIND_FLUID) {
        if (!APPLY) vort[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        return;
    }
    vorticity_particle<APPLY>(i, pc, a, c, vel, vort, [&](const float4 &s, float t2, auto &&term) {
        if (c.cap == 0 || (UNIFORM && !neighbor_ok(pc, pc))) return;
        auto other = [&](uint32_t q) { return APPLY ? vort[q] : vel[q]; };
        auto same = [&](uint32_t q) { return UNIFORM || a.classes[a.cls[q]].fluid_mat == pc.fluid_mat; };
        if (APPLY && a.nbr) {
            // the list the curl pass wrote: the same neighbors in the same order (positions unchanged)
            const uint32_t cnt = a.nbr_cnt[i];
            for (uint32_t k = 0; k < cnt; ++k) {
                const uint32_t q = a.nbr[(size_t)k * c.n + i];
                const float4 pj = a.pos[q];
                term(same(q), s.x - pj.x, s.y - pj.y, s.z - pj.z, other(q));
            }
            return;
        }
        uint32_t cnt = 0;
        walk_runs(a.cellc[i], run_table(a), c, [&](uint32_t q) {
            if (q == i) return true;
            if (!UNIFORM && !neighbor_ok(pc, a.classes[a.cls[q]])) return true;
            const float4 pj = a.pos[q];
            if (pj.w <= kEps) return true;
            const float dx = s.x - pj.x, dy = s.y - pj.y, dz = s.z - pj.z;
            if (!(dot3(dx, dy, dz, dx, dy, dz) < t2)) return true;
            if (!APPLY && a.nbr) a.nbr[(size_t)cnt * c.n + i] = q;  // for the confinement pass
            term(same(q), dx, dy, dz, other(q));
            return ++cnt < c.cap;
        });
        if (!APPLY && a.nbr) a.nbr_cnt[i] = cnt;
    });
}

template <bool UNIFORM, bool APPLY>
__global__ __launch_bounds__(kBlock) void k_fluid_vorticity(FluidArgs a, SubstepConsts c, float4 *__restrict__ vel,
                                                            float4 *__restrict__ vort)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < c.n) vorticity_global<UNIFORM, APPLY>(i, a, c, vel, vort);
}

// FluidAnisotropyJacobiRotate, physics_fluid_anisotropy_common.hlsli:28-74 (rsqrt read as
// 1/sqrt): the rotation in the (P, Q) plane that zeroes A[P][Q], accumulated into R.
template <int P, int Q>
__device__ __forceinline__ void jacobi_rotate(float (&A)[3][3], float (&R)[3][3])
{
    constexpr int K = 3 - P - Q;
    const float apq = A[P][Q];
    if (fabsf(apq) <= 1.0e-20f) return;
    const float d = fdiv(A[P][P] - A[Q][Q], 2.0f * apq);
    float t = fdiv(1.0f, fabsf(d) + fsqrt(d * d + 1.0f));
    if (d < 0.0f) t = -t;
    const float cs = fdiv(1.0f, fsqrt(t * t + 1.0f));
    const float sn = t * cs;
    A[P][P] = A[P][P] + t * apq;
    A[Q][Q] = A[Q][Q] - t * apq;
    A[P][Q] = 0.0f;
    A[Q][P] = 0.0f;
    const float akp = cs * A[K][P] + sn * A[K][Q];
    const float akq = -sn * A[K][P] + cs * A[K][Q];
    A[K][P] = akp;
    A[P][K] = akp;
    A[K][Q] = akq;
    A[Q][K] = akq;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float rkp = cs * R[k][P] + sn * R[k][Q];
        const float rkq = -sn * R[k][P] + cs * R[k][Q];
        R[k][P] = rkp;
        R[k][Q] = rkq;
    }
}

template <int A_, int B_>
__device__ __forceinline__ void sort_pair(float (&ev)[3], float (&ax)[3][3])
{
    if (ev[A_] < ev[B_]) {
        const float t = ev[A_];
        ev[A_] = ev[B_];
        ev[B_] = t;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const float u = ax[A_][c];
            ax[A_][c] = ax[B_][c];
            ax[B_][c] = u;
        }
    }
}

// Render anisotropy: physics_fluid_build_render_anisotropy.cs.hlsl:34-171 with
// physics_fluid_anisotropy_common.hlsli:9-156 (rcp and rsqrt read as correctly rounded 1/x and
// 1/sqrt), over the post-update list taken twice: the weighted mean of the listed
// neighbors, then their weighted covariance; four largest-pivot Jacobi rotations, axes sorted by
// decreasing eigenvalue, scales 1.1 sqrt(eigenvalue) clamped to [r, 2r].  A pinned fluid particle
// has no list (the reference reads a count its build never wrote there) and gets the isotropic
// frame.  Written in particle-index order: out[k * n + particle] for axis k.  each(first, s, t2, f)
// calls f(neighbor position) for every listed neighbor.
template <class Each>
__device__ __forceinline__ void aniso_particle(uint32_t i, const ParticleClass &pc, size_t pid, bool listed,
                                               const FluidArgs &a, const SubstepConsts &c, float4 *out, Each &&each)
{
    const size_t n = c.npid;
    const float radius = fmaxd(pc.radius, 1.0e-4f);
    float ax[3][3] = {{1.0f, 0.0f, 0.0f}, {0.0f, 1.0f, 0.0f}, {0.0f, 0.0f, 1.0f}};
    float sc[3] = {radius, radius, radius};
    if (pc.kind == CN_PARTICLE_KIND_FLUID) {
        const cn_fluid_material &m = a.fm[pc.fluid_mat];
        const float support = fmaxd(m.smoothing_radius, radius);
        const float inv = fdiv(1.0f, support);
        const float iso = fmaxd(1.0f * radius, radius);
        const float4 s = a.pos[i];
        const float t2 = a.fc[pc.fluid_mat].t2;
        const bool walk = s.w > kEps && listed;
        // f(neighbor position, weight) per contributing entry of the list
        auto weighed = [&](bool first, auto &&f) {
            each(first, s, t2, [&](const float4 &pj) {
                const float dx = s.x - pj.x, dy = s.y - pj.y, dz = s.z - pj.z;
                const float d2 = dot3(dx, dy, dz, dx, dy, dz);
                if (d2 > 0.0f) {
                    const float dist = fsqrt(d2);
                    if (dist < support) {
                        const float x = dist * inv;
                        f(pj, 1.0f - x * x * x);
                    }
                }
            });
        };
        float mx = 0.0f, my = 0.0f, mz = 0.0f, wsum = 0.0f;
        if (walk)
            weighed(true, [&](const float4 &pj, float w) {
                wsum = wsum + w;
                mx = mx + pj.x * w;
                my = my + pj.y * w;
                mz = mz + pj.z * w;
            });
        if (!(wsum <= 0.0f)) {
            mx = fdiv(mx, wsum);
            my = fdiv(my, wsum);
            mz = fdiv(mz, wsum);
            float C[3][3] = {{0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f}};
            weighed(false, [&](const float4 &pj, float w) {
                const float cc[3] = {pj.x - mx, pj.y - my, pj.z - mz};
#pragma unroll
                for (int r = 0; r < 3; ++r)
#pragma unroll
                    for (int q = 0; q < 3; ++q) C[r][q] = C[r][q] + w * cc[r] * cc[q];
            });
#pragma unroll
            for (int r = 0; r < 3; ++r)
#pragma unroll
                for (int q = 0; q < 3; ++q) C[r][q] = fdiv(C[r][q], wsum);
            C[0][1] = C[1][0] = 0.5f * (C[0][1] + C[1][0]);
            C[0][2] = C[2][0] = 0.5f * (C[0][2] + C[2][0]);
            C[1][2] = C[2][1] = 0.5f * (C[1][2] + C[2][1]);
            // FluidAnisotropyEigenDecomposition, physics_fluid_anisotropy_common.hlsli:76-122
            float R[3][3] = {{1.0f, 0.0f, 0.0f}, {0.0f, 1.0f, 0.0f}, {0.0f, 0.0f, 1.0f}};
            for (int it = 0; it < 4; ++it) {
                int pair = 0;
                float mxv = fabsf(C[0][1]);
                const float a02 = fabsf(C[0][2]);
                if (a02 > mxv) {
                    pair = 1;
                    mxv = a02;
                }
                const float a12 = fabsf(C[1][2]);
                if (a12 > mxv) {
                    pair = 2;
                    mxv = a12;
                }
                if (mxv < 1.0e-15f) break;
                if (pair == 0)
                    jacobi_rotate<0, 1>(C, R);
                else if (pair == 1)
                    jacobi_rotate<0, 2>(C, R);
                else
                    jacobi_rotate<1, 2>(C, R);
            }
            float ev[3] = {fmaxd(C[0][0], 0.0f), fmaxd(C[1][1], 0.0f), fmaxd(C[2][2], 0.0f)};
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const float vx = R[0][k], vy = R[1][k], vz = R[2][k];
                const float l2 = dot3(vx, vy, vz, vx, vy, vz);
                if (l2 > 1.0e-8f) {
                    const float rl = fdiv(1.0f, fsqrt(l2));
                    ax[k][0] = vx * rl;
                    ax[k][1] = vy * rl;
                    ax[k][2] = vz * rl;
                }
            }
            sort_pair<0, 1>(ev, ax);
            sort_pair<0, 2>(ev, ax);
            sort_pair<1, 2>(ev, ax);
#pragma unroll
            for (int k = 0; k < 3; ++k) sc[k] = fmind(fmaxd(fsqrt(ev[k]) * 1.1f, 1.0f * radius), 2.0f * radius);
        } else {
            sc[0] = sc[1] = sc[2] = iso;
        }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) out[k * n + pid] = make_float4(ax[k][0], ax[k][1], ax[k][2], sc[k]);
}

// The same over the run table: the list stored where a list buffer is given, walked again otherwise.
template <bool UNIFORM>
__device__ __forceinline__ void aniso_global(uint32_t i, const FluidArgs &a, const SubstepConsts &c,
                                             const uint32_t *id, float4 *out)
{
    const ParticleClass pc = a.classes[UNIFORM ? 0u : a.cls[i]];
    if (!a.active[pc.scene]) return;
    const bool listed = c.cap > 0 && (!UNIFORM || neighbor_ok(pc, pc));
    aniso_particle(i, pc, id[i], listed, a, c, out, [&](bool first, const float4 &s, float t2, auto &&f) {
        if (!first && a.nbr) {
            const uint32_t cnt = a.nbr_cnt[i];
            for (uint32_t k = 0; k < cnt; ++k) f(a.pos[a.nbr[(size_t)k * c.n + i]]);
            return;
        }
        uint32_t cnt = 0;
        walk_runs(a.cellc[i], run_table(a), c, [&](uint32_t q) {
            if (q == i) return true;
            if (!UNIFORM && !neighbor_ok(pc, a.classes[a.cls[q]])) return true;
            const float4 pj = a.pos[q];
            if (pj.w <= kEps) return true;
            const float dx = s.x - pj.x, dy = s.y - pj.y, dz = s.z - pj.z;
            if (!(dot3(dx, dy, dz, dx, dy, dz) < t2)) return true;
            if (first && a.nbr) a.nbr[(size_t)cnt * c.n + i] = q;
            f(pj);
            return ++cnt < c.cap;
        });
        if (first && a.nbr) a.nbr_cnt[i] = cnt;
    });
}

// FLUID = false: the particles the tiled launch leaves out.
template <bool UNIFORM, bool FLUID>
__global__ __launch_bounds__(kBlock) void k_fluid_render_aniso(FluidArgs a, SubstepConsts c,
                                                               const uint32_t *__restrict__ id,
                                                               float4 *__restrict__ out)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= c.n) return;
    if (!FLUID && a.classes[a.cls[i]].kind == CN_PARTICLE_KIND_FLUID) return;
    aniso_global<UNIFORM>(i, a, c, id, out);
}

// The vorticity and anisotropy passes over the staged halos of the cell blocks, whose cells are the
// substep's: final positions in LDS (with the velocities for the curl, |curl| in w for the
// confinement), the neighbors found there and kept as a list of staged entries, which the confinement
// pass reads again in the same staging.  Walked particle by particle through the run table, every
// candidate cost a dependent load and a branch: 270 us for the curl of 200,000 particles and 207 us for
// the anisotropy, against 79 and 89 us; the confinement (41 us, 38 from a list of slots) only follows
// the curl's list.  What bounds them now: the walk's distance tests (all 27 cells: the passes'
// bound on how far a particle has moved from its cell is not looked at), and in the confinement the latency of a block's
// staging, some two blocks to each workgroup the chip holds.
// Blocks with a halo larger than the tile, or without a descriptor, walk the run table.
constexpr int kPostCurl = 0, kPostConfine = 1, kPostAniso = 2;
template <bool UNIFORM, int PASS>
__global__ __launch_bounds__(kTileBlock) __attribute__((amdgpu_waves_per_eu(kDeltaWaves))) void k_fluid_post_tiled(
    FluidArgs a, SubstepConsts c, float4 *__restrict__ vel, float4 *__restrict__ vort, const uint32_t *__restrict__ id,
    float4 *__restrict__ out)
{
    extern __shared__ float4 dyn[];
    __shared__ uint32_t hoff[kHalo + 1];
    __shared__ uint32_t hstart[kHalo];
    constexpr bool CURL = PASS == kPostCurl, CONFINE = PASS == kPostConfine;
    const uint32_t room = a.tile + kTilePad, tid = threadIdx.x, nblk = a.nblk[1];
    float4 *lpos = dyn;
    float4 *lvel = lpos + room;
    uint32_t *lcls = reinterpret_cast<uint32_t *>(lvel + (CURL ? room : 0u));
    // each die takes a run of consecutive blocks, whose halos overlap
    const uint32_t die = blockIdx.x % kXcds, wgs = (gridDim.x + kXcds - 1u - die) / kXcds;
    const uint32_t per = (nblk + kXcds - 1u) / kXcds, end = min(nblk, per * (die + 1u));
    TileState ts;
    for (uint32_t blk = per * die + blockIdx.x / kXcds; blk < end; blk += wgs) {
        tile_load(ts, blk, hoff, hstart, 0u, a, c);
        __syncthreads();
        if (ts.skip) {
            __syncthreads();
            continue;
        }
        if (!ts.lds) {
            for (uint32_t i = ts.p0 + tid; i < ts.p1; i += kTileBlock) {
                if constexpr (PASS == kPostAniso) {
                    if (a.classes[UNIFORM ? 0u : a.cls[i]].kind == CN_PARTICLE_KIND_FLUID)
                        aniso_global<UNIFORM>(i, a, c, id, out);
                } else {
                    vorticity_global<UNIFORM, CONFINE>(i, a, c, vel, vort);
                }
            }
            __syncthreads();
            continue;
        }
        const uint32_t total = hoff[kHalo], fill = total * kEntryScale, ref = UNIFORM ? 0u : a.cls[ts.p0];
        bool mixed = false;
        float4 lv[kStageCells], le[kStageCells];
        float lw[kStageCells];
        uint32_t lq[kStageCells];
        stage_halo(
            hoff, hstart,
            [&](uint32_t u, uint32_t q) {
                lv[u] = a.pos[q];
                if (CURL) le[u] = vel[q];
                if (CONFINE) lw[u] = vort[q].w;
                if (!UNIFORM) lq[u] = a.cls[q];
            },
            [&](uint32_t u, uint32_t f, uint32_t) {
                // component by component: the arrays stay in registers
                if (CONFINE) {
                    lpos[f] = make_float4(lv[u].x, lv[u].y, lv[u].z, lw[u]);
                } else {
                    const bool far = lv[u].w <= kEps;
                    lpos[f] = make_float4(far ? kFarAway : lv[u].x, far ? kFarAway : lv[u].y, far ? kFarAway : lv[u].z, 0.0f);
                }
                if (CURL) lvel[f] = make_float4(le[u].x, le[u].y, le[u].z, 0.0f);
                if (!UNIFORM) {
                    lcls[f] = lq[u];
                    mixed |= lq[u] != ref;
                }
            });
        if (tid == 0) {  // what the filling entry names
            lpos[total] = make_float4(kFarAway, kFarAway, kFarAway, 0.0f);
            if (CURL) lvel[total] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (!UNIFORM) lcls[total] = ref;
        }
        const int any_mixed = __syncthreads_or(mixed ? 1 : 0);  // also the barrier after staging
        const bool bu = UNIFORM || !any_mixed;
        for (uint32_t i = ts.p0 + tid; i < ts.p1; i += kTileBlock) {
            const ParticleClass pc = a.classes[UNIFORM ? 0u : a.cls[i]];
            if (pc.kind != CN_PARTICLE_KIND_FLUID) continue;
            const bool listed = c.cap > 0 && (!bu || neighbor_ok(pc, pc));
            uint2 *li = list_words(a.list, i, list_rows(c.cap));
            auto find = [&](const float4 &s, float t2) -> uint32_t {
                const int4 ci = a.cellc[i];
                const int hc = halo_cell(ts, ci);
                const uint32_t fs = hoff[hc] + (i - hstart[hc]);
                DensitySelf x;
                x.s = s;
                x.pc = pc;
                RowCull rc = row_cull(s, ci, 0.0f, 0.0f, 3.4e38f);  // every cell
                ListOut lo(li, c.cap);
                if (bu) scan_rows<true>(hoff, hc, fs, lpos, lcls, x, t2, lo, a, rc);
                else scan_rows<false>(hoff, hc, fs, lpos, lcls, x, t2, lo, a, rc);
                return lo.finish(fill);
            };
            uint32_t words = 0;
            auto entries = [&](auto &&f) {
                if (!words) return;
                each_word(li, words, [&](uint2 w) {
                    uint32_t e[4];
                    word_entries(w, e);
#pragma unroll
                    for (uint32_t u = 0; u < 4; ++u) f(e[u]);
                });
            };
            if constexpr (PASS == kPostAniso) {
                aniso_particle(i, pc, id[i], listed, a, c, out, [&](bool first, const float4 &s, float t2, auto &&f) {
                    if (first) words = find(s, t2);
                    entries([&](uint32_t e) { f(at16(lpos, e)); });
                });
            } else {
                vorticity_particle<CONFINE>(i, pc, a, c, vel, vort, [&](const float4 &s, float t2, auto &&term) {
                    if (!listed) return;
                    if (CONFINE) {
                        words = a.lcnt[i];
                    } else {
                        words = find(s, t2);
                        a.lcnt[i] = words;
                    }
                    entries([&](uint32_t e) {
                        const float4 pj = at16(lpos, e);
                        term(bu || a.classes[at4(lcls, e)].fluid_mat == pc.fluid_mat, s.x - pj.x, s.y - pj.y, s.z - pj.z,
                             CONFINE ? pj : at16(lvel, e));
                    });
                });
            }
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------------------------
// launches
// ---------------------------------------------------------------------------------------------
static FluidArgs fluid_args(const SceneBuffers &s, const SubstepConsts &c, uint32_t it, int din)
{
    FluidArgs a;
    const int cur = s.cur;
    a.pos = s.pos[cur];
    a.cls = s.cls[cur];
    a.cellc = s.cellc;
    a.bnd = s.bnd;
    a.bndl = s.bndl;
    a.din = s.dacc[din];
    a.dout = s.dacc[1 - din];
    a.cur = s.curpos;
    a.cs = s.cs;
    a.nc = s.nc;
    a.nbr = s.nbr;
    a.nbr_cnt = s.nbr_cnt;
    a.list = s.list;
    a.lcnt = s.lcnt;
    a.slist = s.slist;
    a.scnt = s.scnt;
    a.run_key = s.run_key;
    a.run_start = s.run_start;
    a.run_info = s.run_info;
    a.run_info_out = s.run_info;
    a.run_count = s.run_count;
    a.bucket = s.bucket;
    a.bucket_shift = c.bucket_shift;
    a.blk_first_run = s.blk_first_run;
    a.nblk = s.nblk;
    a.blk_halo = s.blk_halo;
    a.wide_blk = s.wide_blk;
    a.iter_state = s.iter_state;
    a.classes = s.classes;
    a.fm = s.fluid_mats;
    a.fc = s.fluid_consts;
    a.col = s.colliders;
    a.scenes = s.scenes;
    a.active = s.scene_active;
    a.meta = s.meta;
    a.it = it;
    a.tile = 0;
    a.wide_only = 0;
    return a;
}

static uint32_t grid_of(uint32_t n) { return (n + kBlock - 1) / kBlock; }

// LDS budget of one tiled workgroup (the static halo table and counters take some 2 KiB more).  In a
// large scene three workgroups of the density pass and two of the delta pass share a CU's 160 KiB; a
// scene whose cell blocks leave a CU one or two workgroups (256 and 512 blocks, of some 400 particles in
// a fluid at rest) lets each have what the others would not use, so that fewer blocks need the wide
// layout or the run table.  A scene of few particles in many blocks (a spray, a thin sheet, many small
// scenes) does not: 90,000 particles in 7,000 blocks took 16.9 ms a step with a CU
// to each workgroup, and take 11.5.
static uint32_t lds_budget(const SubstepConsts &c, uint32_t share)
{
    const uint32_t by_n = c.n <= 96u * 1024u ? 1u : (c.n <= 192u * 1024u ? 2u : 3u);
    const uint32_t fits = std::max(by_n, c.blocks <= 256u ? 1u : (c.blocks <= 512u ? 2u : 3u));
    return 156u * 1024u / std::min(share, fits) - 2u * 1024u;
}

static bool tiled(const SubstepConsts &c, uint32_t it) { return c.key_mode == CN_KEY_MORTON && it < kIterStateWords; }

// persistent grid: workgroups in flight on all dies, each pulling cell blocks from the queues
static uint32_t persistent_grid(const SubstepConsts &c)
{
    return std::min<uint32_t>(std::max<uint32_t>(c.grid_max, kXcds), std::max<uint32_t>(kXcds, (c.n + 127u) / 128u));
}

// Halo capacities: the density pass stages positions (and classes, kTilePad spare entries each),
// the delta pass records, previous deltas, normals and classes, the wide delta pass the same
// without previous deltas but with a slot map.  density >= wide >= delta, so every block the delta
// passes stage was staged (and listed in halo offsets) by the density pass.
void fluid_tiles(SubstepConsts &c)
{
    const uint32_t cls = c.fluid_uniform ? 0u : 4u, nc = c.tension ? 16u : 0u, dens = lds_budget(c, 3), lds = lds_budget(c, 2);
    const uint32_t most = std::min<uint32_t>(c.tile_max, kTileMost);
    c.tile_dens = std::min<uint32_t>(most, dens / (16u + cls) - kTilePad);
    c.tile_wide = std::min<uint32_t>(c.tile_dens, lds / (20u + nc + cls) - 1u);
    c.tile_delta = c.viscous ? std::min<uint32_t>(c.tile_wide, lds / (32u + nc + cls) - 1u) : c.tile_wide;
}

void launch_blk_halo(const SceneBuffers &s, const SubstepConsts &c, hipStream_t st)
{
    const FluidArgs a = fluid_args(s, c, 0, 0);
    const uint32_t g = std::min<uint32_t>(std::max<uint32_t>(c.blk_cap, 1u), 4096u);
    hipLaunchKernelGGL(k_blk_halo, dim3(g), dim3(kBlock), 0, st, a, c);
}

// One of a tiled pass's class instantiations: one class in the launch, one per scene with fluid,
// or classes per particle.
template <void (*ONE)(FluidArgs, SubstepConsts), void (*BLOCK)(FluidArgs, SubstepConsts),
          void (*MIXED)(FluidArgs, SubstepConsts)>
static void launch_tiled(const SubstepConsts &c, dim3 grid, dim3 block, size_t lds, hipStream_t st, const FluidArgs &a)
{
    if (c.uniform_class)
        hipLaunchKernelGGL(ONE, grid, block, lds, st, a, c);
    else if (c.fluid_uniform)
        hipLaunchKernelGGL(BLOCK, grid, block, lds, st, a, c);
    else
        hipLaunchKernelGGL(MIXED, grid, block, lds, st, a, c);
}

void launch_fluid_density(const SceneBuffers &s, const SubstepConsts &c, uint32_t it, int din, hipStream_t st)
{
    FluidArgs a = fluid_args(s, c, it, din);
    if (tiled(c, it)) {
        const uint32_t per = 16u + (c.fluid_uniform ? 0u : 4u);
        a.tile = c.tile_dens;
        const size_t lds = (size_t)(a.tile + kTilePad) * per;
        const dim3 grid(persistent_grid(c)), block(kTileBlock);
        if (c.superset && it == 0) {
            launch_tiled<k_fluid_density_tiled<kClsOne, kDensBuild>, k_fluid_density_tiled<kClsBlock, kDensBuild>,
                         k_fluid_density_tiled<kClsMixed, kDensBuild>>(c, grid, block, lds, st, a);
        } else if (c.superset) {
            launch_tiled<k_fluid_density_tiled<kClsOne, kDensReuse>, k_fluid_density_tiled<kClsBlock, kDensReuse>,
                         k_fluid_density_tiled<kClsMixed, kDensReuse>>(c, grid, block, lds, st, a);
        } else {
            launch_tiled<k_fluid_density_tiled<kClsOne, kDensPlain>, k_fluid_density_tiled<kClsBlock, kDensPlain>,
                         k_fluid_density_tiled<kClsMixed, kDensPlain>>(c, grid, block, lds, st, a);
        }
    } else {
        if (c.uniform_class)
            hipLaunchKernelGGL(k_fluid_density_global<true>, dim3(grid_of(c.n)), dim3(kBlock), 0, st, a, c);
        else
            hipLaunchKernelGGL(k_fluid_density_global<false>, dim3(grid_of(c.n)), dim3(kBlock), 0, st, a, c);
    }
}

void launch_fluid_delta(const SceneBuffers &s, const SubstepConsts &c, uint32_t it, int din, hipStream_t st)
{
    FluidArgs a = fluid_args(s, c, it, din);
    if (tiled(c, it)) {
        const uint32_t cls = c.fluid_uniform ? 0u : 4u, nc = c.tension ? 16u : 0u;
        const dim3 grid(persistent_grid(c)), block(kTileBlock);
        // The neighbors' previous deltas are read by the viscosity and CFL terms.  Without a viscous
        // material only the CFL term can want them, which it does in the rare iteration that moved a
        // particle by half its CFL radius: every block takes the wide layout in one launch.
        if (it > 0 && !c.viscous) {
            a.tile = c.tile_wide;
            launch_tiled<k_fluid_delta_tiled<kClsOne, true>, k_fluid_delta_tiled<kClsBlock, true>,
                         k_fluid_delta_tiled<kClsMixed, true>>(c, grid, block, (size_t)(a.tile + 1u) * (20u + nc + cls), st, a);
            return;
        }
        // first iteration: no previous delta, so the delta pass stages as much as the wide one
        a.tile = it > 0 ? c.tile_delta : c.tile_wide;
        size_t lds = (size_t)(a.tile + 1u) * (16u + (it > 0 ? 16u : 0u) + nc + cls);
        launch_tiled<k_fluid_delta_tiled<kClsOne, false>, k_fluid_delta_tiled<kClsBlock, false>,
                     k_fluid_delta_tiled<kClsMixed, false>>(c, grid, block, lds, st, a);
        if (it > 0 && c.tile_wide > c.tile_delta) {
            a.tile = c.tile_wide;
            a.wide_only = 1;
            lds = (size_t)(a.tile + 1u) * (20u + nc + cls);
            launch_tiled<k_fluid_delta_tiled<kClsOne, true>, k_fluid_delta_tiled<kClsBlock, true>,
                         k_fluid_delta_tiled<kClsMixed, true>>(c, grid, block, lds, st, a);
        }
    } else {
        if (c.uniform_class)
            hipLaunchKernelGGL(k_fluid_delta_global<true>, dim3(grid_of(c.n)), dim3(kBlock), 0, st, a, c);
        else
            hipLaunchKernelGGL(k_fluid_delta_global<false>, dim3(grid_of(c.n)), dim3(kBlock), 0, st, a, c);
    }
}

// Halo capacity of the vorticity and anisotropy passes: two workgroups a CU, records of positions and
// velocities (the curl's; the confinement pass has to stage the blocks that the curl pass listed).
static uint32_t post_tile(const SubstepConsts &c)
{
    const uint32_t cls = c.uniform_class ? 0u : 4u;
    return std::min<uint32_t>(std::min<uint32_t>(c.tile_max, kTileMost), lds_budget(c, 2) / (32u + cls) - kTilePad);
}

void launch_fluid_vorticity(const SceneBuffers &s, const SubstepConsts &c, hipStream_t st)
{
    FluidArgs a = fluid_args(s, c, 0, 0);
    float4 *vel = s.vel[s.cur];
    float4 *vort = s.cs;  // free between the last delta pass of a substep and the next density pass
    if (tiled(c, 0)) {
        const uint32_t cls = c.uniform_class ? 0u : 4u;
        a.tile = post_tile(c);
        const size_t lds = (size_t)(a.tile + kTilePad) * (16u + cls), more = (size_t)(a.tile + kTilePad) * 16u;
        const dim3 grid(persistent_grid(c)), block(kTileBlock);
        const uint32_t *id = nullptr;
        float4 *out = nullptr;
        if (c.uniform_class) {
            hipLaunchKernelGGL((k_fluid_post_tiled<true, kPostCurl>), grid, block, lds + more, st, a, c, vel, vort, id, out);
            hipLaunchKernelGGL((k_fluid_post_tiled<true, kPostConfine>), grid, block, lds, st, a, c, vel, vort, id, out);
        } else {
            hipLaunchKernelGGL((k_fluid_post_tiled<false, kPostCurl>), grid, block, lds + more, st, a, c, vel, vort, id, out);
            hipLaunchKernelGGL((k_fluid_post_tiled<false, kPostConfine>), grid, block, lds, st, a, c, vel, vort, id, out);
        }
    } else if (c.uniform_class) {
        hipLaunchKernelGGL((k_fluid_vorticity<true, false>), dim3(grid_of(c.n)), dim3(kBlock), 0, st, a, c, vel, vort);
        hipLaunchKernelGGL((k_fluid_vorticity<true, true>), dim3(grid_of(c.n)), dim3(kBlock), 0, st, a, c, vel, vort);
    } else {
        hipLaunchKernelGGL((k_fluid_vorticity<false, false>), dim3(grid_of(c.n)), dim3(kBlock), 0, st, a, c, vel, vort);
        hipLaunchKernelGGL((k_fluid_vorticity<false, true>), dim3(grid_of(c.n)), dim3(kBlock), 0, st, a, c, vel, vort);
    }
}

void launch_fluid_render_aniso(const SceneBuffers &s, const SubstepConsts &c, float4 *out, hipStream_t st)
{
    FluidArgs a = fluid_args(s, c, 0, 0);
    const uint32_t *id = s.id[s.cur];
    const dim3 each(grid_of(c.n));
    if (tiled(c, 0)) {
        a.tile = post_tile(c);
        const size_t lds = (size_t)(a.tile + kTilePad) * (16u + (c.uniform_class ? 0u : 4u));
        const dim3 grid(persistent_grid(c)), block(kTileBlock);
        float4 *none = nullptr;
        if (c.uniform_class) {
            hipLaunchKernelGGL((k_fluid_post_tiled<true, kPostAniso>), grid, block, lds, st, a, c, none, none, id, out);
        } else {
            hipLaunchKernelGGL((k_fluid_post_tiled<false, kPostAniso>), grid, block, lds, st, a, c, none, none, id, out);
            hipLaunchKernelGGL((k_fluid_render_aniso<false, false>), each, dim3(kBlock), 0, st, a, c, id, out);
        }
    } else if (c.uniform_class) {
        hipLaunchKernelGGL((k_fluid_render_aniso<true, true>), each, dim3(kBlock), 0, st, a, c, id, out);
    } else {
        hipLaunchKernelGGL((k_fluid_render_aniso<false, true>), each, dim3(kBlock), 0, st, a, c, id, out);
    }
}

void launch_fluid_lists(const SceneBuffers &s, const SubstepConsts &c, hipStream_t st)
{
    const FluidArgs a = fluid_args(s, c, 0, 0);
    if (c.uniform_class)
        hipLaunchKernelGGL(k_fluid_lists<true>, dim3(grid_of(c.n)), dim3(kBlock), 0, st, a, c);
    else
        hipLaunchKernelGGL(k_fluid_lists<false>, dim3(grid_of(c.n)), dim3(kBlock), 0, st, a, c);
}

}  // namespace cn
