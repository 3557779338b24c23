// cn_internal.h -- declarations shared by the library's translation units (not installed).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <future>
#include <system_error>
#include <vector>

#include "cn_device.h"

namespace cn {

constexpr uint32_t kIterStateWords = 64;  // iterations with tiled fluid passes (later ones walk the run table)
constexpr uint32_t kXcds = 8;             // accelerator dies; each has its own L2 and block-queue counter
// iter_state words: block-queue counters of the density and delta passes (kXcds per iteration,
// each on a 128-byte line of its own: the workgroups of every die pop their blocks with atomics
// at the memory side, which serialise per line), the queue counter of the wide-tile delta pass per
// iteration and the wide-block count (all cleared once per substep), then the largest |delta|^2
// bits of each iteration
constexpr uint32_t kQueueStride = 32;  // words between two block-queue counters
constexpr uint32_t kStateDensity = 0;
constexpr uint32_t kStateDelta = kIterStateWords * kXcds * kQueueStride;
constexpr uint32_t kStateWideQueue = 2 * kIterStateWords * kXcds * kQueueStride;
constexpr uint32_t kStateWideCount = kStateWideQueue + kIterStateWords;
constexpr uint32_t kStateMaxDisp = kStateWideCount + 1;
constexpr uint32_t kStateWords = kStateMaxDisp + kIterStateWords;
// per-block halo descriptor: start slot and exclusive particle offset of each of the 6x6x6 halo
// cells (x fastest), the halo particle total, a purity flag, the block's particle range and the
// cell coordinates of its low corner
constexpr uint32_t kHalo = 216;
constexpr uint32_t kHdStart = 0;
constexpr uint32_t kHdOff = kHalo;              // kHalo + 1 offsets, the last one the total
constexpr uint32_t kHdFlags = 2 * kHalo + 1;
constexpr uint32_t kHdP0 = kHdFlags + 1;
constexpr uint32_t kHdP1 = kHdFlags + 2;
constexpr uint32_t kHdBase = kHdFlags + 3;      // 3 words
constexpr uint32_t kHdScene = kHdFlags + 6;
constexpr uint32_t kHdPairs = kHdFlags + 7;     // 1: a contact pair can exist between particles of the halo
constexpr uint32_t kHdSuper = kHdFlags + 8;     // 1: every particle of the block has its candidate list
constexpr uint32_t kHdFluidOnly = kHdFlags + 9;  // the scene's fluid_only
constexpr uint32_t kHaloStride = 448;
static_assert(kHdFluidOnly < kHaloStride, "the descriptor's words fit its stride");
// kHdFlags value of a block in a scene without fluid particles or contact pairs (no halo written)
constexpr uint32_t kHdNoFluid = 2u;
// candidate contact partners a particle keeps per substep; more are counted as overflows
constexpr uint32_t kContactPartners = 32;
constexpr uint32_t kMetaWords = 16;  // device diagnostics words
// candidate list slots of a fluid particle: its neighbors within h + skin at iteration 0
// (skin = kSkinFrac h), reused by a later iteration of the substep while its own displacement since
// iteration 0 plus the largest one in its block's halo stays below the skin
constexpr uint32_t kSuperSlots = 96;
constexpr float kSkinFrac = 0.05f;
// Per-slot lists of 16-bit entries are stored four to a word, in groups of kListGroup consecutive
// slots: word w of slot i sits (i / kListGroup) * kListGroup * rows entries into the buffer, then
// w * kListGroup + i % kListGroup words on, so one wave's words are 512 consecutive bytes.
constexpr uint32_t kListGroup = 64;
__host__ __device__ inline uint32_t list_rows(uint32_t entries) { return (entries + 3u) & ~3u; }
// byte offset of word 0 of slot i; rows is a multiple of four
__host__ __device__ inline size_t list_word_base(uint32_t i, uint32_t rows)
{
    return (size_t)(i / kListGroup) * kListGroup * rows * sizeof(uint16_t) + (i % kListGroup) * (4 * sizeof(uint16_t));
}
__host__ __device__ inline size_t list_slots(size_t n) { return (n + kListGroup - 1) / kListGroup * kListGroup; }
// entries of a list buffer: the slots' rows, and two words per lane that a list's reader may load
// past the last one
inline size_t list_entries(size_t n, uint32_t entries)
{
    return list_slots(n) * list_rows(entries ? entries : 1u) + 2 * 4 * kListGroup;
}
// Bytes of the entries themselves (slots x entries) that cn_scene_reserve and the candidate lists
// allow a pool: larger workloads are split into pools.
constexpr uint64_t kListBytesMax = 0xffffffffull - 0x100000ull;
// halo particles a list entry can name (a byte offset of 16-byte records), less the filling entry
constexpr uint32_t kTileMost = 4095;
// w of a fluid solver position (SceneBuffers::curpos) that no neighbor list takes: zero inverse mass.
// Otherwise w is D, the bound on the particle's displacement since the substep's first iteration.
constexpr float kNoMass = -1.0f;

// What follows from a fluid material's smoothing radius, computed on the host with the operations
// the kernels would use.
struct FluidConst {
    float t2;     // smallest d^2 whose correctly rounded root is >= h: d2 < t2 <=> sqrt(d2) < h
    float h;      // max(smoothing radius, 1e-4)
    float kw;     // spiky_coef(h)
    float ih;     // 1 / h
    float ts2;    // squared candidate radius, h + skin
    float rs;     // its root
    float allow;  // bound on D_i + D_j under which the candidate lists stay complete
    float pad;
};

// ---- radix sort (cn_sort.hip) ----
constexpr uint32_t kDirectTiles = 128;  // tiles whose counts a scatter workgroup sums itself
size_t sort_scratch_words(uint32_t n);  // for every sort of at most n pairs
uint32_t sort_rounds(uint32_t n);   // a tile holds 256 x rounds pairs
bool sort_one_group(uint32_t n);    // sorted in one launch, without counts
uint2 *radix_sort_pairs(uint2 *buf_a, uint2 *buf_b, uint32_t n, uint32_t key_bits, uint32_t *scratch, bool counted,
                        hipStream_t stream);
void radix_sort_arrays(uint32_t *keys, uint32_t *vals, uint2 *buf_a, uint2 *buf_b, uint32_t n, uint32_t key_bits,
                       uint32_t *scratch, hipStream_t stream);

// Device pointers of one resident scene (single scene or one slot pool).
// Device forms of the soft constraints: the caller's records (cn_soft_edge, cn_soft_bend,
// cn_cloth_dihedral, cn_soft_tet) without their padding, with the compliance and the tet rest volume
// clamped at zero on upload (the solves use only max(value, 0)) and a disabled edge marked by a NaN
// compliance, so a solve reads 16-24 bytes per constraint instead of 32.
struct EdgeDev {
    uint32_t a, b;
    float rest_length, compliance;
};
struct BendDev {
    uint32_t p0, p1, p2;
    float rest_angle, compliance;
};
struct DihedralDev {
    uint32_t e0, e1, o0, o1;
    float rest_angle, compliance;
};
struct TetDev {
    uint32_t p[4];
    float rest_volume, compliance;
};

// One constraint's position correction for one of its vertices (12 bytes: the records are written
// by the constraint solves and summed per vertex, so their size is most of the soft phase's traffic).
struct CorrRec {
    float x, y, z;
};

// ---- tiled soft-constraint passes (cn_tiles.hip, cn_soft.hip) ----
// A tile: up to kSoftTile constrained particles of one scene, close in space.  Per constraint group
// (edges; bends and dihedrals; tets) a workgroup loads the tile's particles and those its constraints
// reach (the halo), solves every constraint that touches one of its particles, and sums its own
// particles' correction records, all in LDS.
// Constrained particles of a tile.  Up to kSoftFew of them tiles of 256 would leave CUs with fewer than
// two, and what a pass takes is a tile's latency: half the particles a tile take a 32^3 tet block from
// 785 to 708 us a step and a 253 x 253 cloth from 767 to 747.  Past that the larger tiles' fewer border
// constraints count: 48 mixed scenes 4,807 against 4,868 us.
constexpr uint32_t kSoftTile = 256, kSoftFew = 2 * 256 * kSoftTile;
constexpr uint32_t kSoftTileLds = 76u * 1024u;  // two workgroups per CU
constexpr uint32_t kTileOwner = 0x80000000u;    // constraint word: this tile writes its lambda
constexpr uint16_t kTileNoRec = 0xffffu;        // record slot of a vertex that is not the tile's own
struct SoftTile {
    uint32_t own0, nown;    // its particles: own[own0 ..), ascending
    uint32_t halo0, nhalo;  // the others it reads: halo[halo0 ..)
    uint32_t ent0, nent;    // its constraints: con / verts / slots
    uint32_t start0, nrec;  // its particles' first records: starts[start0 .. start0 + nown]
    uint32_t scene;
};
struct SoftTilesHost {
    struct Group {
        std::vector<SoftTile> tiles;
        std::vector<uint32_t> con, verts, slots;  // per entry: constraint, arity / 2 words of 16-bit pairs
        std::vector<uint32_t> halo;
        std::vector<uint16_t> starts;
        uint32_t lds = 0;                         // bytes of the largest tile
    };
    std::vector<uint32_t> own;
    std::vector<uint32_t> stages;  // per scene: bit g: it has constraints of group g
    Group group[3];
};
// The constraints of the three groups (bends before dihedrals) and their vertices.
struct SoftTopology {
    const EdgeDev *edges;
    const BendDev *bends;
    const DihedralDev *dihedrals;
    const TetDev *tets;
    uint32_t nb;
    uint32_t count[3];
    uint32_t vertex(int g, uint32_t c, uint32_t k) const
    {
        if (g == 0) return k == 0 ? edges[c].a : edges[c].b;
        if (g == 2) return tets[c].p[k];
        if (c < nb) return k == 0 ? bends[c].p0 : (k == 1 ? bends[c].p1 : (k == 2 ? bends[c].p2 : 0xffffffffu));
        const DihedralDev &d = dihedrals[c - nb];
        return k == 0 ? d.e0 : (k == 1 ? d.e1 : (k == 2 ? d.o0 : d.o1));
    }
};

// f on a thread of its own; when none is to be had, at the time its result is asked for
template <typename F>
auto run_aside(F f) -> std::future<decltype(f())>
{
    try {
        return std::async(std::launch::async, f);
    } catch (const std::system_error &) {
        return std::async(std::launch::deferred, f);
    }
}
bool build_soft_tiles(uint32_t n, const float *pos, const std::vector<uint32_t> &soft, const uint32_t *pid_scene,
                      uint32_t nscenes, const SoftTopology &topo, SoftTilesHost &out);

struct SceneBuffers {
    uint32_t n = 0;                 // slots of the per-slot arrays in use
    uint32_t npid = 0;              // particles of the pool (particle-index arrays hold npid entries)
    // particle state in slot order, double-buffered across the per-substep reorder
    float4 *pos[2] = {nullptr, nullptr};
    float4 *vel[2] = {nullptr, nullptr};
    uint32_t *cls[2] = {nullptr, nullptr};
    uint32_t *id[2] = {nullptr, nullptr};
    int cur = 0;
    float4 *prev[2] = {nullptr, nullptr};  // position before the last predict, in slot order
    int4 *cellc = nullptr;          // cell coordinates of each slot (w unused)
    uint32_t *bnd = nullptr;        // candidate colliders: bitmask over the scene's visit order, or a
                                    // list count (kBndList) with the entries in bndl
    uint16_t *bndl = nullptr;       // kBndListCap candidate colliders per slot (scenes of more than
                                    // kMaskColliders colliders; null when the pool has none)
    // broadphase
    uint2 *kv[2] = {nullptr, nullptr};
    uint32_t *sort_scratch = nullptr;
    uint32_t *elem_run = nullptr;
    uint32_t *run_key = nullptr;
    uint32_t *run_start = nullptr;  // n + 1
    int4 *run_info = nullptr;       // (cx, cy, cz, kRunPure | run_class or 0)
    uint32_t *bucket = nullptr;     // (1 << bucket_bits) + 1
    uint32_t bucket_bits = 0;
    uint2 *tile_counts = nullptr;   // runs and blocks per 1024-key tile (scanned when there are many)
    uint32_t *perm = nullptr;       // slot -> old slot (large scenes)
    uint32_t *run_count = nullptr;  // [0] runs, [1] some cell lies outside its scene's window (kRunWords)
    // fluid solve
    float4 *dacc[2] = {nullptr, nullptr};
    float4 *curpos = nullptr;       // (x* + delta, D or kNoMass): neighbor positions of the walk
    float4 *cs = nullptr;           // (x* + delta, density constraint): neighbor records of the delta pass
    float4 *nc = nullptr;           // surface normal * tension (only with surface tension)
    uint32_t *blk_first_run = nullptr;  // first run of each Morton 4x4x4 block, then the run count
    uint32_t *nblk = nullptr;       // [0] Morton blocks, [1] blocks of scenes with fluid (a prefix)
    uint32_t *blk_halo = nullptr;   // kHaloStride words per block, for the first blk_cap blocks
    uint32_t blk_cap = 0;
    uint32_t *wide_blk = nullptr;   // blocks whose halo fits the wide delta tile only (blk_cap)
    uint32_t *iter_state = nullptr; // kStateWords: block-queue counters and max |delta|^2 per iteration
    FluidConst *fluid_consts = nullptr;  // per fluid material
    uint16_t *list = nullptr;       // fluid neighbor lists as halo offsets, in slot groups
    uint16_t *slist = nullptr;      // candidate lists of iteration 0 as halo offsets, in slot groups
    uint32_t *scnt = nullptr;       // per slot: its staged entry and the words of its candidate list
    // constraint adjacency in particle-index order (pool indices): particle i's adjacent
    // particles are adj_idx[adj_off[i] .. adj_off[i] + adj_cnt[i]); null when no scene has any
    uint32_t *adj_off = nullptr;
    uint32_t *adj_cnt = nullptr;
    uint32_t *adj_idx = nullptr;
    uint32_t *lcnt = nullptr;       // per slot: its staged entry, the list the delta pass walks and its words
    uint32_t *nbr = nullptr;        // neighbor lists of the pass entry, k-major: nbr[k * n + i]
    uint32_t *nbr_cnt = nullptr;
    size_t nbr_alloc = 0;
    uint32_t cap = 0;
    // particle-particle contacts (allocated when the scene has a solid particle)
    uint32_t *ct_list = nullptr;    // candidate partner slots, k-major: ct_list[k * n + i]
    uint32_t *ct_count = nullptr;
    float4 *ct_rec = nullptr;       // (normal, penetration) of each candidate's last contact, k-major
    uint32_t *ct_bits = nullptr;    // bit k: candidate k's last contact is active
    float4 *ct_corr = nullptr;      // summed correction of the last contact pass
    float4 *ct_gen = nullptr;       // position of each solid's last particle-rigid contact generation
    size_t ct_alloc = 0;
    // index-order exports
    float4 *out_pos = nullptr;
    float4 *out_vel = nullptr;
    float4 *out_prev = nullptr;
    float4 *aniso = nullptr;        // render anisotropy: axis1 | axis2 | axis3, n each, particle order
    size_t aniso_alloc = 0;
    // tables
    ParticleClass *classes = nullptr;
    uint32_t nclasses = 0;
    uint32_t fluid_uniform = 0;     // every scene with fluid has one particle class
    cn_fluid_material *fluid_mats = nullptr;
    float4 *part_mats = nullptr;
    Collider *colliders = nullptr;
    uint32_t ncolliders = 0;
    ColGroup *col_groups = nullptr;  // per scene of more than kMaskColliders colliders, from grp0
    SceneInfo *scenes = nullptr;    // one record per scene of the pool
    uint32_t nscenes = 0;
    uint32_t *scene_active = nullptr;  // per scene: 1 = stepped by cn_step, 0 = state left untouched
    uint32_t *pid_scene = nullptr;     // scene of each particle index
    // diagnostics (device): [0] max required neighbors, [1] truncations, [2..3] neighbor total,
    // [4] contact partner overflows, [5] LDS blocks, [6] run-table blocks, [7] max |delta|^2 bits,
    // [8] longest run of equal keys, [9] candidate-list reuses; kMetaWords words
    uint32_t *meta = nullptr;
    // soft constraints
    uint32_t *slot_of = nullptr;
    float4 *posi = nullptr;         // positions of the constrained particles in particle-index order
                                    // during the soft phase of an iteration: two buffers of npid
    uint32_t *soft_ids = nullptr;   // the constrained particles, ascending
    uint32_t *rigid_pick = nullptr; // per constrained particle: its particle-rigid work of the substep
    uint32_t nsoft = 0;
    EdgeDev *edges = nullptr;
    BendDev *bends = nullptr;
    DihedralDev *dihedrals = nullptr;
    TetDev *tets = nullptr;
    uint32_t ne = 0, nb = 0, nd = 0, nt = 0;
    float *lam = nullptr;           // edges | bends + dihedrals | tets
    CorrRec *corr = nullptr;        // correction records of edges | bends + dihedrals | tets, each group
                                    // in its incidence (CSR) order, then one spare record
    size_t corr_off[3] = {0, 0, 0};
    // tiled soft passes (null: some particle has too many constraints for a tile)
    SoftTile *soft_tiles = nullptr;      // the groups' tiles back to back
    uint32_t soft_ntiles[3] = {0, 0, 0}, soft_lds[3] = {0, 0, 0};
    uint32_t *soft_own = nullptr, *soft_halo = nullptr;
    uint16_t *soft_starts = nullptr;
    uint32_t *soft_ent = nullptr;        // con, verts, slots of the three groups
    size_t soft_ent_off[3][3] = {};
    float2 *soft_prm = nullptr;          // (rest value, compliance) of edges | bends + dihedrals | tets
    float *lam2 = nullptr;               // the other buffer of lam: a pass reads one and writes the other
    uint32_t *inc = nullptr;        // three CSR incidence structures back to back, then the record maps
    size_t inc_off[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
};

// ---- broadphase + fluid launches (cn_kernels.hip) ----
constexpr uint32_t kRunWords = 2;
// returns whether the lowest digit's sort counts were taken too
bool launch_keys(const SceneBuffers &s, const SubstepConsts &c, hipStream_t st);
// lookups: the run table will be searched (fluid, or contact candidates)
void launch_runs(SceneBuffers &s, const SubstepConsts &c, const uint2 *sorted, uint32_t key_bits, bool lookups,
                 hipStream_t st);
void launch_reorder(SceneBuffers &s, const SubstepConsts &c, const uint2 *sorted, hipStream_t st);
void fluid_tiles(SubstepConsts &c);
void launch_blk_halo(const SceneBuffers &s, const SubstepConsts &c, hipStream_t st);
void launch_fluid_density(const SceneBuffers &s, const SubstepConsts &c, uint32_t it, int din, hipStream_t st);
void launch_fluid_delta(const SceneBuffers &s, const SubstepConsts &c, uint32_t it, int din, hipStream_t st);
void launch_fluid_lists(const SceneBuffers &s, const SubstepConsts &c, hipStream_t st);
// vorticity confinement on the finalized positions and velocities of the substep
void launch_fluid_vorticity(const SceneBuffers &s, const SubstepConsts &c, hipStream_t st);
// render anisotropy of the finalized positions into out (3 n float4, particle-index order)
void launch_fluid_render_aniso(const SceneBuffers &s, const SubstepConsts &c, float4 *out, hipStream_t st);
void launch_finalize(const SceneBuffers &s, const SubstepConsts &c, int din, hipStream_t st);
void launch_export(const SceneBuffers &s, bool state, bool prev, hipStream_t st);
void launch_set_state(SceneBuffers &s, uint32_t first, uint32_t count, const float4 *P, const float4 *V,
                      hipStream_t st);
void launch_fill(uint32_t *p, uint32_t words, uint32_t value, hipStream_t st);

// ---- particle-particle contacts (cn_contact.hip) ----
void launch_contact_partners(const SceneBuffers &s, const SubstepConsts &c, hipStream_t st);
void launch_contact_iteration(const SceneBuffers &s, const SubstepConsts &c, int din, hipStream_t st);
void launch_contact_velocity(const SceneBuffers &s, const SubstepConsts &c, hipStream_t st);
void launch_rigid_velocity(const SceneBuffers &s, const SubstepConsts &c, uint32_t iters, hipStream_t st);
// the particle-rigid contacts of scenes solved in particle-index order, on the soft phase's positions:
// the substep's choice of work per particle, then (where the last tiled pass does not do it) an
// iteration; solved: soft iterations since the gather (tiled passes; 0 otherwise)
struct RigidPidArgs;
RigidPidArgs rigid_pid_args(const SceneBuffers &s, uint32_t solved);
void launch_rigid_pick(const SceneBuffers &s, const SubstepConsts &c, hipStream_t st);
void launch_rigid_pid(const SceneBuffers &s, const SubstepConsts &c, uint32_t solved, hipStream_t st);
void launch_tick_gather(const SceneBuffers &pool, const SceneBuffers &tick, const uint4 *seg, uint32_t nseg,
                        hipStream_t st);
void launch_tick_scatter(const SceneBuffers &pool, const SceneBuffers &tick, const uint4 *seg, uint32_t nseg,
                         hipStream_t st);

// ---- XPBD soft constraints (cn_soft.hip) ----
struct SoftArgs {
    float4 *pos;               // slot order
    float4 *posi;              // particle-index order (constrained particles) while the soft passes run
    const uint32_t *soft_ids;  // constrained particles
    uint32_t nsoft;
    const uint32_t *slot_of;   // particle index -> slot
    const uint32_t *id;        // slot -> particle index
    uint32_t n;
    float dt, relax;
    const EdgeDev *edges;
    uint32_t ne;
    float *lam_e;
    CorrRec *corr_e;           // correction records in incidence order
    const uint32_t *map_e;     // 2 per edge: the position of its vertex records in corr_e
    const BendDev *bends;
    uint32_t nb;
    const DihedralDev *dih;
    uint32_t nd;
    float *lam_b;              // bends then dihedrals
    CorrRec *corr_b;
    const uint32_t *map_b;     // 4 per bend / dihedral (a bend's fourth is the spare record)
    const TetDev *tets;
    uint32_t nt;
    float *lam_t;
    CorrRec *corr_t;
    const uint32_t *map_t;     // 4 per tet
    const uint32_t *inc_e_start;  // incidence ranges: a particle's records are corr_x[start[p], start[p + 1])
    const uint32_t *inc_b_start;
    const uint32_t *inc_t_start;
    const uint32_t *active;    // per scene
    const uint32_t *pid_scene; // particle index -> scene
    const SceneInfo *scenes;
    // tiled passes: a scene's positions alternate between two buffers of n, one step per group it has
    // constraints of; solved counts the iterations since the gather
    const SoftTile *tiles;     // null: the passes over the whole pool
    uint32_t ntiles[3], lds[3];
    const uint32_t *own, *halo;
    const uint16_t *starts;
    const uint32_t *con[3], *verts[3], *slots[3];
    const float2 *prm[3];
    float *lam_in[3], *lam_out[3];
    uint32_t keep_tets;        // the last iteration of a step: every tet's records go to corr_t
    uint32_t solved;
    uint32_t all_live;         // every scene takes part in the step (no per-particle check)
    uint32_t first;            // first iteration of a substep: every lambda starts at zero (read as
                               // zero, and written by every constraint, also where it does nothing)
};
// gather / scatter: copy the constrained particles' positions from slot order before the solves and
// back after them (needed only around iterations where another pass moves those particles)
// solve = false: only the gather and / or the scatter
void launch_soft_iteration(SoftArgs &a, const SceneBuffers &s, const SubstepConsts &c, bool rigid, bool gather, bool scatter, bool solve, hipStream_t st);

// per-pass entries in the reference's data order (cn_passes.hip)
void launch_ref_keys(const float4 *pos, uint32_t n, float inv_cell, uint32_t *keys, int32_t *cells,
                     hipStream_t st);
void launch_ref_cell_ranges(const uint32_t *sorted_keys, uint32_t n, uint32_t capacity, uint32_t *ranges,
                            hipStream_t st);

}  // namespace cn
