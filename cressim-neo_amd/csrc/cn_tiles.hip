// cn_tiles.hip -- host side of the tiled soft-constraint passes: the constrained particles cut into
// spatial tiles, and per tile and constraint group what a workgroup needs to solve every constraint
// that touches one of the tile's particles with its positions and correction records in LDS.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <future>
#include <vector>

#include "cn_internal.h"

namespace cn {

namespace {

// A box of fewer particles, or a run of tiles with fewer constraints, is not worth a thread (some 20 us).
constexpr size_t kAsideParticles = 8192, kAsideEntries = 65536;

// Cuts ids[lo, hi) into ceil((hi - lo) / most) spatially compact tiles of at most `most` particles by
// halving the box along its longest side, whole tiles to each half; sorts each tile and writes the tiles' ends.  The first
// halves of a large box are cut on threads of their own.
void cut(std::vector<uint32_t> &ids, size_t lo, size_t hi, uint32_t most, const float *pos, uint32_t *ends)
{
    const size_t n = hi - lo;
    if (n <= most) {
        std::sort(ids.begin() + lo, ids.begin() + hi);
        *ends = (uint32_t)hi;
        return;
    }
    float mn[3] = {3.4e38f, 3.4e38f, 3.4e38f}, mx[3] = {-3.4e38f, -3.4e38f, -3.4e38f};
    auto at = [&](uint32_t p, int a) {
        const float v = pos[4ull * p + a];
        return std::isfinite(v) ? v : 0.0f;
    };
    for (size_t k = lo; k < hi; ++k)
        for (int a = 0; a < 3; ++a) {
            mn[a] = std::min(mn[a], at(ids[k], a));
            mx[a] = std::max(mx[a], at(ids[k], a));
        }
    int ax = 0;
    for (int a = 1; a < 3; ++a)
        if (mx[a] - mn[a] > mx[ax] - mn[ax]) ax = a;
    const size_t tiles = (n + most - 1) / most, mid = lo + (tiles / 2) * most;
    std::nth_element(ids.begin() + lo, ids.begin() + mid, ids.begin() + hi, [&](uint32_t x, uint32_t y) {
        const float a = at(x, ax), b = at(y, ax);
        return a < b || (a == b && x < y);
    });
    if (n < kAsideParticles) {
        cut(ids, lo, mid, most, pos, ends);
        cut(ids, mid, hi, most, pos, ends + tiles / 2);
    } else {
        std::future<void> half = run_aside([&, lo, mid] { cut(ids, lo, mid, most, pos, ends); });
        cut(ids, mid, hi, most, pos, ends + tiles / 2);
        half.get();
    }
}

constexpr uint32_t kNone = 0xffffffffu;

struct Cut {
    const std::vector<uint32_t> &own;    // the particles, tile by tile
    const std::vector<uint32_t> &first;  // the tiles' first ones, then their number
    const std::vector<uint32_t> &tile_of, &in_tile;
    const uint32_t *pid_scene;
    const std::vector<uint32_t> &stages;
    uint32_t n;
};

// Whether a group's tiles fit a workgroup's LDS; never: one particle's constraints alone do not.
enum class Fit { yes, no, never };

// The tiles of one constraint group.
template <int GROUP>
Fit build_group(const Cut &cut, const SoftTopology &topo, SoftTilesHost::Group &G)
{
    constexpr uint32_t A = GROUP == 0 ? 2u : 4u;
    G = SoftTilesHost::Group{};
    const uint32_t nc = topo.count[GROUP], ntile = (uint32_t)cut.first.size() - 1;
    if (!nc) return Fit::yes;
    // the distinct tiles of a constraint's vertices, the first vertex's first
    auto tiles_of = [&](uint32_t c, uint32_t (&p)[4], uint32_t (&ts)[4]) {
        uint32_t m = 0;
        for (uint32_t k = 0; k < A; ++k) {
            p[k] = topo.vertex(GROUP, c, k);
            if (p[k] == kNone) continue;
            const uint32_t t = cut.tile_of[p[k]];
            bool seen = false;
            for (uint32_t q = 0; q < m; ++q) seen |= ts[q] == t;
            if (!seen) ts[m++] = t;
        }
        return m;
    };
    // a constraint goes to every tile that holds one of its vertices, in constraint order
    std::vector<uint32_t> ent(ntile + 1, 0u), deg(cut.n, 0u);
    uint32_t p[4], ts[4];
    for (uint32_t c = 0; c < nc; ++c) {
        const uint32_t m = tiles_of(c, p, ts);
        for (uint32_t q = 0; q < m; ++q) ++ent[ts[q] + 1];
        for (uint32_t k = 0; k < A; ++k)
            if (p[k] != kNone) ++deg[p[k]];
    }
    {
        // the particle of the most constraints: its records, its position and those of its partners
        const uint32_t hub = (uint32_t)(std::max_element(deg.begin(), deg.end()) - deg.begin());
        const size_t records = deg[hub] * sizeof(CorrRec) + sizeof(float4);
        if (records + (size_t)deg[hub] * (A - 1) * sizeof(float4) > kSoftTileLds) {
            std::vector<uint32_t> partners;
            for (uint32_t c = 0; c < nc; ++c) {
                bool of = false;
                for (uint32_t k = 0; k < A; ++k) of |= topo.vertex(GROUP, c, k) == hub;
                for (uint32_t k = 0; of && k < A; ++k)
                    if (const uint32_t q = topo.vertex(GROUP, c, k); q != kNone && q != hub) partners.push_back(q);
            }
            std::sort(partners.begin(), partners.end());
            partners.erase(std::unique(partners.begin(), partners.end()), partners.end());
            if (records + partners.size() * sizeof(float4) > kSoftTileLds) return Fit::never;
        }
    }
    for (uint32_t t = 0; t < ntile; ++t) ent[t + 1] += ent[t];
    G.con.resize(ent[ntile]);
    G.verts.resize((size_t)ent[ntile] * (A / 2));
    G.slots.resize((size_t)ent[ntile] * (A / 2));
    {
        std::vector<uint32_t> at(ent.begin(), ent.end() - 1);
        for (uint32_t c = 0; c < nc; ++c) {
            const uint32_t m = tiles_of(c, p, ts);
            // the tile of the first vertex owns the constraint: it writes the new lambda
            for (uint32_t q = 0; q < m; ++q) G.con[at[ts[q]]++] = c | (q == 0 ? kTileOwner : 0u);
        }
    }
    // The tiles' entries, in runs of tiles on threads of their own: a particle's cursor belongs to its tile.
    std::vector<uint32_t> cursor(std::move(deg));
    struct Run {
        std::vector<SoftTile> tiles;
        std::vector<uint32_t> halo;
        std::vector<uint16_t> starts;
        uint32_t lds = 0;
        bool fits = true;
    };
    auto fill = [&](uint32_t t0, uint32_t t1) {
        Run R;
        std::vector<uint32_t> stamp(cut.n, kNone), local(cut.n);
        for (uint32_t t = t0; t < t1; ++t) {
            const uint32_t f = cut.first[t], scene = cut.pid_scene[cut.own[f]];
            if (!(cut.stages[scene] & (1u << GROUP))) continue;
            SoftTile d{};
            d.own0 = f;
            d.nown = cut.first[t + 1] - f;
            d.halo0 = (uint32_t)R.halo.size();
            d.ent0 = ent[t];
            d.nent = ent[t + 1] - ent[t];
            d.start0 = (uint32_t)R.starts.size();
            d.scene = scene;
            uint64_t rec = 0;
            for (uint32_t k = 0; k < d.nown; ++k) {  // cursor: a particle's records, then its next one
                const uint32_t q = cut.own[f + k], m = cursor[q];
                R.starts.push_back((uint16_t)std::min<uint64_t>(rec, 0xffffu));
                cursor[q] = (uint32_t)rec;
                rec += m;
            }
            R.starts.push_back((uint16_t)std::min<uint64_t>(rec, 0xffffu));
            R.fits &= rec * sizeof(CorrRec) <= kSoftTileLds;
            if (!R.fits) break;
            d.nrec = (uint32_t)rec;
            for (uint32_t e = d.ent0; e < d.ent0 + d.nent; ++e) {
                const uint32_t c = G.con[e] & ~kTileOwner;
                uint32_t v[4], s[4];
                for (uint32_t k = 0; k < A; ++k) {
                    const uint32_t q = topo.vertex(GROUP, c, k);
                    v[k] = 0;
                    s[k] = kTileNoRec;
                    if (q == kNone) continue;
                    if (cut.tile_of[q] == t) {
                        v[k] = cut.in_tile[q];
                        s[k] = cursor[q]++;
                    } else {
                        if (stamp[q] != t) {
                            stamp[q] = t;
                            local[q] = d.nown + (uint32_t)(R.halo.size() - d.halo0);
                            R.halo.push_back(q);
                        }
                        v[k] = std::min<uint32_t>(local[q], 0xffffu);
                    }
                }
                for (uint32_t k = 0; k < A; k += 2) {
                    G.verts[(size_t)e * (A / 2) + k / 2] = v[k] | (v[k + 1] << 16);
                    G.slots[(size_t)e * (A / 2) + k / 2] = s[k] | (s[k + 1] << 16);
                }
            }
            d.nhalo = (uint32_t)R.halo.size() - d.halo0;
            const size_t bytes = (size_t)(d.nown + d.nhalo) * sizeof(float4) + (size_t)rec * sizeof(CorrRec);
            R.fits &= bytes <= kSoftTileLds;
            if (!R.fits) break;
            R.lds = std::max(R.lds, (uint32_t)bytes);
            R.tiles.push_back(d);
        }
        return R;
    };
    std::vector<std::future<Run>> runs;
    const uint32_t nrun = (uint32_t)std::min<size_t>({4, ntile, ent[ntile] / kAsideEntries + 1});
    for (uint32_t r = 1; r < nrun; ++r)
        runs.push_back(run_aside([&, r] { return fill(ntile * (uint64_t)r / nrun, ntile * (uint64_t)(r + 1) / nrun); }));
    Run R = fill(0, ntile / nrun);
    for (uint32_t r = 0; r < nrun; ++r) {
        if (r) R = runs[r - 1].get();
        for (SoftTile &d : R.tiles) {
            d.halo0 += (uint32_t)G.halo.size();
            d.start0 += (uint32_t)G.starts.size();
        }
        G.tiles.insert(G.tiles.end(), R.tiles.begin(), R.tiles.end());
        G.halo.insert(G.halo.end(), R.halo.begin(), R.halo.end());
        G.starts.insert(G.starts.end(), R.starts.begin(), R.starts.end());
        G.lds = std::max(G.lds, R.lds);
        if (!R.fits) return Fit::no;  // the runs still filling end before this returns
    }
    return Fit::yes;
}

}  // namespace

// False when some particle has more incident constraints than a workgroup's LDS holds.
bool build_soft_tiles(uint32_t n, const float *pos, const std::vector<uint32_t> &soft, const uint32_t *pid_scene,
                      uint32_t nscenes, const SoftTopology &topo, SoftTilesHost &out)
{
    out = SoftTilesHost{};
    out.stages.assign(nscenes, 0u);
    for (int g = 0; g < 3; ++g)
        for (uint32_t c = 0; c < topo.count[g]; ++c) out.stages[pid_scene[topo.vertex(g, c, 0)]] |= 1u << g;
    std::vector<uint32_t> tile_of(n, kNone), in_tile(n), first;
    for (uint32_t most = soft.size() <= kSoftFew ? kSoftTile / 2 : kSoftTile; most >= 8u; most /= 2) {
        // tiles, scene by scene (soft is ascending, and so are its scenes)
        out.own.assign(soft.begin(), soft.end());
        first.assign(1, 0u);
        for (size_t lo = 0; lo < soft.size();) {
            size_t hi = lo;
            while (hi < soft.size() && pid_scene[soft[hi]] == pid_scene[soft[lo]]) ++hi;
            const size_t t = first.size();
            first.resize(t + (hi - lo + most - 1) / most);
            cut(out.own, lo, hi, most, pos, first.data() + t);
            lo = hi;
        }
        for (size_t t = 0; t + 1 < first.size(); ++t) {
            const uint32_t f = first[t], e = first[t + 1];
            for (uint32_t k = f; k < e; ++k) {
                tile_of[out.own[k]] = (uint32_t)t;
                in_tile[out.own[k]] = k - f;
            }
        }
        const Cut c{out.own, first, tile_of, in_tile, pid_scene, out.stages, n};
        // the groups are independent: the edges' and the bends' beside the tets'
        std::future<Fit> e = run_aside([&] { return build_group<0>(c, topo, out.group[0]); });
        std::future<Fit> b = run_aside([&] { return build_group<1>(c, topo, out.group[1]); });
        const Fit fit[3] = {build_group<2>(c, topo, out.group[2]), e.get(), b.get()};
        if (std::count(fit, fit + 3, Fit::yes) == 3) return true;
        if (std::count(fit, fit + 3, Fit::never)) return false;
    }
    return false;
}

}  // namespace cn
