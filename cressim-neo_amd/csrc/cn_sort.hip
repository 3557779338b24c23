// cn_sort.hip -- stable LSD radix sort of (key, value) uint32 pairs for gfx950.
//
// Replaces the reference's 32-pass one-bit split sort (physics_pass_dispatcher.cpp:3963-4063,
// physics_radix_{classify,finalize,scatter}.cs.hlsl) with 8-bit digits: per digit pass a histogram per
// tile (LDS atomics), the tiles' bases, and a scatter whose waves rank their own items with wave64
// ballots.  Any stable LSD sort yields the same order as the reference's stable one-bit sort, so keys
// and permutation are bit-identical to it.
//
// What bounds it: launches and latency below some 100,000 pairs, the scattered 8-byte stores above.
//   - at most kOneGroup pairs: every pass in one workgroup's LDS, one launch
//   - few tiles (kDirectTiles): a scatter workgroup sums the tiles' counts itself, two launches a
//     pass, with tiles of 1,024 pairs so that small sorts still spread over the chip
//   - more: a row scan per digit between the two, tiles of 2,048 and then 4,096 pairs (sort_rounds)
// A wave ranks its items against its own counters, so a tile takes three workgroup barriers whatever
// its rounds (with counters of the workgroup it took three per round of 256 items: 16.1 us a pass
// over 1,000,003 pairs).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "cn_internal.h"

namespace cn {

constexpr int kSortThreads = 256;
constexpr int kSortWaves = kSortThreads / 64;
constexpr uint32_t kOneGroup = 4096;
constexpr int kOneThreads = 1024;

// Pairs as records, or as two arrays (the caller's of the pair entry points).
struct PairIn {
    const uint2 *kv;
    const uint32_t *keys, *vals;  // used when kv is null
    __device__ __forceinline__ uint32_t key(uint32_t i) const { return kv ? kv[i].x : keys[i]; }
    __device__ __forceinline__ uint2 get(uint32_t i) const { return kv ? kv[i] : make_uint2(keys[i], vals[i]); }
};
struct PairOut {
    uint2 *kv;
    uint32_t *keys, *vals;
    __device__ __forceinline__ void put(uint32_t i, uint2 p) const
    {
        if (kv) {
            kv[i] = p;
        } else {
            keys[i] = p.x;
            vals[i] = p.y;
        }
    }
};

// Rounds of a tile: small tiles while their counts are summed directly, and in larger sorts as many
// as leave every CU a few workgroups (a wave's ranks are a serial chain, some 300 ns a round).  The keys
// and three passes over 2,500,000 particles take 99 us with 8 rounds and 106 with 16, over 4,194,304 141
// either way, over 8,000,000 251 and 246.
// The tiles grow at these sizes, so their number falls there: sort_scratch_words looks at both.
constexpr uint32_t kRoundsFour = 1024u * kDirectTiles, kRoundsEight = 4u * 1024u * 1024u;
uint32_t sort_rounds(uint32_t n)
{
    return n <= kRoundsFour ? 4u : (n <= kRoundsEight ? 8u : 16u);
}
static uint32_t sort_tiles(uint32_t n)
{
    const uint32_t tile = kSortThreads * sort_rounds(n);
    return (n + tile - 1) / tile;
}
bool sort_one_group(uint32_t n) { return n <= kOneGroup; }

// Words of the counts: [tile][digit] when the scatter sums them (direct), [digit][tile] for the row scan.
template <int R>
__global__ __launch_bounds__(kSortThreads) void k_radix_hist(PairIn in, uint32_t n, uint32_t shift, uint32_t nb,
                                                             uint32_t direct, uint32_t *__restrict__ counts)
{
    __shared__ uint32_t hist[256];
    const uint32_t t = threadIdx.x, b = blockIdx.x;
    const uint32_t base = b * (kSortThreads * R);
    uint32_t d[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t e = base + r * kSortThreads + t;
        d[r] = e < n ? (in.key(e) >> shift) & 0xffu : kInvalid;
    }
    hist[t] = 0;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r)
        if (d[r] != kInvalid) atomicAdd(&hist[d[r]], 1u);
    __syncthreads();
    counts[direct ? b * 256u + t : t * nb + b] = hist[t];
}

// One workgroup per digit: exclusive scan of the digit's row of per-tile counts, row total out.
__global__ __launch_bounds__(kSortThreads) void k_radix_rowscan(uint32_t *__restrict__ counts, uint32_t nb,
                                                                uint32_t *__restrict__ totals)
{
    __shared__ uint32_t sh[kSortWaves];
    const uint32_t d = blockIdx.x;
    const uint32_t t = threadIdx.x;
    uint32_t *row = counts + (size_t)d * nb;
    uint32_t carry = 0;
    for (uint32_t c0 = 0; c0 < nb; c0 += kSortThreads * 4) {
        uint32_t v[4];
        uint32_t local = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t idx = c0 + t * 4 + k;
            v[k] = idx < nb ? row[idx] : 0u;
            local += v[k];
        }
        uint32_t total;
        uint32_t run = carry + block_exclusive_scan(local, sh, total);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t idx = c0 + t * 4 + k;
            if (idx < nb) row[idx] = run;
            run += v[k];
        }
        carry += total;
    }
    if (t == 0) totals[d] = carry;
}

// The lanes of the wave that hold digit d, among the valid ones.
__device__ __forceinline__ uint64_t digit_peers(uint32_t d, bool valid)
{
    uint64_t match = __ballot(valid);
#pragma unroll
    for (int bit = 0; bit < 8; ++bit) {
        const bool on = (d >> bit) & 1u;
        const uint64_t bal = __ballot(on);
        match &= on ? bal : ~bal;
    }
    return match;
}

// Ranks one item per lane among the wave's items of its digit so far: cnt, the wave's counters.
__device__ __forceinline__ uint32_t wave_rank(uint32_t d, bool valid, uint32_t lane, uint32_t *cnt)
{
    const uint64_t peers = digit_peers(d, valid);
    const uint32_t before = (uint32_t)__popcll(peers & ((1ull << lane) - 1ull));
    const uint32_t first = valid ? cnt[d] : 0u;
    // every peer has read the counter before the first of them advances it (LDS operations of a wave
    // complete in order; the fences keep the compiler to it)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (valid && before == 0u) cnt[d] = first + (uint32_t)__popcll(peers);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    return first + before;
}

template <int R>
__global__ __launch_bounds__(kSortThreads) void k_radix_scatter(PairIn in, PairOut out, uint32_t n, uint32_t shift,
                                                                uint32_t nb, uint32_t direct,
                                                                const uint32_t *__restrict__ counts,
                                                                const uint32_t *__restrict__ totals)
{
    __shared__ uint32_t cnt[kSortWaves][256];
    __shared__ uint32_t sh[kSortWaves];
    const uint32_t t = threadIdx.x, b = blockIdx.x;
    const uint32_t lane = t & 63u, wave = t >> 6;
    // a wave's items are one contiguous stretch of the tile: tile order is wave, round, lane
    const uint32_t first = b * (kSortThreads * R) + wave * (64u * R);
    uint2 items[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t e = first + r * 64u + lane;
        items[r] = e < n ? in.get(e) : make_uint2(0u, 0u);
    }
    // digit t's pairs in all tiles and in the tiles before this one
    uint32_t total = 0, before = 0;
    if (direct) {
#pragma unroll 8
        for (uint32_t k = 0; k < nb; ++k) {
            const uint32_t v = counts[k * 256u + t];
            total += v;
            before += k < b ? v : 0u;
        }
    } else {
        total = totals[t];
        before = counts[t * nb + b];
    }
#pragma unroll
    for (int w = 0; w < kSortWaves; ++w) cnt[w][t] = 0;
    uint32_t all;
    const uint32_t base = block_exclusive_scan(total, sh, all) + before;  // also the barrier after clearing
    uint32_t rank[R];
#pragma unroll
    for (int r = 0; r < R; ++r)
        rank[r] = wave_rank((items[r].x >> shift) & 0xffu, first + r * 64u + lane < n, lane, cnt[wave]);
    __syncthreads();
    {
        uint32_t run = base;
#pragma unroll
        for (int w = 0; w < kSortWaves; ++w) {
            const uint32_t c = cnt[w][t];
            cnt[w][t] = run;
            run += c;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r)
        if (first + r * 64u + lane < n) out.put(cnt[wave][(items[r].x >> shift) & 0xffu] + rank[r], items[r]);
}

// Every pass over at most kOneGroup pairs in one workgroup: ranks as above, the pairs exchanged through LDS.
__global__ __launch_bounds__(kOneThreads) void k_radix_one_group(PairIn in, PairOut out, uint32_t n, uint32_t key_bits)
{
    constexpr int R = kOneGroup / kOneThreads, W = kOneThreads / 64;
    __shared__ uint32_t cnt[W][256];
    __shared__ uint32_t sh[W];
    __shared__ uint2 pairs[kOneGroup];
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    const uint32_t first = wave * (64u * R);
    uint2 items[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t e = first + r * 64u + lane;
        items[r] = e < n ? in.get(e) : make_uint2(0u, 0u);
    }
    for (uint32_t shift = 0; shift < key_bits; shift += 8) {
        for (uint32_t k = t; k < W * 256u; k += kOneThreads) (&cnt[0][0])[k] = 0;
        __syncthreads();
        uint32_t rank[R];
#pragma unroll
        for (int r = 0; r < R; ++r)
            rank[r] = wave_rank((items[r].x >> shift) & 0xffu, first + r * 64u + lane < n, lane, cnt[wave]);
        __syncthreads();
        uint32_t total = 0;
        if (t < 256)
#pragma unroll
            for (int w = 0; w < W; ++w) total += cnt[w][t];
        uint32_t all, run = block_exclusive_scan_wide<kOneThreads>(total, sh, all);
        if (t < 256)
#pragma unroll
            for (int w = 0; w < W; ++w) {
                const uint32_t c = cnt[w][t];
                cnt[w][t] = run;
                run += c;
            }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (first + r * 64u + lane < n) pairs[cnt[wave][(items[r].x >> shift) & 0xffu] + rank[r]] = items[r];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const uint32_t e = first + r * 64u + lane;
            if (e < n) items[r] = pairs[e];
        }
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t e = first + r * 64u + lane;
        if (e < n) out.put(e, items[r]);
    }
}

// Scratch words of every sort of at most n pairs: a smaller sort has more tiles than n's where n lies
// past a size at which the tiles grow (4,000,000 pairs have 1,954, 5,000,000 have 1,221).
size_t sort_scratch_words(uint32_t n)
{
    uint32_t tiles = sort_tiles(n);
    for (uint32_t most : {kRoundsFour, kRoundsEight}) tiles = std::max(tiles, sort_tiles(std::min(n, most)));
    return (size_t)256 * tiles + 256;
}

template <int R>
static void radix_pass(const PairIn &in, const PairOut &out, uint32_t n, uint32_t shift, uint32_t *scratch, bool counted,
                       hipStream_t stream)
{
    const uint32_t nb = (n + kSortThreads * R - 1) / (kSortThreads * R);
    const uint32_t direct = nb <= kDirectTiles ? 1u : 0u;
    uint32_t *totals = scratch + (size_t)256 * nb;
    if (!counted)
        hipLaunchKernelGGL(k_radix_hist<R>, dim3(nb), dim3(kSortThreads), 0, stream, in, n, shift, nb, direct, scratch);
    if (!direct) hipLaunchKernelGGL(k_radix_rowscan, dim3(256), dim3(kSortThreads), 0, stream, scratch, nb, totals);
    hipLaunchKernelGGL(k_radix_scatter<R>, dim3(nb), dim3(kSortThreads), 0, stream, in, out, n, shift, nb, direct, scratch,
                       totals);
}

// Sorts by the low key_bits of the keys; passes alternate between a and b, the first reads `in`, the
// last writes `last` when that is given.  Returns where the result is.
static uint2 *sort_passes(PairIn in, uint2 *a, uint2 *b, const PairOut *last, uint32_t n, uint32_t key_bits,
                          uint32_t *scratch, bool counted, hipStream_t stream)
{
    if (sort_one_group(n)) {
        hipLaunchKernelGGL(k_radix_one_group, dim3(1), dim3(kOneThreads), 0, stream, in,
                           last ? *last : PairOut{b, nullptr, nullptr}, n, key_bits);
        return b;
    }
    const uint32_t rounds = sort_rounds(n);
    uint2 *dst = b;
    for (uint32_t shift = 0; shift < key_bits; shift += 8) {
        const bool end = shift + 8 >= key_bits;
        const PairOut out = end && last ? *last : PairOut{dst, nullptr, nullptr};
        const bool have = counted && shift == 0;
        if (rounds == 4u) radix_pass<4>(in, out, n, shift, scratch, have, stream);
        else if (rounds == 8u) radix_pass<8>(in, out, n, shift, scratch, have, stream);
        else radix_pass<16>(in, out, n, shift, scratch, have, stream);
        in = PairIn{dst, nullptr, nullptr};
        dst = dst == b ? a : b;
    }
    return const_cast<uint2 *>(in.kv);
}

// Sorts n pairs by the low key_bits of .x, stably.  buf_a holds the input; the result ends in
// the returned buffer (buf_a or buf_b).  scratch needs sort_scratch_words(n) uint32 words.  counted: the
// lowest digit's counts are in scratch already (SortCounts).
uint2 *radix_sort_pairs(uint2 *buf_a, uint2 *buf_b, uint32_t n, uint32_t key_bits, uint32_t *scratch, bool counted,
                        hipStream_t stream)
{
    if (n <= 1) return buf_a;
    return sort_passes(PairIn{buf_a, nullptr, nullptr}, buf_a, buf_b, nullptr, n, key_bits, scratch, counted, stream);
}

// The same over two separate arrays in place: the first pass reads them, the last one writes them.
void radix_sort_arrays(uint32_t *keys, uint32_t *vals, uint2 *buf_a, uint2 *buf_b, uint32_t n, uint32_t key_bits,
                       uint32_t *scratch, hipStream_t stream)
{
    if (n <= 1) return;
    const PairOut last{nullptr, keys, vals};
    sort_passes(PairIn{nullptr, keys, vals}, buf_a, buf_b, &last, n, key_bits, scratch, false, stream);
}

}  // namespace cn
