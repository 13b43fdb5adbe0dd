// Team form of the fused kernels, for large launches whose items touch many streams (an all-reduce reads 8 buffers and
// writes 8, an all-gather reads 1 and writes 8).
//
// The plain fused kernels let every workgroup read a tile and write it straight away, so at any moment each XCD of the
// chip has reads and writes of all its workgroups in flight.  This part moves more bytes when an XCD does one thing at
// a time (measured on MI355X, 8 x 256 MiB read and 8 x 256 MiB written: 5.3 - 5.6 TB/s with reads and writes
// interleaved per workgroup, 5.9 - 6.0 TB/s when the 32 workgroups of an XCD read together and then write together;
// 1 read : 8 writes 4.9 against 5.9 TB/s).  So here the workgroups of one XCD form a team:
//   read phase   every workgroup evaluates up to kTeamTiles tiles (every 32nd tile of the team's region, so an XCD
//                works on one contiguous stretch of the tile space) and parks the results in LDS.  A round is
//                read with all its loads issued together (a copy) or source by source with the
//                partial results in LDS (a chain; a chain of chains), see BySource() below
//   barrier      among the team's workgroups only; the other XCDs run on, in whatever phase they are
//   write phase  every workgroup writes its parked tiles to their destinations, destination by destination
// Workgroup b belongs to XCD b % 8 (workgroups are dealt to the XCDs round robin).  If they are not, or if the team is
// not resident all at once, only the speed changes: nothing passes between workgroups through the barrier, it only
// aligns them in time, every wait is bounded, and after one wait that ran out a team stops waiting for that launch.
//
// The counters live in device memory that starts out zero; the last workgroup of a launch to finish puts them back to
// zero, so the next launch (or a replay of a HIP graph) finds them as the first one did.
#pragma once
#include "kernels_impl.h"

namespace hcclamd {

constexpr uint32_t kTeamVecPerTile = kTileBytes / 16;
constexpr uint64_t kTeamWaitTicks = 20000;                       // 200 us of the 100 MHz clock

// All atomics here are relaxed and at agent scope: they are carried out in memory, beyond the XCDs' separate L2 caches,
// and order nothing else (no data is handed from workgroup to workgroup).
__device__ __forceinline__ uint32_t TeamLoad(const uint32_t *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void TeamStore(uint32_t *p, uint32_t v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t TeamAdd(uint32_t *p, uint32_t v)
{
    return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The team's region for its next round.  Every workgroup of the team asks on its own; whoever comes first to the
// round's slot claims it (0 -> 1), draws the next region from the launch's ticket counter and leaves the answer
// (region + 2) in the slot.  The others wait for that answer: the claimer is running and needs nobody to get there,
// so the wait ends whether or not the rest of the grid is resident.  `seen` is what an earlier look at the slot showed.
__device__ __forceinline__ uint32_t TeamNextRegion(uint32_t *slot, uint32_t *ticket, uint32_t seen)
{
    uint32_t v = seen;
    for (;;) {
        if (v >= 2u) {
            return v - 2u;
        }
        if (v == 0u) {
            // (also reached when the slot was put back to zero under a waiting workgroup: two launches of one prepared
            // collective running at the same time share this block; each region is then still worked on at least once)
            uint32_t expected = 0u;
            if (__hip_atomic_compare_exchange_strong(slot, &expected, 1u, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
                v = TeamAdd(ticket, 1u) + kTeamXcds + 2u;      // regions 0 .. kTeamXcds - 1 are the first round's
                TeamStore(slot, v);
            } else {
                v = expected;
            }
            continue;
        }
        __builtin_amdgcn_s_sleep(2);
        v = TeamLoad(slot);
    }
}

// Arrival at the team's barrier, then (thread 0) the question for the next region while the others arrive, then the
// wait: bounded, and given up for the rest of the launch once it has run out (kTeamGaveUpBit in the arrival word).
// `meanwhile` runs between a workgroup's arrival and its wait.
// Every access here is a trip to memory and back, a few microseconds under load, and whatever the last workgroup to
// arrive does here delays its whole team: it learns from its own arrival that nobody is missing, and it has
// normally seen the next region already (`seen`: a look at the slot taken before its last tile).
template <typename Meanwhile>
__device__ __forceinline__ uint32_t TeamBarrier(uint32_t *c, uint32_t target, uint32_t *slot, uint32_t *ticket, uint32_t seen,
    uint32_t *nextShared, Meanwhile meanwhile)
{
    __syncthreads();
    uint32_t v = 0;
    if (threadIdx.x == 0) {
        v = TeamAdd(c + kTeamArrive, 1u) + 1u;
    }
    meanwhile();
    if (threadIdx.x == 0) {
        *nextShared = TeamNextRegion(slot, ticket, seen);
        if ((v & ~kTeamGaveUpBit) < target && (v & kTeamGaveUpBit) == 0u) {
            const uint64_t t0 = wall_clock64();
            for (;;) {
                v = TeamLoad(c + kTeamArrive);
                if ((v & ~kTeamGaveUpBit) >= target || (v & kTeamGaveUpBit) != 0u) {
                    break;
                }
                if (wall_clock64() - t0 > kTeamWaitTicks) {
                    __hip_atomic_fetch_or(c + kTeamArrive, kTeamGaveUpBit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
            }
        }
    }
    __syncthreads();
    return *nextShared;
}

// The last workgroup of the launch to finish puts every counter and slot back to zero.  Counted in two levels (the last
// of a team reports for the team): atomics on one address are carried out one after the other, a hundred nanoseconds
// and more each, and a whole grid counting on one word is most of a small launch's time.
__device__ __forceinline__ void TeamLeave(uint32_t *teamCtr, uint32_t *ctr, uint32_t teamSize, uint32_t nregions)
{
    __shared__ uint32_t last;
    __syncthreads();
    if (threadIdx.x == 0) {
        last = 0u;
        if (TeamAdd(ctr + kTeamLeft, 1u) + 1u == teamSize) {
            last = TeamAdd(teamCtr + kTeamFinished, 1u) + 1u == kTeamXcds ? 1u : 0u;
        }
    }
    __syncthreads();
    if (last) {       // everybody else is past every barrier and every slot
        uint32_t *slots = teamCtr + kTeamHeaderWords + 2u * nregions;
        for (uint32_t i = threadIdx.x; i < kTeamXcds * (nregions + 1u); i += kBlockThreads) {
            TeamStore(slots + i, 0u);
        }
        if (threadIdx.x < kTeamXcds) {
            TeamStore(teamCtr + threadIdx.x * kTeamCtrStride + kTeamArrive, 0u);
            TeamStore(teamCtr + threadIdx.x * kTeamCtrStride + kTeamLeft, 0u);
        }
        if (threadIdx.x == 0) {
            TeamStore(teamCtr + kTeamTicket, 0u);
            TeamStore(teamCtr + kTeamFinished, 0u);
        }
    }
}

// One parked tile to one destination.
template <uint32_t POLICY>
__device__ __forceinline__ void TeamDrain(const LdsV4 *park, void *o)
{
    const uint32_t tid = threadIdx.x;
    const BufferRsrc r = MakeBuffer(o, kTileBytes);
    V4 w[kVecPerLane];
#pragma unroll
    for (uint32_t u = 0; u < kVecPerLane; u++) {
        w[u] = park[u * kBlockThreads + tid];
    }
#pragma unroll
    for (uint32_t u = 0; u < kVecPerLane; u++) {
        BufferStore16<POLICY>(r, (u * kBlockThreads + tid) * 16u, w[u]);
    }
}

// A workgroup's tiles of one round: every teamSize-th tile of the team's region, so that the team reads, and later writes,
// one stretch of teamSize tiles of every stream at a time instead of teamSize stretches apart (8 ranks x 256 MiB: 1.5 %
// faster).  They may belong to several items.
struct TeamRound {
    const FusedDesc *items;
    uint32_t nitems, tilesPerItem;
    uint32_t first, n, teamSize;
    uint32_t *heldItem;      // LDS: the tiles' items, for the write phase
    uint32_t *peek, *seen;   // thread 0 looks at the slot of the next round once the round's last loads are on their way
    __device__ __forceinline__ uint32_t Tile(uint32_t q) const { return first + q * teamSize; }
    // Item of tile q in d, which holds the item of the tile before it (q > 0).
    __device__ __forceinline__ void Item(uint32_t q, FusedDesc &d, uint32_t &idx, uint32_t &end) const
    {
        const uint32_t tile = Tile(q);
        if (q == 0 || tile >= end) {
            idx = ItemOfTile(items, nitems, tile, tilesPerItem);
            d = items[idx];
            end = d.tile0 + uint32_t(d.bytes / kTileBytes);
        }
        if (threadIdx.x == 0) {
            heldItem[q] = idx;
        }
    }
    __device__ __forceinline__ void Peek() const
    {
        if (threadIdx.x == 0) {
            *seen = TeamLoad(peek);
        }
    }
};

// N tiles from tile q0 of a round on, as the loads by source need them: the first entry of each one's item in the source pool,
// and its offset from the item's pointers.
template <uint32_t N> struct TeamPlaces {
    uint32_t base[N];
    uint64_t off[N];
    uint64_t accLeft[N];
    __device__ __forceinline__ void Find(const TeamRound &r, uint32_t q0, FusedDesc &d, uint32_t &idx, uint32_t &end)
    {
#pragma unroll
        for (uint32_t q = 0; q < N; q++) {
            r.Item(q0 + q, d, idx, end);
            base[q] = d.srcBase;
            off[q] = uint64_t(r.Tile(q0 + q) - d.tile0) * kTileBytes;
            accLeft[q] = d.accLeftMask;
        }
    }
};

// Eval: Read(round, srcPool, extra, park) evaluates the round's tiles and leaves the vectors of tile q at
// park[q * kTeamVecPerTile]; the static Rest(d, ends, srcPool, extra, dstPool) handles an item's rest or its ends there and then.
//
// The whole tiles are cut into regions (first tile, number of tiles), a table the host wrote behind the counters:
// workgroup i of a team of n takes the tiles first + i, first + i + n, ... of the team's region.  Team x starts
// with region x; the later ones are drawn from a counter as the teams get there, and the last regions are smaller,
// so that the XCDs, which do not all move data at the same rate, finish together.
template <typename Eval>
__device__ __forceinline__ void TeamBody(const FusedDesc *__restrict__ items, uint32_t nitems, uint32_t nall, uint32_t nwhole, uint32_t ntiles,
    const void *const *__restrict__ srcPool, void *const *__restrict__ dstPool, uint32_t tilesPerItem,
    uint32_t *__restrict__ teamCtr, const void *extra)
{
    extern __shared__ V4 teamLds[];
    __shared__ uint32_t heldItem[kTeamTiles];
    __shared__ uint32_t nextShared;
    LdsV4 *park = (LdsV4 *)teamLds;

    const uint32_t xcd = blockIdx.x % kTeamXcds, inTeam = blockIdx.x / kTeamXcds, teamSize = gridDim.x / kTeamXcds;
    const uint32_t nregions = teamCtr[kTeamRegionCount];
    const TeamRegion *regions = reinterpret_cast<const TeamRegion *>(teamCtr + kTeamHeaderWords);
    uint32_t *slots = teamCtr + kTeamHeaderWords + 2u * nregions + xcd * (nregions + 1u);
    uint32_t *ctr = teamCtr + xcd * kTeamCtrStride;
    uint32_t nextRest = blockIdx.x;
    auto rests = [&]() __attribute__((always_inline)) {
        for (; nextRest < ntiles - nwhole; nextRest += gridDim.x) {
            const bool ends = nextRest >= nall;
            const FusedDesc d = items[ends ? nextRest - nall : nextRest];
            Eval::Rest(d, ends, srcPool + d.srcBase, extra, dstPool + d.dstBase);
        }
    };
    uint32_t target = 0;
    uint32_t region = xcd;
    for (uint32_t round = 0; region < nregions; round++) {
        const TeamRegion reg = regions[region];
        const uint32_t n = inTeam < reg.count ? (reg.count - 1 - inTeam) / teamSize + 1 : 0;
        uint32_t seen = 0;
        if (n != 0) {
            const TeamRound r = {items, nitems, tilesPerItem, reg.first + inTeam, n, teamSize, heldItem, slots + round, &seen};
            Eval::Read(r, srcPool, extra, park);
        }
        target += teamSize;
        // The items' rests and ends, a few short pieces, cost no time of their own there.  (Every team has a round: the
        // host makes at least kTeamXcds regions.  One call: called twice, this is not inlined.)
        region = TeamBarrier(ctr, target, slots + round, teamCtr + kTeamTicket, seen, &nextShared, rests);
        // Every lane reads back the vectors it parked itself.  A workgroup's tiles mostly belong to one item, so its
        // descriptor and the destination pointer are kept from tile to tile.
        for (uint32_t k = 0, more = n; more != 0; k++) {
            uint32_t cur = ~0u;
            FusedDesc w;
            char *o = nullptr;
            more = 0;
            for (uint32_t q = 0; q < n; q++) {
                const uint32_t item = __builtin_amdgcn_readfirstlane(heldItem[q]);
                if (item != cur) {
                    cur = item;
                    w = items[cur];
                    o = k < w.ndst ? static_cast<char *>(dstPool[w.dstBase + k]) : nullptr;
                    more |= k + 1 < w.ndst ? 1u : 0u;
                }
                if (o == nullptr) {
                    continue;
                }
                char *to = o + uint64_t(reg.first + inTeam + q * teamSize - w.tile0) * kTileBytes;
                if (w.flags & kFusedOrdinaryStores) {
                    TeamDrain<STORE_ORDINARY>(park + q * kTeamVecPerTile, to);
                } else if (w.flags & kFusedNtStores) {
                    TeamDrain<STORE_NT>(park + q * kTeamVecPerTile, to);
                } else {
                    TeamDrain<STORE_STREAMED>(park + q * kTeamVecPerTile, to);
                }
            }
        }
        // the next round's results must not land in LDS before this round's have been read
        __syncthreads();
    }
    TeamLeave(teamCtr, ctr, teamSize, nregions);
}

// ---- what a tile's value is, per kernel family --------------------------------------------------------------------
// A bf16 combine is a dozen instructions per element pair (widen, combine, round); between a set's loads and the next
// request for that set they cost more than the order of the reads gains (8 ranks x 256 MiB, source by source against
// tile by tile: fp32 sum 0.708 / 0.719 ms, int32 0.705 / 0.720, int64 product 0.725 / 0.749, fp16 sum 0.716 / 0.720,
// int8 the same, bf16 sum 0.737 / 0.734, bf16 max 0.762 / 0.753).
template <typename T> struct ReadsBySource { static constexpr bool value = true; };
template <> struct ReadsBySource<Bf16Bits> { static constexpr bool value = false; };

// One register set: N whole tiles of their items' source j.
template <uint32_t N>
__device__ __forceinline__ void TeamLoadSet(V4 (&v)[N][kVecPerLane], const TeamPlaces<N> &at, const void *const *__restrict__ srcPool, uint32_t j)
{
#pragma unroll
    for (uint32_t q = 0; q < N; q++) {
        const char *s = static_cast<const char *>(srcPool[at.base[q] + j]) + at.off[q];
#pragma unroll
        for (uint32_t u = 0; u < kVecPerLane; u++) {
            v[q][u] = Load16<ACC_VEC16_ANY>(s, (u * kBlockThreads + threadIdx.x) * 16u);
        }
    }
}
template <uint32_t U> __device__ __forceinline__ void TeamPark(LdsV4 *park, uint32_t first, const V4 (&x)[U])
{
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
        park[(first + u) * kBlockThreads + threadIdx.x] = x[u];
    }
}

// Tile by tile, from tile q on: tile(d, off, where the values go) for each.
template <typename Tile> __device__ __forceinline__ void TeamByTile(const TeamRound &r, uint32_t q, LdsV4 *park, Tile tile)
{
    FusedDesc d;
    uint32_t idx = 0, end = 0;
    for (; q < r.n; q++) {
        if (q + 1 == r.n) {
            // a look at the slot of the next round, in flight together with the last tile's loads: a workgroup
            // that is behind the others finds the answer there
            r.Peek();
        }
        r.Item(q, d, idx, end);
        tile(d, uint64_t(r.Tile(q) - d.tile0) * kTileBytes, park + q * kTeamVecPerTile);
    }
}

template <typename T, int OP> struct TeamChainEval {
    // Source j into the partial results: source 0 starts them.  A tile's partial results are fetched from LDS together,
    // so that their latencies overlap.
    template <uint32_t N>
    static __device__ __forceinline__ void FoldSet(const V4 (&v)[N][kVecPerLane], const TeamPlaces<N> &at, uint32_t j, LdsV4 *park)
    {
        const uint32_t tid = threadIdx.x;
        if (j == 0) {
#pragma unroll
            for (uint32_t q = 0; q < N; q++) {
                TeamPark(park + q * kTeamVecPerTile, 0, v[q]);
            }
            return;
        }
#pragma unroll
        for (uint32_t q = 0; q < N; q++) {
            V4 a[kVecPerLane];
#pragma unroll
            for (uint32_t u = 0; u < kVecPerLane; u++) {
                a[u] = park[q * kTeamVecPerTile + u * kBlockThreads + tid];
            }
            if (OrderMatters<T, OP>::value && ((at.accLeft[q] >> j) & 1ull)) {      // the same for the whole wave
#pragma unroll
                for (uint32_t u = 0; u < kVecPerLane; u++) {
                    a[u] = Combine16<T, OP>(a[u], v[q][u]);
                }
            } else {
#pragma unroll
                for (uint32_t u = 0; u < kVecPerLane; u++) {
                    a[u] = Combine16<T, OP>(v[q][u], a[u]);
                }
            }
            TeamPark(park + q * kTeamVecPerTile, 0, a);
        }
    }
    // A whole round at once, whichever items its tiles belong to.  The team reads source by source -- at any moment its loads go to one stretch of N x 32 tiles of one buffer instead of 32 tiles of each of
    // the item's buffers -- and the partial results rest in LDS, folded in the chain's order, so the bits are those of
    // the tile-by-tile evaluation.  Two register sets of N x 4 vectors: while one source is folded, the next one's
    // loads are in flight, and the one after that is requested as soon as the fold has freed its set (8 ranks x
    // 256 MiB, stand-alone: 691 us this way, 770 us with one set, 705 us tile by tile).
    // Straight-line code for a source count fixed at compile time, in which every wait is for exactly the loads it
    // needs, measured the same and takes three times as long to build.
    template <uint32_t N>
    static __device__ __forceinline__ void BySource(const TeamRound &r, const void *const *__restrict__ srcPool, LdsV4 *park)
    {
        FusedDesc d;
        uint32_t idx = 0, end = 0;
        TeamPlaces<N> at;
        at.Find(r, 0, d, idx, end);
        const uint32_t nsrc = d.nsrc;
        V4 va[N][kVecPerLane], vb[N][kVecPerLane];
        TeamLoadSet<N>(va, at, srcPool, 0);
        TeamLoadSet<N>(vb, at, srcPool, 1);
        uint32_t j = 0;
#pragma nounroll
        for (; j + 4 <= nsrc; j += 2) {
            FoldSet<N>(va, at, j, park);
            TeamLoadSet<N>(va, at, srcPool, j + 2);
            FoldSet<N>(vb, at, j + 1, park);
            TeamLoadSet<N>(vb, at, srcPool, j + 3);
        }
        // two or three sources left, the first two of them loaded or on their way
        const bool three = nsrc - j == 3;
        FoldSet<N>(va, at, j, park);
        if (three) {
            TeamLoadSet<N>(va, at, srcPool, j + 2);
        }
        r.Peek();
        FoldSet<N>(vb, at, j + 1, park);
        if (three) {
            FoldSet<N>(va, at, j + 2, park);
        }
    }
    static __device__ __forceinline__ void Read(const TeamRound &r, const void *const *__restrict__ srcPool, const void *, LdsV4 *park)
    {
        if constexpr (ReadsBySource<T>::value && sizeof(T) != 1 && !FoldLane<T, OP>::kChecked) {    // (those fold in registers, see FoldLane)
            if (r.n >= kTeamTiles / 2 && (r.items[0].flags & kFusedAlike)) {
                switch (r.n) {
                    case 4: BySource<4>(r, srcPool, park); break;
                    case 5: BySource<5>(r, srcPool, park); break;
                    case 6: BySource<6>(r, srcPool, park); break;
                    case 7: BySource<7>(r, srcPool, park); break;
                    default: BySource<8>(r, srcPool, park); break;
                }
                return;
            }
        }
        // Up to 8 source pointers are kept in registers from tile to tile: fetched per tile they are a chain
        // of dependent loads in front of the tile's data, with nothing else on the CU to hide it.
        const void *sp[8];
        uint32_t held = ~0u;
        uint32_t pos[kChainVec];
        TilePositions(pos);
        TeamByTile(r, 0, park, [&](const FusedDesc &d, uint64_t off, LdsV4 *to) {
            V4 acc[kChainVec];
            if (d.nsrc <= 8) {
                if (d.srcBase != held) {
                    held = d.srcBase;
#pragma unroll
                    for (uint32_t j = 0; j < 8; j++) {
                        sp[j] = srcPool[d.srcBase + j];       // (more lies behind the pool)
                    }
                }
                ChainFew<FoldLane<T, OP>, T, OP, kChainVec>(d.nsrc, d.accLeftMask, sp, off, pos, acc);
            } else {
                ChainMany<typename FoldLane<T, OP>::Exact, T, OP, kChainVec>(d.nsrc, d.accLeftMask, srcPool + d.srcBase, off, pos, acc);
            }
            TeamPark(to, 0, acc);
        });
    }
    static __device__ __forceinline__ void Rest(const FusedDesc &d, bool ends, const void *const *__restrict__ src, const void *, void *const *__restrict__ dst)
    {
        ChainRest<T, OP>(d, ends, src, dst);
    }
};

struct TeamCopyEval {
    // The loads of all tiles are issued before the first of them is parked, instead of tile after tile with an LDS write between them.
    // A full round whose first source lies off a word boundary is fetched in words (WordVec): all-gather of odd blocks of
    // 2-byte elements, us, 128-bit loads / words: 8 ranks x 8 MiB 109.4 / 108.0, 16 MiB 211.7 / 207.9; 16 ranks x 8 MiB 380.7 / 371.2.
    template <uint32_t N, typename L = MoveLane>
    static __device__ __forceinline__ void Together(const TeamRound &r, const void *const *__restrict__ srcPool, LdsV4 *park)
    {
        FusedDesc d;
        uint32_t idx = 0, end = 0;
        TeamPlaces<N> at;
        at.Find(r, 0, d, idx, end);
        typename L::Raw v[N][kVecPerLane];
#pragma unroll
        for (uint32_t q = 0; q < N; q++) {
            const char *s = static_cast<const char *>(srcPool[at.base[q]]) + at.off[q];
#pragma unroll
            for (uint32_t u = 0; u < kVecPerLane; u++) {
                v[q][u] = L::Load(s, (u * kBlockThreads + threadIdx.x) * 16u);
            }
        }
        r.Peek();
#pragma unroll
        for (uint32_t q = 0; q < N; q++) {
            V4 x[kVecPerLane];
#pragma unroll
            for (uint32_t u = 0; u < kVecPerLane; u++) {
                x[u] = L::Value(v[q][u], srcPool[at.base[q]]);
            }
            TeamPark(park + q * kTeamVecPerTile, 0, x);
        }
    }
    static __device__ __forceinline__ void Read(const TeamRound &r, const void *const *__restrict__ srcPool, const void *, LdsV4 *park)
    {
        switch (r.n) {
            case 1: Together<1>(r, srcPool, park); break;
            case 2: Together<2>(r, srcPool, park); break;
            case 3: Together<3>(r, srcPool, park); break;
            case 4: Together<4>(r, srcPool, park); break;
            case 5: Together<5>(r, srcPool, park); break;
            case 6: Together<6>(r, srcPool, park); break;
            case 7: Together<7>(r, srcPool, park); break;
            default:
                if (r.items[ItemOfTile(r.items, r.nitems, r.first, r.tilesPerItem)].flags & kFusedWordSources) {
                    Together<8, WordLane<uint8_t, ROP_SUM>>(r, srcPool, park);
                } else {
                    Together<8>(r, srcPool, park);
                }
                break;
        }
    }
    static __device__ __forceinline__ void Rest(const FusedDesc &d, bool ends, const void *const *__restrict__ src, const void *, void *const *__restrict__ dst)
    {
        CopyRest(d, ends, src[0], dst);
    }
};

template <typename T, int OP> struct TeamTreeEval {
    static __device__ __forceinline__ void Read(const TeamRound &r, const void *const *__restrict__ srcPool, const void *, LdsV4 *park)
    {
        uint32_t pos[kChainVec];
        TilePositions(pos);
        TeamByTile(r, 0, park, [&](const FusedDesc &d, uint64_t off, LdsV4 *to) {
            V4 x[kChainVec];
            TreeValue<VecLane<T, OP>, kChainVec>(d, srcPool + d.srcBase, off, pos, x);
            TeamPark(to, 0, x);
        });
    }
    static __device__ __forceinline__ void Rest(const FusedDesc &d, bool ends, const void *const *__restrict__ src, const void *, void *const *__restrict__ dst)
    {
        TreeRest<T, OP>(d, ends, src, dst);
    }
};

// extra = the launch's op words (they follow the item table)
template <typename T, int OP, bool ROUNDS> struct TeamStackEval {
    // A whole round source by source, as the chain's (TeamChainEval::BySource), for expressions that never hold more than
    // two partial results while a source is being read (a chain of chains: the two-level all-reduce): the lower one in
    // LDS, the upper one in registers.  Three sets of eight tiles are more registers than a wave has, so the round goes
    // in halves of four tiles, through one pipeline: the second half's first sources are requested while the first
    // half's last ones are folded.  Measured (8 ranks, fp32 sum, us, tile by tile / this way): two servers of four, 64 MiB
    // per rank 198.0 / 180.8 (5.4 / 5.9 TB/s), 256 MiB 745 - 755 / 721; the 8-rank ring's chain of 64 MiB takes 176.  What
    // bounds it now is what bounds the chain, the write phase.  Without the piece cut all types but bf16 gain, 64 MiB: fp16
    // 200.6 / 183.7, int8 209.5 / 186.8, int32 199.9 / 183.9, uint64 197.4 / 177.6, fp64 194.0 / 177.4, maximum of fp32 226.4 / 191.9.
    // Its registers cost the tiles that are not read this way: 8-byte types and 8-bit products have a kernel without it
    // (ROUNDS) for launches with few such rounds (exec.cc).
    static constexpr uint32_t kHalf = kTeamTiles / 2;
    typedef V4 Set[kHalf][kVecPerLane];
    static __device__ __forceinline__ void FoldUpper(Set &v, const Set &under, bool underLeft)
    {
#pragma unroll
        for (uint32_t q = 0; q < kHalf; q++) {
#pragma unroll
            for (uint32_t u = 0; u < kVecPerLane; u++) {
                v[q][u] = underLeft ? Combine16<T, OP>(under[q][u], v[q][u]) : Combine16<T, OP>(v[q][u], under[q][u]);
            }
        }
    }
    static __device__ __forceinline__ void FoldLower(Set &v, const LdsV4 *park, bool underLeft)
    {
#pragma unroll
        for (uint32_t q = 0; q < kHalf; q++) {
            V4 a[kVecPerLane];
#pragma unroll
            for (uint32_t u = 0; u < kVecPerLane; u++) {
                a[u] = park[q * kTeamVecPerTile + u * kBlockThreads + threadIdx.x];
            }
#pragma unroll
            for (uint32_t u = 0; u < kVecPerLane; u++) {
                v[q][u] = underLeft ? Combine16<T, OP>(a[u], v[q][u]) : Combine16<T, OP>(v[q][u], a[u]);
            }
        }
    }
    // Pushes a source and folds as its op word says (`depth`: partial results held).
    static __device__ __forceinline__ void Push(Set &v, uint32_t op, Set &upper, LdsV4 *park, uint32_t &depth)
    {
        uint32_t nfold = op & 7u, left = OrderMatters<T, OP>::value ? op >> 8 : ~0u;
        if (depth == 2 && nfold != 0) {
            if (left & 1u) {      // the same for the whole wave
                FoldUpper(v, upper, true);
            } else {
                FoldUpper(v, upper, false);
            }
            left >>= 1;
            nfold--;
            depth = 1;
        }
        if (depth == 1 && nfold != 0) {
            if (left & 1u) {
                FoldLower(v, park, true);
            } else {
                FoldLower(v, park, false);
            }
            depth = 0;
        }
        if (depth == 0) {
#pragma unroll
            for (uint32_t q = 0; q < kHalf; q++) {
#pragma unroll
                for (uint32_t u = 0; u < kVecPerLane; u++) {
                    park[q * kTeamVecPerTile + u * kBlockThreads + threadIdx.x] = v[q][u];
                }
            }
        } else {
#pragma unroll
            for (uint32_t q = 0; q < kHalf; q++) {
#pragma unroll
                for (uint32_t u = 0; u < kVecPerLane; u++) {
                    upper[q][u] = v[q][u];
                }
            }
        }
        depth++;
    }
    // The first four tiles of a round, or all eight: each four of one item (one program), and the same number of sources.
    static __device__ __forceinline__ bool Fits(const TeamRound &r)
    {
        uint32_t nsrc = 0;
        for (uint32_t q = 0; q + kHalf <= r.n && (q == 0 || r.n == kTeamTiles); q += kHalf) {
            const FusedDesc d = r.items[ItemOfTile(r.items, r.nitems, r.Tile(q), r.tilesPerItem)];
            if (d.nsrc < 2 || d.nleaf > 3 || r.Tile(q + kHalf - 1) >= d.tile0 + uint32_t(d.bytes / kTileBytes) || (q != 0 && d.nsrc != nsrc)) {
                return false;
            }
            nsrc = d.nsrc;
        }
        return true;
    }
    template <uint32_t HALVES>
    static __device__ __forceinline__ void BySource(const TeamRound &r, const void *const *__restrict__ srcPool, const uint32_t *__restrict__ opPool,
        LdsV4 *park)
    {
        FusedDesc d;
        uint32_t idx = 0, end = 0;
        TeamPlaces<kHalf> at[HALVES];
        uint32_t ops[HALVES];
#pragma unroll
        for (uint32_t h = 0; h < HALVES; h++) {
            at[h].Find(r, h * kHalf, d, idx, end);
            ops[h] = d.srcBase;
        }
        const uint32_t nsrc = d.nsrc, total = nsrc * HALVES;
        Set va, vb, upper;
        uint32_t depth = 0;
        auto load = [&](Set &v, uint32_t j) {
            if (HALVES == 2 && j >= nsrc) {
                TeamLoadSet<kHalf>(v, at[HALVES - 1], srcPool, j - nsrc);
            } else {
                TeamLoadSet<kHalf>(v, at[0], srcPool, j);
            }
        };
        auto push = [&](Set &v, uint32_t j) {
            const uint32_t half = HALVES == 2 && j >= nsrc ? 1u : 0u;
            depth = j == half * nsrc ? 0u : depth;
            Push(v, opPool[(half != 0 ? ops[HALVES - 1] : ops[0]) + j - half * nsrc], upper, park + half * kHalf * kTeamVecPerTile, depth);
        };
        load(va, 0);
        load(vb, 1);
        uint32_t j = 0;
#pragma nounroll
        for (; j + 4 <= total; j += 2) {
            push(va, j);
            load(va, j + 2);
            push(vb, j + 1);
            load(vb, j + 3);
        }
        // two or three left, the first two of them loaded or on their way
        const bool three = total - j == 3;
        push(va, j);
        if (three) {
            load(va, j + 2);
        }
        r.Peek();
        push(vb, j + 1);
        if (three) {
            push(va, j + 2);
        }
    }
    static __device__ __forceinline__ void Read(const TeamRound &r, const void *const *__restrict__ srcPool, const void *extra, LdsV4 *park)
    {
        const uint32_t *opPool = static_cast<const uint32_t *>(extra);
        uint32_t q = 0;
        if constexpr (ROUNDS && ReadsBySource<T>::value) {
            if (r.n >= kHalf && Fits(r)) {
                if (r.n == kTeamTiles) {
                    BySource<2>(r, srcPool, opPool, park);
                    return;
                }
                BySource<1>(r, srcPool, opPool, park);
                q = kHalf;
            }
        }
        uint32_t pos[kChainVec];
        TilePositions(pos);
        TeamByTile(r, q, park, [&](const FusedDesc &d, uint64_t off, LdsV4 *to) {
            StackTile<T, OP, kStackTeamBatch>(d, srcPool + d.srcBase, opPool + d.srcBase, off, pos,
                [&](uint32_t h, const auto &x) { TeamPark(to, h, x); });
        });
    }
    static __device__ __forceinline__ void Rest(const FusedDesc &d, bool ends, const void *const *__restrict__ src, const void *extra, void *const *__restrict__ dst)
    {
        StackRest<T, OP>(d, ends, src, static_cast<const uint32_t *>(extra) + d.srcBase, dst);
    }
};

// Same tables and arguments as the plain fused kernels, plus the team block (counters, region table, slots; layout in
// kernels.h).  Launched with one workgroup per CU
// (a multiple of kTeamXcds workgroups) and kTeamDynamicLds bytes of dynamic LDS.
template <typename T, int OP>
__global__ void __launch_bounds__(kBlockThreads) TeamChainKernel(const FusedDesc *__restrict__ items, uint32_t nitems, uint32_t nall, uint32_t nwhole,
    uint32_t ntiles, const void *const *__restrict__ srcPool, void *const *__restrict__ dstPool, uint32_t tilesPerItem,
    uint32_t *__restrict__ teamCtr)
{
    TeamBody<TeamChainEval<T, OP>>(items, nitems, nall, nwhole, ntiles, srcPool, dstPool, tilesPerItem, teamCtr, nullptr);
}

template <int Variant>
__global__ void __launch_bounds__(kBlockThreads) TeamCopyKernel(const FusedDesc *__restrict__ items, uint32_t nitems, uint32_t nall, uint32_t nwhole,
    uint32_t ntiles, const void *const *__restrict__ srcPool, void *const *__restrict__ dstPool, uint32_t tilesPerItem,
    uint32_t *__restrict__ teamCtr)
{
    TeamBody<TeamCopyEval>(items, nitems, nall, nwhole, ntiles, srcPool, dstPool, tilesPerItem, teamCtr, nullptr);
}

template <typename T, int OP>
__global__ void __launch_bounds__(kBlockThreads) TeamTreeKernel(const FusedDesc *__restrict__ items, uint32_t nitems, uint32_t nall, uint32_t nwhole,
    uint32_t ntiles, const void *const *__restrict__ srcPool, void *const *__restrict__ dstPool, uint32_t tilesPerItem,
    uint32_t *__restrict__ teamCtr)
{
    TeamBody<TeamTreeEval<T, OP>>(items, nitems, nall, nwhole, ntiles, srcPool, dstPool, tilesPerItem, teamCtr, nullptr);
}

template <typename T, int OP, bool ROUNDS>
__global__ void __launch_bounds__(kBlockThreads) TeamStackKernel(const FusedDesc *__restrict__ items, uint32_t nitems, uint32_t nall, uint32_t nwhole,
    uint32_t ntiles, const void *const *__restrict__ srcPool, void *const *__restrict__ dstPool, uint32_t tilesPerItem,
    uint32_t *__restrict__ teamCtr)
{
    TeamBody<TeamStackEval<T, OP, ROUNDS>>(items, nitems, nall, nwhole, ntiles, srcPool, dstPool, tilesPerItem, teamCtr, items + nall);
}

}  // namespace hcclamd
