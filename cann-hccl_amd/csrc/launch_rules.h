// Rules of the executor on sizes and alignment: how a stretch of bytes is cut, which tiles the teams take, how results
// are stored.  Pure C++: no HIP calls, so the rules can be checked without a GPU.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <vector>

#include "kernels.h"

namespace hcclamd {

// Which pointers a stretch's head brings to a 16-byte boundary.
enum AnchorRule : int {
    ANCHOR_FIRST = 0,   // the first one, the destination: the step kernel's vector stores are aligned ones, and what a step
                        // stores the next one reads (ring reduce-scatter step by step, 8 ranks, bf16, sends 2 bytes off, us,
                        // this way / the largest group: 2 MiB 25.4 / 26.3, 8 MiB 44.5 / 45.9, sends and results off 26.9 / 27.8)
    ANCHOR_MOST = 1     // the largest group that agrees (of two equal ones the one with the first pointer): a fused
                        // reduce-scatter of odd blocks reads all its sources aligned and writes its one destination unaligned
};

// A stretch of bytes cut into an element-wise head, a 16-byte vector body and an element-wise tail.
struct Cut {
    uint64_t head, body, tail;
    bool aligned;          // every pointer is on a 16-byte boundary where the body starts
};

// Cuts [0, bytes), given the addresses involved (the first one is a destination; all are multiples of the element size).
// The head brings the anchor's pointers to a 16-byte boundary; those that are then not on one
// too are accessed with unaligned 128-bit accesses.
// The head of a long stretch reaches to a 128-byte boundary of those pointers:
// a wave stores 1 KiB at a time, and when those stores straddle memory lines every line is written in
// two pieces (measured, 8-rank fp32 all-reduce of 256 MiB per rank with all buffers 16 bytes off a
// 128-byte boundary: 0.97 ms fused against 0.76 ms aligned).
inline Cut CutByAlignment(const std::vector<uintptr_t> &addrs, uint64_t bytes, AnchorRule rule)
{
    size_t count[16] = {0};
    for (uintptr_t a : addrs) {
        count[a & 15]++;
    }
    uintptr_t anchor = addrs[0];
    for (uintptr_t a : addrs) {
        anchor = rule == ANCHOR_MOST && count[a & 15] > count[anchor & 15] ? a : anchor;
    }
    const uint64_t align = bytes >= 4 * uint64_t(kTileBytes) + 128 ? 128 : 16;
    const uint64_t head = std::min<uint64_t>(bytes, (align - (anchor & (align - 1))) & (align - 1));
    const uint64_t body = (bytes - head) & ~uint64_t(15);
    return Cut{head, body, bytes - head - body, count[anchor & 15] == addrs.size()};
}

// The team kernels are chosen for launches of at least this many halves of a round of whole tiles.  All-reduce, us, plain / team: 8 ranks,
// fp32, 12 MiB (768 tiles) 36.0 / 36.6, 16 MiB (1024, half a round) 49.5 / 46.2, 24 MiB 72.4 / 68.2, 32 MiB 96.3 / 88.0, 48 MiB 145.4 /
// 137.3; 32 ranks, bf16 halving-doubling (a round is 1024 tiles), 4 MiB (256) 45.3 / 46.6, 8 MiB (512) 95.1 / 87.8, 16 MiB 209 / 172.5.
constexpr uint32_t kTeamMinHalfRounds = 1;
// Items with fewer than 12 sources and destinations (4 ranks, fp32): 16 MiB 24.3 / 26.1, 32 MiB (a round) 48.0 / 47.4, 48 MiB 70.5 / 74.8,
// 64 MiB 93.6 / 95.1, 128 MiB (4 rounds) 188.5 / 183.3.
constexpr uint32_t kTeamMinHalfRoundsFew = 8;
// One source and many destinations, all-gather: 8 ranks 3 MiB (1536 tiles) 29.2 / 39.4, 4 MiB (2048, a round) 41.6 / 52.0, 5 MiB 64.5 / 68.4,
// 2 bytes off a boundary 71.7 / 69.9, 6 MiB 86.4 / 79.8, 8 MiB 120.9 / 105.5; 16 ranks 1 MiB (1024) 38.5 / 52.5, 2 MiB 104.6 / 99.0; 9 ranks 4 MiB 66.8 /
// 67.6.  (The line was drawn when the plain kernel's results were not written through, 4 MiB 60.0 / 54.2; between a round and
// the memory-side cache's size the plain form is now the faster one.)
constexpr uint32_t kTeamMinHalfRoundsCopy = 2;
// One source and 4 to 6 destinations: items on whole 128-byte lines (they have neither head nor tail) / others.  Few streams suffer less from one another, so the team's order pays
// later; but its time hardly depends on where the buffers lie, while the plain form's does (three sets of buffers in turn, plain with eight workgroups per CU /
// team, several placements; rounds): 4 ranks 16 MiB (2) 62 / 65, 32 MiB (4) 122 ... 131 / 118, 40 MiB 144 / 144, 48 MiB 166 ... 191 / 171 ... 173, 64 MiB (8) 255 / 226,
// 128 MiB (16) 487 / 440; 5 ranks 16 MiB (2.5) 86.9 / 89.3, 27 MiB (4.2) 150 ... 166 / 145, 60 MiB 329 ... 339 / 307; 6 ranks 16 MiB (3) 115 ... 121 / 120, 22 MiB
// (4.1) 166 / 159, 55 MiB 404 / 382.  Off a boundary: 4 ranks 26 MiB 91 ... 94 / 102, 40 MiB (5) 147 / 154, 64 MiB (8) 245 ... 255 / 243, 80 MiB 287 / 299, 100 MiB
// 389 / 374; 5 ranks 40 MiB (6.25) 206 ... 231 / 217 ... 220, 60 MiB (9.4) 314 / 320; 6 ranks 24 MiB (4.5) 183 / 184, 30 MiB 215 / 225, 40 MiB (7.5) 311 / 301.
// Broadcasts, whose one item is read from one buffer, gain more from the same lines on (plain / team, three sets of buffers and every rank as the root in turn): 5 ranks 128 MiB
// (4) 129.2 / 116.2, 256 MiB 267 / 219, 600 MiB 635 / 497; 6 ranks 160.0 / 135.2, 322 / 259, 760 / 588; 7 ranks 188.2 / 154.8, 382 / 298, 893 / 684; off a boundary, 256 MiB (8)
// 5 ranks 267 / 221, 6 ranks 321 / 261, 7 ranks 384 / 301.
constexpr uint32_t kTeamMinHalfRoundsCopyFew = 8, kTeamMinHalfRoundsCopyFewUneven = 16;

// Whether a launch whose items with whole tiles have `bytes` in all runs that long.  (By bytes, not by tiles: a buffer that starts
// off a boundary leaves every item a tile short, and many short pieces are no round.)
inline bool TeamRounds(uint64_t bytes, uint32_t halfRounds, uint32_t roundTiles, uint32_t workgroups)
{
    return 2 * bytes >= uint64_t(halfRounds) * roundTiles * workgroups * kTileBytes;
}

// The regions the teams of a launch draw (kernels_team.h): roundTiles tiles per workgroup; over the last quarter of the
// tiles the size is halved whenever fewer than 8 regions of the current size are left.  The XCDs do not all move data at
// the same rate, and with regions that get smaller towards the end they finish together (measured, 8 x 256 MiB fp32
// all-reduce: 727 us with 64 equal regions dealt out in order, 714 us with the shrinking tail
// drawn from the counter; shrinking earlier costs more than it brings, small regions run slower --
// the more so since rounds of many whole tiles are read in one piece: with "fewer than 16"
// all-gather and broadcast took 2 % longer, the all-reduces 1 %).
// Less than two rounds (by `bytes`, see TeamRounds: a buffer off a boundary by a few bytes is dealt out like one on it; 8 ranks
// x 64 MiB 12 bytes off a boundary 177.9 us, by whole tiles 186.4): a full one and what is left dealt out evenly, or one round of
// what there is.  All-reduce of 8 ranks, fp32, us, this way / two equal rounds / the rule above: 40 MiB 113.5 / 118.6 / 111.7,
// 48 MiB 136.6 / 140.2 / 147.4, 56 MiB 161.9 / 161.8 / 158.4; all-gather 8 x 6 MiB 80.7 / - / 92.0.
inline std::vector<TeamRegion> TeamRegions(uint32_t tiles, uint64_t bytes, uint32_t roundTiles, uint32_t perTeam)
{
    std::vector<TeamRegion> regions;
    const bool even = !TeamRounds(bytes, 4, roundTiles, perTeam * kTeamXcds);
    uint32_t per = roundTiles;
    for (uint32_t at = 0; at < tiles;) {
        const uint32_t left = tiles - at;
        if (even) {
            const uint32_t teamsLeft = kTeamXcds - uint32_t(regions.size()) % kTeamXcds;
            const uint32_t n = std::min(roundTiles * perTeam, (left + teamsLeft - 1) / teamsLeft);
            regions.push_back(TeamRegion{at, n});
            at += n;
            continue;
        }
        if (uint64_t(at) * 4 >= uint64_t(tiles) * 3) {
            while (per > 1 && uint64_t(per) * perTeam * 8 > left) {
                per /= 2;
            }
        }
        const uint32_t n = std::min(left, per * perTeam);
        regions.push_back(TeamRegion{at, n});
        at += n;
    }
    while (regions.size() < kTeamXcds) {
        regions.push_back(TeamRegion{tiles, 0});     // every team has a round (the items behind the whole tiles are handled there)
    }
    return regions;
}

constexpr uint64_t kMemorySideCacheBytes = 256ull << 20;

// Whether a launch of the plain copy kernel writes its results through (StorePolicy, kernels_impl.h) instead of non-temporally:
// `traffic` bytes read and written by the launch, `written` of them written, `moved` read and written by the whole collective, whose
// launches all store alike.  One destination: never.  On the same buffers again and again it pays (all-to-all-v of 16 ranks, 210 MiB,
// non-temporal / through, us, 37.1 / 36.6; uniform all-to-all 8 ranks 32 MiB 84.5 / 75.7), on four sets of buffers in turn it does not: 16 ranks
// 210 MiB 39.1 / 45.9, 480 MiB 85.0 / 91.8, 8 ranks 314 MiB 55.8 / 59.3, 64 ranks 412 MiB 90.9 / 102.4.  Several, up to 512 MiB in all (all-gather,
// same buffers; four sets in turn): 2 ranks 10 MiB 10.4 / 7.4; 11.8 / 12.0, 64 MiB (384 MiB moved) 67.7 / 60.1; 79.4 / 78.8, 3 ranks 8 MiB 17.2 / 12.0; 18.7 /
// 18.0, 8 ranks 2 MiB 28.2 / 20.1; 27.4 / 26.9, 16 ranks 1 MiB 53.7 / 38.7; 54.6 / 53.8.  Beyond, the one loses what the other
// gains: 2 ranks 128 MiB (768) 139.5 / 143.8, 3 ranks 48 MiB (576) 107.8 / 111.7 -- unless every
// block goes to four destinations or more: 5 ranks 24 MiB (720) 150.5 / 147.6, 6 ranks 24 MiB (1008) 217.8 / 210.7; 219.9 / 213.1.
inline bool CopiesWriteThrough(uint64_t traffic, uint64_t written, uint64_t moved)
{
    return 2 * written > traffic && (moved <= 2 * kMemorySideCacheBytes || 5 * written >= 4 * traffic);
}

// The same for a launch of the plain reducing kernels: many sources into one destination, up to 512 MiB in all.
inline bool ResultsWriteThrough(uint64_t traffic, uint64_t written, uint64_t moved)
{
    return 3 * written <= traffic && moved <= 2 * kMemorySideCacheBytes;
}

// How a launch of a fused collective stores (flags of its items).  setting: "fused_stores", -1 "auto", 0 "nt", 1 "ordinary".
inline uint32_t StoreFlags(int setting, bool reduces, bool team, uint64_t traffic, uint64_t written, uint64_t moved)
{
    if (setting >= 0) {
        return setting == 1 ? kFusedOrdinaryStores : kFusedNtStores;
    }
    if (team) {
        return 0;
    }
    return (reduces ? ResultsWriteThrough(traffic, written, moved) : CopiesWriteThrough(traffic, written, moved)) ? kFusedThroughStores : kFusedNtStores;
}

// What the width of a launch of the plain fused kernels goes by, summed over a collective's items.
struct FusedShape {
    double streamBytes = 0;     // read and written
    double storeBytes = 0;      // written
    double bytes = 0;           // of the items themselves
    bool reduces = false, chains = false;          // a reduction; of chains (else of trees or stack programs)
    bool allGather = false, reduceScatter = false;
    bool bf16Selects = false;   // maximum or minimum of bf16
    uint32_t sources = 0;       // of an item
    uint32_t unit = 1;          // bytes of an element
    uint64_t capBytes = 0;      // read and written by one launch, 0: by all
    uint32_t numCu = 256;
};

// Workgroups per CU.  Streaming kernels on this part run best with few, fat workgroups as long as a
// lane keeps enough memory operations in flight: 1 workgroup per CU when an item touches 8 or
// more streams (sources + destinations), more when it touches fewer (measured on MI355X: 8 -> 8
// all-reduce and 1 -> 8 all-gather best at 1 per CU, the 2 -> 1 step kernel at 2 per CU).
inline uint32_t FusedPerCu(const FusedShape &f)
{
    constexpr double kMiB = 1024.0 * 1024.0;
    const double streams = f.bytes > 0 ? f.streamBytes / f.bytes : 2.0;   // loads + stores per lane and vector
    uint32_t perCu = streams >= 8.0 ? 1u : (streams >= 3.0 ? 2u : 4u);
    // Many sources into one destination (reduce-scatter, reduce).  Beyond the memory-side cache few workgroups keep the
    // sources' streams apart, below it many hide the latency of a combine, which for elements of one and two bytes takes
    // several instructions.  Three sets of buffers in turn, us, 1 / 2 / 8 per CU: 8 ranks in a ring bf16 sum of 64 MiB 93.2 / 98 / 99.3,
    // 256 MiB 376 / - / 401, fp32 93.0 / 97.3 / 96.5, int8 96.8 / 95.6 / 98.7; 16 ranks x 32 MiB fp16 87 / - / 94; bf16 of 48 MiB 73.3 / 70.1 / 72.0, of 32
    // MiB 49.5 / 49.0 / 47.5; 4 ranks x 128 MiB bf16 105.6 / 108.9 / -, fp32 105.4 / 110.1 / -, but 5 ranks x 100 MiB 110.3 / 101.3 / -.
    // Many more sources (MiB read in all): fp32 reduce, 24 ranks 600 MiB 103.8 / 103.5, 32 ranks 2400 MiB 413.6 / 408.6, 48 ranks 408.2 / 391.1, 64 ranks 402.8 / 386.4,
    // reduce-scatter, 24 ranks 441.2 / 435.3, 40 ranks 2600 MiB 454.9 / 448.8, 60 ranks 496.7 / 482.7 (16 ranks 436.0 / 435.1).  Reduce-scatters, whose many items are short
    // then: bf16, 28 ranks 2600 MiB 434 / 458 / 494, 48 ranks 440 / 458 / 470, 52 ranks 439 / 452 / 463, 56 ranks 512 / 521 / 509, 60 ranks 514 / 517 / 500, 64 ranks 560
    // MiB 143 / 142 / 134, 2600 MiB 500 / 513 / 487; int8, 36 ranks 537 / 449 / 469, 40 ranks 539 / 427 / 454, 44 ranks 900 MiB 189 / 173 / 158, 1500 MiB 288 / 262 / 247, 48 ranks
    // 400 MiB 98 / 87 / 76, 2600 MiB 520 / 472 / 438, 64 ranks 593 / 533 / 465.
    // Seven sources are streams enough for two (bf16 540 MiB 103.1 / 96.2 / 98.3, 1500 MiB 291.8 / 268.7 / 274.7, 2600 MiB 502 / 477 / 489, fp32 900 MiB 167.0 / 157.5 / 160.4, reduce, fp32 540 MiB 97.7 / 93.0 / 96.2).
    // Maxima and minima of bf16 go by a rule of several instructions beyond 8 sources: 10 ranks 900 MiB 175.6 / 164.4 / 168.4, 24 ranks 2600 MiB 488 / 460 / 471, 40 ranks 900 MiB 186 / 167 / 169, 48 ranks
    // 165.7 / 159.0 / 157.4, 2600 MiB 489 / 473 / 466, 52 ranks 900 MiB 174.6 / 157.4 / 152.7, 8 ranks 163.9 / 158.0 / 159.2, but a reduce of 8 155.1 / 156.9 / 160.5, of 16 167.9 / 159.3 / 161.5, of 48 160.2 / 156.6 / 154.1.
    // Such elements, and those of one byte, do best with eight somewhat longer the more sources there are (2 / 8 per CU): int8 28 ranks 400 MiB 67.7 / 72.1, 32 ranks 330 MiB 59.7 / 54.4, 400 MiB 66.2 / 64.0,
    // 430 MiB 72.1 / 77.9, 36 ranks 400 MiB 70.5 / 66.3, 460 MiB 76.9 / 81.8, 40 ranks 400 MiB 74.1 / 67.1, 500 MiB 84.8 / 87.0; bf16 maximum 32 ranks 330 MiB 60.1 / 57.6, 430 MiB 75.3 / 80.7, 40 ranks 74.3 / 70.9, 500
    // MiB 86.3 / 94.2; reduce, int8, 48 ranks 400 MiB 83.1 / 72.1, 540 MiB 92.5 / 85.7, 64 ranks 112.7 / 96.4, bf16 maximum 48 ranks 450 MiB 86.8 / 82.1, 64 ranks 540 MiB 111.7 / 103.3.
    const bool manyToOne = f.reduces && f.storeBytes * 5.0 <= f.streamBytes;
    const bool toOne = manyToOne && f.chains && (perCu == 1 || (streams <= 5.0 && f.streamBytes > 512.0 * kMiB));
    if (toOne) {
        const bool costly = f.unit == 1 || f.bf16Selects;
        if (costly && ((f.sources >= 32 && f.streamBytes <= 416.0 * kMiB) || (f.sources > 40 && f.streamBytes <= 640.0 * kMiB) ||
            (f.reduceScatter && f.sources > (f.unit == 1 ? 40u : 44u)))) {
            perCu = 8u;
        } else if (f.streamBytes > 512.0 * kMiB) {
            const bool two = f.sources == 7 || (costly && (f.unit == 1 || f.sources > (f.reduceScatter ? 7u : 8u))) || (f.unit > 2 && f.sources >= 24);
            perCu = two ? 2u : f.unit == 2 && f.reduceScatter && f.sources > 52 ? 8u : 1u;
        } else {
            perCu = f.streamBytes > 320.0 * kMiB ? 2u : f.unit <= 2 ? 8u : 2u;
        }
    }
    // Trees and stack programs, whose combines are more of the work, gain nothing from few (fp32 tree of 8 x 64 MiB 1 / 2 per CU 101 / 99) and keep many for
    // elements of one and two bytes up to about a gigabyte (two servers, 8 ranks, bf16 40 MiB 2 / 8 per CU 63.8 / 62.2).
    const double launchBytes = f.capBytes != 0 ? std::min(f.streamBytes, double(f.capBytes)) : f.streamBytes;
    if (manyToOne && !toOne && perCu == 1 && f.unit <= 2 && launchBytes <= 1280.0 * kMiB) {
        perCu = 8;
    }
    // Blocks of several sources into two or more destinations each (all-gather) without the teams: many workgroups as long as the results stay in
    // the memory-side cache, and again far beyond it where there are fewer than 7 destinations (three sets in turn, us, 1 or 2 / 8 per CU,
    // bytes moved in parentheses: 8 ranks 256 KiB 4.6 / 4.1, 2 MiB 26.4 / 25.6, 3 MiB 42.7 / 40.5; 4 ranks 4 MiB (80 MiB) 13.7 / 13.0, 8 MiB (160)
    // 30.9 / 30.1, 16 MiB (320) 61.5 / 63, 40 MiB (800) 150 / 144; 3 ranks 8 MiB (96) 17.2 / 16.3, 13 MiB (156) 30.3 / 31.2, 24 MiB (288) 54.6 / 55.7,
    // 64 MiB (768) 145 / 138, 96 MiB 213 ... 239 / 217 ... 229; 5 ranks 7 MiB (210) 43.0 / 43.5, 40 MiB (1200) 215 / 206; 2 ranks 64 MiB (384) 73 / 70.5, 112 MiB
    // (672) 129 / 121, 128 MiB 139 / 140).  A broadcast sweeps one source and is left at two: 3 ranks 32 MiB 14.3 / 15.2, 4 ranks 256 MiB 176 / 185, 6 ranks 100
    // MiB 110 / 113.
    const double cached = (streams >= 8.0 ? 256.0 : 128.0) * kMiB;
    if (f.allGather && streams >= 3.0 && (streams <= 3.0 || f.streamBytes <= cached || (streams < 8.0 && f.streamBytes > 512.0 * kMiB))) {
        perCu = 8u;
    }
    // Plain copies (one source, one destination) go through the copy kernel, which really gets the
    // occupancy it is launched with; with non-temporal stores more workgroups only widen the range
    // of addresses written at a time, which this memory system likes less (measured, 8 ranks:
    // uniform all-to-all of 32 MiB per pair 752 us at 1 or 2 per CU, 835 us at 4, 850 us at 8;
    // 16-rank all-to-all-v, 106 MB of ragged segments: 55.6 / 40.5 / 42.5 / 41.3 us at 1 / 2 / 4 / 8).
    if (!f.reduces && streams < 3.0) {
        perCu = 2u;
    }
    // few tiles per workgroup: a second workgroup per CU evens out the tail (measured: 16-rank
    // ring all-reduce of 32 MiB per rank 241 us at 1 per CU, 220 us at 2), eight do so better between 3 and 16 tiles per CU
    // (at 2 / 8: 4 ranks 32 MiB 47.1 / 44.5, 48 MiB 70.1 / 69.0; 8 ranks 15.9 MiB bf16 maximum 46.4 / 43.8; 16 ranks 12 MiB 71.1 / 67.2;
    // 8 ranks 10 MiB, 2.5 tiles, 29.0 / 30.8; 4 ranks 64 MiB equal, int8 26 MiB 37.3 / 39.0), trees and stack programs only up to 4 (halving-doubling: 4 ranks
    // bf16 12.8 MiB 21.0 / 20.1, 16 MiB 23.5 / 24.2, 24 MiB 35.8 / 36.4, 32 MiB 47.5 / 48.5, 16 ranks 12.8 MiB 85.0 / 84.4; two servers: 4 ranks 12.8 MiB
    // 21.0 / 20.1, 16 MiB 23.5 / 24.1, 32 MiB 47.4 / 48.5).
    if (perCu == 1 && !toOne && f.bytes / kTileBytes < 32.0 * f.numCu) {
        const double tilesPerCu = f.bytes / kTileBytes / f.numCu;
        perCu = f.reduces && f.unit > 1 && tilesPerCu >= 3.0 && tilesPerCu < (f.chains ? 16.0 : 4.0) ? 8 : 2;
    }
    return perCu;
}

}  // namespace hcclamd
