// Small collectives: from a plan to one launch whose descriptors ride in the kernel arguments (kernels_direct.h).
#include <algorithm>
#include <cstring>

#include "runtime.h"

namespace hcclamd {

namespace {

// Where the tile kernels become the better form: they keep four times as much in flight per lane, which pays once every
// CU has work.  Three sets of buffers in turn, us, tile kernels / this form (the usual ones packed):
//   all-reduce, 8 ranks, ring, bf16 512 KiB 5.7 / 3.6, 1 MiB 6.3 / 3.7, fp32 5.3 / 3.7, 5.9 / 3.6; 16 ranks, fp32 9.1 / 4.5, 10.3 / 6.2; halving-doubling, bf16, 12
//     ranks 256 KiB 9.3 / 4.5, 1 MiB 10.6 / 6.5, 24 ranks 17.3 / 5.5, 19.8 / 9.7
//   reduce-scatter, 8 ranks, bf16 (bytes received by all ranks): 1 MiB 5.3 / 3.5, 2 MiB 6.2 / 4.1, 4 MiB 7.8 / 7.2
//   all-gather (read and written): 8 ranks 5 MiB 4.2 / 3.4, 20 MiB 4.3 / 4.4; 16 ranks 5.1 / 4.4, 5.3 / 4.5
constexpr uint64_t kDirectMaxBytes = uint64_t(1) << 20;       // of a reduction's results
constexpr uint64_t kDirectMaxToOne = uint64_t(4) << 20;       // the same where each has one destination
// Blocks of whole 16-byte vectors of more than three sources, in types that combine in an instruction or two: beyond this line the
// packed form alone goes on (PackedFits).  Tile kernels / this form, us, one destination per result:
//   reduce-scatter, 2.5 MiB: fp32, 4 ranks 4.2 / 3.3, 16 ranks 9.2 / 8.2, 32 ranks 15.9 / 14.7; int64, 32 ranks 15.7 / 14.7
//   reduce, fp32, 2.5 MiB: 8 ranks 5.9 / 4.7, 32 ranks 15.6 / 14.9
// Up to the larger limit this form stays ahead for bf16 of up to 8 ranks and for 8-bit elements (4 MiB: bf16, 4 ranks 5.2 / 4.3, 8 ranks 7.6 / 7.5; int8, 8 ranks 7.9 / 7.6, 12
// ranks 3.5 MiB 10.2 / 9.9, 4 MiB 10.6 / 11.4, 32 ranks 23.3 / 21.7, 24.4 / 27.8), for ragged blocks of few ranks (int8, 8 ranks 3.5 MiB 8.0 / 7.9, 32 ranks 3 MiB 23.7 / 23.3, 3.5
// MiB 25.0 / 26.8) and for three sources or fewer (3 ranks, 4 MiB 4.7 / 3.9).
// Copies, also from one to one, are ahead up to their limit (20 MiB read and written: broadcast, 2 ranks 5.3 / 5.1, 32 ranks 7.7 / 5.6, send 5.0 / 4.6, scatter 5.1 / 5.0 ... 5.3), and a
// call with new buffers uploads nothing; with known buffers a small one costs 0.2 more than with tables (its arguments are 1.3 KB).
constexpr uint64_t kDirectMaxToOneEven = uint64_t(5) << 19;
constexpr uint64_t kDirectMaxToOneBf16 = uint64_t(13) << 18, kDirectMaxToOneBf16Ragged = uint64_t(11) << 18;
constexpr uint64_t kDirectMaxTraffic = uint64_t(20) << 20;    // read and written by a collective that only moves data
// The rule looks at the call alone: a collective that is too large is told apart before anything is looked up or planned
// for it (with a look into the plan, a caller with more distinct requests than this form's table holds paid for a plan on
// every call: 400 large all-reduces in turn, 8 ranks, 13.5 us of host time per call instead of 6.1).

template <uint32_t CAP> void PutIndex(uint32_t *list, uint32_t at, uint32_t index) { list[at >> 2] |= index << (8u * (at & 3u)); }

// Fills the arguments of a launch of `CAP`; false where the plan does not fit.
template <uint32_t CAP> bool FillDirect(const Plan &plan, DirectLaunch *d)
{
    d->image.assign(sizeof(DirectArgs<CAP>), 0);
    DirectArgs<CAP> *args = reinterpret_cast<DirectArgs<CAP> *>(d->image.data());
    d->bases.clear();
    auto baseOf = [&](const Ref &r, uint32_t *index) {
        for (size_t i = 0; i < d->bases.size(); i++) {
            if (d->bases[i].first == r.rank && d->bases[i].second == r.buf) {
                *index = uint32_t(i);
                return true;
            }
        }
        if (d->bases.size() == kDirectBases<CAP>) {
            return false;
        }
        *index = uint32_t(d->bases.size());
        d->bases.emplace_back(r.rank, r.buf);
        return true;
    };
    if (plan.fused.empty() || plan.fused.size() > kDirectItems<CAP>) {
        return false;
    }
    uint64_t longest = 0;
    for (size_t n = 0; n < plan.fused.size(); n++) {
        const FusedItem &f = plan.fused[n];
        DirectItem<CAP> &it = args->item[n];
        const bool tree = f.kind == FK_TREE, stack = f.kind == FK_STACK;
        if (f.dst.empty() || f.dst.size() > CAP || (stack && (CAP > 8 || f.src.size() > 8)) || (tree && f.nleaf > CAP) ||
            (!tree && f.src.size() > CAP)) {
            return false;
        }
        longest = std::max(longest, f.bytes);
        it.bytes = uint32_t(f.bytes);
        it.ndst = f.dst.size();
        it.kind = tree ? DIRECT_TREE : (stack ? DIRECT_STACK : DIRECT_CHAIN);
        it.nleaf = f.nleaf;
        const uint64_t srcOff = f.src[0].off, dstOff = f.dst[0].off;
        // every source at one offset of its buffer, every destination at one offset of its; what the kernels add to a
        // base pointer is a 32-bit number
        if (srcOff + f.bytes > 0x7fffffffull || dstOff + f.bytes > 0x7fffffffull) {
            return false;
        }
        it.srcOff = uint32_t(srcOff);
        it.dstOff = uint32_t(dstOff);
        uint32_t index = 0;
        for (size_t k = 0; k < f.dst.size(); k++) {
            if (f.dst[k].off != dstOff || !baseOf(f.dst[k], &index)) {
                return false;
            }
            PutIndex<CAP>(it.dst, uint32_t(k), index);
        }
        it.nsrc = f.src.size();
        for (size_t k = 0; k < f.src.size(); k++) {
            const bool valid = f.srcValid[k] != 0;
            if (valid && (f.src[k].off != srcOff || !baseOf(f.src[k], &index))) {
                return false;
            }
            if (!tree) {
                PutIndex<CAP>(it.src, uint32_t(k), index);
                if (f.kind == FK_CHAIN && f.accLeft[k]) {
                    it.accLeft |= 1u << k;
                }
                if (stack) {
                    it.ops[(k >> 1) % (sizeof(it.ops) / 4)] |= uint32_t(f.ops[k]) << (16u * (k & 1u));
                }
            } else if ((k & 1u) == 0) {
                PutIndex<CAP>(it.src, uint32_t(k / 2), index);
            } else if (f.nleaf <= kDirectSecond<CAP>) {
                PutIndex<CAP>(it.src, kDirectSecond<CAP> + uint32_t(k / 2), index);     // (repeats the first where absent)
                it.second |= (valid ? 1u : 0u) << (k / 2);
            } else if (valid) {
                return false;
            }
        }
        for (size_t k = f.src.size(); stack && k < 8; k++) {
            PutIndex<CAP>(it.src, uint32_t(k), index);
        }
    }
    d->gridX = 1 + uint32_t((longest + kDirectChunk - 1) / kDirectChunk);
    d->gridY = uint32_t(plan.fused.size());
    return true;
}

}  // namespace

bool DirectFits(int coll, uint32_t p, uint64_t bytes, int dtype)
{
    const bool even = bytes % 16 == 0 && p > 3 && dtype != HCCL_DATA_TYPE_INT8 && dtype != HCCL_DATA_TYPE_UINT8 && dtype != HCCL_DATA_TYPE_BFP16;
    const uint64_t toOne = even ? kDirectMaxToOneEven : kDirectMaxToOne;
    switch (coll) {
        case COLL_ALLREDUCE: return bytes <= (p > 1 ? kDirectMaxBytes : toOne);
        case COLL_REDUCESCATTER: return bytes <= toOne / p;
        case COLL_REDUCE: return bytes <= toOne;
        case COLL_ALLGATHER: return bytes <= kDirectMaxTraffic / p / (p + 1);
        case COLL_BROADCAST: return bytes <= kDirectMaxTraffic / p;
        case COLL_SCATTER: return bytes <= kDirectMaxTraffic / p / 2;
        case COLL_SENDRECV: return bytes <= kDirectMaxTraffic / 2;
        default: return false;
    }
}

// bf16, of which every combining rounds: with 16 and more sources the waves of this form come to wait for it where the tile kernels' larger ones still have loads in flight.  This form's
// time as a share of the tiles', reduce-scatter of whole vectors / of others / reduce, sum: 16 ranks 3 MiB 0.92 / 1.03 / 0.92, 3.25 MiB 0.97 / 1.05 / 1.01, 3.75 MiB 1.07 / 1.21 / 1.10; 24 ranks 2.75 MiB
// 0.87 / 0.99 / 0.85, 3 MiB 0.90 / 1.15 / 0.91, 3.5 MiB 1.02 / 1.14 / 1.04; 32 ranks 3 MiB 0.90 / 1.05 / 0.92, 3.25 MiB 0.97 / 1.09 / 1.00, 4 MiB 1.11 / 1.44 / 1.07.  Fewer ranks stay ahead up to 4 MiB (9 ranks
// 3.5 MiB 0.93 / 0.97 / 0.91, 12 ranks 3.25 MiB 0.91 / 0.93 / 0.94, 4 MiB 0.99 / 1.02 / 1.02, 14 ranks 1.01 / 1.00 / 1.04), and so do maxima and minima, which round nothing (16 ranks 3.5 MiB 0.88 / 0.98 /
// 0.90, 32 ranks 0.92 / 1.03 / 0.91), but for blocks of parts of vectors of 28 and more (28 ranks 3.25 MiB 0.98, 3.5 MiB 1.17, 32 ranks 3.25 MiB 0.96, 4 MiB 1.33).
bool CombiningBound(int coll, uint32_t p, uint64_t bytes, int dtype, int op)
{
    if ((coll != COLL_REDUCESCATTER && coll != COLL_REDUCE) || p < 16 || dtype != HCCL_DATA_TYPE_BFP16) {
        return false;
    }
    const bool selects = op == HCCL_REDUCE_MAX || op == HCCL_REDUCE_MIN, ragged = coll == COLL_REDUCESCATTER && bytes % 16 != 0;
    if (selects && (!ragged || p < 28)) {
        return false;
    }
    return (coll == COLL_REDUCESCATTER ? bytes * p : bytes) > (ragged && !selects ? kDirectMaxToOneBf16Ragged : kDirectMaxToOneBf16);
}

// Beyond those limits, where the items are alike (PackDirect): waves of 1 or 4 KiB keep every CU equally busy where the tile kernels' tiles of
// 16 KiB do not, that is where there are few of them, or a few more than one, two or three for each CU (on 256 CUs 4, 8, 12 MiB): a CU takes some 4 us for a tile
// that is read from 8 buffers and stored to 8.  So the windows are in sixteenths of a tile for each CU, 256 KiB on 256 CUs.  Measured there, three sets of buffers in turn, us, tile kernels / packed with KiB / packed with 4 KiB:
//   all-reduce, 2 ranks: 4 MiB 4.5 / 3.6 / 3.6, 6 MiB 5.7 / 5.1 / 4.5, 8 MiB 6.0 / 6.0 / 5.8, 24 MiB 18.0 / 16.6 / 17.1, 48 MiB 33.8 / 31.9 / 33.5
//     4 ranks: 3 MiB 5.2 / 4.5 / 4.6, 4.25 MiB 8.0 / 6.9 / 6.0, 6 MiB 8.7 / 9.4 / 7.6, 7 MiB 9.5 / 10.4 / 9.8, 8 MiB 10.6 / 12.2 / 12.0, 9 MiB
//       14.1 / 13.9 / 13.8, 14 MiB 21.7 / 19.9 / 20.1, 24 MiB 35.9 / 32.1 / 31.6, 28 MiB 40.7 / 41.1 / 40.9
//     8 ranks: 1.5 MiB 6.4 / 4.6 / 5.5, 2 MiB 7.0 / 6.0 / 6.1, 2.5 MiB 7.5 / 7.7 / 7.0, 3 MiB 8.3 / 9.7 / 7.8 (bf16 maximum 8.6 / - / 9.5), 4 MiB 10.7 / 12.5 / 10.5,
//       4.25 MiB 14.3 / 13.2 / 11.5, 5 MiB 15.8 / 15.1 / 12.8, 6 MiB 16.7 / 17.6 / 16.5, 8 MiB 21.1 / 22.4 / 22.0, 8.5 MiB 26.4 / 24.2 / 24.5, 12 MiB
//       34.7 / 33.7 / 33.2, 14 MiB 41.7 / 44.0 / 42.8
//     16 ranks: 1.5 MiB 11.0 / 9.5 / 10.2, 2 MiB 12.3 / 13.3 / 11.1, 3 MiB 16.0 / 18.1 / 15.6 (bf16 17.5 / - / 17.7), 4.25 MiB 27.7 / 24.6 / 22.9, 5 MiB
//       29.6 / 27.5 / 25.7, 6 MiB 33.3 / 35.3 / 31.2 (fp16, bf16 up to 33), 8.5 MiB 54.5 / 57.3 / 53.1; 32 ranks 1.5 MiB 21.3 / 17.7 / -
//   reduce-scatter (bytes received by all ranks), blocks of whole vectors: 2 ranks 6 MiB 4.5 / 4.0, 14 MiB 8.5 / 7.9, 16 MiB 9.1 / 9.0, 20 MiB 11.7 / 11.1, 64 MiB
//     32.2 / 30.1; 4 ranks 5 MiB 6.1 / 5.1, 7 MiB 7.0 / 6.6 (int8 6.4 MiB 6.5 / 6.9), 8 MiB 7.6 / 7.7, 9 MiB 9.8 / 8.1, 11 MiB 10.5 / 10.2, 12 MiB 11.0 / 11.4; 8 ranks 3 MiB
//     6.3 / 5.3, 4 MiB 7.3 / 7.0, 5 MiB 9.4 / 8.2, 6 MiB 10.1 / 9.7 (int8 5.7 MiB 9.8 / 10.6), 7 MiB 11.2 / 10.9, 8 MiB 12.1 / 13.5; 16 ranks 1 MiB 7.7 / 5.1, 2 MiB 8.6 / 8.3 (bf16
//     10.1 / 8.4), 3 MiB 9.8 / 9.7, 4.05 MiB (fp16) 12.4 / 14.0, 4.25 MiB 15.5 / 13.5, 5 MiB 16.4 / 15.3, 6 MiB 17.8 / 20.4
//   other blocks: 2 ranks 14 MiB 8.9 / 8.8, 4 ranks 6 MiB 6.9 / 6.8, 8 ranks 3 MiB 6.7 / 5.9, 4 MiB 8.5 / 7.8, 5 MiB 9.8 / 9.0, 16 ranks 2 MiB 9.2 / 7.9,
//     3 MiB 10.3 / 10.7.  Waves of 4 KiB bring nothing where every block has one destination (8 ranks bf16 pairwise, 4 MiB 6.9 / 7.7).
// Two kinds of calls gain less and stay out: 16 ranks' all-reduce of a 16-bit floating-point type between 1.5 and 4 MiB, whose waves of 4 KiB wait for their own
// arithmetic (1.75 MiB bf16 sum 12.4 / 12.1, fp16 minimum of the uncut mesh 12.2 / 16.1; beyond 4 MiB the tiles wait longer: 4.25 MiB bf16 sum 27.1 / 23.2, maximum
// 25.8 / 22.9, halving-doubling 30.8 / 24.2, 5.44 MiB 31.5 / 29.3, 31.3 / 30.5, 33.6 / 30.8), and bytes off a vector boundary (8 ranks 4.75 MiB 9.3 / 10.1).
namespace {

enum PackedCalls : uint8_t {
    ALL_REDUCE_HALVES = 1, ALL_REDUCE_OTHERS = 2, ALL_REDUCE = 3,     // of fp16 and bf16; of other types
    BLOCKS_WHOLE = 4, BLOCKS_WHOLE_BYTES = 32, BLOCKS = 36,           // reduce-scatter, blocks of whole 16-byte vectors; of 8-bit elements
    BLOCKS_BYTES = 8, BLOCKS_OTHERS = 16, BLOCKS_RAGGED = 24          // other blocks, of 8-bit elements; of other types
};
struct PackedWindow {
    uint8_t calls, least, most;      // ranks
    uint16_t above, upTo;            // bytes of an all-reduce, received by all ranks of a reduce-scatter
    uint16_t upToOff;                // where sends and results lie off half a memory line
};
constexpr PackedWindow kPackedWindows[] = {
    {ALL_REDUCE, 2, 2, 0, 192, 64},
    {ALL_REDUCE, 3, 3, 0, 14, 14},
    {ALL_REDUCE, 4, 4, 0, 24, 21}, {ALL_REDUCE, 4, 4, 32, 96, 32},
    {ALL_REDUCE, 5, 7, 0, 9, 9},
    {ALL_REDUCE, 8, 8, 0, 11, 11}, {ALL_REDUCE, 8, 8, 16, 22, 21}, {ALL_REDUCE, 8, 8, 32, 48, 42},
    {ALL_REDUCE, 9, 32, 0, 6, 6}, {ALL_REDUCE_OTHERS, 16, 16, 6, 11, 11}, {ALL_REDUCE, 16, 16, 16, 22, 21},
    {BLOCKS, 2, 2, 0, 60, 60}, {BLOCKS, 2, 2, 64, 256, 64},
    {BLOCKS, 3, 3, 0, 24, 24},
    {BLOCKS, 4, 4, 0, 24, 24}, {BLOCKS_WHOLE, 4, 4, 24, 30, 26}, {BLOCKS, 4, 4, 32, 44, 41},
    {BLOCKS, 5, 7, 0, 18, 18},
    {BLOCKS, 8, 8, 0, 21, 21}, {BLOCKS_WHOLE, 8, 8, 21, 24, 21},
    {BLOCKS, 16, 16, 0, 11, 11}, {BLOCKS, 16, 16, 17, 20, 20},
    {BLOCKS_RAGGED, 2, 2, 0, 56, 56},
    {BLOCKS_RAGGED, 3, 4, 0, 24, 24},
    {BLOCKS_RAGGED, 5, 8, 0, 14, 14}, {BLOCKS_OTHERS, 8, 8, 16, 20, 20},
    {BLOCKS_RAGGED, 16, 16, 0, 10, 10},
};
uint64_t SixteenthTiles(uint32_t numCu) { return uint64_t(numCu) * kTileBytes / 16; }

}  // namespace

// Buffers off a boundary.  The tile kernels bring their vectors to one, the packed ones access them as they come, which costs little as long as they lie on
// 4 bytes: tiles / packed, all-reduce, bf16, 8 ranks 2.5 MiB on 512 bytes 7.8 / 7.4, 4 bytes off 7.9 / 7.8, 2 bytes off 7.9 / 11.7, 5 MiB 15.6 / 13.3, 15.7 / 14.0, 15.7 / 19.0.  Of an
// all-reduce it takes sends and results off 4 bytes for packed to fall behind (8 ranks 2.5 MiB, only sends 7.9 / 7.6, only results 7.9 / 6.4), and then not below some size: 2 ranks
// 3 MiB 0.87 of the tiles' time, 4 MiB 1.02 ... 1.10; 3 ranks 2.25 MiB 0.95 ... 1.00, 3.25 MiB 1.2; 4 ranks 1.75 MiB 0.75 ... 0.94, 2.25 MiB 1.12 ... 1.19; 6 and 8 ranks 1.5 MiB 0.94 ... 1.00,
// 8 ranks 1.75 MiB 1.06 ... 1.10; 12 to 32 ranks 1.25 MiB 0.82 ... 1.02, 16 ranks 1.5 MiB 0.99 ... 1.12.  A reduce-scatter of whole vectors reads its sources off 4 bytes whatever its results: 2 ranks
// 3 MiB 0.88 ... 1.00, 5 MiB 0.94 ... 1.05; 3 ranks 2 MiB 0.80 ... 0.95, 2.5 MiB 1.09, 5 MiB 0.98 ... 1.11; 4 to 16 ranks 3 MiB 0.90 ... 1.04, 4 ranks 4 MiB 1.03 ... 1.19, 8 ranks 3.5 MiB 1.06 ... 1.11,
// 5.5 MiB 1.16 ... 1.22.  Blocks of parts of vectors lie off by themselves, and their windows hold wherever the buffers lie.
// Stores that straddle memory lines cost something at any size: sends and results off half a line leave the upper ends of the larger windows to the tiles (packed as a share of the tiles' time, random sizes,
// types and placements; all-reduce, 4 ranks 20 ... 24 quarters of a MiB on / off lines 0.91 / 1.00, 32 ... 96 0.92 / 1.02, 8 ranks 45 ... 48 0.93 / 1.06, 16 ranks 21 and 22 0.94 / 1.04, 2 ranks 190 0.90 / 1.02;
// reduce-scatter, 4 ranks 26 ... 30 1.02 / 1.07, 41 ... 44 0.99 / 1.07, 8 ranks 21 ... 24 1.00 / 1.06, 2 ranks 200 0.96 / 1.04).  In place, where reads and stores of one line are by different waves, more: 2 ranks 9 ... 19 1.04, 3 ranks 8 ... 10
// 1.03, 12 ... 14 1.08, 4 ranks 8 ... 16 1.03 ... 1.20, 6 ranks 8 and 9 1.03, 8 ranks 8 ... 11 1.07, 16 ranks 6 ... 11 1.06 ... 1.17, 16 ... 22 0.98 ... 1.17.
bool PackedFits(int coll, uint32_t p, uint64_t bytes, int dtype, uint32_t numCu, uint64_t sends, uint64_t recvs, bool inPlace)
{
    uint8_t call = 0;
    uint64_t total = bytes;
    if (coll == COLL_ALLREDUCE) {
        call = dtype == HCCL_DATA_TYPE_FP16 || dtype == HCCL_DATA_TYPE_BFP16 ? ALL_REDUCE_HALVES : ALL_REDUCE_OTHERS;
    } else if (coll == COLL_REDUCESCATTER) {
        const bool bytesOnly = dtype == HCCL_DATA_TYPE_INT8 || dtype == HCCL_DATA_TYPE_UINT8;
        call = bytes % 16 == 0 ? (bytesOnly ? BLOCKS_WHOLE_BYTES : BLOCKS_WHOLE) : (bytesOnly ? BLOCKS_BYTES : BLOCKS_OTHERS);
        total *= p;
    }
    const uint64_t unit = SixteenthTiles(numCu);
    const bool off = (sends & 3u) != 0 && (coll == COLL_ALLREDUCE ? (recvs & 3u) != 0 : call == BLOCKS_WHOLE || call == BLOCKS_WHOLE_BYTES);
    const bool offLine = (sends & 63u) != 0 && (recvs & 63u) != 0;
    uint64_t most = 0;
    if (off) {
        most = coll != COLL_ALLREDUCE ? (p == 3 ? 8 : 12) : (p == 2 ? 12 : p <= 4 ? 7 : p <= 8 ? 6 : 5);
    } else if (offLine && inPlace && coll == COLL_ALLREDUCE) {
        most = p == 2 ? 12 : p == 3 ? 8 : p == 4 ? 7 : p <= 7 ? 8 : p == 8 ? 7 : p == 16 ? 5 : 0;
    }
    if (most != 0 && total > most * unit) {
        return false;
    }
    for (const PackedWindow &w : kPackedWindows) {
        if ((w.calls & call) != 0 && p >= w.least && p <= w.most && total > w.above * unit && total <= (offLine ? w.upToOff : w.upTo) * unit) {
            return true;
        }
    }
    return false;
}

bool BuildDirect(const Plan &plan, bool reduceColl, int dtype, int op, DirectLaunch *d)
{
    d->func = nullptr;
    uint64_t bytes = 0;
    for (const FusedItem &f : plan.fused) {
        bytes += f.bytes;
    }
    if (!plan.fusedOk || bytes == 0) {
        return false;
    }
    const bool narrow = FillDirect<8>(plan, d);
    if (!narrow && !FillDirect<32>(plan, d)) {
        return false;
    }
    const KernelKind kind = narrow ? KK_DIRECT : KK_DIRECT_WIDE;
    d->sendBytes = plan.sendBytes;
    d->recvBytes = plan.recvBytes;
    d->func = reduceColl ? LookupKernel(dtype, op, kind) : LookupCopyKernel(kind);
    return d->func != nullptr;
}

namespace {

// Whether the KiB of an item go to the XCDs in fours (KiBOf, kernels_direct.h): `total` bytes in `items` items of more than 8 ranks.  Us, workgroups of 4 KiB / of
// KiB one by one / in fours: reduce of 2 MiB, fp32, 16 ranks 7.4 / 7.7 / 6.9, 24 ranks 9.9 / 10.8 / 9.8, 32 ranks 12.8 / 13.9 / 12.7, bf16, 16 ranks 7.1 / 8.0 / 7.5; but 12 ranks,
// whose buffers of 1.5 and 2 MiB stay apart, 5.1 / 4.6 / 4.8 and 5.5 / 5.3 / 5.6.  Reduce-scatter (results in all), fp32, 12 ranks 2 MiB 6.5 / 6.3 / 5.8, 2.5 MiB 7.0 / 7.3 /
// 6.8, 16 ranks 2 MiB 8.1 / 7.7 / 6.9, 24 ranks 2.5 MiB 12.5 / 12.8 / 11.8; bf16, 12 ranks 3.5 MiB 10.0 / 10.0 / 9.4, but 16 ranks 2.5 MiB 8.5 / 8.7 / 8.8, 3.5 MiB 11.4 / 11.7 /
// 12.1.  All-reduce, 32 ranks 512 KiB 8.1 / 7.7 / 6.8 (with both batches of sources in flight); 16 ranks 768 KiB 6.3 / 5.0 / 5.2.  Up to 8 sources it makes no difference;
// copies lose (20 MiB read and written 4.2 / 4.6).
bool PackedInFours(uint32_t p, uint32_t items, bool toOne, uint64_t total, int dtype)
{
    if (p > 16 || !toOne) {
        return p > 16;
    }
    const bool halves = dtype == HCCL_DATA_TYPE_FP16 || dtype == HCCL_DATA_TYPE_BFP16;
    return items > 1 ? p < 16 || !halves || total <= uint64_t(9) << 18 : p == 16;
}

// Arguments of `P` ranks out of items of `nsrc` sources each, already found alike.
template <uint32_t P> void FillPacked(const Plan &plan, const std::vector<uint32_t> &order, uint32_t info, DirectLaunch *d)
{
    d->packed.assign(sizeof(PackedArgs<P>), 0);
    PackedArgs<P> *args = reinterpret_cast<PackedArgs<P> *>(d->packed.data());
    const FusedItem &f = plan.fused[0], &last = plan.fused[plan.fused.size() - 1];
    args->first = uint32_t(f.bytes);
    args->last = uint32_t(last.bytes);
    if (plan.fused.size() > 1) {
        args->srcStep = uint32_t(plan.fused[1].src[0].off);
        args->dstStep = uint32_t(plan.fused[1].dst[0].off);
    }
    args->info = info;
    for (size_t j = 0; j < order.size(); j++) {
        args->order[P > 16 ? j / 4 : j / 8] |= order[j] << (P > 16 ? 8 * (j % 4) : 4 * (j % 8));
    }
    d->packedRanks = P;
}

// base + (offset << shift) for every rank's pointer; false where the offsets do not fit 32 bits.
template <uint32_t P> bool FillOffsets(DirectLaunch *d, uint32_t ranks, const std::vector<void *> &send, const std::vector<void *> &recv)
{
    PackedArgs<P> *args = reinterpret_cast<PackedArgs<P> *>(d->packed.data());
    uint64_t least = ~uint64_t(0), most = 0, bits = 0;
    for (uint32_t r = 0; r < ranks; r++) {
        for (const void *v : {send[r], recv[r]}) {
            const uint64_t at = reinterpret_cast<uint64_t>(v);
            least = std::min(least, at);
            most = std::max(most, at);
            bits |= at;
        }
    }
    // (an alignment of the addresses themselves is one of their differences; beyond 4 KiB a larger shift brings nothing)
    const uint32_t shift = uint32_t(__builtin_ctzll(bits | 4096));
    least &= ~uint64_t(4095);
    if (((most - least) >> shift) > 0xffffffffull) {
        return false;
    }
    args->base = least;
    args->info = (args->info & ~(63u << kPackedShift)) | (shift << kPackedShift);
    for (uint32_t r = 0; r < ranks; r++) {
        args->off[r] = uint32_t((reinterpret_cast<uint64_t>(send[r]) - least) >> shift);
        args->off[P + r] = uint32_t((reinterpret_cast<uint64_t>(recv[r]) - least) >> shift);
    }
    return true;
}

}  // namespace

void PackDirect(const Plan &plan, bool reduceColl, int dtype, int op, DirectLaunch *d, uint32_t numCu)
{
    const uint32_t p = plan.p, n = uint32_t(plan.fused.size());
    if (p > 32 || n == 0 || n > p) {
        return;
    }
    const FusedItem &f = plan.fused[0];
    const bool tree = f.kind == FK_TREE;
    if (f.kind == FK_STACK) {
        return;
    }
    // the sources of an item: a tree's leaves one behind the other, all of them pairs or none
    auto sources = [&](const FusedItem &it, std::vector<uint32_t> *ranks) {
        ranks->clear();
        const bool pairs = tree && it.srcValid[1] != 0;
        for (size_t k = 0; k < it.src.size(); k++) {
            const bool here = !tree || (k & 1u) == 0 || pairs;
            if ((it.srcValid[k] != 0) != here) {
                return false;
            }
            if (here) {
                if (it.src[k].buf != BUF_SEND) {
                    return false;
                }
                ranks->push_back(it.src[k].rank);
            }
        }
        return true;
    };
    std::vector<uint32_t> order, ranks;
    if (!sources(f, &order) || order.empty() || order.size() > 32 || (tree && ((order.size() & (order.size() - 1)) != 0 || order.size() < 2))) {
        return;
    }
    const bool toOne = f.dst.size() == 1 && p > 1;
    bool left = true, ring = true, ends = false;      // chain: every source behind the first is the right operand; all but the second the left one
    const uint64_t srcStep = n > 1 ? plan.fused[1].src[0].off : 0, dstStep = n > 1 ? plan.fused[1].dst[0].off : 0;
    uint64_t longest = 0;
    for (uint32_t i = 0; i < n; i++) {
        const FusedItem &it = plan.fused[i];
        if (it.kind != f.kind || (i + 1 < n && it.bytes != f.bytes) || it.bytes > 0x7fffffffull || !sources(it, &ranks) || ranks.size() != order.size() ||
            it.dst.size() != (toOne ? 1 : p)) {
            return;
        }
        for (size_t j = 0; j < ranks.size(); j++) {
            const uint32_t want = tree ? order[j] ^ i : (order[j] + i) % p;
            if (ranks[j] != want) {
                return;
            }
        }
        for (size_t k = 0; k < it.src.size(); k++) {
            if (it.srcValid[k] != 0 && it.src[k].off != i * srcStep) {
                return;
            }
        }
        uint64_t seen = 0;
        for (size_t k = 0; k < it.dst.size(); k++) {
            if (it.dst[k].buf != BUF_RECV || it.dst[k].off != i * dstStep || (toOne && it.dst[k].rank != i)) {
                return;
            }
            seen |= uint64_t(1) << it.dst[k].rank;
        }
        if (!toOne && seen != (uint64_t(1) << p) - 1) {
            return;
        }
        for (size_t j = 1; !tree && j < it.accLeft.size(); j++) {
            left = left && it.accLeft[j] != 0;
            ring = ring && (it.accLeft[j] != 0) == (j == 1);
        }
        ends = ends || it.bytes % 16 != 0;
        longest = std::max(longest, it.bytes);
    }
    // (the offsets of the last item and its length are 32-bit numbers of the plan's, which BuildDirect has looked at)
    if (!tree && order.size() > 1 && !left && !ring) {
        return;
    }
    uint64_t total = 0;
    for (const FusedItem &it : plan.fused) {
        total += it.bytes;
    }
    const bool fours = reduceColl && p > 8 && PackedInFours(p, n, toOne, total, dtype);
    const uint32_t info = uint32_t(order.size()) << kPackedSources | n << kPackedItems | p << kPackedModulus | (tree ? kPackedTree : 0u) |
        (toOne ? kPackedToOne : 0u) | (fours ? kPackedFours : 0u) | (ends ? kPackedEnds : 0u) | (!tree && !left ? kPackedRing : 0u);
    KernelKind kind = KK_PACKED_8;
    if (p <= 8) {
        FillPacked<8>(plan, order, info, d);
    } else if (p <= 16) {
        FillPacked<16>(plan, order, info, d);
        kind = KK_PACKED_16;
    } else {
        FillPacked<32>(plan, order, info, d);
        kind = KK_PACKED_32;
    }
    const uint32_t shape = PackedShape(uint32_t(order.size()));
    bool wide = false;
    if (reduceColl && shape < kPackedShapes && order.size() == p) {       // (of two sources, added and exclusive-ored are the same)
        kind = KernelKind((tree ? KK_PACKED_TREE : (left ? KK_PACKED_CHAIN : KK_PACKED_RING)) + shape);
        // waves of 4 KiB where PackedFits' figures say so
        wide = !toOne && total > (p <= 8 ? 8 : 6) * SixteenthTiles(numCu) && total <= 32 * SixteenthTiles(numCu);
    }
    d->packedWide = wide;
    const uint32_t chunk = wide ? kPackedWideChunk : kDirectChunk;
    kind = wide ? KernelKind(kind + KK_PACKED_WIDE) : kind;
    d->packedGridX = uint32_t(longest / chunk + (longest % chunk >= 16 ? 1 : 0)) + (ends ? 1u : 0u);
    d->packedFunc = reduceColl ? LookupKernel(dtype, op, kind) : LookupCopyKernel(kind);
    // Both batches of many sources in flight, but for large all-reduces whose combining takes an instruction or two, where the waves a CU holds count for more (share of the time batch after
    // batch: fp32, 32 ranks 1 MiB 0.94, 1.12 MiB 1.09, 1.5 MiB 1.17, 24 ranks 1.5 MiB 1.04; bf16 sum, 32 ranks 1.5 MiB 0.93, int8 0.89), and for maxima and minima of 32 halves, whose registers leave no
    // room for it (all-reduce of bf16, 512 KiB 1.26, fp16 1.13).
    const bool halves = dtype == HCCL_DATA_TYPE_FP16 || dtype == HCCL_DATA_TYPE_BFP16, selects = op == HCCL_REDUCE_MAX || op == HCCL_REDUCE_MIN;
    const bool costly = dtype == HCCL_DATA_TYPE_INT8 || dtype == HCCL_DATA_TYPE_UINT8 || (dtype == HCCL_DATA_TYPE_BFP16 && !selects);
    if (reduceColl && !tree && order.size() >= 24 && !(order.size() == 32 && halves && selects) && (toOne || costly || total <= 4 * SixteenthTiles(numCu))) {
        d->packedTwoFunc = LookupKernel(dtype, op, KernelKind(KK_PACKED_TWO + (order.size() == 32 ? 1 : 0)));
    }
}

bool FillBases(DirectLaunch *d, const std::vector<void *> &send, const std::vector<void *> &recv)
{
    uint64_t *base = reinterpret_cast<uint64_t *>(d->image.data());     // DirectArgs<>::base comes first
    bool same = true;
    for (size_t i = 0; i < d->bases.size(); i++) {
        const uint64_t p = reinterpret_cast<uint64_t>((d->bases[i].second == BUF_SEND ? send : recv)[d->bases[i].first]);
        same = same && base[i] == p;
        base[i] = p;
    }
    if (d->packedFunc != nullptr && !same) {
        const uint32_t ranks = uint32_t(send.size());
        d->usePacked = d->packedRanks == 8 ? FillOffsets<8>(d, ranks, send, recv)
                                           : (d->packedRanks == 16 ? FillOffsets<16>(d, ranks, send, recv) : FillOffsets<32>(d, ranks, send, recv));
    }
    return same;
}

}  // namespace hcclamd
