// Device-side contract between the executor and the gfx950 kernels.
//
// These kernels stand where the reference has its closed Reducer / Sender / Transport leaf
// (call sites ALG/base/alg_template/temp_reduce_scatter/reduce_scatter_ring.cc:31-87) and its AIV
// copy / atomic-reduce kernels (ALG/base/alg_aiv_template/aiv_communication_base.h:367-485):
// element-wise dst = a (+) b and plain copies between rank buffers, all in one GPU's HBM.
#pragma once
#include <cstdint>

namespace hcclamd {

// One workgroup iteration handles one tile: 256 lanes x 16 bytes x 4.
constexpr uint32_t kTileBytes = 16384;
constexpr uint32_t kBlockThreads = 256;

// How a step's bytes may be accessed.
enum AccessMode : uint32_t {
    ACC_VEC16 = 0,      // every pointer 16-byte aligned, byte count a multiple of 16
    ACC_VEC16_ANY = 1,  // multiple of 16, the destination 16-byte aligned, the sources at any element boundary
    ACC_ELEM = 2        // element by element (heads, tails)
};

// dst = a            when b == nullptr
// dst = a (+) b      otherwise (a = the rank's own operand, b = the peer's)
struct StepDesc {
    void *dst;
    const void *a;
    const void *b;
    uint64_t bytes;
    uint32_t tile0;     // index of this step's first tile inside the launch
    uint32_t mode;      // AccessMode
};

// Fused item: read nsrc sources once, combine in the schedule's order, write ndst destinations.
//   chain : acc = src[0]; for j = 1..nsrc-1: acc = bit j of accLeftMask ? acc (+) src[j] : src[j] (+) acc
//   tree  : nleaf leaves, leaf i = src[2i] (+) src[2i+1] (src[2i+1] may be null); then
//           v[i] = v[i] (+) v[i+w] for w = 1, 2, 4, ... ; result v[0]
//   stack : any other expression.  Sources in evaluation order; after pushing src[j] the two topmost
//           values are folded ops[j] & 7 times, bit 8 + i of ops[j] set = the lower value is the left
//           operand of fold i.  The launch's op words (one uint32 per source-pool entry, same index)
//           follow its item table in memory; nleaf holds the stack depth the program needs.
// An item is one entry of the table and one list of pointers, which say where its body starts: a multiple of 16 bytes, in whole
// tiles and a rest shorter than one.  In front of the body and behind it lie its ends, done element by element.  (The tables
// of a collective travel to the device in front of it, and those of the call that allocates nothing have to fit 256 KiB.)
struct FusedDesc {
    uint64_t bytes;     // of the body
    uint64_t accLeftMask;
    uint32_t tile0;
    uint16_t head;      // bytes in front of the body, fewer than 128
    uint16_t tail;      // bytes behind it, fewer than 16
    uint32_t nsrc;
    uint32_t ndst;
    uint32_t srcBase;   // index into the source pointer pool
    uint32_t dstBase;   // index into the destination pointer pool
    uint32_t nleaf;
    uint32_t flags;     // kFused...
};

// flags of a fused item.  Stores: one of the first two and kFusedNtStores (StorePolicy, kernels_impl.h), or, in the team kernels, none.
constexpr uint32_t kFusedOrdinaryStores = 1u;  // write-back
constexpr uint32_t kFusedThroughStores = 2u;   // written through to memory, without the non-temporal hint (plain kernels)
constexpr uint32_t kFusedWordSources = 4u;     // 8-bit chains, copies: a source's body starts off a 4-byte boundary
constexpr uint32_t kFusedPairs = 8u;           // trees: some leaf has a second source
constexpr uint32_t kFusedNtStores = 32u;       // non-temporal
constexpr uint32_t kFusedAlike = 16u;          // chains: all items of the launch have the same number of sources, two or more

// flags of the step kernel
constexpr uint32_t kStepOrdinaryStores = 1u;   // write-back stores instead of non-temporal ones in the fast loop
constexpr uint32_t kStepReverse = 2u;          // the fast loop walks every step from its last tile to its first

// Small-segment gather (pure data movement, one source and one destination per segment, any byte alignment of
// either): one wave moves one segment through its share of the workgroup's LDS.
struct SegDesc {
    const void *src;
    void *dst;
    uint64_t bytes;     // <= kGatherMaxBytes
    uint64_t pad;
};
constexpr uint32_t kGatherMaxBytes = 8192;

// An all-to-all-v as its callers describe it (kernels_a2av.h): up to P ranks, counts and displacements in elements.
template <uint32_t P> struct A2avTable {
    uint64_t send[P], recv[P];
    uint32_t rowStart[P];      // first piece of receiver j's blocks; behind the last receiver the number of pieces
    uint32_t count[P * P];     // [receiver][sender]
    uint32_t to[P * P];        // [receiver][sender]: displacement in the receive buffer
    uint32_t from[P * P];      // [receiver][sender]: displacement in the send buffer
};
// A block goes in pieces of (1 << shift) bytes, counted from the memory line of 128 bytes that its place in the receive buffer begins
// in; the pieces are numbered receiver by receiver, sender by sender.  A launch takes pieces [first, end).
struct A2avRange {
    uint32_t first, end;
    uint32_t unitShift, shift;
};
template <uint32_t P> struct A2avArgs {
    A2avTable<P> table;
    A2avRange range;
};
static_assert(sizeof(A2avArgs<16>) <= 4096, "kernel arguments");
constexpr uint32_t kA2avLine = 128;
constexpr uint32_t kA2avShift = 12;      // pieces of 4 KiB, four vectors per lane

enum KernelKind : int {
    KK_STEP = 0, KK_CHAIN = 1, KK_TREE = 2, KK_STACK = 3,
    KK_TEAM_CHAIN = 4, KK_TEAM_TREE = 5, KK_TEAM_STACK = 6,   // team forms of the fused kernels, see below
    KK_DIRECT = 7, KK_DIRECT_WIDE = 8,                         // small collectives, see below
    KK_TEAM_STACK_TILES = 9,                                   // the team's stack kernel without its rounds read source by source
    KK_CHAIN_SLOW = 10,                                        // the chain kernel with two sources in flight
    KK_PACKED_8 = 11, KK_PACKED_16 = 12, KK_PACKED_32 = 13,    // small collectives whose items are alike, by the most ranks they take
    KK_PACKED_CHAIN = 14,                                      // the same for 2, 4, 8, 16 sources (kinds 14 ... 17): chains whose sources
                                                               // are the right operands,
    KK_PACKED_RING = 18,                                       // chains whose sources behind the second one are the left operands,
    KK_PACKED_TREE = 22,                                       // trees;
    KK_PACKED_WIDE = 12,                                       // added to one of the last 12 kinds: four vectors per lane
    KK_PACKED_TWO = 38,                                        // chains of 24 ... 31 sources, both batches of them in flight; of 32 (39)
    KK_COUNT = 40,
    KK_GATHER = 40,                                            // copy kernel table only, like these:
    KK_A2AV = 41,                                              // all-to-all-v from the callers' tables in device memory, of 8, 16, 32, 64
                                                               // ranks: workgroups of one wave (kinds 41 ... 44), of four (45 ... 48);
    KK_A2AV_ARGS = 49                                          // in the kernel arguments, of 8, 16 ranks: one wave (49, 50), four (51, 52)
};
constexpr uint32_t kPackedShapes = 4;
// Index of a number of sources among those that have a kernel of their own, kPackedShapes where it has none.
constexpr uint32_t PackedShape(uint32_t nsrc) { return nsrc == 2 ? 0 : nsrc == 4 ? 1 : nsrc == 8 ? 2 : nsrc == 16 ? 3 : kPackedShapes; }

// Team form of a fused kernel: the workgroups of one XCD read their tiles together, park the results in LDS, and write
// them together (kernels_team.h).  Launched with a multiple of kTeamXcds workgroups (one per CU) and kTeamDynamicLds
// bytes of dynamic LDS; takes one more argument, the launch's team block in device memory, which belongs to this launch
// alone.  Layout, in uint32 words:
//   [x * kTeamCtrStride + kTeamArrive]   x < kTeamXcds: barrier arrivals of team x; kTeamGaveUpBit set once a wait ran out
//   [x * kTeamCtrStride + kTeamLeft]     workgroups of team x that have finished
//   [kTeamTicket]       regions handed out beyond the first kTeamXcds
//   [kTeamFinished]     teams that have finished
//   [kTeamRegionCount]  number of regions n (written by the host, never changed)
//   [kTeamHeaderWords ...]            n x TeamRegion (written by the host, never changed)
//   [kTeamHeaderWords + 2 n ...]      kTeamXcds x (n + 1) slots: the region of team x's round r + 1, plus 2; 1 = being drawn
// Everything but the count and the table starts out zero, and the kernel leaves it zero again.
constexpr uint32_t kTeamTiles = 8;        // tiles a workgroup can park per round
constexpr uint32_t kTeamXcds = 8;
constexpr uint32_t kTeamCtrStride = 32;   // words per XCD (128 bytes, a memory line of its own)
constexpr uint32_t kTeamArrive = 0, kTeamLeft = 1;
constexpr uint32_t kTeamGaveUpBit = 0x80000000u;
constexpr uint32_t kTeamTicket = kTeamXcds * kTeamCtrStride, kTeamFinished = kTeamTicket + 1, kTeamRegionCount = kTeamTicket + 2;
constexpr uint32_t kTeamHeaderWords = kTeamTicket + 4;
constexpr uint32_t kTeamDynamicLds = kTeamTiles * kTileBytes;
struct TeamRegion {
    uint32_t first;   // first tile
    uint32_t count;   // tiles, at most kTeamTiles for each workgroup of a team
};
inline uint32_t TeamBlockWords(uint32_t nregions) { return kTeamHeaderWords + 2u * nregions + kTeamXcds * (nregions + 1u); }

// Small collectives (kernels_direct.h): the whole description of a launch rides in its kernel arguments.  All sources of
// an item lie at the same offset of their buffers and all destinations at the same offset of theirs.
constexpr uint32_t kDirectThreads = 64;                  // a workgroup is one wave,
constexpr uint32_t kDirectChunk = kDirectThreads * 16;   // of an item it takes these bytes,
constexpr uint32_t kPackedWideChunk = 4 * kDirectChunk;  // or these
enum DirectKind : uint32_t { DIRECT_CHAIN = 0, DIRECT_TREE = 1, DIRECT_STACK = 2 };

// CAP = 8: up to 8 sources and destinations per item; CAP = 32: up to 32 (no stack programs).
template <uint32_t CAP> struct DirectItem {
    uint32_t bytes;
    uint32_t srcOff, dstOff;
    uint32_t nsrc, ndst;
    uint32_t kind;
    uint32_t nleaf;          // tree: number of leaves
    uint32_t accLeft;        // chain: bit j as in FusedDesc::accLeftMask
    uint32_t second;         // tree: bit i = leaf i is src[i] (+) src[kDirectSecond + i]
    uint32_t src[CAP > 8 ? 8 : 4];     // base indexes, a byte each.  chain: sources; tree: first sources of the leaves, their
                                       // second ones (repeating the first where there is none) from kDirectSecond on;
                                       // stack: sources, the last one repeated up to 8
    uint32_t dst[CAP / 4];             // base indexes of the destinations, 0 behind the last one
    uint32_t ops[CAP > 8 ? 1 : 4];     // stack: a halfword per source
};
template <uint32_t CAP> constexpr uint32_t kDirectSecond = CAP > 8 ? 16 : 8;
template <uint32_t CAP> constexpr uint32_t kDirectItems = CAP > 8 ? 32 : 16;
template <uint32_t CAP> constexpr uint32_t kDirectBases = CAP > 8 ? 64 : 16;
template <uint32_t CAP> struct DirectArgs {
    uint64_t base[kDirectBases<CAP>];
    DirectItem<CAP> item[kDirectItems<CAP>];
};
static_assert(sizeof(DirectArgs<32>) <= 4096, "kernel arguments");

// The same for items that are alike, the usual collective: item i reads the send buffers at i * srcStep and writes the receive
// buffers at i * dstStep, all of them or the one of rank i, and its list of sources is item 0's with i added to every rank (chains:
// ring, mesh) or exclusive-ored (trees: halving-doubling).  P: the most ranks.  A rank's pointer is base + (off << shift).
template <uint32_t P> struct PackedArgs {
    uint64_t base;
    uint32_t first, last;              // bytes of an item, of the last one
    uint32_t srcStep, dstStep;
    uint32_t info;                     // kPacked... fields
    uint32_t order[P > 16 ? 8 : P / 8];   // item 0's sources: a byte each, four bits up to 16 ranks
    uint32_t off[2 * P];               // send buffers, then receive buffers
};
// A launch costs the host more with every line of arguments, most of all beyond the second one (8 ranks, 128 bytes and up).  Empty
// kernels one after the other, us, 64, 104, 136, 264, 1352 bytes of arguments: 2.6, 2.8, 3.4, 3.5, 4.1 (2.2, 2.2, 2.35, 2.35, 2.4 while the
// calling thread happens to run where the arguments' memory is near).
static_assert(sizeof(PackedArgs<8>) <= 104, "two lines of kernel arguments");
constexpr uint32_t kPackedSources = 0, kPackedItems = 6, kPackedModulus = 12, kPackedShift = 18;   // lowest bits of the fields of six bits
constexpr uint32_t kPackedTree = 1u << 24;      // pairwise bottom-up over the sources; else a chain
constexpr uint32_t kPackedToOne = 1u << 25;     // one destination, the item's rank; else one to every rank of the modulus
constexpr uint32_t kPackedEnds = 1u << 26;      // some item ends in a part of a vector
constexpr uint32_t kPackedFours = 1u << 28;     // KiB in fours to the XCDs (more than 8 ranks)
constexpr uint32_t kPackedRing = 1u << 27;      // chain: sources behind the second one are the left operands; else the right ones

// Kernel entry for (data type, reduce op, kind); nullptr if the combination is not built.
// Signatures:
//   KK_STEP            (const StepDesc *steps, uint32_t nsteps, uint32_t nwhole, uint32_t ntiles, uint32_t flags)
//                      steps whose tiles are all whole and ACC_VEC16 come first: tiles [0, nwhole)
//   KK_CHAIN / KK_CHAIN_SLOW / KK_TREE / KK_STACK
//                      (const FusedDesc *items, uint32_t nitems, uint32_t nall, uint32_t nwhole, uint32_t ntiles,
//                       const void *const *srcPool, void *const *dstPool, uint32_t tilesPerItem)
//                      tiles [0, nwhole) are the whole tiles of the first nitems of the nall items; tile nwhole + i is the rest of
//                      item i's body, tile nwhole + nall + i its ends (ntiles: as many of these as any item needs, empty ones included);
//                      tilesPerItem: whole tiles of each of the first nitems items (the last one at most as many), 0 = they differ.
//                      Up to seven pointers behind an item's list of sources may be read (and are not used): the destinations'
//                      pool lies behind the sources', and the tables end on a multiple of 256 bytes.
//   KK_TEAM_*          the same and (uint32_t *teamBlock)
//   KK_PACKED_n        (PackedArgs<n>; those of 2, 4 and 8 sources PackedArgs<8>, of 16 PackedArgs<16>; KK_PACKED_TWO PackedArgs<32>), grid (chunks of the longest item's whole vectors, items), with kPackedEnds one more in x, the first one, for the bytes
//                      behind an item's last whole vector
//   KK_DIRECT / KK_DIRECT_WIDE   (DirectArgs<8> / DirectArgs<32>), grid (1 + chunks of the longest item, items): blockIdx.x == 0
//                      is for the bytes behind an item's last whole vector
const void *LookupKernel(int hcclDataType, int hcclReduceOp, KernelKind kind);

//   KK_GATHER          (const SegDesc *segs, uint32_t nsegs)
//                      copy kernel table only
//   KK_A2AV            (const A2avTable<P> *table, A2avRange); KK_A2AV_ARGS (A2avArgs<P>); any number of workgroups
//                      copy kernel table only
// Byte-wise variants for pure data movement (all-gather, all-to-all-v): KK_STEP, KK_CHAIN, KK_TEAM_CHAIN, KK_GATHER,
// KK_DIRECT, KK_DIRECT_WIDE and KK_PACKED_n.
const void *LookupCopyKernel(KernelKind kind);

}  // namespace hcclamd
