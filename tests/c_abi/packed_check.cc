// The packed arguments of small collectives (cann-hccl_amd/csrc/direct.cc, PackDirect) against the planner, on the host: a seeded
// walk over requests and buffers.  The arguments are read back as the kernels of kernels_direct.h read them, to addresses, and
// every item has to be the plan's: the same expression over the same addresses, the same destinations.  A usual collective
// (ring, uncut mesh, halving-doubling over a power of two) has to be taken.  argv[1] = requests.  Prints how many went which way.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <set>
#include <string>
#include <vector>

#include "runtime.h"

namespace hcclamd {
static const char g_kernels[KK_COUNT] = {};
const void *LookupKernel(int, int, KernelKind kind) { return &g_kernels[kind]; }
const void *LookupCopyKernel(KernelKind kind) { return &g_kernels[kind]; }
}  // namespace hcclamd

using namespace hcclamd;

namespace {

long g_wide = 0, g_fours = 0;
uint64_t g_state = 0x9E3779B97F4A7C15ull;
uint64_t Below(uint64_t n)
{
    g_state = g_state * 6364136223846793005ull + 1442695040888963407ull;
    return n == 0 ? 0 : (g_state >> 29) % n;
}

std::string At(uint64_t a) { return std::to_string(a); }
std::string Both(const std::string &a, const std::string &b) { return "(" + a + "+" + b + ")"; }
std::string Pairwise(std::vector<std::string> v)
{
    for (size_t w = 1; w < v.size(); w <<= 1) {
        for (size_t i = 0; i + w < v.size(); i += 2 * w) {
            v[i] = Both(v[i], v[i + w]);
        }
    }
    return v[0];
}

struct Item {
    uint64_t bytes = 0;
    std::string value;
    std::set<uint64_t> dst;
};

Item OfPlan(const FusedItem &f, const std::vector<void *> &send, const std::vector<void *> &recv)
{
    auto where = [&](const Ref &r) { return reinterpret_cast<uint64_t>((r.buf == BUF_SEND ? send : recv)[r.rank]) + r.off; };
    Item it;
    it.bytes = f.bytes;
    for (const Ref &d : f.dst) {
        it.dst.insert(where(d));
    }
    if (f.kind == FK_TREE) {
        std::vector<std::string> leaf;
        for (uint32_t i = 0; i < f.nleaf; i++) {
            leaf.push_back(f.srcValid[2 * i + 1] ? Both(At(where(f.src[2 * i])), At(where(f.src[2 * i + 1]))) : At(where(f.src[2 * i])));
        }
        it.value = Pairwise(leaf);
        return it;
    }
    it.value = At(where(f.src[0]));
    for (size_t j = 1; j < f.src.size(); j++) {
        it.value = f.accLeft[j] ? Both(it.value, At(where(f.src[j]))) : Both(At(where(f.src[j])), it.value);
    }
    return it;
}

template <uint32_t P> Item OfArguments(const PackedArgs<P> &k, uint32_t i, bool *ok)
{
    auto field = [&](uint32_t at) { return (k.info >> at) & 63u; };
    auto pointer = [&](uint32_t n) {
        *ok = *ok && n < 2 * P;
        return k.base + (uint64_t(k.off[n % (2 * P)]) << field(kPackedShift));
    };
    const uint32_t nsrc = field(kPackedSources), mod = field(kPackedModulus);
    *ok = *ok && nsrc >= 1 && nsrc <= P && mod <= P && i < mod;
    std::vector<std::string> src;
    for (uint32_t j = 0; j < nsrc; j++) {
        const uint32_t o = P > 16 ? (k.order[j / 4] >> (8 * (j % 4))) & 0xff : (k.order[j / 8] >> (4 * (j % 8))) & 15;
        const uint32_t r = (k.info & kPackedTree) ? o ^ i : (o + i >= mod ? o + i - mod : o + i);
        *ok = *ok && r < mod;
        src.push_back(At(pointer(r) + uint64_t(i) * k.srcStep));
    }
    Item it;
    it.bytes = i + 1 == field(kPackedItems) ? k.last : k.first;
    if (k.info & kPackedTree) {
        *ok = *ok && (nsrc & (nsrc - 1)) == 0 && nsrc >= 2;
        it.value = Pairwise(src);
    } else {
        it.value = src[0];
        for (uint32_t j = 1; j < nsrc; j++) {
            const bool left = !(k.info & kPackedRing) || j < 2;
            it.value = left ? Both(it.value, src[j]) : Both(src[j], it.value);
        }
    }
    for (uint32_t n = 0; n < ((k.info & kPackedToOne) ? 1 : mod); n++) {
        it.dst.insert(pointer(P + ((k.info & kPackedToOne) ? i : n)) + uint64_t(i) * k.dstStep);
    }
    return it;
}

template <uint32_t P> bool Same(const Plan &plan, const DirectLaunch &d, const std::vector<void *> &send, const std::vector<void *> &recv)
{
    if (d.packed.size() != sizeof(PackedArgs<P>)) {
        return false;
    }
    const PackedArgs<P> &k = *reinterpret_cast<const PackedArgs<P> *>(d.packed.data());
    // the kernel: one of its own for 2, 4, 8 or 16 sources of as many ranks, else the one for the arguments
    const uint32_t nsrc = (k.info >> kPackedSources) & 63u, mod = (k.info >> kPackedModulus) & 63u, shape = PackedShape(nsrc);
    int kind = P == 8 ? KK_PACKED_8 : P == 16 ? KK_PACKED_16 : KK_PACKED_32;
    if (shape < kPackedShapes && nsrc == mod) {
        kind = int(shape) + ((k.info & kPackedTree) ? KK_PACKED_TREE : (k.info & kPackedRing) ? KK_PACKED_RING : KK_PACKED_CHAIN);
        if (P != (nsrc == 16 ? 16 : 8)) {
            return false;
        }
        // of several MiB to many destinations: four vectors per lane
        uint64_t total = 0;
        for (const FusedItem &f : plan.fused) {
            total += f.bytes;
        }
        if (!(k.info & kPackedToOne) && total > (nsrc == 16 ? 3u << 19 : 2u << 20) && total <= 8u << 20) {
            kind += KK_PACKED_WIDE;
            g_wide++;
        }
    }
    const uint32_t chunk = kind >= KK_PACKED_CHAIN + KK_PACKED_WIDE ? 4096 : 1024;
    if (d.packedFunc != LookupKernel(0, 0, KernelKind(kind))) {
        return false;
    }
    const uint32_t ends = (k.info & kPackedEnds) ? 1 : 0;
    g_fours += (k.info & kPackedFours) != 0;
    bool ok = (P > 8 || !(k.info & kPackedFours)) && ((k.info >> kPackedItems) & 63u) == plan.fused.size() && d.gridY == plan.fused.size();
    for (uint32_t i = 0; ok && i < plan.fused.size(); i++) {
        const Item a = OfPlan(plan.fused[i], send, recv), b = OfArguments<P>(k, i, &ok);
        ok = ok && a.bytes == b.bytes && a.value == b.value && a.dst == b.dst && (a.bytes % 16 == 0 || ends) &&
            uint64_t(d.packedGridX - ends) * chunk >= a.bytes / 16 * 16;
    }
    return ok;
}

#define CHECK(c)                                             \
    do {                                                     \
        if (!(c)) {                                          \
            std::printf("line %d: not so: %s\n", __LINE__, #c); \
            std::exit(1);                                    \
        }                                                    \
    } while (0)

// Both sides of the lines up to which a call goes out with its records in the arguments.
void CheckLimits()
{
    const uint64_t mib = uint64_t(1) << 20;
    for (uint32_t p : {2u, 8u, 9u, 14u, 16u, 27u, 28u, 32u}) {
        for (int dtype : {HCCL_DATA_TYPE_BFP16, HCCL_DATA_TYPE_INT8, HCCL_DATA_TYPE_FP32}) {
            for (int op : {HCCL_REDUCE_SUM, HCCL_REDUCE_PROD, HCCL_REDUCE_MAX, HCCL_REDUCE_MIN}) {
                const bool bf16 = dtype == HCCL_DATA_TYPE_BFP16 && p >= 16, even = dtype == HCCL_DATA_TYPE_FP32 && p > 3;
                const bool selects = op == HCCL_REDUCE_MAX || op == HCCL_REDUCE_MIN;
                const uint64_t whole = even ? 5 * mib / 2 : bf16 && !selects ? 13 * mib / 4 : 4 * mib;
                const uint64_t ragged = !bf16 ? 4 * mib : !selects ? 11 * mib / 4 : p >= 28 ? 13 * mib / 4 : 4 * mib;
                auto fits = [&](int coll, uint64_t bytes) { return DirectFits(coll, p, bytes, dtype) && !CombiningBound(coll, p, bytes, dtype, op); };
                CHECK(fits(COLL_REDUCE, whole) && !fits(COLL_REDUCE, whole + 16));
                CHECK(fits(COLL_REDUCESCATTER, whole / p / 16 * 16) && !fits(COLL_REDUCESCATTER, whole / p / 16 * 16 + 16));
                CHECK(fits(COLL_REDUCESCATTER, ragged / p / 16 * 16 - 4) && !fits(COLL_REDUCESCATTER, ragged / p / 16 * 16 + 20));
                CHECK(!CombiningBound(COLL_ALLREDUCE, p, 8 * mib, dtype, op));
            }
        }
    }
}

// Both sides of the windows in which the packed form goes on, by sixteenths of a tile for each CU.
void CheckWindows()
{
    struct Line {
        int coll;
        uint32_t least, most;
        int dtype;
        bool ragged;
        std::vector<uint32_t> edges;      // out, in, out, ...
    };
    const int ar = COLL_ALLREDUCE, rs = COLL_REDUCESCATTER, fp32 = HCCL_DATA_TYPE_FP32, int8 = HCCL_DATA_TYPE_INT8;
    const std::vector<Line> lines = {
        {ar, 2, 2, fp32, false, {192}}, {ar, 3, 3, fp32, false, {14}}, {ar, 4, 4, fp32, false, {24, 32, 96}}, {ar, 5, 7, fp32, false, {9}},
        {ar, 8, 8, int8, false, {11, 16, 22, 32, 48}}, {ar, 9, 15, fp32, false, {6}}, {ar, 16, 16, fp32, false, {11, 16, 22}},
        {ar, 16, 16, HCCL_DATA_TYPE_BFP16, false, {6, 16, 22}}, {ar, 16, 16, HCCL_DATA_TYPE_FP16, false, {6, 16, 22}}, {ar, 17, 32, fp32, false, {6}},
        {rs, 2, 2, fp32, false, {60, 64, 256}}, {rs, 3, 3, fp32, false, {24}}, {rs, 4, 4, fp32, false, {30, 32, 44}}, {rs, 4, 4, int8, false, {24, 32, 44}}, {rs, 5, 7, fp32, false, {18}},
        {rs, 8, 8, fp32, false, {24}}, {rs, 8, 8, int8, false, {21}}, {rs, 9, 15, fp32, false, {}}, {rs, 16, 16, fp32, false, {11, 17, 20}}, {rs, 17, 32, fp32, false, {}},
        {rs, 2, 2, fp32, true, {56}}, {rs, 3, 4, int8, true, {24}}, {rs, 5, 7, fp32, true, {14}}, {rs, 8, 8, fp32, true, {14, 16, 20}},
        {rs, 8, 8, int8, true, {14}}, {rs, 9, 15, fp32, true, {}}, {rs, 16, 16, fp32, true, {10}}, {rs, 17, 32, fp32, true, {}},
    };
    for (uint32_t numCu : {256u, 128u, 32u}) {
        const uint64_t sixteenth = uint64_t(numCu) * 1024;
        for (const Line &l : lines) {
            for (uint32_t p = l.least; p <= l.most; p++) {
                const uint64_t share = l.coll == rs ? p : 1;
                auto in = [&](uint64_t bytes) { return PackedFits(l.coll, p, bytes - (l.ragged ? 12 : 0), l.dtype, numCu); };
                bool inside = !l.edges.empty();
                CHECK(in(4096) == inside);
                for (uint32_t e : l.edges) {
                    const uint64_t upTo = e * sixteenth / share / 16 * 16;
                    CHECK(in(upTo) == inside);
                    inside = !inside;
                    CHECK(in(upTo + (l.ragged ? 32 : 16)) == inside);
                }
                CHECK(!in(uint64_t(1) << 32));
            }
        }
        CHECK(!PackedFits(COLL_ALLREDUCE, 1, 4096, fp32, numCu) && !PackedFits(COLL_ALLREDUCE, 33, 4096, fp32, numCu) && !PackedFits(COLL_REDUCE, 8, 4096, fp32, numCu));
    }
}

// Buffers off a boundary, both sides of the lines that hold for them.
void CheckOffBoundary()
{
    const uint64_t q = 256 * 1024;
    const int ar = COLL_ALLREDUCE, rs = COLL_REDUCESCATTER, type = HCCL_DATA_TYPE_BFP16;
    auto in = [&](int coll, uint32_t p, uint64_t quarters, uint64_t more, uint64_t sends, uint64_t recvs) {
        return PackedFits(coll, p, (quarters * q / (coll == rs ? p : 1)) / 16 * 16 + more, type, 256, 0x7f0000000000ull | sends, 0x7f0000000000ull | recvs);
    };
    const uint32_t allReduce[][2] = {{2, 12}, {3, 7}, {4, 7}, {6, 6}, {8, 6}, {12, 5}, {16, 5}, {32, 5}};
    for (const auto &l : allReduce) {
        CHECK(in(ar, l[0], l[1], 0, 2, 2) && !in(ar, l[0], l[1], 16, 2, 2) && !in(ar, l[0], l[1], 16, 3, 1));
        CHECK(in(ar, l[0], l[1], 16, 4, 4) && in(ar, l[0], l[1], 16, 2, 4) && in(ar, l[0], l[1], 16, 8, 1));
    }
    CHECK(!in(ar, 4, 20, 0, 6, 2) && in(ar, 4, 20, 0, 4, 4) && !in(ar, 8, 20, 0, 1, 1) && in(ar, 8, 20, 0, 1, 0) && !in(ar, 8, 40, 0, 2, 2) && in(ar, 8, 40, 0, 4, 4));
    const uint32_t blocks[][2] = {{2, 12}, {3, 8}, {4, 12}, {6, 12}, {8, 12}};
    for (const auto &l : blocks) {
        CHECK(in(rs, l[0], l[1], 0, 2, 0) && !in(rs, l[0], l[1], 16, 2, 0) && in(rs, l[0], l[1], 16, 0, 2) && in(rs, l[0], l[1], 16, 4, 4) && in(rs, l[0], l[1], 2, 2, 2));
    }
    CHECK(!in(rs, 16, 18, 0, 6, 0) && in(rs, 16, 18, 0, 4, 0) && !in(rs, 8, 20, 0, 2, 0));
    // off half a memory line the upper ends go, in place more
    CHECK(in(ar, 2, 64, 0, 4, 4) && !in(ar, 2, 64, 16, 4, 4) && in(ar, 2, 64, 16, 64, 4) && in(ar, 2, 64, 16, 4, 0) && !in(ar, 4, 80, 0, 16, 16) && in(ar, 4, 80, 0, 64, 64));
    CHECK(in(rs, 2, 200, 0, 0, 16) && !in(rs, 2, 200, 0, 8, 16) && in(rs, 2, 200, 0, 64, 16));
    const uint32_t ends[][5] = {{uint32_t(ar), 4, 24, 21, 0}, {uint32_t(ar), 8, 22, 21, 0}, {uint32_t(ar), 8, 48, 42, 0}, {uint32_t(ar), 16, 22, 21, 0}, {uint32_t(rs), 4, 30, 26, 0},
                                {uint32_t(rs), 4, 44, 41, 0}, {uint32_t(rs), 8, 24, 21, 0}};
    for (const auto &l : ends) {
        CHECK(in(l[0], l[1], l[2], 0, 0, 0) && !in(l[0], l[1], l[2], 16, 0, 0) && in(l[0], l[1], l[3], 0, 4, 4) && !in(l[0], l[1], l[3], 16, 4, 4) && in(l[0], l[1], l[3], 16, 64, 4));
    }
    auto inPlace = [&](uint32_t p, uint64_t quarters, uint64_t more, uint64_t at) {
        return PackedFits(ar, p, quarters * q + more, type, 256, 0x7f0000000000ull | at, 0x7f0000000000ull | at, true);
    };
    const uint32_t same[][2] = {{2, 12}, {3, 8}, {4, 7}, {6, 8}, {8, 7}, {16, 5}};
    for (const auto &l : same) {
        CHECK(inPlace(l[0], l[1], 0, 4) && !inPlace(l[0], l[1], 16, 4) && !inPlace(l[0], l[1], 16, 16) && inPlace(l[0], l[1], 16, 64));
    }
    CHECK(inPlace(12, 6, 0, 4) && inPlace(32, 6, 0, 16) && !inPlace(4, 15, 0, 4) && !inPlace(8, 20, 0, 4) && in(ar, 8, 20, 0, 4, 4));
}

}  // namespace

int main(int argc, char **argv)
{
    CheckLimits();
    CheckWindows();
    CheckOffBoundary();
    const long want = argc > 1 ? std::atol(argv[1]) : 3000;
    long taken[3] = {0, 0, 0}, unlike = 0, apart = 0, trees = 0, inPlace = 0;
    for (long n = 0; n < want;) {
        PlanRequest rq;
        const int colls[] = {COLL_ALLREDUCE, COLL_ALLREDUCE, COLL_REDUCESCATTER, COLL_ALLGATHER, COLL_BROADCAST, COLL_REDUCE, COLL_SCATTER};
        rq.coll = CollKind(colls[Below(Below(4) ? 4 : 7)]);
        const Algo algos[] = {ALGO_RING, ALGO_RING, ALGO_MESH, ALGO_MESH_ATOMIC, ALGO_RHD};
        rq.algo = algos[Below(5)];
        rq.p = uint32_t(Below(3) ? 1 + Below(8) : 1 + Below(40));
        if (rq.algo == ALGO_MESH && rq.p > 12) {
            rq.p = uint32_t(2 + Below(11));
        }
        if (rq.coll == COLL_SCATTER) {
            rq.algo = ALGO_MESH;
        }
        if (Below(8) == 0 && rq.p % 2 == 0 && rq.p > 2) {
            rq.servers = 2;
        }
        const uint32_t units[] = {1, 2, 4, 8};
        rq.unit = units[Below(4)];
        rq.root = uint32_t(Below(rq.p));
        const bool same = rq.coll == COLL_BROADCAST || (rq.coll == COLL_ALLREDUCE && Below(2));
        rq.alias.assign(rq.p, same ? 1 : 0);
        rq.count = 1 + Below(Below(2) ? 300 : Below(4) ? 40000 / rq.p : 12000000 / rq.unit);
        Plan plan;
        std::string err;
        DirectLaunch d;
        if (BuildPlan(rq, &plan, &err) != 0 || !BuildDirect(plan, true, 4, 0, &d)) {
            continue;
        }
        n++;
        PackDirect(plan, true, 4, 0, &d);
        // (sums of fp32: both batches of many sources in flight, up to 1 MiB where there is more than one destination)
        uint64_t total = 0;
        for (const FusedItem &f : plan.fused) {
            total += f.bytes;
        }
        const FusedItem &item = plan.fused[0];
        const bool two = d.packedFunc != nullptr && item.kind == FK_CHAIN && item.src.size() >= 24 && (item.dst.size() == 1 || total <= 1u << 20);
        if (d.packedTwoFunc != (two ? LookupKernel(0, 0, KernelKind(item.src.size() == 32 ? KK_PACKED_TWO + 1 : KK_PACKED_TWO)) : nullptr)) {
            std::printf("coll %d p %u total %llu: the kernel for %u sources\n", int(rq.coll), rq.p, (unsigned long long)total, item.src.size());
            return 1;
        }
        const bool usual = rq.p <= 32 && rq.servers == 1 &&
            ((rq.coll == COLL_ALLGATHER) || ((rq.coll == COLL_ALLREDUCE || rq.coll == COLL_REDUCESCATTER) &&
                (rq.algo == ALGO_RING || rq.algo == ALGO_MESH_ATOMIC || (rq.algo == ALGO_RHD && (rq.p & (rq.p - 1)) == 0))));
        if (usual && rq.p > 1 && d.packedFunc == nullptr) {
            std::printf("coll %d algo %d p %u count %llu unit %u: not taken\n", int(rq.coll), int(rq.algo), rq.p, (unsigned long long)rq.count, rq.unit);
            return 1;
        }
        // several sets of buffers: near one another, at odd addresses, and, now and then, too far apart for 32 bits
        for (int set = 0; set < 3; set++) {
            const uint64_t align[] = {512, 1, 4096, 2, 16, 256};
            const uint64_t grain = align[Below(6)], reach = set == 2 ? uint64_t(1) << (33 + Below(13)) : uint64_t(1) << (24 + Below(8));
            std::vector<void *> send(rq.p), recv(rq.p);
            for (uint32_t r = 0; r < rq.p; r++) {
                send[r] = reinterpret_cast<void *>(0x7f0000000000ull + Below(reach) / grain * grain);
                recv[r] = same ? send[r] : reinterpret_cast<void *>(0x7f0000000000ull + Below(reach) / grain * grain);
            }
            const bool hit = FillBases(&d, send, recv);
            if (hit && set == 0) {
                std::printf("a first call's buffers counted as seen\n");
                return 1;
            }
            if (!d.usePacked) {
                apart += d.packedFunc != nullptr;
                if (d.packedFunc != nullptr && set < 2) {
                    std::printf("buffers within 2 GiB not taken\n");
                    return 1;
                }
                continue;
            }
            const bool ok = d.packedRanks == 8 ? Same<8>(plan, d, send, recv) : d.packedRanks == 16 ? Same<16>(plan, d, send, recv) : Same<32>(plan, d, send, recv);
            if (!ok || rq.p > d.packedRanks) {
                std::printf("coll %d algo %d p %u servers %u count %llu unit %u: the arguments are not the plan's items\n", int(rq.coll), int(rq.algo), rq.p,
                    rq.servers, (unsigned long long)rq.count, rq.unit);
                return 1;
            }
            inPlace += same;
        }
        unlike += d.packedFunc == nullptr;
        trees += d.packedFunc != nullptr && plan.fused[0].kind == FK_TREE;
        if (d.packedFunc != nullptr) {
            taken[d.packedRanks == 8 ? 0 : d.packedRanks == 16 ? 1 : 2]++;
        }
    }
    std::printf("OK up to 8 ranks %ld 16 ranks %ld 32 ranks %ld trees %ld in place %ld unlike %ld too far apart %ld wide %ld in fours %ld\n", taken[0], taken[1], taken[2], trees,
        inPlace, unlike, apart, g_wide, g_fours);
    return 0;
}
