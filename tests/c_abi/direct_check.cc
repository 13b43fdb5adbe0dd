// Small collectives (cann-hccl_amd/csrc/direct.cc) against the planner, on the host: a seeded walk over requests.
//   - DirectFits weighs a collective from its call alone; what it takes the collective to move has to be what the plan moves.
//   - The kernel arguments that BuildDirect makes are read back as the kernels of kernels_direct.h read them; every item has
//     to be the plan's item: the same expression over the same ranges, the same destinations.
//   - Where a plan is turned away, one of the records' limits has to be exceeded.
// argv[1] = requests.  Prints how many went which way.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <string>
#include <vector>

#include "runtime.h"

namespace hcclamd {
// the kernels are not linked: any address that tells narrow from wide
static const char g_narrow = 0, g_wide = 0;
const void *LookupKernel(int, int, KernelKind kind) { return kind == KK_DIRECT ? &g_narrow : &g_wide; }
const void *LookupCopyKernel(KernelKind kind) { return kind == KK_DIRECT ? &g_narrow : &g_wide; }
}  // namespace hcclamd

using namespace hcclamd;

namespace {

uint64_t g_state = 0x9E3779B97F4A7C15ull;
uint64_t Below(uint64_t n)
{
    g_state = g_state * 6364136223846793005ull + 1442695040888963407ull;
    return n == 0 ? 0 : (g_state >> 29) % n;
}

std::string Range(uint32_t rank, uint32_t buf, uint64_t off)
{
    return std::to_string(rank) + (buf == BUF_SEND ? "s" : "r") + "@" + std::to_string(off);
}
std::string Range(const Ref &r) { return Range(r.rank, r.buf, r.off); }
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

// The stack machine of both descriptions: source j is pushed, then ops[j] & 7 folds.
template <typename Src, typename Op> std::string Stack(uint32_t nsrc, Src src, Op op, size_t *depth)
{
    std::vector<std::string> st;
    for (uint32_t j = 0; j < nsrc; j++) {
        st.push_back(src(j));
        *depth = std::max(*depth, st.size());
        for (uint32_t f = 0; f < (op(j) & 7u) && st.size() >= 2; f++) {
            const std::string top = st.back();
            st.pop_back();
            st.back() = ((op(j) >> (8 + f)) & 1u) ? Both(st.back(), top) : Both(top, st.back());
        }
    }
    return st.size() == 1 ? st[0] : "unfinished";
}

std::string OfPlan(const FusedItem &f)
{
    if (f.kind == FK_TREE) {
        std::vector<std::string> leaf;
        for (uint32_t i = 0; i < f.nleaf; i++) {
            leaf.push_back(f.srcValid[2 * i + 1] ? Both(Range(f.src[2 * i]), Range(f.src[2 * i + 1])) : Range(f.src[2 * i]));
        }
        return Pairwise(leaf);
    }
    if (f.kind == FK_STACK) {
        size_t depth = 0;
        return Stack(uint32_t(f.src.size()), [&](uint32_t j) { return Range(f.src[j]); }, [&](uint32_t j) { return uint32_t(f.ops[j]); }, &depth);
    }
    std::string acc = Range(f.src[0]);
    for (size_t j = 1; j < f.src.size(); j++) {
        acc = f.accLeft[j] ? Both(acc, Range(f.src[j])) : Both(Range(f.src[j]), acc);
    }
    return acc;
}

template <uint32_t CAP> struct View {
    const DirectArgs<CAP> *args;
    const DirectItem<CAP> *it;
    const DirectLaunch *d;
    bool ok = true;
    uint32_t Index(const uint32_t *list, uint32_t words, uint32_t j)
    {
        const uint32_t i = (j >> 2) < words ? (list[j >> 2] >> (8u * (j & 3u))) & 0xffu : ~0u;
        ok = ok && i < d->bases.size() && i < kDirectBases<CAP>;
        return ok ? i : 0;
    }
    std::string Src(uint32_t j)
    {
        const auto &b = d->bases[Index(it->src, sizeof(it->src) / 4, j)];
        return Range(b.first, b.second, it->srcOff);
    }
    std::string Dst(uint32_t k)
    {
        const auto &b = d->bases[Index(it->dst, sizeof(it->dst) / 4, k)];
        return Range(b.first, b.second, it->dstOff);
    }
    std::string Value()
    {
        if (it->kind == DIRECT_CHAIN) {
            std::string acc = Src(0);
            for (uint32_t j = 1; j < it->nsrc; j++) {
                acc = ((it->accLeft >> j) & 1u) ? Both(acc, Src(j)) : Both(Src(j), acc);
            }
            ok = ok && it->nsrc >= 1 && it->nsrc <= CAP;
            return acc;
        }
        if (it->kind == DIRECT_TREE) {
            ok = ok && (it->nleaf == 1 || it->nleaf == 2 || it->nleaf == 4 || it->nleaf == 8 || (CAP > 8 && (it->nleaf == 16 || it->nleaf == 32))) &&
                (it->nleaf <= kDirectSecond<CAP> || it->second == 0);
            std::vector<std::string> leaf;
            for (uint32_t i = 0; i < it->nleaf; i++) {
                const std::string a = Src(i);
                if (it->second != 0) {
                    Src(kDirectSecond<CAP> + i);      // the kernel reads it whether there is one or not
                }
                leaf.push_back(((it->second >> i) & 1u) ? Both(a, Src(kDirectSecond<CAP> + i)) : a);
            }
            return Pairwise(leaf);
        }
        ok = ok && it->kind == DIRECT_STACK && CAP == 8 && it->nsrc <= 8;
        for (uint32_t j = 0; j < 8; j++) {
            Src(j);
        }
        size_t depth = 0;
        const std::string v = Stack(it->nsrc, [&](uint32_t j) { return Src(j); },
            [&](uint32_t j) { return (it->ops[(j >> 1) % (sizeof(it->ops) / 4)] >> (16u * (j & 1u))) & 0xffffu; }, &depth);
        ok = ok && depth <= 4;                         // what DirectStack has room for
        return v;
    }
};

template <uint32_t CAP> bool Same(const Plan &plan, const DirectLaunch &d)
{
    if (d.image.size() != sizeof(DirectArgs<CAP>) || d.gridY != plan.fused.size() || d.gridY > kDirectItems<CAP>) {
        return false;
    }
    const DirectArgs<CAP> *args = reinterpret_cast<const DirectArgs<CAP> *>(d.image.data());
    for (size_t n = 0; n < plan.fused.size(); n++) {
        const FusedItem &f = plan.fused[n];
        View<CAP> v{args, &args->item[n], &d};
        if (v.it->bytes != f.bytes || v.it->ndst != f.dst.size() || uint64_t(d.gridX - 1) * kDirectChunk < f.bytes || v.Value() != OfPlan(f)) {
            return false;
        }
        for (uint32_t k = 0; k < v.it->ndst; k++) {
            if (v.Dst(k) != Range(f.dst[k])) {
                return false;
            }
        }
        for (uint32_t k = 0; k < (v.it->ndst + 7) / 8 * 8; k++) {
            v.Dst(k);                                  // fetched eight at a time
        }
        if (!v.ok) {
            return false;
        }
    }
    return true;
}

// Whether the records of `CAP` hold the plan.
template <uint32_t CAP> bool Fits(const Plan &plan)
{
    std::vector<std::pair<uint32_t, uint8_t>> bases;
    auto base = [&](const Ref &r) {
        if (std::find(bases.begin(), bases.end(), std::make_pair(r.rank, r.buf)) == bases.end()) {
            bases.emplace_back(r.rank, r.buf);
        }
    };
    for (const FusedItem &f : plan.fused) {
        const uint32_t sources = f.kind == FK_TREE ? f.nleaf : uint32_t(f.src.size());
        if (sources > CAP || f.dst.size() > CAP || (f.kind == FK_STACK && CAP > 8)) {
            return false;
        }
        for (size_t k = 0; k < f.src.size(); k++) {
            if (f.srcValid[k]) {
                base(f.src[k]);
                if (f.src[k].off != f.src[0].off || (f.kind == FK_TREE && f.nleaf > kDirectSecond<CAP> && (k & 1) != 0)) {
                    return false;
                }
            }
        }
        for (const Ref &r : f.dst) {
            base(r);
            if (r.off != f.dst[0].off) {
                return false;
            }
        }
    }
    return plan.fused.size() <= kDirectItems<CAP> && bases.size() <= kDirectBases<CAP>;
}

}  // namespace

int main(int argc, char **argv)
{
    const long want = argc > 1 ? std::atol(argv[1]) : 3000;
    // results, results to one destination each, the same of whole vectors, traffic
    const uint64_t limits[] = {uint64_t(1) << 20, uint64_t(4) << 20, uint64_t(5) << 19, uint64_t(20) << 20};
    long narrow = 0, wide = 0, trees = 0, seconds = 0, stacks = 0, away = 0, large = 0, edges = 0;
    for (long n = 0; n < want;) {
        PlanRequest rq;
        const int colls[] = {COLL_ALLREDUCE, COLL_ALLREDUCE, COLL_ALLREDUCE, COLL_REDUCESCATTER, COLL_ALLGATHER, COLL_BROADCAST, COLL_REDUCE, COLL_SCATTER,
            COLL_SENDRECV};
        rq.coll = CollKind(colls[Below(9)]);
        const Algo algos[] = {ALGO_RING, ALGO_RING, ALGO_MESH, ALGO_MESH_ATOMIC, ALGO_RHD};
        rq.algo = algos[Below(5)];
        rq.p = uint32_t(Below(3) ? 1 + Below(8) : 1 + Below(40));
        if (rq.algo == ALGO_MESH && rq.p > 12) {
            rq.p = uint32_t(2 + Below(11));
        }
        if (rq.coll == COLL_SCATTER) {
            rq.algo = Below(2) ? ALGO_MESH : ALGO_RING;
        } else if (rq.coll >= COLL_SENDRECV) {
            rq.algo = ALGO_RING;
        }
        if (Below(3) == 0 && rq.coll != COLL_SENDRECV) {
            const uint32_t s = uint32_t(2 + Below(3));
            if (rq.p % s == 0 && rq.p > s) {
                rq.servers = s;
                rq.level0Rings = rq.p / s == 8 && Below(2) ? 4 : uint32_t(Below(2));
            }
        }
        const int dtype = int(Below(12));
        const uint32_t units[] = {1, 2, 4, 2, 4, 8, 8, 1, 2, 4, 8, 2};
        rq.unit = units[dtype];
        rq.root = uint32_t(Below(rq.p));
        rq.peer = rq.coll == COLL_SENDRECV && rq.p > 1 ? (rq.root + 1 + uint32_t(Below(rq.p - 1))) % rq.p : 0;
        rq.alias.assign(rq.p, 0);
        if ((rq.coll == COLL_ALLREDUCE && Below(2)) || rq.coll == COLL_BROADCAST) {
            rq.alias.assign(rq.p, 1);
        }
        // mostly small counts of every length; every fourth one at the limit of its collective
        const uint64_t weight = rq.coll == COLL_ALLGATHER ? uint64_t(rq.p) * (rq.p + 1) : rq.coll == COLL_BROADCAST ? rq.p
            : rq.coll == COLL_SCATTER ? uint64_t(rq.p) * 2 : rq.coll == COLL_SENDRECV ? 2 : rq.coll == COLL_REDUCESCATTER ? rq.p : 1;
        const bool copies = rq.coll == COLL_ALLGATHER || rq.coll == COLL_BROADCAST || rq.coll == COLL_SCATTER || rq.coll == COLL_SENDRECV;
        const bool toOne = !copies && (rq.coll != COLL_ALLREDUCE || rq.p == 1);
        uint64_t limit = copies ? limits[3] : toOne ? limits[1 + Below(2)] : limits[0];
        const uint64_t most = limit / weight / rq.unit;
        const bool edge = Below(4) == 0;
        rq.count = edge ? most + Below(2) : 1 + Below(Below(2) ? 500 : most);
        if (toOne) {
            const bool wide = dtype != HCCL_DATA_TYPE_INT8 && dtype != HCCL_DATA_TYPE_UINT8 && dtype != HCCL_DATA_TYPE_BFP16;
            limit = limits[rq.count * rq.unit % 16 == 0 && rq.p > 3 && wide ? 2 : 1];
        }
        Plan plan;
        std::string err;
        if (BuildPlan(rq, &plan, &err) != 0) {
            continue;                                   // a combination the planner does not take
        }
        n++;
        const uint64_t bytes = rq.count * rq.unit;
        const bool fits = DirectFits(rq.coll, rq.p, bytes, dtype);
        const bool reduceColl = !copies;
        if (plan.fusedOk) {
            uint64_t results = 0, traffic = 0;
            for (const FusedItem &f : plan.fused) {
                results += f.bytes;
                traffic += f.bytes * (1 + f.dst.size());
            }
            // (nothing to move for one rank in place)
            if (!plan.fused.empty() && (copies ? traffic : results) != weight * bytes) {
                std::printf("coll %d p %u servers %u count %llu: weighed as %llu, moves %llu\n", int(rq.coll), rq.p, rq.servers,
                    (unsigned long long)rq.count, (unsigned long long)(weight * bytes), (unsigned long long)(copies ? traffic : results));
                return 1;
            }
        }
        if (fits != (weight * bytes <= limit)) {
            std::printf("coll %d p %u bytes %llu: DirectFits says %d\n", int(rq.coll), rq.p, (unsigned long long)bytes, int(fits));
            return 1;
        }
        edges += edge;
        if (!fits) {
            large++;
            continue;
        }
        DirectLaunch d;
        const bool built = BuildDirect(plan, reduceColl, 4, 0, &d);
        if (built != (plan.fusedOk && !plan.fused.empty() && (Fits<8>(plan) || Fits<32>(plan)))) {
            std::printf("coll %d algo %d p %u servers %u count %llu: built %d\n", int(rq.coll), int(rq.algo), rq.p, rq.servers, (unsigned long long)rq.count, built);
            return 1;
        }
        if (!built) {
            away++;
            continue;
        }
        const bool isNarrow = d.func == LookupCopyKernel(KK_DIRECT);
        if (isNarrow != Fits<8>(plan) || !(isNarrow ? Same<8>(plan, d) : Same<32>(plan, d)) || d.sendBytes != plan.sendBytes ||
            d.recvBytes != plan.recvBytes) {
            std::printf("coll %d algo %d p %u servers %u level0 %u count %llu unit %u: the arguments are not the plan's items\n", int(rq.coll), int(rq.algo),
                rq.p, rq.servers, rq.level0Rings, (unsigned long long)rq.count, rq.unit);
            return 1;
        }
        (isNarrow ? narrow : wide)++;
        for (const FusedItem &f : plan.fused) {
            trees += f.kind == FK_TREE;
            stacks += f.kind == FK_STACK;
            seconds += f.kind == FK_TREE && std::count(f.srcValid.begin(), f.srcValid.end(), uint8_t(1)) > int(f.nleaf);
        }
    }
    std::printf("OK narrow %ld wide %ld tree items %ld with second sources %ld stack items %ld turned away %ld too large %ld at a limit %ld\n", narrow,
        wide, trees, seconds, stacks, away, large, edges);
    return 0;
}
