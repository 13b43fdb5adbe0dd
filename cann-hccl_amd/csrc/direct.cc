// Small collectives: from a plan to one launch whose descriptors ride in the kernel arguments (kernels_direct.h).
#include <algorithm>
#include <cstring>

#include "runtime.h"

namespace hcclamd {

namespace {

// Where the tile kernels become the better form: they keep four times as much in flight per lane, which pays once every
// CU has work.  Measured (us per collective among others, tile kernels / this form):
//   all-reduce, 8 ranks, bf16 ring: 512 KiB 5.9 / 3.6, 1 MiB 7.1 / 5.3, 2 MiB 8.2 / 8.0, 4 MiB 12.1 / 13.9;
//     fp32 ring 1 MiB 6.0 / 5.7, 2 MiB 7.0 / 7.9; 16 ranks 1 MiB 10.7 / 8.7, 2 MiB 12.9 / 14.8;
//     halving-doubling, bf16, 24 ranks 256 KiB 16.9 / 6.5, 1 MiB 20.8 / 13.7
//   reduce-scatter, 8 ranks, bf16 (bytes received by all ranks): 2 MiB 6.8 / 4.9, 4 MiB 8.2 / 7.7, 8 MiB 13.5 / 13.5
//   all-gather (bytes sent by all ranks): 8 ranks 2 MiB 4.3 / 4.1, 4 MiB 6.9 / 6.9, 8 MiB 12.6 / 14.3;
//     16 ranks 1 MiB 5.1 / 4.2, 2 MiB 6.7 / 6.8
constexpr uint64_t kDirectMaxBytes = uint64_t(1) << 20;       // of a reduction's results
constexpr uint64_t kDirectMaxToOne = uint64_t(4) << 20;       // the same where each has one destination
// Blocks of whole 16-byte vectors of more than three sources, in types that combine in an instruction or two: the tile
// kernels get ahead sooner there.  Tile kernels / this form, us, new data for every call, one destination per result:
//   reduce-scatter, fp32: 4 ranks 2.5 MiB 5.1 / 5.1, 4 MiB 6.1 / 6.2; 16 ranks 2.5 MiB 10.4 / 9.7, 3 MiB 11.3 / 11.9;
//     32 ranks 2.5 MiB 17.6 / 16.5, 4 MiB 23.5 / 24.8; int64 32 ranks 3 MiB 18.5 / 20.5
//   reduce, fp32: 8 ranks 2.5 MiB 6.8 / 6.3, 4 MiB 8.5 / 8.8; 32 ranks 2.5 MiB 17.2 / 16.3, 4 MiB 22.8 / 25.4
// Up to the larger limit this form stays ahead for bf16 and 8-bit elements (32 ranks, 4 MiB: bf16 27.6 / 25.1, int8 26.3 / 25.1)
// and for ragged blocks, whose ends the tile kernels take element by element (fp32, 32 ranks, 4 MiB 62.9 / 27.6), and for three sources or fewer (3 ranks, 4 MiB 6.2 / 5.4).
// Copies, also from one to one, are ahead up to their limit for 2 to 32 ranks (scatter of 10 MiB 6.4 / 6.0).
constexpr uint64_t kDirectMaxToOneEven = uint64_t(5) << 19;
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

bool FillBases(DirectLaunch *d, const std::vector<void *> &send, const std::vector<void *> &recv)
{
    uint64_t *base = reinterpret_cast<uint64_t *>(d->image.data());     // DirectArgs<>::base comes first
    bool same = true;
    for (size_t i = 0; i < d->bases.size(); i++) {
        const uint64_t p = reinterpret_cast<uint64_t>((d->bases[i].second == BUF_SEND ? send : recv)[d->bases[i].first]);
        same = same && base[i] == p;
        base[i] = p;
    }
    return same;
}

}  // namespace hcclamd
