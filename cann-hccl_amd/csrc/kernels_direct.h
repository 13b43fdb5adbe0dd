// Small collectives: one launch whose descriptors ride in the kernel arguments.
//
// A small collective is latency and nothing else.  The tile kernels reach their data through a chain of dependent
// loads (argument -> item table -> pointer pool -> data) and wait for one destination pointer after the other, and
// their tables have to be in device memory first.  Here an item's record lies at a place that follows from the block
// index, all of its pointers are fetched together, and the data loads of up to 16 sources are issued back to back
// without a branch between them (the number of sources picks straight-line code; a guard per source makes the compiler
// wait for each load).  What a launch takes on the device, us, first in first out, 8 ranks: an empty kernel 1.6, all-reduce of fp32 8 KiB per
// rank 3.5 with a branch per destination, a trip per pointer, and all shapes in one kernel, 2.2 this way; bf16 64 KiB 3.6 / 2.5, 1 MiB 5.9 / 3.4.
// No table is uploaded or kept, so a call with new buffers costs what a repeated one does.
//
// A workgroup is one wave and handles 1 KiB of one item (blockIdx.y), one 16-byte vector per lane: what a CU has in flight limits it, so
// the work has to spread evenly over the CUs.  8 ranks, fp32, workgroups of 4 KiB / 2 KiB / 1 KiB: 64 KiB 2.5 / 2.2 / 2.2, 1.25 MiB 4.4 / 3.9 / 3.3,
// 2.25 MiB 7.6 / 7.1 / 6.5 (2 MiB, a whole number of 4 KiB to a CU: 5.6 / 5.9 / 5.8).  Accesses are unaligned 128-bit ones (the instruction is the same
// one), so one form serves every alignment; the bytes behind the last whole vector go element by element to a workgroup of their own
// (blockIdx.x == 0), side by side with the others.
//
// Two kinds of arguments: a record per item, and for items that are alike, the usual collective, one record for all (PackedArgs).
#pragma once
#include <type_traits>

#include "kernels_impl.h"

namespace hcclamd {

// The kernel arguments where they lie (constant memory): read through the parameter itself, the wide form is copied to
// private memory first.
#define HCCL_CONSTANT __attribute__((address_space(4)))
// All of these, fetched before anything behind it: on its own the compiler waits for one before it asks for the next.
template <uint32_t N, typename W> __device__ __forceinline__ void Fetched(const W (&w)[N])
{
    if constexpr (N == 1) {
        asm volatile("" ::"s"(w[0]));
    } else if constexpr (N < 4) {
        asm volatile("" ::"s"(w[0]), "s"(w[1]), "s"(w[N - 1]));
    } else if constexpr (N < 8) {
        asm volatile("" ::"s"(w[0]), "s"(w[1]), "s"(w[2]), "s"(w[3]), "s"(w[N > 4 ? 4 : 0]), "s"(w[N > 5 ? 5 : 0]), "s"(w[N > 6 ? 6 : 0]));
    } else if constexpr (N == 8) {
        asm volatile("" ::"s"(w[0]), "s"(w[1]), "s"(w[2]), "s"(w[3]), "s"(w[4]), "s"(w[5]), "s"(w[6]), "s"(w[7]));
    } else {
        static_assert(N == 16, "how many are fetched together");
        asm volatile("" ::"s"(w[0]), "s"(w[1]), "s"(w[2]), "s"(w[3]), "s"(w[4]), "s"(w[5]), "s"(w[6]), "s"(w[7]), "s"(w[8]), "s"(w[9]),
            "s"(w[10]), "s"(w[11]), "s"(w[12]), "s"(w[13]), "s"(w[14]), "s"(w[15]));
    }
}

template <uint32_t CAP> struct DirectView {
    typedef uint64_t Word;       // what there is of a pointer in the arguments
    static constexpr bool kMany = CAP > 8;
    const DirectArgs<CAP> HCCL_CONSTANT *args;
    const DirectItem<CAP> HCCL_CONSTANT *it;
    __device__ __forceinline__ DirectView()
    {
        args = (const DirectArgs<CAP> HCCL_CONSTANT *)__builtin_amdgcn_kernarg_segment_ptr();
        it = &args->item[blockIdx.y];
        // the words every item needs, in one go: fetched where they are used they are one trip to memory each
        asm volatile("" ::"s"(it->bytes), "s"(it->srcOff), "s"(it->dstOff), "s"(it->nsrc), "s"(it->ndst), "s"(it->kind), "s"(it->src[0]),
            "s"(it->src[1]), "s"(it->dst[0]), "s"(it->dst[1]));
    }
    __device__ __forceinline__ uint32_t Bytes() const { return it->bytes; }
    __device__ __forceinline__ uint32_t SrcOff() const { return it->srcOff; }
    __device__ __forceinline__ uint32_t DstOff() const { return it->dstOff; }
    __device__ __forceinline__ uint32_t Sources() const { return it->nsrc; }
    __device__ __forceinline__ uint32_t Destinations() const { return it->ndst; }
    // base pointer of entry j of the list of sources / destinations (base indexes, four to a word)
    __device__ __forceinline__ Word Src(uint32_t j) const { return args->base[(it->src[j >> 2] >> (8u * (j & 3u))) & 0xffu]; }
    __device__ __forceinline__ Word Dst(uint32_t k) const { return args->base[(it->dst[k >> 2] >> (8u * (k & 3u))) & 0xffu]; }
    __device__ __forceinline__ uint64_t Pointer(Word w) const { return w; }
};
template <uint32_t P> struct PackedView {
    typedef uint32_t Word;
    static constexpr bool kMany = P > 8;
    static constexpr uint32_t kRanks = P;
    const PackedArgs<P> HCCL_CONSTANT *k;
    __device__ __forceinline__ PackedView()
    {
        k = (const PackedArgs<P> HCCL_CONSTANT *)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" ::"s"(k->base), "s"(k->first), "s"(k->last), "s"(k->srcStep), "s"(k->dstStep), "s"(k->info), "s"(k->order[0]));
    }
    __device__ __forceinline__ uint32_t Field(uint32_t at) const { return (k->info >> at) & 63u; }
    __device__ __forceinline__ uint32_t Bytes() const
    {
        // (a choice between the two is turned into one between their addresses, another trip)
        const uint32_t f = k->first, l = k->last;
        return l ^ ((f ^ l) & (blockIdx.y + 1 == Field(kPackedItems) ? 0u : ~0u));
    }
    __device__ __forceinline__ uint32_t SrcOff() const { return blockIdx.y * k->srcStep; }
    __device__ __forceinline__ uint32_t DstOff() const { return blockIdx.y * k->dstStep; }
    __device__ __forceinline__ uint32_t Sources() const { return Field(kPackedSources); }
    __device__ __forceinline__ uint32_t Destinations() const { return k->info & kPackedToOne ? 1u : Field(kPackedModulus); }
    __device__ __forceinline__ uint64_t Pointer(Word w) const { return k->base + (uint64_t(w) << Field(kPackedShift)); }
    __device__ __forceinline__ uint32_t Order(uint32_t j) const
    {
        return P > 16 ? (k->order[(j >> 2) & 7u] >> (8u * (j & 3u))) & 0xffu : (k->order[(j >> 3) & (P / 8 - 1)] >> (4u * (j & 7u))) & 15u;
    }
    // source j of a chain, of a tree
    __device__ __forceinline__ Word Src(uint32_t j) const
    {
        const uint32_t sum = Order(j) + blockIdx.y, mod = Field(kPackedModulus);
        return k->off[min(sum, sum - mod)];       // (below the modulus the difference wraps around)
    }
    __device__ __forceinline__ Word Leaf(uint32_t j) const { return k->off[Order(j) ^ blockIdx.y]; }
    __device__ __forceinline__ Word Dst(uint32_t n) const { return k->off[P + (k->info & kPackedToOne ? blockIdx.y : n)]; }
};

// Which KiB of its item a workgroup takes.  Many sources (kPackedFours, direct.cc): four in a row go to one XCD (workgroup b runs on XCD b % 8), in groups of 32,
// as they did with workgroups of 4 KiB; where the sources lie a power of two apart, an XCD that takes every eighth KiB of each meets the same few channels with all of them.
__device__ __forceinline__ uint32_t KiBOf(uint32_t x, uint32_t bytes, bool inFours)
{
    return inFours && ((x | 31u) + 1u) * kDirectChunk <= bytes ? (x & ~31u) + (x & 7u) * 4u + ((x >> 3) & 3u) : x;
}

// N sources from source j0 on into acc; FIRST: the first of them starts it.  left(j): the value so far is the left operand.
template <typename L, typename T, int OP, uint32_t N, bool FIRST, typename View, typename Left>
__device__ __forceinline__ void DirectBatch(const View &view, uint32_t j0, uint32_t off, typename L::Val &acc, Left left)
{
    typename View::Word p[N];
#pragma unroll
    for (uint32_t j = 0; j < N; j++) {
        p[j] = view.Src(j0 + j);
    }
    Fetched(p);
    typename L::Val v[N];
#pragma unroll
    for (uint32_t j = 0; j < N; j++) {
        v[j] = L::Load(reinterpret_cast<const void *>(view.Pointer(p[j])), off);
    }
    PinAccesses();
#pragma unroll
    for (uint32_t j = 0; j < N; j++) {
        if (FIRST && j == 0) {
            acc = v[0];
        } else if (OrderMatters<T, OP>::value && !left(j0 + j)) {
            acc = L::Combine(v[j], acc);
        } else {
            acc = L::Combine(acc, v[j]);
        }
    }
}

// The first N + M sources, all in flight before the first is combined.  With the second batch asked for behind the first one's combining, us, one after the other / this
// way: all-reduce, bf16, 32 ranks 512 KiB 7.9 / 6.9, 768 KiB 10.2 / 9.1, 24 ranks 1 MiB 10.8 / 9.1; reduce-scatter of 32 ranks, results of 2 MiB in all 14.4 / 12.3; fp32, 32
// ranks' reduce of 1 MiB 7.5 / 6.7.
template <typename L, typename T, int OP, uint32_t N, uint32_t M, typename View, typename First, typename Later>
__device__ __forceinline__ void DirectTwoBatches(const View &view, uint32_t off, typename L::Val &acc, First first, Later later)
{
    typename View::Word p[N], q[M];
#pragma unroll
    for (uint32_t j = 0; j < N; j++) {
        p[j] = view.Src(j);
    }
    Fetched(p);
    typename L::Val v[N], w[M];
#pragma unroll
    for (uint32_t j = 0; j < N; j++) {
        v[j] = L::Load(reinterpret_cast<const void *>(view.Pointer(p[j])), off);
    }
#pragma unroll
    for (uint32_t j = 0; j < M; j++) {
        q[j] = view.Src(N + j);
    }
    Fetched(q);
#pragma unroll
    for (uint32_t j = 0; j < M; j++) {
        w[j] = L::Load(reinterpret_cast<const void *>(view.Pointer(q[j])), off);
    }
    PinAccesses();
    acc = v[0];
#pragma unroll
    for (uint32_t j = 1; j < N; j++) {
        acc = OrderMatters<T, OP>::value && !first(j) ? L::Combine(v[j], acc) : L::Combine(acc, v[j]);
    }
#pragma unroll
    for (uint32_t j = 0; j < M; j++) {
        acc = OrderMatters<T, OP>::value && !later(N + j) ? L::Combine(w[j], acc) : L::Combine(acc, w[j]);
    }
}

// The sources from j on, fewer than 8.
template <typename L, typename T, int OP, typename View, typename Later>
__device__ __forceinline__ void DirectRest(const View &view, uint32_t j, uint32_t off, typename L::Val &acc, Later later)
{
    switch (view.Sources() - j) {
        case 1: DirectBatch<L, T, OP, 1, false>(view, j, off, acc, later); break;
        case 2: DirectBatch<L, T, OP, 2, false>(view, j, off, acc, later); break;
        case 3: DirectBatch<L, T, OP, 3, false>(view, j, off, acc, later); break;
        case 4: DirectBatch<L, T, OP, 4, false>(view, j, off, acc, later); break;
        case 5: DirectBatch<L, T, OP, 5, false>(view, j, off, acc, later); break;
        case 6: DirectBatch<L, T, OP, 6, false>(view, j, off, acc, later); break;
        case 7: DirectBatch<L, T, OP, 7, false>(view, j, off, acc, later); break;
        default: break;
    }
}

// first(j), later(j): whether the value so far is the left operand, for the sources loaded first and for those behind them.  TWO: of 24 sources and more both batches in flight; else one after
// the other.
template <typename L, typename T, int OP, bool TWO, typename View, typename First, typename Later>
__device__ __forceinline__ typename L::Val DirectChain(const View &view, uint32_t off, First first, Later later)
{
    typename L::Val acc;
    const uint32_t nsrc = view.Sources();
    if (__builtin_expect(nsrc == 8, 1)) {
        DirectBatch<L, T, OP, 8, true>(view, 0, off, acc, first);
        return acc;
    }
    switch (nsrc) {
        case 1: DirectBatch<L, T, OP, 1, true>(view, 0, off, acc, first); return acc;
        case 2: DirectBatch<L, T, OP, 2, true>(view, 0, off, acc, first); return acc;
        case 3: DirectBatch<L, T, OP, 3, true>(view, 0, off, acc, first); return acc;
        case 4: DirectBatch<L, T, OP, 4, true>(view, 0, off, acc, first); return acc;
        case 5: DirectBatch<L, T, OP, 5, true>(view, 0, off, acc, first); return acc;
        case 6: DirectBatch<L, T, OP, 6, true>(view, 0, off, acc, first); return acc;
        case 7: DirectBatch<L, T, OP, 7, true>(view, 0, off, acc, first); return acc;
        default: break;
    }
    if constexpr (View::kMany) {
        uint32_t j = 8;
        if (TWO && nsrc >= 32) {
            DirectTwoBatches<L, T, OP, 16, 16>(view, off, acc, first, later);
            j = 32;
        } else if (TWO && nsrc >= 24) {
            DirectTwoBatches<L, T, OP, 16, 8>(view, off, acc, first, later);
            j = 24;
        } else if (nsrc >= 16) {
            DirectBatch<L, T, OP, 16, true>(view, 0, off, acc, first);
            j = 16;
        } else {
            DirectBatch<L, T, OP, 8, true>(view, 0, off, acc, first);
        }
        if constexpr (!TWO) {
#pragma nounroll
            for (; j + 16 <= nsrc; j += 16) {
                DirectBatch<L, T, OP, 16, false>(view, j, off, acc, later);
            }
        }
        if (j + 8 <= nsrc) {
            DirectBatch<L, T, OP, 8, false>(view, j, off, acc, later);
            j += 8;
        }
        DirectRest<L, T, OP>(view, j, off, acc, later);
    }
    return acc;
}

// N values pairwise, bottom-up, into the first of them.
template <typename L, uint32_t N> __device__ __forceinline__ void DirectPairwise(typename L::Val (&v)[N])
{
#pragma unroll
    for (uint32_t w = 1; w < N; w <<= 1) {
#pragma unroll
        for (uint32_t i = 0; i + w < N; i += 2 * w) {
            v[i] = L::Combine(v[i], v[i + w]);
        }
    }
}

// G leaves from leaf i0 on, folded pairwise.  `second` of the item: the leaves that are two sources combined; the list of second
// sources repeats the first one where there is none, so that its loads need no guard.
template <typename L, uint32_t CAP, uint32_t G>
__device__ __forceinline__ typename L::Val DirectLeaves(const DirectView<CAP> &view, uint32_t i0, uint32_t off)
{
    uint64_t p[G];
#pragma unroll
    for (uint32_t i = 0; i < G; i++) {
        p[i] = view.Src(i0 + i);
    }
    Fetched(p);
    typename L::Val v[G];
#pragma unroll
    for (uint32_t i = 0; i < G; i++) {
        v[i] = L::Load(reinterpret_cast<const void *>(p[i]), off);
    }
    if (view.it->second != 0) {
        typename L::Val w[G];
#pragma unroll
        for (uint32_t i = 0; i < G; i++) {
            p[i] = view.Src(kDirectSecond<CAP> + i0 + i);
        }
        Fetched(p);
#pragma unroll
        for (uint32_t i = 0; i < G; i++) {
            w[i] = L::Load(reinterpret_cast<const void *>(p[i]), off);
        }
        PinAccesses();
#pragma unroll
        for (uint32_t i = 0; i < G; i++) {
            if ((view.it->second >> (i0 + i)) & 1u) {
                v[i] = L::Combine(v[i], w[i]);
            }
        }
    }
    PinAccesses();
    DirectPairwise<L, G>(v);
    return v[0];
}

template <typename L, uint32_t CAP>
__device__ __forceinline__ typename L::Val DirectTree(const DirectView<CAP> &view, uint32_t off)
{
    switch (view.it->nleaf) {
        case 1: return DirectLeaves<L, CAP, 1>(view, 0, off);
        case 2: return DirectLeaves<L, CAP, 2>(view, 0, off);
        case 4: return DirectLeaves<L, CAP, 4>(view, 0, off);
        case 8: return DirectLeaves<L, CAP, 8>(view, 0, off);
        default: break;
    }
    if constexpr (CAP > 8) {
        typename L::Val v = DirectLeaves<L, CAP, 16>(view, 0, off);
        if (view.it->nleaf == 32) {
            v = L::Combine(v, DirectLeaves<L, CAP, 16>(view, 16, off));
        }
        return v;
    } else {
        return typename L::Val();
    }
}

// Any other expression of at most 8 sources: the stack machine of StackVecPass over one value per lane.  Such an expression
// needs no more than 4 values on the stack (a fifth takes 16 sources).
template <typename L, typename T, int OP, uint32_t CAP>
__device__ __forceinline__ typename L::Val DirectStack(const DirectView<CAP> &view, uint32_t off)
{
    constexpr bool DEEP = false;
    uint64_t p[8];
#pragma unroll
    for (uint32_t j = 0; j < 8; j++) {      // the list repeats its last source up to 8
        p[j] = view.Src(j);
    }
    Fetched(p);
    typename L::Val v[8];
#pragma unroll
    for (uint32_t j = 0; j < 8; j++) {
        v[j] = L::Load(reinterpret_cast<const void *>(p[j]), off);
    }
    PinAccesses();
    typename L::Val top = v[0], b0 = top, b1 = top, b2 = top, b3 = top, b4 = top, b5 = top, b6 = top;   // (b3 ... b6 only named)
    uint32_t depth = 0;
    const uint32_t nsrc = view.it->nsrc;
#pragma unroll
    for (uint32_t j = 0; j < 8; j++) {
        if (j < nsrc) {
            const uint32_t op = (view.it->ops[j >> 1] >> (16u * (j & 1u))) & 0xffffu;
            if (depth > 0) {
                HCCL_STACK_PUT(depth - 1, top)
            }
            top = v[j];
            depth++;
            const uint32_t nfold = op & 7u;
#pragma nounroll
            for (uint32_t f = 0; f < nfold && depth >= 2; f++) {
                typename L::Val under;
                HCCL_STACK_GET(depth - 2, under)
                if (!OrderMatters<T, OP>::value || ((op >> (8 + f)) & 1u)) {
                    top = L::Combine(under, top);
                } else {
                    top = L::Combine(top, under);
                }
                depth--;
            }
        }
    }
    return top;
}

template <typename L, typename T, int OP, uint32_t CAP>
__device__ __forceinline__ typename L::Val DirectValue(const DirectView<CAP> &view, uint32_t off)
{
    if (view.it->kind == DIRECT_CHAIN) {
        auto left = [&](uint32_t j) { return ((view.it->accLeft >> j) & 1u) != 0; };
        return DirectChain<L, T, OP, true>(view, off, left, left);
    }
    if (CAP > 8 || view.it->kind == DIRECT_TREE) {
        return DirectTree<L, CAP>(view, off);
    }
    return DirectStack<L, T, OP, CAP>(view, off);
}

// G sources from source j0 on, pairwise.
template <typename L, uint32_t P, uint32_t G>
__device__ __forceinline__ typename L::Val PackedLeaves(const PackedView<P> &view, uint32_t j0, uint32_t off)
{
    uint32_t p[G];
#pragma unroll
    for (uint32_t i = 0; i < G; i++) {
        p[i] = view.Leaf(j0 + i);
    }
    Fetched(p);
    typename L::Val v[G];
#pragma unroll
    for (uint32_t i = 0; i < G; i++) {
        v[i] = L::Load(reinterpret_cast<const void *>(view.Pointer(p[i])), off);
    }
    PinAccesses();
    DirectPairwise<L, G>(v);
    return v[0];
}
template <typename L, typename T, int OP, uint32_t P>
__device__ __forceinline__ typename L::Val DirectValue(const PackedView<P> &view, uint32_t off)
{
    if (__builtin_expect((view.k->info & kPackedTree) != 0, 0)) {
        switch (view.Sources()) {
            case 2: return PackedLeaves<L, P, 2>(view, 0, off);
            case 4: return PackedLeaves<L, P, 4>(view, 0, off);
            case 8: return PackedLeaves<L, P, 8>(view, 0, off);
            default: break;
        }
        if constexpr (P > 8) {
            typename L::Val v = PackedLeaves<L, P, 16>(view, 0, off);
            if (P > 16 && view.Sources() == 32) {
                v = L::Combine(v, PackedLeaves<L, P, 16>(view, 16, off));
            }
            return v;
        } else {
            return typename L::Val();
        }
    }
    auto yes = [](uint32_t) { return true; };
    if (OrderMatters<T, OP>::value && (view.k->info & kPackedRing) != 0) {
        return DirectChain<L, T, OP, false>(view, off, [](uint32_t j) { return j < 2; }, [](uint32_t) { return false; });
    }
    return DirectChain<L, T, OP, false>(view, off, yes, yes);
}

// A lane's vector to every destination: N at a time without a branch between them, those behind the last one dropped by the
// range check of their buffers.  A branch per destination is a jump to a line of code that has to be fetched, and a pointer fetched
// where it is used a trip to the arguments.  Written through: plain non-temporal stores take half as long again at 1 MiB per rank.
template <uint32_t N, typename View>
__device__ __forceinline__ void DirectStoreTo(const View &view, uint32_t k0, uint32_t ndst, uint32_t at, V4 r)
{
    const uint32_t bytes = view.Bytes() & ~15u, to = view.DstOff();
    typename View::Word o[N];
#pragma unroll
    for (uint32_t k = 0; k < N; k++) {
        o[k] = view.Dst(k0 + k);      // (the lists are padded)
    }
    Fetched(o);
#pragma unroll
    for (uint32_t k = 0; k < N; k++) {
        BufferStore16<STORE_THROUGH>(MakeBuffer(reinterpret_cast<void *>(view.Pointer(o[k]) + to), k0 + k < ndst ? bytes : 0u), at, r);
    }
}
template <typename View>
__device__ __forceinline__ void DirectStore(const View &view, uint32_t at, V4 r)
{
    const uint32_t ndst = view.Destinations();
    if (__builtin_expect(ndst > 4, 1)) {
        DirectStoreTo<8>(view, 0, ndst, at, r);
        if constexpr (View::kMany) {
#pragma nounroll
            for (uint32_t k0 = 8; k0 < ndst; k0 += 8) {
                DirectStoreTo<8>(view, k0, ndst, at, r);
            }
        }
    } else if (ndst == 1) {
        DirectStoreTo<1>(view, 0, ndst, at, r);
    } else {
        DirectStoreTo<4>(view, 0, ndst, at, r);
    }
}

// The item's whole vectors, a lane's at byte `at`, or the element behind them that is this lane's.
template <typename T, int OP, typename View> __device__ __forceinline__ void DirectVector(const View &view, uint32_t at)
{
    if (at + 16u <= view.Bytes()) {
        DirectStore(view, at, DirectValue<VecLane<T, OP>, T, OP>(view, view.SrcOff() + at));
    }
}
template <typename View, typename Value> __device__ __forceinline__ void DirectEnd(const View &view, Value value)
{
    typedef decltype(value(0u)) T;
    const uint32_t rest = view.Bytes() & 15u, mine = threadIdx.x * uint32_t(sizeof(T));
    if (mine < rest) {
        const uint32_t at = view.Bytes() - rest + mine, ndst = view.Destinations();
        const T r = value(view.SrcOff() + at);
#pragma nounroll
        for (uint32_t k = 0; k < ndst; k++) {
            StoreElem<T>(reinterpret_cast<void *>(view.Pointer(view.Dst(k))), view.DstOff() + at, r);
        }
    }
}

template <typename T, int OP, uint32_t CAP>
__global__ void __launch_bounds__(kDirectThreads) DirectKernel(const DirectArgs<CAP>)
{
    const DirectView<CAP> view;
    if (blockIdx.x != 0) {
        DirectVector<T, OP>(view, KiBOf(blockIdx.x - 1, view.Bytes(), CAP > 8 && view.Destinations() == 1) * kDirectChunk + threadIdx.x * 16u);
    } else {
        DirectEnd(view, [&](uint32_t off) { return DirectValue<ElemLane<T, OP>, T, OP>(view, off); });
    }
}
template <typename T, int OP, uint32_t P>
__global__ void __launch_bounds__(kDirectThreads) PackedKernel(const PackedArgs<P>)
{
    const PackedView<P> view;
    const uint32_t ends = view.k->info & kPackedEnds ? 1u : 0u;
    if (blockIdx.x >= ends) {
        DirectVector<T, OP>(view, KiBOf(blockIdx.x - ends, view.Bytes(), P > 8 && (view.k->info & kPackedFours) != 0) * kDirectChunk + threadIdx.x * 16u);
    } else {
        DirectEnd(view, [&](uint32_t off) { return DirectValue<ElemLane<T, OP>, T, OP>(view, off); });
    }
}

// Chains of 24 ... 32 sources with both batches in flight, in a kernel of their own: in one with the others its registers and its code, which the way of fewer sources leads
// around, cost those more than it gains here.  as a share of the time batch after batch, apart / in one kernel: 17
// ranks' bf16 sum 768 KiB reduce-scatter 1.01 / 1.09, reduce 1.03 / 1.10, all-reduce 1.01 / 1.07, 20 ranks' all-reduce of 512 KiB 0.99 / 1.13; what it brings 24 to 32: reduce-scatter
// of 512 KiB to 1 MiB bf16 0.78 ... 0.88, int8 0.83 ... 0.97, fp32 0.89 ... 0.97, reduce 0.76 ... 0.85, 0.82 ... 0.97, 0.87 ... 1.00.
template <typename L, typename T, int OP, bool ALL, typename First, typename Later>
__device__ __forceinline__ typename L::Val PackedTwoChain(const PackedView<32> &view, uint32_t off, First first, Later later)
{
    typename L::Val acc;
    if constexpr (ALL) {
        DirectTwoBatches<L, T, OP, 16, 16>(view, off, acc, first, later);
    } else {
        DirectTwoBatches<L, T, OP, 16, 8>(view, off, acc, first, later);
        DirectRest<L, T, OP>(view, 24, off, acc, later);
    }
    return acc;
}
template <typename L, typename T, int OP, bool ALL> __device__ __forceinline__ typename L::Val PackedTwoValue(const PackedView<32> &view, uint32_t off)
{
    if (OrderMatters<T, OP>::value && (view.k->info & kPackedRing) != 0) {
        return PackedTwoChain<L, T, OP, ALL>(view, off, [](uint32_t j) { return j < 2; }, [](uint32_t) { return false; });
    }
    auto yes = [](uint32_t) { return true; };
    return PackedTwoChain<L, T, OP, ALL>(view, off, yes, yes);
}
// ALL: 32 sources, else 24 ... 31.
template <typename T, int OP, bool ALL> __global__ void __launch_bounds__(kDirectThreads) PackedTwoKernel(const PackedArgs<32>)
{
    const PackedView<32> view;
    const uint32_t ends = view.k->info & kPackedEnds ? 1u : 0u;
    if (blockIdx.x >= ends) {
        const uint32_t at = KiBOf(blockIdx.x - ends, view.Bytes(), (view.k->info & kPackedFours) != 0) * kDirectChunk + threadIdx.x * 16u;
        if (at + 16u <= view.Bytes()) {
            DirectStore(view, at, PackedTwoValue<VecLane<T, OP>, T, OP, ALL>(view, view.SrcOff() + at));
        }
    } else {
        DirectEnd(view, [&](uint32_t off) { return PackedTwoValue<ElemLane<T, OP>, T, OP, ALL>(view, off); });
    }
}

// The usual numbers of sources, each with a kernel of its own, in which the way of a vector is one stretch of code: with all numbers
// and shapes in one kernel the way leads over half a dozen jumps to lines that have to be fetched.  8 ranks, device time per launch, us,
// one kernel / this way: fp32 8 KiB 2.5 / 2.1, 64 KiB 2.9 / 2.4, 1 MiB 3.4 / 3.0; bf16 2.8 / 2.4, 3.2 / 2.7, 3.7 / 3.3.
// (Two sources have one order for every shape: the first is the left operand.)
enum PackedOrder : int { PACKED_LEFT = 0, PACKED_RING = 1, PACKED_TREE = 2 };
template <typename L, typename T, int OP, uint32_t N, int SHAPE, typename View>
__device__ __forceinline__ typename L::Val PackedValue(const View &view, uint32_t off)
{
    if constexpr (SHAPE == PACKED_TREE) {
        return PackedLeaves<L, View::kRanks, N>(view, 0, off);
    } else {
        typename L::Val acc;
        DirectBatch<L, T, OP, N, true>(view, 0, off, acc, [](uint32_t j) { return SHAPE == PACKED_LEFT || j < 2; });
        return acc;
    }
}
template <typename T, int OP, uint32_t P, uint32_t N, int SHAPE>
__global__ void __launch_bounds__(kDirectThreads) PackedShapeKernel(const PackedArgs<P>)
{
    const PackedView<P> view;
    const uint32_t ends = view.k->info & kPackedEnds ? 1u : 0u;
    if (blockIdx.x >= ends) {
        const uint32_t at = KiBOf(blockIdx.x - ends, view.Bytes(), P > 8 && (view.k->info & kPackedFours) != 0) * kDirectChunk + threadIdx.x * 16u;
        if (at + 16u <= view.Bytes()) {
            DirectStore(view, at, PackedValue<VecLane<T, OP>, T, OP, N, SHAPE>(view, view.SrcOff() + at));
        }
    } else {
        DirectEnd(view, [&](uint32_t off) { return PackedValue<ElemLane<T, OP>, T, OP, N, SHAPE>(view, off); });
    }
}

// The same with four vectors per lane, for collectives of 2 ... 8 MiB with many destinations: bound by how many stores a CU has on their way, not by
// latency, and four vectors of one source and one destination lie behind one another, so that a wave stores whole 4 KiB.  All reads of a wave
// are in flight before the first is combined.  8 ranks, fp32, 4.25 MiB: tile kernel 14.3 us, a vector per lane 13.2, four 11.5; 16 ranks 27.7, 24.6, 22.9.
template <typename L, typename T, int OP, uint32_t N, int SHAPE, typename View>
__device__ __forceinline__ void PackedValues(const View &view, const uint32_t (&at)[4], V4 (&x)[4])
{
    typename View::Word p[N];
#pragma unroll
    for (uint32_t j = 0; j < N; j++) {
        p[j] = SHAPE == PACKED_TREE ? view.Leaf(j) : view.Src(j);
    }
    Fetched(p);
    const void *src[N];
#pragma unroll
    for (uint32_t j = 0; j < N; j++) {
        src[j] = reinterpret_cast<const void *>(view.Pointer(p[j]));
    }
    if constexpr (SHAPE == PACKED_TREE) {
        typedef VecLane<T, OP> Tree;
        V4 v[N][4];
        ChainLoad<Tree, N, 4>(src, view.SrcOff(), at, v);
#pragma unroll
        for (uint32_t w = 1; w < N; w <<= 1) {
#pragma unroll
            for (uint32_t i = 0; i + w < N; i += 2 * w) {
#pragma unroll
                for (uint32_t u = 0; u < 4; u++) {
                    v[i][u] = Tree::Combine(v[i][u], v[i + w][u]);
                }
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < 4; u++) {
            x[u] = v[0][u];
        }
    } else {
        ChainWhole<L, T, OP, N, 4>(src, view.SrcOff(), at, SHAPE == PACKED_RING ? uint64_t(2) : ~uint64_t(0), x);
    }
}
// A lane's vectors to every destination, as DirectStore.
template <uint32_t N, typename View>
__device__ __forceinline__ void PackedStoreTo(const View &view, uint32_t k0, uint32_t ndst, const uint32_t (&pos)[4], const V4 (&x)[4])
{
    const uint32_t bytes = view.Bytes() & ~15u, to = view.DstOff();
    typename View::Word o[N];
#pragma unroll
    for (uint32_t k = 0; k < N; k++) {
        o[k] = view.Dst(k0 + k);
    }
    Fetched(o);
#pragma unroll
    for (uint32_t k = 0; k < N; k++) {
        const BufferRsrc r = MakeBuffer(reinterpret_cast<void *>(view.Pointer(o[k]) + to), k0 + k < ndst ? bytes : 0u);
#pragma unroll
        for (uint32_t u = 0; u < 4; u++) {
            BufferStore16<STORE_THROUGH>(r, pos[u], x[u]);
        }
    }
}
template <typename View> __device__ __forceinline__ void PackedStore(const View &view, const uint32_t (&pos)[4], const V4 (&x)[4])
{
    const uint32_t ndst = view.Destinations();
    if (ndst == 1) {
        PackedStoreTo<1>(view, 0, ndst, pos, x);
        return;
    }
#pragma nounroll
    for (uint32_t k0 = 0; k0 < ndst; k0 += 4) {
        PackedStoreTo<4>(view, k0, ndst, pos, x);
    }
}
// Positions of a lane's vectors, and where it reads: behind the last whole vector that one again, dropped by the stores' range check.
__device__ __forceinline__ void PackedPositions(uint32_t chunk, uint32_t bytes, uint32_t (&pos)[4], uint32_t (&at)[4])
{
#pragma unroll
    for (uint32_t u = 0; u < 4; u++) {
        pos[u] = chunk * kPackedWideChunk + u * kDirectChunk + threadIdx.x * 16u;
        at[u] = min(pos[u], (bytes & ~15u) - 16u);
    }
}
template <typename T, int OP, uint32_t P, uint32_t N, int SHAPE>
__global__ void __launch_bounds__(kDirectThreads) PackedWideKernel(const PackedArgs<P>)
{
    typedef FoldLane<T, OP> Few;
    typedef typename Few::Exact Many;
    const PackedView<P> view;
    const uint32_t ends = view.k->info & kPackedEnds ? 1u : 0u, bytes = view.Bytes();
    if (blockIdx.x >= ends) {
        const uint32_t chunk = blockIdx.x - ends;
        if (chunk * kPackedWideChunk < (bytes & ~15u)) {
            uint32_t pos[4], at[4];
            V4 x[4];
            PackedPositions(chunk, bytes, pos, at);
            PackedValues<std::conditional_t<(N > 8), Many, Few>, T, OP, N, SHAPE>(view, at, x);
            PackedStore(view, pos, x);
        }
    } else {
        DirectEnd(view, [&](uint32_t off) { return PackedValue<ElemLane<T, OP>, T, OP, N, SHAPE>(view, off); });
    }
}

// Pure data movement: one source per item.
template <typename View> __device__ __forceinline__ void DirectMove(const View &view, uint32_t at)
{
    if (at + 16u <= view.Bytes()) {
        DirectStore(view, at, MoveLane::Load(reinterpret_cast<const void *>(view.Pointer(view.Src(0))), view.SrcOff() + at));
    }
}
template <typename View> __device__ __forceinline__ void DirectMoveEnd(const View &view)
{
    DirectEnd(view, [&](uint32_t off) { return LoadElem<uint8_t>(reinterpret_cast<const void *>(view.Pointer(view.Src(0))), off); });
}
template <uint32_t CAP>
__global__ void __launch_bounds__(kDirectThreads) DirectCopyKernel(const DirectArgs<CAP>)
{
    const DirectView<CAP> view;
    if (blockIdx.x != 0) {
        DirectMove(view, (blockIdx.x - 1) * kDirectChunk + threadIdx.x * 16u);
    } else {
        DirectMoveEnd(view);
    }
}
template <uint32_t P>
__global__ void __launch_bounds__(kDirectThreads) PackedCopyKernel(const PackedArgs<P>)
{
    const PackedView<P> view;
    const uint32_t ends = view.k->info & kPackedEnds ? 1u : 0u;
    if (blockIdx.x >= ends) {
        DirectMove(view, (blockIdx.x - ends) * kDirectChunk + threadIdx.x * 16u);
    } else {
        DirectMoveEnd(view);
    }
}

}  // namespace hcclamd
