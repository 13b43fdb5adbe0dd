// Small collectives: one launch whose descriptors ride in the kernel arguments.
//
// A small collective is latency and nothing else.  The tile kernels reach their data through a chain of dependent
// loads (argument -> item table -> pointer pool -> data) and wait for one destination pointer after the other, and
// their tables have to be in device memory first.  Here an item's record lies at a place that follows from the block
// index, all of its pointers are fetched together, and the data loads of up to 16 sources are issued back to back
// without a branch between them (the number of sources picks straight-line code; a guard per source makes the compiler
// wait for each load).  Measured on MI355X, time of the kernel, tile form / this form: 8 ranks, ring all-reduce, fp32
// 8 KiB per rank 4.5 / 3.5 us, bf16 8 KiB 5.8 / 3.2, bf16 512 KiB 6.1 / 3.6; 24 ranks, halving-doubling, bf16 256 KiB
// 19.7 / 7.6.  An empty kernel takes 2; what is left is two trips to the arguments, one to the data, and the stores.
// No table is uploaded or kept, so a call with new buffers costs what a repeated one does (8 ranks x 8 KiB through ctypes,
// 200 sets of buffers used once each: 6.1 us per call, 5.9 repeated; through tables 11.1 and 6.0).
//
// A workgroup handles 4 KiB of one item (blockIdx.y), one 16-byte vector per lane: four times as many workgroups as the
// tile kernels use.  Accesses are unaligned 128-bit ones (the instruction is the same one), so one form serves every
// alignment; the bytes behind the last whole vector go element by element to a workgroup of their own (blockIdx.x == 0), side by side with the others.
#pragma once
#include "kernels_impl.h"

namespace hcclamd {

// The kernel arguments where they lie (constant memory): read through the parameter itself, the wide form is copied to
// private memory first.
#define HCCL_CONSTANT __attribute__((address_space(4)))
template <uint32_t CAP> struct DirectView {
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
    // base pointer of entry j of the list of sources / destinations (base indexes, four to a word)
    __device__ __forceinline__ uint64_t Src(uint32_t j) const { return args->base[(it->src[j >> 2] >> (8u * (j & 3u))) & 0xffu]; }
    __device__ __forceinline__ uint64_t Dst(uint32_t k) const { return args->base[(it->dst[k >> 2] >> (8u * (k & 3u))) & 0xffu]; }
};

// N sources from source j0 on into acc.
template <typename L, typename T, int OP, uint32_t CAP, uint32_t N>
__device__ __forceinline__ void DirectBatch(const DirectView<CAP> &view, uint32_t j0, uint32_t off,
    typename L::Val &acc)
{
    uint64_t p[N];
#pragma unroll
    for (uint32_t j = 0; j < N; j++) {
        p[j] = view.Src(j0 + j);
    }
    typename L::Val v[N];
#pragma unroll
    for (uint32_t j = 0; j < N; j++) {
        v[j] = L::Load(reinterpret_cast<const void *>(p[j]), off);
    }
    PinAccesses();
    acc = j0 == 0 ? v[0] : ((OrderMatters<T, OP>::value && !((view.it->accLeft >> j0) & 1u)) ? L::Combine(v[0], acc) : L::Combine(acc, v[0]));
#pragma unroll
    for (uint32_t j = 1; j < N; j++) {
        if (OrderMatters<T, OP>::value && !((view.it->accLeft >> (j0 + j)) & 1u)) {
            acc = L::Combine(v[j], acc);
        } else {
            acc = L::Combine(acc, v[j]);
        }
    }
}

template <typename L, typename T, int OP, uint32_t CAP>
__device__ __forceinline__ typename L::Val DirectChain(const DirectView<CAP> &view, uint32_t off)
{
    typename L::Val acc;
    const uint32_t nsrc = view.it->nsrc;
    uint32_t j = 0;
    if (CAP > 8) {
#pragma nounroll
        for (; j + 16 <= nsrc; j += 16) {
            DirectBatch<L, T, OP, CAP, 16>(view, j, off, acc);
        }
    }
    if (j + 8 <= nsrc) {
        DirectBatch<L, T, OP, CAP, 8>(view, j, off, acc);
        j += 8;
    }
    switch (nsrc - j) {
        case 1: DirectBatch<L, T, OP, CAP, 1>(view, j, off, acc); break;
        case 2: DirectBatch<L, T, OP, CAP, 2>(view, j, off, acc); break;
        case 3: DirectBatch<L, T, OP, CAP, 3>(view, j, off, acc); break;
        case 4: DirectBatch<L, T, OP, CAP, 4>(view, j, off, acc); break;
        case 5: DirectBatch<L, T, OP, CAP, 5>(view, j, off, acc); break;
        case 6: DirectBatch<L, T, OP, CAP, 6>(view, j, off, acc); break;
        case 7: DirectBatch<L, T, OP, CAP, 7>(view, j, off, acc); break;
        default: break;
    }
    return acc;
}

// G leaves from leaf i0 on, folded pairwise.  `second` of the item: the leaves that are two sources combined; the list of second
// sources repeats the first one where there is none, so that its loads need no guard.
template <typename L, uint32_t CAP, uint32_t G>
__device__ __forceinline__ typename L::Val DirectLeaves(const DirectView<CAP> &view, uint32_t i0, uint32_t off)
{
    typename L::Val v[G];
#pragma unroll
    for (uint32_t i = 0; i < G; i++) {
        v[i] = L::Load(reinterpret_cast<const void *>(view.Src(i0 + i)), off);
    }
    if (view.it->second != 0) {
        typename L::Val w[G];
#pragma unroll
        for (uint32_t i = 0; i < G; i++) {
            w[i] = L::Load(reinterpret_cast<const void *>(view.Src(kDirectSecond<CAP> + i0 + i)), off);
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
#pragma unroll
    for (uint32_t w = 1; w < G; w <<= 1) {
#pragma unroll
        for (uint32_t i = 0; i + w < G; i += 2 * w) {
            v[i] = L::Combine(v[i], v[i + w]);
        }
    }
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
    typename L::Val v[8];
#pragma unroll
    for (uint32_t j = 0; j < 8; j++) {      // the list repeats its last source up to 8
        v[j] = L::Load(reinterpret_cast<const void *>(view.Src(j)), off);
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

// The first 8 destinations, fetched before the data (the list is padded: no guards).
template <uint32_t CAP>
__device__ __forceinline__ void DirectFetchDst(const DirectView<CAP> &view, uint32_t k0, uint64_t (&o)[8])
{
#pragma unroll
    for (uint32_t k = 0; k < 8; k++) {
        o[k] = view.Dst(k0 + k);
    }
}

template <typename L, uint32_t CAP>
__device__ __forceinline__ void DirectStore(const DirectView<CAP> &view, uint64_t (&o)[8], uint32_t at, typename L::Val r)
{
    const uint32_t ndst = view.it->ndst, to = view.it->dstOff + at;
    for (uint32_t k0 = 0;;) {
#pragma unroll
        for (uint32_t k = 0; k < 8; k++) {
            if (k0 + k < ndst) {
                L::Store(reinterpret_cast<void *>(o[k]), to, r);
            }
        }
        k0 += 8;
        if (CAP <= 8 || k0 >= ndst) {
            break;
        }
        DirectFetchDst<CAP>(view, k0, o);
    }
}

// One lane's position: its value, and where that goes.
template <typename L, typename T, int OP, uint32_t CAP>
__device__ __forceinline__ void DirectLane(const DirectView<CAP> &view, uint32_t at)
{
    const uint32_t off = view.it->srcOff + at;
    uint64_t o[8];
    DirectFetchDst<CAP>(view, 0, o);
    typename L::Val r;
    if (view.it->kind == DIRECT_CHAIN) {
        r = DirectChain<L, T, OP, CAP>(view, off);
    } else if (CAP > 8 || view.it->kind == DIRECT_TREE) {
        r = DirectTree<L, CAP>(view, off);
    } else {
        r = DirectStack<L, T, OP, CAP>(view, off);
    }
    DirectStore<L, CAP>(view, o, at, r);
}

template <typename L, uint32_t CAP>
__device__ __forceinline__ void DirectMove(const DirectView<CAP> &view, uint32_t at)
{
    uint64_t o[8];
    DirectFetchDst<CAP>(view, 0, o);
    const typename L::Val r = L::Load(reinterpret_cast<const void *>(view.Src(0)), view.it->srcOff + at);
    DirectStore<L, CAP>(view, o, at, r);
}

template <typename T, int OP, uint32_t CAP>
__global__ void __launch_bounds__(kBlockThreads) DirectKernel(const DirectArgs<CAP>)
{
    const DirectView<CAP> view;
    if (blockIdx.x != 0) {
        const uint32_t at = (blockIdx.x - 1) * kDirectChunk + threadIdx.x * 16u;
        if (at + 16u <= view.it->bytes) {
            DirectLane<VecLane<T, OP>, T, OP, CAP>(view, at);
        }
    } else {
        const uint32_t rest = view.it->bytes & 15u;
        if (threadIdx.x * uint32_t(sizeof(T)) < rest) {
            DirectLane<ElemLane<T, OP>, T, OP, CAP>(view, view.it->bytes - rest + threadIdx.x * uint32_t(sizeof(T)));
        }
    }
}

// Pure data movement: one source per item.
template <uint32_t CAP>
__global__ void __launch_bounds__(kBlockThreads) DirectCopyKernel(const DirectArgs<CAP>)
{
    const DirectView<CAP> view;
    if (blockIdx.x != 0) {
        const uint32_t at = (blockIdx.x - 1) * kDirectChunk + threadIdx.x * 16u;
        if (at + 16u <= view.it->bytes) {
            DirectMove<VecLane<uint8_t, ROP_SUM>, CAP>(view, at);
        }
    } else {
        const uint32_t rest = view.it->bytes & 15u;
        if (threadIdx.x < rest) {
            DirectMove<ElemLane<uint8_t, ROP_SUM>, CAP>(view, view.it->bytes - rest + threadIdx.x);
        }
    }
}

}  // namespace hcclamd
