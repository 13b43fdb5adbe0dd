// All-to-all-v straight from the tables of its callers: a block's source, destination and length follow from three numbers of
// theirs, so nothing is planned, cut or laid out for the device; 12 bytes per pair of ranks travel to it, a new call's of up to 16 ranks in the
// kernel arguments.
//
// A wave takes a piece of 4 KiB of a block at a time.  It finds it by itself: the lanes
// hold the first piece of every receiver's blocks (at most 64 receivers, one per lane), then that receiver's row of the tables, whose
// pieces they add up; the row of the next piece is on its way while this one is copied.
// Pieces begin on a memory line of the destination, so all stores but those of a block's ends are aligned; loads go to any address.
#pragma once
#include "kernels_direct.h"

namespace hcclamd {

// The sum of the lanes up to this one.
__device__ __forceinline__ uint32_t WaveSum(uint32_t v)
{
    // within rows of 16 lanes (row_shr), then the last lane of a row into the next one, of the first half into the second (row_bcast)
    v += uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x111, 0xf, 0xf, false));
    v += uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x112, 0xf, 0xf, false));
    v += uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x114, 0xf, 0xf, false));
    v += uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x118, 0xf, 0xf, false));
    v += uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x142, 0xa, 0xf, false));
    v += uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x143, 0xc, 0xf, false));
    return v;
}
__device__ __forceinline__ uint32_t OfLane(uint32_t v, uint32_t lane) { return uint32_t(__builtin_amdgcn_readlane(int(v), int(lane))); }
__device__ __forceinline__ uint64_t OfLane(uint64_t v, uint32_t lane)
{
    return uint64_t(OfLane(uint32_t(v >> 32), lane)) << 32 | OfLane(uint32_t(v), lane);
}

template <uint32_t P> struct A2avRow {
    typedef const A2avTable<P> HCCL_GLOBAL *Table;
    uint32_t piece, start;     // the piece, the first one of its receiver
    uint64_t recv;
    uint32_t count, to, from;  // of this lane's sender
    uint64_t send;
    // `starts`: every lane's receiver's first piece
    __device__ __forceinline__ void Load(Table t, uint32_t starts, uint32_t q)
    {
        const uint32_t lane = threadIdx.x & 63u, i = lane < P ? lane : P - 1;
        const uint32_t j = uint32_t(__popcll(__ballot(starts <= q))) - 1u;
        piece = q;
        start = OfLane(starts, j);
        recv = t->recv[j];
        count = t->count[j * P + i];
        to = t->to[j * P + i];
        from = t->from[j * P + i];
        send = t->send[i];
    }
    __device__ __forceinline__ void Taken() { asm volatile("" : "+v"(count), "+v"(to), "+v"(from), "+v"(send)::"memory"); }
};

struct A2avPiece {
    uint64_t src, dst;
    uint32_t bytes;
};
template <uint32_t P> __device__ __forceinline__ A2avPiece A2avFind(const A2avRow<P> &r, const A2avRange &range)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t bytes = lane < P ? r.count << range.unitShift : 0u;
    const uint64_t dst = r.recv + (uint64_t(r.to) << range.unitShift), src = r.send + (uint64_t(r.from) << range.unitShift);
    const uint32_t off = uint32_t(dst) & (kA2avLine - 1);
    const uint32_t size = 1u << range.shift;
    const uint32_t n = bytes == 0 ? 0u : (off + bytes + size - 1) >> range.shift;
    const uint32_t upTo = WaveSum(n), before = upTo - n, x = r.piece - r.start;
    const uint32_t i = uint32_t(__popcll(__ballot(before <= x))) - 1u;      // (the last of the blocks that begin there: one with a piece)
    const uint32_t k = x - OfLane(before, i), o = OfLane(off, i), b = OfLane(bytes, i);
    const uint32_t lo = k == 0 ? 0u : (k << range.shift) - o, end = ((k + 1) << range.shift) - o;
    return A2avPiece{OfLane(src, i) + lo, OfLane(dst, i) + lo, (end < b ? end : b) - lo};
}

// A wave copies a piece: V vectors per lane, and the bytes in front of the first whole vector of the destination and behind the last one by
// lanes 0 and 16 on.  The next piece's row is asked for before the loads and taken before the stores: a wait for it behind those would be one for
// them too.
template <uint32_t P, uint32_t LANES, uint32_t POLICY>
__device__ __forceinline__ void A2avBody(const A2avTable<P> HCCL_GLOBAL *t, const A2avRange &range)
{
    constexpr uint32_t kWaves = LANES / 64, V = (1u << kA2avShift) / 1024;
    const uint32_t lane = threadIdx.x & 63u, stride = gridDim.x * kWaves;
    const uint32_t starts = lane < P ? t->rowStart[lane] : ~0u;
    uint32_t q = range.first + blockIdx.x * kWaves + (kWaves > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0u);
    if (q >= range.end) {
        return;
    }
    A2avRow<P> row;
    row.Load(t, starts, q);
    row.Taken();
    for (;;) {
        const A2avPiece p = A2avFind<P>(row, range);
        q += stride;
        const bool more = q < range.end;
        if (more) {
            row.Load(t, starts, q);
        }
        const uint32_t head = min(uint32_t(-p.dst) & 15u, p.bytes), body = (p.bytes - head) & ~15u, tail = p.bytes - head - body;
        const uint32_t end = lane < 16 ? lane : head + body + lane - 16;        // of the piece, in bytes
        const bool ends = lane < 16 ? lane < head : lane < 16 + tail;
        uint8_t e = 0;
        if (ends) {
            e = LoadElem<uint8_t>(reinterpret_cast<const void *>(p.src), end);
        }
        // (where there is no whole vector: the one that holds the first byte, dropped)
        const uint64_t from = body != 0 ? p.src + head : p.src & ~uint64_t(15);
        const uint32_t last = body != 0 ? body - 16 : 0u;
        V4 v[V];
#pragma unroll
        for (uint32_t u = 0; u < V; u++) {
            v[u] = Load16<ACC_VEC16_ANY>(reinterpret_cast<const void *>(from), min((u * 64 + lane) * 16, last));
        }
        HoldBack(v);
        row.Taken();
        const BufferRsrc r = MakeBuffer(reinterpret_cast<void *>(p.dst + head), body);
#pragma unroll
        for (uint32_t u = 0; u < V; u++) {
            BufferStore16<POLICY>(r, (u * 64 + lane) * 16, v[u]);
        }
        if (ends) {
            StoreElem<uint8_t>(reinterpret_cast<void *>(p.dst), end, e);
        }
        if (!more) {
            break;
        }
    }
}

template <uint32_t P, uint32_t LANES, uint32_t POLICY> __global__ void __launch_bounds__(LANES) A2avArgsKernel(const A2avArgs<P>)
{
    const A2avArgs<P> HCCL_CONSTANT *k = (const A2avArgs<P> HCCL_CONSTANT *)__builtin_amdgcn_kernarg_segment_ptr();
    A2avBody<P, LANES, POLICY>((const A2avTable<P> HCCL_GLOBAL *)&k->table, A2avRange{k->range.first, k->range.end, k->range.unitShift, k->range.shift});
}
template <uint32_t P, uint32_t LANES, uint32_t POLICY>
__global__ void __launch_bounds__(LANES) A2avTableKernel(const A2avTable<P> *table, A2avRange range)
{
    A2avBody<P, LANES, POLICY>((const A2avTable<P> HCCL_GLOBAL *)table, range);
}

}  // namespace hcclamd
