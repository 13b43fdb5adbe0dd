// Rules of the executor on sizes and alignment: how a stretch of bytes is cut, how results are stored.  Pure C++: no HIP
// calls, so the rules can be checked without a GPU.
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

constexpr uint64_t kMemorySideCacheBytes = 256ull << 20;

// Whether a launch of the plain copy kernel writes its results through (StorePolicy, kernels_impl.h) instead of non-temporally:
// `traffic` bytes read and written by the launch, `written` of them written, `moved` read and written by the whole collective, whose
// launches all store alike.  Up to 512 MiB in all, us, non-temporal / through: all-gather 2 ranks 10 MiB 10.4 / 7.4, 64 MiB
// (384 MiB moved) 67.7 / 60.1; 3 ranks 8 MiB 17.2 / 12.0, 32 MiB (384) 71.5 / 59.9; 8 ranks 2 MiB 28.2 / 20.1; 16 ranks 1 MiB 53.7 / 38.7;
// uniform all-to-all 8 ranks 8 MiB 21.3 / 20.3, 32 MiB (512) 84.5 / 75.7.  Beyond, the one loses what the other
// gains: 2 ranks 128 MiB (768) 139.5 / 143.8, 3 ranks 48 MiB (576) 107.8 / 111.7, all-to-all 64 MiB (1024) 170.0 / 172.5 -- unless every
// block goes to four destinations or more: 5 ranks 24 MiB (720) 150.5 / 147.6, 6 ranks 24 MiB (1008) 217.8 / 210.7, 32 MiB 295 / 281.
inline bool CopiesWriteThrough(uint64_t traffic, uint64_t written, uint64_t moved)
{
    return moved <= 2 * kMemorySideCacheBytes || 5 * written >= 4 * traffic;
}

}  // namespace hcclamd
