// All-to-all-v straight from the tables of its callers (kernels_a2av.h): the ranks' rows are taken over as they come, narrowed to 32 bits,
// and that is what the device works from.  A block's place follows from the tables, so there is nothing to plan; what is checked is
// what a plan would have shown: the two sides agree, no two blocks land on the same bytes, no buffer overlaps another one.
//
// The latest calls are kept, tables and buffers, a few of them: a rank's rows are compared with theirs as they come, and a call that
// is one of them in every number is launched as it was.  Measured, us, planned and with tables of descriptors / this way.  The first pass on new tables and
// buffers, through the Python mirror, to completion: 8 ranks 60 / 25, 16 ranks 105 - 130 / 30, 32 ranks 190 - 245 / 50, 64 ranks 570 - 620 / 70.
// Three sets of tables in turn: 64 ranks, blocks of a few hundred bytes 21.6 / 11.8 (128 KiB of tables copied, hashed and compared again; now compared
// only), of 2000 bytes 24.6 / 11.6, of 16 KB 53.3 / 41.7; 16 ranks x 4 KB 8.4 / 5.4, x 20 KB 11.5 / 5.5 (two kernels, for short segments and for tiles; now
// one), x 262 KB 38.4 / 38.4; 32 ranks x 8 KB 13.0 / 7.1, x 64 KB 45.6 / 39.0, x 262 KB 151.9 / 152.1.
//
// Left to the general way (the caller expands the rows and plans): values of 2^32 and more, blocks of 2 GiB and more, blocks that overlap in a receive
// buffer, send buffers that overlap receive buffers, a stream that is being captured, and every setting that asks for another kernel.
#include <algorithm>
#include <cstdlib>
#include <cstring>

#include "log.h"
#include "noalloc.h"
#include "runtime.h"

namespace hcclamd {

namespace {

#define HIP_OK(expr)                                                                                  \
    do {                                                                                              \
        hipError_t e_ = (expr);                                                                       \
        if (e_ != hipSuccess) {                                                                       \
            HCCL_LOG_ERROR("%s failed: %s", #expr, hipGetErrorString(e_));                            \
            return HCCL_E_RUNTIME;                                                                    \
        }                                                                                             \
    } while (0)

// How wide (bytes moved in all).  Three sets of buffers and tables in turn, us, 16 workgroups of one wave per CU, written through / two of four waves, non-temporal / one of
// them.  While what is read and written stays in the memory-side cache, the first: lognormal blocks, 16 ranks 26 MiB 10.7 / 11.8 / 12.1, 60 MiB 21.7 / 23.3 / 23.7, 90 MiB 31.0 / 33.5
// / 33.7, 95 MiB 33.1 / 35.1 / -, 100 MiB 36.7 / 37.0 / -, 105 MiB 39.3 / 38.3 / -; 64 ranks 90 MiB 32.8 / 36.6 / 36.9, 100 MiB 39.9 / 40.7 / -, 110 MiB 44.7 / 44.3 / -; uniform,
// 8 ranks 60 MiB 20.3 / 22.1 / 22.5, 95 MiB 31.9 / 33.5 / -, 100 MiB 34.5 / 35.3 / -, 105 MiB 37.9 / 37.0 / -.  Beyond, two up to 128 MiB.
// From there on two for uniform blocks of up to 16 ranks, which the workgroups then take in step, one for others (planned copies / two / one): uniform, 4 ranks 512 MiB 86.1 / 87.4 / 88.0 (one way), 1000 MiB
// 168.3 / 172.1 / 173.5, 8 ranks 512 MiB 86.2 / 87.3 / 88.7, 16 ranks 92.6 / 91.7 / 94.4, 32 ranks 1000 MiB 175.1 / 179.4 / 177.8; lognormal, 2 ranks 95.0 / 97.7 / 96.2 and 183.4 / 187.4 / 185.0, 4 ranks 100.2 / 102.1 /
// 100.1, 196.3 / 199.7 / 196.2, 8 ranks 99.8 / 101.1 / 98.4, 192.3 / 196.8 / 191.4, 16 ranks 98.3 / 98.9 / 96.2, 187.8 / 190.9 / 185.1, 32 ranks 103.1 / 103.0 / 100.1, 194.9 / 197.5 / 190.1, 64 ranks 214 / 206 / 199.
constexpr uint64_t kOneWaveTotal = uint64_t(96) << 20, kTwoPerCuTotal = uint64_t(128) << 20;
constexpr uint64_t kLaunchTotal = uint64_t(256) << 20;    // in one launch (as other collectives that hop from buffer to buffer)

// The image's tables, wherever they lie for the group's number of ranks.
struct View {
    uint32_t stride;
    uint64_t *send, *recv;
    uint32_t *rowStart, *count, *to, *from;
};
template <uint32_t P> View ViewOf(A2avSet *s)
{
    A2avTable<P> *t = reinterpret_cast<A2avTable<P> *>(s->image.data());
    return View{P, t->send, t->recv, t->rowStart, t->count, t->to, t->from};
}
uint32_t RanksOf(uint32_t p) { return p <= 8 ? 8 : (p <= 16 ? 16 : (p <= 32 ? 32 : 64)); }
View ViewOf(A2avSet *s, uint32_t p)
{
    switch (RanksOf(p)) {
        case 8: return ViewOf<8>(s);
        case 16: return ViewOf<16>(s);
        case 32: return ViewOf<32>(s);
        default: return ViewOf<64>(s);
    }
}
size_t TableBytes(uint32_t p)
{
    switch (RanksOf(p)) {
        case 8: return sizeof(A2avTable<8>);
        case 16: return sizeof(A2avTable<16>);
        case 32: return sizeof(A2avTable<32>);
        default: return sizeof(A2avTable<64>);
    }
}
size_t ImageBytes(uint32_t p) { return p <= 8 ? sizeof(A2avArgs<8>) : (p <= 16 ? sizeof(A2avArgs<16>) : TableBytes(p)); }

// p numbers into 32 bits; what they hold beyond that.
uint64_t Narrow(const uint64_t *row, uint32_t *to, uint32_t p)
{
    uint64_t beyond = 0;
    for (uint32_t i = 0; i < p; i++) {
        to[i] = uint32_t(row[i]);
        beyond |= row[i];
    }
    return beyond >> 32;
}
uint64_t Differ(const uint64_t *row, const uint32_t *have, uint32_t p)
{
    uint64_t d = 0;
    for (uint32_t i = 0; i < p; i++) {
        d |= row[i] ^ have[i];
    }
    return d;
}

// The set in which this call is written down: one that is not among those it has agreed with so far, the one longest unused.
uint32_t Victim(const Group *g)
{
    uint32_t best = 0;
    uint64_t oldest = ~uint64_t(0);
    for (uint32_t k = 0; k < kA2avSets; k++) {
        const A2avSet &s = g->a2avSets[k];
        const uint64_t used = s.valid ? s.lastUse : 0;
        if (!((g->a2avAlive >> k) & 1u) && used < oldest) {
            oldest = used;
            best = k;
        }
    }
    return best;
}

// What a rank passed, into set s.
bool TakeRow(Group *g, A2avSet *s, uint32_t r, void *send, void *recv, const uint64_t *const rows[4])
{
    const View v = ViewOf(s, g->p);
    v.send[r] = reinterpret_cast<uint64_t>(send);
    v.recv[r] = reinterpret_cast<uint64_t>(recv);
    uint64_t beyond = Narrow(rows[0], s->sent.data() + size_t(r) * g->p, g->p);
    beyond |= Narrow(rows[1], s->place.data() + size_t(r) * g->p, g->p);
    beyond |= Narrow(rows[2], v.count + size_t(r) * v.stride, g->p);
    beyond |= Narrow(rows[3], v.to + size_t(r) * v.stride, g->p);
    return beyond == 0;
}
bool SameRow(Group *g, A2avSet *s, uint32_t r, const void *send, const void *recv, const uint64_t *const rows[4])
{
    const View v = ViewOf(s, g->p);
    return v.send[r] == reinterpret_cast<uint64_t>(send) && v.recv[r] == reinterpret_cast<uint64_t>(recv) &&
        Differ(rows[3], v.to + size_t(r) * v.stride, g->p) == 0 && Differ(rows[2], v.count + size_t(r) * v.stride, g->p) == 0 &&
        Differ(rows[1], s->place.data() + size_t(r) * g->p, g->p) == 0 && Differ(rows[0], s->sent.data() + size_t(r) * g->p, g->p) == 0;
}
void CopyRow(const Group *g, A2avSet *from, A2avSet *to, uint32_t r)
{
    const View a = ViewOf(from, g->p), b = ViewOf(to, g->p);
    const size_t n = g->p * sizeof(uint32_t);
    b.send[r] = a.send[r];
    b.recv[r] = a.recv[r];
    std::memcpy(to->sent.data() + size_t(r) * g->p, from->sent.data() + size_t(r) * g->p, n);
    std::memcpy(to->place.data() + size_t(r) * g->p, from->place.data() + size_t(r) * g->p, n);
    std::memcpy(b.count + size_t(r) * b.stride, a.count + size_t(r) * a.stride, n);
    std::memcpy(b.to + size_t(r) * b.stride, a.to + size_t(r) * a.stride, n);
}

// alltoall_operator.cc:49-72: what i sends to j must be what j expects from i.
HcclResult SidesAgree(const Group *g, const A2avSet &s, const View &v)
{
    constexpr uint32_t kBlock = 16;      // (one of the two tables is walked across its rows)
    const uint32_t p = g->p;
    uint32_t differ = 0;
    for (uint32_t i0 = 0; i0 < p; i0 += kBlock) {
        for (uint32_t j0 = 0; j0 < p; j0 += kBlock) {
            for (uint32_t i = i0; i < std::min(i0 + kBlock, p); i++) {
                for (uint32_t j = j0; j < std::min(j0 + kBlock, p); j++) {
                    differ |= s.sent[size_t(i) * p + j] ^ v.count[size_t(j) * v.stride + i];
                }
            }
        }
    }
    for (uint32_t i = 0; i < p && differ != 0; i++) {
        for (uint32_t j = 0; j < p; j++) {
            if (s.sent[size_t(i) * p + j] != v.count[size_t(j) * v.stride + i]) {
                HCCL_LOG_ERROR("AlltoAllV: rank %u sends %u elements to rank %u, which expects %u", i, s.sent[size_t(i) * p + j], j,
                    v.count[size_t(j) * v.stride + i]);
                return HCCL_E_PARA;
            }
        }
    }
    return HCCL_SUCCESS;
}

// Whether no two blocks of a receiver land on the same bytes.  Usually they lie one behind the other.
bool Apart(const uint32_t *to, const uint32_t *count, uint32_t p)
{
    uint32_t bad = 0;
    for (uint32_t i = 0; i + 1 < p; i++) {
        bad |= uint64_t(to[i]) + count[i] > to[i + 1] ? 1u : 0u;
    }
    if (bad == 0) {
        return true;
    }
    std::vector<std::pair<uint64_t, uint64_t>> spans;
    for (uint32_t i = 0; i < p; i++) {
        if (count[i] != 0) {
            spans.emplace_back(to[i], uint64_t(to[i]) + count[i]);
        }
    }
    std::sort(spans.begin(), spans.end());
    for (size_t k = 1; k < spans.size(); k++) {
        if (spans[k - 1].second > spans[k].first) {
            return false;
        }
    }
    return true;
}
uint64_t Extent(const uint32_t *at, const uint32_t *count, uint32_t p)
{
    uint64_t end = 0;
    for (uint32_t i = 0; i < p; i++) {
        const uint64_t e = count[i] != 0 ? uint64_t(at[i]) + count[i] : 0;
        end = e > end ? e : end;
    }
    return end;
}

// Checks the call written down in set s and lays its pieces out.  *general: it goes the general way.
HcclResult Complete(Group *g, A2avSet *s, uint32_t unit, bool *general)
{
    const View v = ViewOf(s, g->p);
    const uint32_t p = g->p, unitShift = uint32_t(__builtin_ctz(unit));
    s->unitShift = unitShift;
    HcclResult r = SidesAgree(g, *s, v);
    if (r != HCCL_SUCCESS) {
        return r;
    }
    uint64_t total = 0;
    uint32_t longest = 0;
    s->sendBytes.resize(p);
    s->recvBytes.resize(p);
    for (uint32_t i = 0; i < p; i++) {
        const uint32_t *count = v.count + size_t(i) * v.stride, *to = v.to + size_t(i) * v.stride, *sent = s->sent.data() + size_t(i) * p;
        s->sendBytes[i] = Extent(s->place.data() + size_t(i) * p, sent, p) * unit;
        s->recvBytes[i] = Extent(to, count, p) * unit;
        if (!Apart(to, count, p)) {
            *general = true;
            return HCCL_SUCCESS;
        }
        for (uint32_t j = 0; j < p; j++) {
            total += count[j];
            longest = std::max(longest, count[j]);
        }
    }
    if (uint64_t(longest) * unit >= uint64_t(1) << 31) {
        *general = true;
        return HCCL_SUCCESS;
    }
    bool needStage = false, gatherInPlace = false;
    r = CheckOverlap(g, s->sendBytes, s->recvBytes, &needStage, &gatherInPlace);
    if (r != HCCL_SUCCESS) {
        return r;
    }
    if (needStage) {
        *general = true;
        return HCCL_SUCCESS;
    }
    constexpr uint32_t kBlock = 16;      // the senders' displacements, by receiver
    for (uint32_t i0 = 0; i0 < p; i0 += kBlock) {
        for (uint32_t j0 = 0; j0 < p; j0 += kBlock) {
            for (uint32_t j = j0; j < std::min(j0 + kBlock, p); j++) {
                for (uint32_t i = i0; i < std::min(i0 + kBlock, p); i++) {
                    v.from[size_t(j) * v.stride + i] = s->place[size_t(i) * p + j];
                }
            }
        }
    }
    const uint32_t size = 1u << kA2avShift;
    uint64_t pieces = 0;
    for (uint32_t j = 0; j < v.stride; j++) {
        v.rowStart[j] = uint32_t(pieces);
        for (uint32_t i = 0; j < p && i < p; i++) {
            const uint32_t bytes = v.count[size_t(j) * v.stride + i] << unitShift;
            const uint32_t off = (uint32_t(v.recv[j]) + (v.to[size_t(j) * v.stride + i] << unitShift)) & (kA2avLine - 1);
            pieces += bytes == 0 ? 0u : (off + uint64_t(bytes) + size - 1) >> kA2avShift;
        }
    }
    if (pieces >= uint64_t(1) << 31) {
        *general = true;
        return HCCL_SUCCESS;
    }
    const bool alike = total == uint64_t(longest) * p * p;
    total *= unit;
    s->pieces = uint32_t(pieces);
    s->width = total <= kOneWaveTotal ? 0 : ((p <= 16 && alike) || total <= kTwoPerCuTotal ? 2 : 1);
    s->launches = uint32_t((total + kLaunchTotal - 1) / kLaunchTotal);
    s->moved = total;
    return HCCL_SUCCESS;
}

}  // namespace

void A2avBegin(Group *g, uint32_t unit)
{
    const GroupConfig &cfg = g->cfg;
    static const bool verifyAll = [] {
        const char *e = std::getenv("HCCL_AMD_PLAN_VERIFY");
        return e != nullptr && e[0] != '\0' && e[0] != '0';
    }();
    g->a2avOpen = cfg.fuse && cfg.direct && cfg.team != 1 && cfg.blocksPerCu == 0 && cfg.launchCapMiB < 0 && cfg.fusedStores < 0 && !verifyAll &&
        unit != 0 && (unit & (unit - 1)) == 0;
    g->a2avAlive = 0;
    g->a2avBuilding = -1;
    g->a2avUnit = unit;
    if (!g->a2avOpen) {
        return;
    }
    g->a2avSets.resize(kA2avSets);
    for (uint32_t k = 0; k < kA2avSets; k++) {
        g->a2avAlive |= g->a2avSets[k].valid && g->a2avSets[k].unitShift == uint32_t(__builtin_ctz(unit)) ? 1u << k : 0u;
    }
}

bool A2avRow(Group *g, uint32_t r, void *send, void *recv, const uint64_t *const rows[4])
{
    if (g->a2avBuilding < 0) {
        const uint32_t before = g->a2avAlive;
        uint32_t alive = 0;
        for (uint32_t k = 0; k < kA2avSets; k++) {
            alive |= ((before >> k) & 1u) && SameRow(g, &g->a2avSets[k], r, send, recv, rows) ? 1u << k : 0u;
        }
        if (alive != 0) {
            g->a2avAlive = alive;
            return true;
        }
        // a new call from here on: the rows so far are those of the sets it agreed with
        const bool first = g->arrived == 0;
        if (first) {
            g->a2avAlive = 0;
        }
        const uint32_t to = Victim(g);
        A2avSet *s = &g->a2avSets[to];
        s->valid = s->general = false;
        s->image.resize(ImageBytes(g->p));
        s->sent.resize(size_t(g->p) * g->p);
        s->place.resize(size_t(g->p) * g->p);
        A2avSet *from = before != 0 ? &g->a2avSets[uint32_t(__builtin_ctz(before))] : s;
        for (uint32_t q = 0; !first && from != s && q < g->p; q++) {
            if (g->here[q] && q != r) {
                CopyRow(g, from, s, q);
            }
        }
        g->a2avBuilding = int(to);
    }
    return TakeRow(g, &g->a2avSets[uint32_t(g->a2avBuilding)], r, send, recv, rows);
}

void A2avExpand(Group *g, uint32_t except)
{
    const uint32_t p = g->p;
    A2avSet *s = g->a2avBuilding >= 0 ? &g->a2avSets[uint32_t(g->a2avBuilding)] : (g->a2avAlive != 0 ? &g->a2avSets[uint32_t(__builtin_ctz(g->a2avAlive))] : nullptr);
    // (rows that are in pend's tables already leave what was found out about those as it is)
    std::vector<uint64_t> *tables[4] = {&g->pend.sendCounts, &g->pend.sdispls, &g->pend.recvCounts, &g->pend.rdispls};
    bool same = true;
    for (std::vector<uint64_t> *t : tables) {
        same = same && t->size() == size_t(p) * p;
        t->resize(size_t(p) * p);
    }
    for (uint32_t r = 0; s != nullptr && r < p; r++) {
        if (!g->here[r] || r == except) {
            continue;
        }
        const View v = ViewOf(s, p);
        const uint32_t *rows[4] = {s->sent.data() + size_t(r) * p, s->place.data() + size_t(r) * p, v.count + size_t(r) * v.stride, v.to + size_t(r) * v.stride};
        for (int k = 0; k < 4; k++) {
            uint64_t *to = tables[k]->data() + size_t(r) * p;
            if (Differ(to, rows[k], p) != 0) {
                std::copy(rows[k], rows[k] + p, to);
                same = false;
            }
        }
    }
    if (!same) {
        g->tablesChecked = false;
        g->lastA2av = nullptr;
    }
    g->a2avOpen = false;
}

HcclResult A2avFinish(Group *g, hipStream_t stream, A2avSet **ready)
{
    *ready = nullptr;
    if (!g->deviceReady) {
        return HCCL_SUCCESS;
    }
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &capture) != hipSuccess || capture != hipStreamCaptureStatusNone) {
        (void)hipGetLastError();
        return HCCL_SUCCESS;
    }
    if (g->a2avBuilding < 0) {
        A2avSet *s = &g->a2avSets[uint32_t(__builtin_ctz(g->a2avAlive))];
        s->hit = true;
        s->lastUse = ++g->a2avClock;
        *ready = s->general ? nullptr : s;
        return HCCL_SUCCESS;
    }
    A2avSet *s = &g->a2avSets[uint32_t(g->a2avBuilding)];
    bool general = false;
    HcclResult r = Complete(g, s, g->a2avUnit, &general);
    if (r != HCCL_SUCCESS) {
        return r;
    }
    if (general) {
        // (its tables and buffers say so: it will go that way whenever it comes back)
        s->valid = s->general = true;
        s->lastUse = ++g->a2avClock;
        return HCCL_SUCCESS;
    }
    s->hit = false;
    *ready = s;
    return HCCL_SUCCESS;
}

namespace {

// Puts the set's tables into device memory, if they are not there, for a launch on `stream`; nothing here waits on the host for other streams' work.
// A set that another call takes over is written anew, behind the launches that read it.  As long as all of a group's calls come on one
// stream, its order sees to that and a call pays for no event.  From the first call on a second stream on, every launch leaves an event behind,
// and sets are written to the other half of the memory: what launches that left no event may still read is never written again.
HcclResult OnDevice(Group *g, A2avSet *s, hipStream_t stream)
{
    const size_t bytes = (TableBytes(g->p) + 255) & ~size_t(255);
    if (g->a2avTables == nullptr) {
        HIP_OK(hipMalloc(&g->a2avTables, 2 * kA2avSets * bytes));
        g->a2avStream = stream;
    }
    g->a2avStreams = g->a2avStreams || g->a2avStream != stream;
    if (s->onDevice) {
        if (s->stream != stream && !s->arrived) {
            if (hipEventQuery(s->uploaded) == hipSuccess) {
                s->arrived = true;
            } else {
                (void)hipGetLastError();
                HIP_OK(hipStreamWaitEvent(stream, s->uploaded, 0));
            }
        }
        return HCCL_SUCCESS;
    }
    if (s->uploaded == nullptr) {
        HIP_OK(hipEventCreateWithFlags(&s->uploaded, hipEventDisableTiming));
    } else if (g->a2avStreams) {
        HIP_OK(hipStreamWaitEvent(stream, s->uploaded, 0));
        for (A2avReader &r : s->readers) {
            if (r.reading) {
                HIP_OK(hipStreamWaitEvent(stream, r.done, 0));
                r.reading = false;
            }
        }
    }
    s->table = static_cast<char *>(g->a2avTables) + (2 * size_t(s - g->a2avSets.data()) + (g->a2avStreams ? 1 : 0)) * bytes;
    StageSlot &slot = g->stageSlots[g->stageNext++ % g->stageSlots.size()];
    if (slot.used) {
        HIP_OK(hipEventSynchronize(slot.done));
    }
    std::memcpy(slot.host, s->image.data(), TableBytes(g->p));
    HIP_OK(UploadFromPinned(s->table, slot.host, TableBytes(g->p), stream));
    HIP_OK(hipEventRecord(slot.done, stream));
    slot.used = true;
    HIP_OK(hipEventRecord(s->uploaded, stream));
    s->stream = stream;
    s->arrived = false;
    s->onDevice = true;
    return HCCL_SUCCESS;
}

// What a launch on `stream` leaves its event in.  A set remembers a few streams; beyond those a launch goes behind the one whose place it takes.
HcclResult Reader(A2avSet *s, hipStream_t stream, A2avReader **reader)
{
    for (A2avReader &r : s->readers) {
        if (r.stream == stream) {
            *reader = &r;
            return HCCL_SUCCESS;
        }
    }
    if (s->readers.size() < kA2avReaders) {
        A2avReader fresh;
        HIP_OK(hipEventCreateWithFlags(&fresh.done, hipEventDisableTiming));
        s->readers.push_back(fresh);
        *reader = &s->readers.back();
    } else {
        *reader = &s->readers[s->nextReader++ % kA2avReaders];
        HIP_OK(hipStreamWaitEvent(stream, (*reader)->done, 0));
    }
    (*reader)->stream = stream;
    return HCCL_SUCCESS;
}

}  // namespace

// Up to 16 ranks a new call's tables travel in the arguments; from its second time on it reads them from device memory: the launch call writes 944
// bytes of arguments to 8 ranks, 3.4 KB to 16, of 24 otherwise.
bool A2avInArguments(const Group *g, const A2avSet *s) { return g->p <= 16 && !s->hit; }

HcclResult A2avLaunch(Group *g, A2avSet *s, hipStream_t stream)
{
    const bool inArguments = A2avInArguments(g, s);
    A2avReader *reader = nullptr;
    if (!s->hit) {
        s->onDevice = false;
    }
    if (!inArguments) {
        HcclResult r = OnDevice(g, s, stream);
        if (r == HCCL_SUCCESS && g->a2avStreams) {
            r = Reader(s, stream, &reader);
        }
        if (r != HCCL_SUCCESS) {
            return r;
        }
    }
    const uint32_t ranks = RanksOf(g->p), which = uint32_t(__builtin_ctz(ranks)) - 3;
    const void *func = LookupCopyKernel(KernelKind(inArguments ? KK_A2AV_ARGS + which + (s->width == 0 ? 0 : 2) : KK_A2AV + which + (s->width == 0 ? 0 : 4)));
    if (func == nullptr) {
        return HCCL_E_NOT_SUPPORT;
    }
    for (uint32_t n = 0; n < s->launches; n++) {
        A2avRange range = {uint32_t(uint64_t(s->pieces) * n / s->launches), uint32_t(uint64_t(s->pieces) * (n + 1) / s->launches), s->unitShift, kA2avShift};
        const uint32_t pieces = range.end - range.first, waves = s->width == 0 ? 1 : kBlockThreads / 64;
        const uint32_t grid = std::min((s->width == 0 ? 16 : s->width) * g->numCu, (pieces + waves - 1) / waves);
        if (grid == 0) {
            continue;
        }
        void *args[2] = {&s->table, &range};
        if (inArguments) {
            std::memcpy(s->image.data() + TableBytes(g->p), &range, sizeof(range));
            args[0] = s->image.data();
        }
        HIP_OK(hipLaunchKernel(func, dim3(grid, 1, 1), dim3(64 * waves, 1, 1), args, 0, stream));
    }
    if (reader != nullptr) {
        HIP_OK(hipEventRecord(reader->done, stream));
        reader->reading = true;
    }
    if (!s->hit) {
        s->valid = true;
        s->lastUse = ++g->a2avClock;
    }
    return HCCL_SUCCESS;
}

}  // namespace hcclamd
