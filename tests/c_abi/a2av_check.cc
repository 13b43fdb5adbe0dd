// The tables of all-to-all-v calls in device memory (cann-hccl_amd/csrc/a2av.cc), on the host: a seeded walk over calls of one group on a
// model of streams and events (the first quarter of them on one stream), in which work is done as late as the orders allow, in any order they leave open.  Whenever a launch is done, the
// tables it reads have to be those of its call.  The calls may not wait for the device, and a call known by its numbers counts as known on whatever
// stream it comes.  argv[1] = ranks, argv[2] = calls, argv[3] = streams, argv[4] = sets of tables in turn.  argv[2] = 0: calls that go the general
// way instead.  Their tables have to come out as the ranks passed them, and what was found out about those has to hold as long as they are the last ones.
// argv[2] = -1: how wide launches are.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <memory>
#include <string>
#include <vector>

#include "noalloc.h"
#include "runtime.h"

namespace {

uint64_t g_state = 0x2545F4914F6CDD1Dull;
uint64_t Below(uint64_t n)
{
    g_state = g_state * 6364136223846793005ull + 1442695040888963407ull;
    return n == 0 ? 0 : (g_state >> 29) % n;
}

struct Op {
    enum { UPLOAD, LAUNCH, RECORD, WAIT } kind;
    const uint8_t *from = nullptr;      // upload
    uint8_t *to = nullptr;              // upload, launch
    size_t bytes = 0;
    std::vector<uint8_t> want;          // launch: the tables it has to find
    uint32_t event = 0;
    uint64_t serial = 0;                // of a record: which one; of a wait: for which one
};
std::map<uintptr_t, std::deque<Op>> g_streams;
struct Event {
    uint64_t recorded = 0, done = 0;
};
std::vector<Event> g_events(1);
long g_deviceWaits = 0, g_hostWaits = 0, g_launches = 0, g_wrong = 0, g_records = 0, g_order = 0, g_inArguments = 0;
bool g_stage = false;                           // the call's buffers overlap
long g_overlapChecks = 0;
const hcclamd::A2avSet *g_ready = nullptr;      // the call being launched
std::vector<uint8_t> g_expected;                // its tables

Event &Of(hipEvent_t e) { return g_events[reinterpret_cast<uintptr_t>(e)]; }
std::deque<Op> &Of(hipStream_t s) { return g_streams[reinterpret_cast<uintptr_t>(s)]; }

bool Step(std::deque<Op> &q)
{
    if (q.empty() || (q.front().kind == Op::WAIT && g_events[q.front().event].done < q.front().serial)) {
        return false;
    }
    const Op &op = q.front();
    if (op.kind == Op::UPLOAD) {
        std::memcpy(op.to, op.from, op.bytes);
    } else if (op.kind == Op::LAUNCH) {
        g_wrong += std::memcmp(op.to, op.want.data(), op.want.size()) != 0;
    } else if (op.kind == Op::RECORD) {
        g_events[op.event].done = std::max(g_events[op.event].done, op.serial);
    }
    q.pop_front();
    return true;
}
// Some work of some streams.
void Progress(uint64_t steps)
{
    for (uint64_t n = 0; n < steps && !g_streams.empty(); n++) {
        auto it = g_streams.begin();
        std::advance(it, Below(g_streams.size()));
        Step(it->second);
    }
}
void Until(const Event &e, uint64_t serial)
{
    for (long n = 0; e.done < serial; n++) {
        Progress(1);
        if (n > 100000000) {
            std::printf("a wait that never ends\n");
            std::exit(1);
        }
    }
}

}  // namespace

extern "C" {
hipError_t hipMalloc(void **p, size_t n) { *p = std::calloc(1, n); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    g_events.emplace_back();
    *e = reinterpret_cast<hipEvent_t>(g_events.size() - 1);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    Op op;
    op.kind = Op::RECORD;
    op.event = uint32_t(reinterpret_cast<uintptr_t>(e));
    op.serial = ++Of(e).recorded;
    Of(s).push_back(op);
    g_records++;
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned)
{
    Op op;
    op.kind = Op::WAIT;
    op.event = uint32_t(reinterpret_cast<uintptr_t>(e));
    op.serial = Of(e).recorded;
    Of(s).push_back(op);
    g_order++;
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) { return Of(e).done == Of(e).recorded ? hipSuccess : hipErrorNotReady; }
hipError_t hipEventSynchronize(hipEvent_t e)
{
    g_hostWaits += Of(e).done != Of(e).recorded;
    Until(Of(e), Of(e).recorded);
    return hipSuccess;
}
hipError_t hipDeviceSynchronize()
{
    g_deviceWaits++;
    for (bool any = true; any;) {
        any = false;
        for (auto &s : g_streams) {
            while (Step(s.second)) {
                any = true;
            }
        }
    }
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *st) { *st = hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "?"; }
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **args, size_t, hipStream_t s)
{
    g_launches++;
    if (args[0] != &g_ready->table) {       // the tables themselves, which a launch copies at once
        g_inArguments++;
        g_wrong += std::memcmp(args[0], g_expected.data(), g_expected.size()) != 0;
        return hipSuccess;
    }
    Op op;
    op.kind = Op::LAUNCH;
    op.to = static_cast<uint8_t *>(g_ready->table);
    op.want = g_expected;
    Of(s).push_back(op);
    return hipSuccess;
}
}

namespace hcclamd {
hipError_t UploadFromPinned(void *dst, const void *pinned, size_t bytes, hipStream_t stream)
{
    Op op;
    op.kind = Op::UPLOAD;
    op.to = static_cast<uint8_t *>(dst);
    op.from = static_cast<const uint8_t *>(pinned);
    op.bytes = bytes;
    Of(stream).push_back(op);
    return hipSuccess;
}
const void *LookupCopyKernel(KernelKind) { return &g_state; }
HcclResult CheckOverlap(const Group *, const std::vector<uint64_t> &, const std::vector<uint64_t> &, bool *stage, bool *own)
{
    g_overlapChecks++;
    *stage = g_stage;
    *own = false;
    return HCCL_SUCCESS;
}
Prepared::~Prepared() = default;
Group::~Group() = default;
}  // namespace hcclamd

using namespace hcclamd;

namespace {

struct Tables {
    std::vector<uint64_t> t[4];      // counts and displacements of the senders, of the receivers
};
Tables Draw(uint32_t p)
{
    Tables c;
    for (std::vector<uint64_t> &t : c.t) {
        t.resize(p * p);
    }
    for (uint64_t &n : c.t[0]) {
        n = Below(5000);
    }
    for (uint32_t i = 0; i < p; i++) {
        uint64_t at = 0, to = 0;
        for (uint32_t j = 0; j < p; j++) {
            c.t[1][i * p + j] = at;
            c.t[3][i * p + j] = to;
            c.t[2][i * p + j] = c.t[0][j * p + i];
            at += c.t[0][i * p + j];
            to += c.t[0][j * p + i];
        }
    }
    return c;
}

// The ranks arrive; false as soon as one's row does not fit.  What Arrive does then, and for the ranks behind it, is done here too.
bool Rows(Group *g, const Tables &c)
{
    const uint32_t p = g->p;
    bool taken = true;
    g->arrived = 0;
    std::fill(g->here.begin(), g->here.end(), 0);
    A2avBegin(g, 4);
    for (uint32_t r = 0; r < p; r++) {
        g->here[r] = 1;
        const uint64_t *rows[4] = {&c.t[0][r * p], &c.t[1][r * p], &c.t[2][r * p], &c.t[3][r * p]};
        if (taken && !A2avRow(g, r, reinterpret_cast<void *>(0x10000000ull + (uint64_t(r) << 24)), reinterpret_cast<void *>(0x7f0000000000ull + (uint64_t(r) << 24)), rows)) {
            A2avExpand(g, r);
            taken = false;
        }
        std::vector<uint64_t> *pend[4] = {&g->pend.sendCounts, &g->pend.sdispls, &g->pend.recvCounts, &g->pend.rdispls};
        for (int k = 0; k < 4 && !taken; k++) {
            uint64_t *row = pend[k]->data() + r * p;
            if (!std::equal(rows[k], rows[k] + p, row)) {
                std::copy(rows[k], rows[k] + p, row);
                g->tablesChecked = false;
                g->lastA2av = nullptr;
            }
        }
        g->arrived++;
    }
    return taken;
}

int General(Group *g)
{
    const uint32_t p = g->p;
    Tables a = Draw(p), b = Draw(p), far = Draw(p);
    far.t[1][(p / 2) * p + 1] = uint64_t(1) << 40;      // (of a block that is empty)
    far.t[0][(p / 2) * p + 1] = far.t[2][1 * p + p / 2] = 0;
    Prepared *const prepared = reinterpret_cast<Prepared *>(uintptr_t(64));
    // which tables, whether their buffers overlap, whether what is known of the last general call's tables has to hold
    const struct {
        const Tables *t;
        bool stage, holds;
    } calls[] = {{&a, true, false}, {&a, true, true}, {&b, false, true}, {&a, true, true}, {&far, false, false}, {&far, false, true}, {&b, false, true}, {&far, false, true},
        {&a, true, false}, {&a, true, true}};
    long checks = 0;
    for (size_t n = 0; n < sizeof(calls) / sizeof(calls[0]); n++) {
        g_stage = calls[n].stage;
        const long before = g_overlapChecks;
        A2avSet *ready = nullptr;
        const bool rows = Rows(g, *calls[n].t);
        if (rows && A2avFinish(g, reinterpret_cast<hipStream_t>(uintptr_t(1)), &ready) != HCCL_SUCCESS) {
            std::printf("general call %zu: refused\n", n);
            return 1;
        }
        checks += g_overlapChecks - before;
        if (calls[n].t == &b) {
            g_ready = ready;
            if (ready != nullptr) {
                g_expected.assign(ready->image.begin(), ready->image.begin() + 16);
            }
            if (ready == nullptr || A2avLaunch(g, ready, reinterpret_cast<hipStream_t>(uintptr_t(1))) != HCCL_SUCCESS) {
                std::printf("general call %zu: an ordinary one not launched\n", n);
                return 1;
            }
            continue;
        }
        if (ready != nullptr || rows != (calls[n].t == &a)) {
            std::printf("general call %zu: taken\n", n);
            return 1;
        }
        if (rows) {
            A2avExpand(g, p);
        }
        const std::vector<uint64_t> *pend[4] = {&g->pend.sendCounts, &g->pend.sdispls, &g->pend.recvCounts, &g->pend.rdispls};
        for (int k = 0; k < 4; k++) {
            if (*pend[k] != calls[n].t->t[k]) {
                std::printf("general call %zu: table %d is not what the ranks passed\n", n, k);
                return 1;
            }
        }
        if ((g->tablesChecked && g->lastA2av == prepared) != calls[n].holds) {
            std::printf("general call %zu: what was known of its tables %s\n", n, calls[n].holds ? "is lost" : "was kept for others");
            return 1;
        }
        g->tablesChecked = true;
        g->lastA2av = prepared;
    }
    // (one look at each of the two sets of tables that fit: a's, b's)
    std::printf("%s looked over %ld\n", checks == 2 ? "OK" : "BAD", checks);
    return checks == 2 ? 0 : 1;
}

// Workgroups per CU on both sides of the lines, 0: sixteen of one wave.  One block longer by four bytes and one shorter: no longer uniform.
int Widths(Group *g)
{
    const uint32_t p = g->p;
    for (uint64_t kib : {uint64_t(90) << 10, uint64_t(100) << 10, uint64_t(124) << 10, uint64_t(140) << 10, uint64_t(500) << 10}) {
        for (bool uniform : {true, false}) {
            Tables c;
            for (std::vector<uint64_t> &t : c.t) {
                t.resize(p * p);
            }
            for (uint64_t &n : c.t[0]) {
                n = kib * 256 / p / p;
            }
            c.t[0][1] += uniform ? 0 : 1;
            c.t[0][p] -= uniform ? 0 : 1;
            for (uint32_t i = 0; i < p; i++) {
                for (uint32_t j = 0; j < p; j++) {
                    c.t[2][i * p + j] = c.t[0][j * p + i];
                    c.t[1][i * p + j] = j == 0 ? 0 : c.t[1][i * p + j - 1] + c.t[0][i * p + j - 1];
                    c.t[3][i * p + j] = j == 0 ? 0 : c.t[3][i * p + j - 1] + c.t[2][i * p + j - 1];
                }
            }
            A2avSet *ready = nullptr;
            if (!Rows(g, c) || A2avFinish(g, reinterpret_cast<hipStream_t>(uintptr_t(1)), &ready) != HCCL_SUCCESS || ready == nullptr) {
                std::printf("%llu KiB: not taken\n", (unsigned long long)kib);
                return 1;
            }
            const uint32_t mib = uint32_t(kib >> 10), want = mib < 96 ? 0 : mib < 128 || (uniform && p <= 16) ? 2 : 1;
            if (ready->width != want) {
                std::printf("%u MiB, uniform %d: %u workgroups per CU\n", mib, int(uniform), ready->width);
                return 1;
            }
        }
    }
    std::printf("OK\n");
    return 0;
}

}  // namespace

int main(int argc, char **argv)
{
    const uint32_t p = uint32_t(argc > 1 ? std::atoi(argv[1]) : 20);
    const long calls = argc > 2 ? std::atol(argv[2]) : 1000;
    const uint64_t streams = uint64_t(argc > 3 ? std::atoi(argv[3]) : 3), sets = uint64_t(argc > 4 ? std::atoi(argv[4]) : 5);
    std::unique_ptr<Group> owner(new Group);
    Group *g = owner.get();
    g->p = p;
    g->deviceReady = true;
    g->here.assign(p, 0);
    g->stageSlots.resize(8);
    for (StageSlot &slot : g->stageSlots) {
        slot.host = std::calloc(1, 128 << 10);
        (void)hipEventCreateWithFlags(&slot.done, 0);
    }
    if (calls <= 0) {
        return calls == 0 ? General(g) : Widths(g);
    }
    const size_t tableBytes = p <= 8 ? sizeof(A2avTable<8>) : p <= 16 ? sizeof(A2avTable<16>) : p <= 32 ? sizeof(A2avTable<32>) : sizeof(A2avTable<64>);
    std::vector<Tables> tables;
    for (uint64_t c = 0; c < sets; c++) {
        tables.push_back(Draw(p));
    }
    long known = 0, shouldKnow = 0;
    std::deque<uint64_t> latest;        // the last distinct calls
    for (long n = 0; n < calls; n++) {
        const uint64_t c = Below(3) ? Below(sets) : uint64_t(n) % sets, stream = n < calls / 4 ? 1 : 1 + (Below(2) ? Below(streams) : uint64_t(n) % streams);
        if (!Rows(g, tables[c])) {
            std::printf("a row not taken\n");
            return 1;
        }
        A2avSet *ready = nullptr;
        if (A2avFinish(g, reinterpret_cast<hipStream_t>(stream), &ready) != HCCL_SUCCESS || ready == nullptr) {
            std::printf("call %ld: not taken\n", n);
            return 1;
        }
        g_ready = ready;
        g_expected.assign(ready->image.begin(), ready->image.begin() + long(tableBytes));
        const auto seen = std::find(latest.begin(), latest.end(), c);
        shouldKnow += seen != latest.end();
        known += ready->hit;
        if (seen != latest.end()) {
            latest.erase(seen);
        }
        latest.push_back(c);
        if (latest.size() > kA2avSets) {
            latest.pop_front();
        }
        if (A2avLaunch(g, ready, reinterpret_cast<hipStream_t>(stream)) != HCCL_SUCCESS) {
            std::printf("call %ld: not launched\n", n);
            return 1;
        }
        if (Below(6) == 0) {
            Progress(Below(16));
        }
    }
    const long records = g_records;
    for (auto &s : g_streams) {
        if (!s.second.empty()) {
            hipEvent_t e;
            (void)hipEventCreateWithFlags(&e, 0);
            (void)hipEventRecord(e, reinterpret_cast<hipStream_t>(s.first));
        }
    }
    const long waits = g_deviceWaits;
    (void)hipDeviceSynchronize();
    for (auto &s : g_streams) {
        if (!s.second.empty()) {
            std::printf("a wait that never ends\n");
            return 1;
        }
    }
    // (tables that fit travel in the arguments, but only of a call that is new)
    const bool ok = g_wrong == 0 && waits == 0 && known == shouldKnow && g_inArguments == (p <= 16 ? calls - known : 0);
    std::printf("%s launches %ld with tables in the arguments %ld wrong %ld device waits %ld known %ld of %ld records %ld orders %ld\n",
        ok ? "OK" : "BAD", g_launches, g_inArguments, g_wrong, waits, known, shouldKnow, records, g_order);
    return ok ? 0 : 1;
}
