// Host-only check of the executor's rules on sizes and alignment (cann-hccl_amd/csrc/launch_rules.h), compiled and run by
// tests/test_launch_rules_cpu.py.
#include <cstdio>
#include <cstdlib>
#include <random>

#include "launch_rules.h"

using namespace hcclamd;

#define CHECK(c)                                              \
    do {                                                      \
        if (!(c)) {                                           \
            std::printf("FAIL line %d: %s\n", __LINE__, #c);  \
            std::exit(1);                                     \
        }                                                     \
    } while (0)

namespace {

std::mt19937_64 rng(20);
uint64_t Draw(uint64_t n) { return rng() % n; }

// Heads, bodies and tails cover the stretch in order, and a body starts where the rule says.
void CheckSplit()
{
    uint64_t bodies = 0, unaligned = 0;
    for (int round = 0; round < 40000; round++) {
        const uint64_t unit = uint64_t(1) << Draw(4);
        std::vector<uintptr_t> addrs(1 + Draw(9));
        const uint64_t residues = 1 + Draw(3);     // few of them, so that groups form
        uint64_t shift[3] = {Draw(128) / unit * unit, Draw(128) / unit * unit, Draw(128) / unit * unit};
        for (uintptr_t &a : addrs) {
            a = (uintptr_t(1) << 40) + Draw(1 << 20) * 128 + shift[Draw(residues)];
        }
        const uint64_t bytes = unit * (Draw(2) != 0 ? Draw(200) : Draw(40000));
        for (AnchorRule rule : {ANCHOR_FIRST, ANCHOR_MOST}) {
            const Cut cut = CutByAlignment(addrs, bytes, rule);
            CHECK(cut.head + cut.body + cut.tail == bytes);
            CHECK(cut.head < 128 && cut.tail < 16 && cut.body % 16 == 0);      // (a fused item's ends are one pass of a workgroup)
            CHECK(cut.head % unit == 0 && cut.tail % unit == 0);
            if (cut.body == 0) {
                continue;
            }
            size_t agree[16] = {0}, most = 0;
            for (uintptr_t a : addrs) {
                most = std::max(most, ++agree[(a + cut.head) & 15]);
            }
            CHECK((agree[0] == addrs.size()) == cut.aligned);
            if (rule == ANCHOR_FIRST) {
                CHECK(((addrs[0] + cut.head) & 15) == 0);      // the step kernel's aligned stores
                CHECK(bytes < 4 * uint64_t(kTileBytes) + 128 || ((addrs[0] + cut.head) & 127) == 0);
            } else {
                CHECK(agree[0] == most);
            }
            bodies++;
            unaligned += cut.aligned ? 0 : 1;
        }
    }
    CHECK(bodies > 30000 && unaligned > 5000);
}

// The regions cover the whole tiles in order, none holds more than its team can park, and every team has one; short of a round
// every team gets as many tiles as the others.
void CheckTeamRegions()
{
    for (int round = 0; round < 20000; round++) {
        const uint32_t roundTiles = 1 + uint32_t(Draw(kTeamTiles)), perTeam = 1 + uint32_t(Draw(40)), all = roundTiles * perTeam * kTeamXcds;
        const uint32_t tiles = uint32_t(Draw(2) != 0 ? Draw(all) : Draw(8 * uint64_t(all)));
        const uint64_t pieces = Draw(uint64_t(tiles) + 1) * Draw(kTileBytes);      // behind the whole tiles: less than a tile for each item
        const std::vector<TeamRegion> regions = TeamRegions(tiles, uint64_t(tiles) * kTileBytes + pieces, roundTiles, perTeam);
        CHECK(regions.size() >= kTeamXcds);
        uint32_t at = 0, least = tiles, most = 0;
        for (const TeamRegion &r : regions) {
            CHECK((r.first == at || r.count == 0) && r.count <= roundTiles * perTeam);
            at += r.count;
            least = std::min(least, r.count);
            most = std::max(most, r.count);
        }
        CHECK(at == tiles && (tiles >= all || most - least <= 1));
    }
}

// The line does not move with a buffer's start or with the number of pieces: the same bytes, cut anywhere.
void CheckTeamRounds()
{
    for (int round = 0; round < 20000; round++) {
        const uint32_t halfRounds = 1 + uint32_t(Draw(8)), roundTiles = 1 + uint32_t(Draw(kTeamTiles)), cus = 8 * (1 + uint32_t(Draw(40))), items = 1 + uint32_t(Draw(64));
        const uint64_t line = uint64_t(halfRounds) * roundTiles * cus * kTileBytes / 2, each = (line + items - 1) / items + kTileBytes;
        const Cut cut = CutByAlignment({(uintptr_t(1) << 40) + Draw(128)}, each, ANCHOR_MOST);
        CHECK(TeamRounds(items * (cut.head + cut.body + cut.tail), halfRounds, roundTiles, cus));
        CHECK(!TeamRounds(line - 1, halfRounds, roundTiles, cus));
    }
}

// All launches of a collective of one shape store alike, however the cap cut it; what the caller has set holds everywhere.
void CheckStores()
{
    for (int round = 0; round < 2000; round++) {
        const bool reduces = Draw(2) != 0;
        const uint64_t nsrc = reduces ? 2 + Draw(16) : 1, ndst = 1 + Draw(8), block = 1 + Draw(uint64_t(200) << 20), items = 1 + Draw(64);
        const uint64_t moved = items * block * (nsrc + ndst);
        const uint32_t whole = StoreFlags(-1, reduces, false, moved, items * block * ndst, moved);
        const bool small = moved <= 2 * kMemorySideCacheBytes;
        CHECK(whole == ((reduces ? small && nsrc >= 2 * ndst : ndst >= 2 && (small || ndst >= 4)) ? kFusedThroughStores : kFusedNtStores));
        for (uint64_t n = 1; n <= items; n++) {
            const uint64_t traffic = n * block * (nsrc + ndst), written = n * block * ndst;
            CHECK(StoreFlags(-1, reduces, false, traffic, written, moved) == whole);
            CHECK(StoreFlags(-1, reduces, true, traffic, written, moved) == 0);
            for (bool team : {false, true}) {
                CHECK(StoreFlags(0, reduces, team, traffic, written, moved) == kFusedNtStores);
                CHECK(StoreFlags(1, reduces, team, traffic, written, moved) == kFusedOrdinaryStores);
            }
        }
    }
}

// Workgroups per CU on either side of the lines.
void CheckWidth()
{
    auto width = [](bool scatter, uint32_t ranks, uint32_t unit, double mibRead, bool bf16Selects = false) {
        FusedShape f;
        f.reduces = f.chains = true;
        f.reduceScatter = scatter;
        f.bf16Selects = bf16Selects;
        f.sources = ranks;
        f.unit = unit;
        f.bytes = mibRead * 1048576.0 / ranks;
        f.storeBytes = f.bytes;
        f.streamBytes = f.bytes * (ranks + 1);
        f.capBytes = scatter ? uint64_t(512) << 20 : 0;
        return FusedPerCu(f);
    };
    for (bool scatter : {false, true}) {
        CHECK(width(scatter, 8, 4, 512) == 1 && width(scatter, 23, 4, 2400) == 1 && width(scatter, 24, 4, 600) == 2 && width(scatter, 64, 8, 2400) == 2);
        CHECK(width(scatter, 8, 2, 512) == 1 && width(scatter, 52, 2, 2400) == 1 && width(scatter, 53, 2, 2400) == (scatter ? 8u : 1u));
        CHECK(width(scatter, 8, 1, 600) == 2 && width(scatter, 40, 1, 2400) == 2 && width(scatter, 41, 1, 2400) == (scatter ? 8u : 2u));
        CHECK(width(scatter, 48, 1, 300) == 8 && width(scatter, 48, 2, 300) == 8 && width(scatter, 48, 4, 300) == 2);
        CHECK(width(scatter, 7, 4, 600) == 2 && width(scatter, 7, 2, 2400) == 2 && width(scatter, 7, 1, 600) == 2 && width(scatter, 7, 2, 200) == 8);
        CHECK(width(scatter, 7, 2, 600, true) == 2 && width(scatter, 8, 2, 600, true) == (scatter ? 2u : 1u) && width(scatter, 9, 2, 600, true) == 2);
        CHECK(width(scatter, 44, 2, 2400, true) == 2 && width(scatter, 45, 2, 2400, true) == (scatter ? 8u : 2u));
        for (bool selects : {false, true}) {
            const uint32_t unit = selects ? 2 : 1;
            CHECK(width(scatter, 31, unit, 330, selects) == 2 && width(scatter, 32, unit, 330, selects) == 8 && width(scatter, 32, unit, 420, selects) == 2);
            CHECK(width(scatter, 40, unit, 450, selects) == 2 && width(scatter, 48, unit, 450, selects) == 8 && width(scatter, 64, unit, 600, selects) == 8);
            CHECK(width(scatter, 64, unit, 700, selects) == (scatter ? 8u : 2u));
        }
        CHECK(width(scatter, 32, 2, 330) == 2 && width(scatter, 48, 2, 450) == 2);
    }
    auto mid = [](bool chains, uint32_t unit, double tilesPerCu) {
        FusedShape f;
        f.reduces = true;
        f.chains = chains;
        f.sources = 4;
        f.unit = unit;
        f.bytes = tilesPerCu * 256 * kTileBytes;
        f.storeBytes = f.bytes * 4;
        f.streamBytes = f.bytes * 8;
        return FusedPerCu(f);
    };
    CHECK(mid(true, 4, 2.9) == 2 && mid(true, 4, 3.1) == 8 && mid(true, 2, 15.9) == 8 && mid(true, 2, 16.1) == 2 && mid(true, 1, 8) == 2 && mid(true, 4, 33) == 1);
    CHECK(mid(false, 4, 2.9) == 2 && mid(false, 4, 3.1) == 8 && mid(false, 2, 3.9) == 8 && mid(false, 2, 4.1) == 2 && mid(false, 4, 15.9) == 2 && mid(false, 1, 3.5) == 2);
}

}  // namespace

int main()
{
    CheckSplit();
    CheckTeamRegions();
    CheckTeamRounds();
    CheckStores();
    CheckWidth();
    std::printf("OK\n");
    return 0;
}
