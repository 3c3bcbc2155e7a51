// Host program of tests/test_team_exchange.py: goes through exchange B of the team form as Cfg lays it out, for both
// network widths, prints every load whose bytes were stored by a wavefront that the reader does not wait for, and compares
// flags with tags over the wrap of their count.
#include <cstdio>
#include <set>
#include <utility>
#include <vector>

#include "bf_team.hip.h"

namespace {

struct Store { int member, wave, at, bytes; };

template <int DM>
int check() {
    typedef bf::team::Cfg<DM> C;
    const int TW = C::TWW, quads = 4, SCALES = bf::T * 4;
    int bad = 0;
    std::vector<Store> stores;
    for (int m = 0; m < C::NWG; m++)
        for (int w = 0; w < C::NW; w++) {
            if (w == 0) stores.push_back({m, w, C::scales_b(m), SCALES});
            if (C::TWO_STEPS) {
                for (int i = 0; i < TW; i++)
                    for (int j = 0; j < quads; j++) stores.push_back({m, w, C::piece_b(m, TW * w + i, j), bf::FRAG});
            } else stores.push_back({m, w, C::WS_B + m * C::ROWS + w * C::ROWS_W, C::ROWS_W});
        }
    for (size_t a = 0; a < stores.size(); a++) {   // places of their own, inside the buffers of the exchange
        const Store& s = stores[a];
        if (s.at < C::WS_B || s.at + s.bytes > C::WS_C || C::WS_C > C::WS_BYTES) bad++, printf("width %d: a store at %d leaves its buffer\n", DM, s.at);
        for (size_t b = 0; b < a; b++)
            if (s.at < stores[b].at + stores[b].bytes && stores[b].at < s.at + s.bytes) bad++, printf("width %d: stores at %d and %d overlap\n", DM, s.at, stores[b].at);
    }
    int loads = 0;
    for (int reader = 0; reader < C::NWG; reader++)
        for (int wave = 0; wave < C::NW; wave++) {
            std::set<int> waited;
            if (C::FLAGS_B > 64) bad++, printf("width %d: %d flags do not fit a wavefront's poll\n", DM, C::FLAGS_B);
            for (int i = 0; i < C::FLAGS_B; i++) waited.insert(C::awaited_b(reader, i));
            std::vector<std::pair<int, int>> reads;   // (place, bytes)
            for (int c = 0; c < C::NWG; c++) {
                reads.push_back({C::scales_b(c), SCALES});
                if (C::TWO_STEPS) reads.push_back({C::piece_b(c, C::tile_b(reader, wave), wave & 3), bf::FRAG});
                else reads.push_back({C::WS_B + c * C::ROWS, C::ROWS});   // four tokens of every tile: a part of every wavefront's store
            }
            for (const auto& r : reads) {
                int covered = 0;
                for (const Store& s : stores) {
                    const int lo = s.at > r.first ? s.at : r.first, hi = s.at + s.bytes < r.first + r.second ? s.at + s.bytes : r.first + r.second;
                    if (lo >= hi) continue;
                    covered += hi - lo;
                    if (!waited.count(C::flag_b(s.member, s.wave)))
                        bad++, printf("width %d: member %d wavefront %d loads %d bytes at %d that member %d wavefront %d stored, without waiting for it\n", DM, reader,
                                      wave, hi - lo, lo, s.member, s.wave);
                }
                if (covered != r.second) bad++, printf("width %d: member %d wavefront %d loads bytes at %d that nobody stored\n", DM, reader, wave, r.first);
                loads++;
            }
        }
    printf("width %d: %d loads, %d faults\n", DM, loads, bad);
    return bad;
}

}  // namespace

// A flag of the exchanges waited for in one launch is the count of this launch or of one before it: raised or not must be told
// apart wherever the count stands, and the heads' flags however many launches they were not raised in.
int check_counts() {
    int bad = 0;
    const unsigned starts[] = {0u, 1u, 0x7ffffff0u, 0x7fffffffu, 0x80000000u, 0xfffffff0u, 0xffffffffu};
    for (unsigned tag0 : starts)
        for (unsigned layer = 1; layer <= 64; layer++) {
            const unsigned tag = tag0 + layer;
            for (unsigned lag = 1; lag <= layer + 64; lag++) bad += bf::team::Reached()(tag - lag, tag) || bf::team::Equal()(tag - lag, tag);
            for (unsigned lag = 1u << 20; lag; lag <<= 1) bad += bf::team::Equal()(tag - lag, tag);
            bad += !bf::team::Reached()(tag, tag) || !bf::team::Equal()(tag, tag);
        }
    printf("counts: %d faults\n", bad);
    return bad;
}

// The launches of a process must leave a unit of every XCD to somebody who completes a team: in the worst case each of
// them has all members of a team but one in place.
int check_units() {
    int bad = 0;
    for (int members : {bf::team::Cfg<256>::NWG, bf::team::Cfg<512>::NWG})
        for (int units = 1; units <= 40; units++)
            for (int queues = 1; queues <= 32; queues++) {
                int left = units;
                for (int i = 0; i < queues; i++) left -= left < members - 1 ? left : members - 1;
                bad += bf::team::units_suffice(queues, members, units) != (left > 0);
            }
    bad += !bf::team::units_suffice(4, bf::team::Cfg<512>::NWG, 32) || bf::team::units_suffice(5, bf::team::Cfg<512>::NWG, 32);
    bad += !bf::team::units_suffice(10, bf::team::Cfg<256>::NWG, 32) || bf::team::units_suffice(11, bf::team::Cfg<256>::NWG, 32);
    printf("units: %d faults\n", bad);
    return bad;
}

int main() {
    if (check_counts() || check_units()) return 1;
    const int narrow = check<256>(), wide = check<512>();
    return narrow || wide;
}
