// Host program of tests/test_duo_start.py: counts, for every wavefront of every launch size, the loads that stand behind the
// first layer's parameters when the kernel waits for those, and prints where the wait would let a parameter be under way.
#include <cstdio>

#include "bf_duo.hip.h"

namespace {

template <bool FP8, int NP>
int check() {
    typedef bf::duo::Cfg<FP8, NP> C;
    int bad = 0, least = 1 << 30, most = 0;
    for (int blocks = 1; blocks <= 600; blocks++)
        for (int block = 0; block < blocks; block++)
            for (int wave = 0; wave < C::NW; wave++) {
                int behind = C::RING;
                for (int j = 0; j < C::WARM; j++) {
                    bool any = false;   // a load that no lane takes part in is not issued
                    for (int lane = 0; lane < 64; lane++) any = any || C::warms(C::warm_line(j, block, blocks, wave, lane), blocks);
                    behind += any;
                }
                least = behind < least ? behind : least;
                most = behind > most ? behind : most;
                bad += behind < C::BEHIND_PARAMETERS;
            }
    printf("%s, %d per workgroup: %d to %d loads behind the parameters, %d allowed under way, %d faults\n", FP8 ? "e4m3" : "int8", NP, least, most,
           C::BEHIND_PARAMETERS, bad);
    return bad;
}

}  // namespace

int main() {
    const int bad = check<false, 1>() + check<false, 2>() + check<true, 1>() + check<true, 2>();
    return bad != 0;
}
