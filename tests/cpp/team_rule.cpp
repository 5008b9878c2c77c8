// Host checks of the one-kernel PCG solve's rules (idp_amd/csrc/team_rule.hpp).
#include <cstdio>
#include <cstdlib>

#include "../../idp_amd/csrc/team_rule.hpp"

#define CHECK(c)                                                         \
    do {                                                                 \
        if (!(c)) {                                                      \
            std::printf("%s:%d: %s\n", __FILE__, __LINE__, #c);          \
            std::exit(1);                                                \
        }                                                                \
    } while (0)

using namespace idp;

// the looks are the two-kernel loop's chunk ends
static void looks()
{
    int b = 0, chunk = 8, look = HAND_FIRST;
    for (int k = 0; k < HAND_LOOKS; ++k) {
        b += chunk;
        chunk = 2 * chunk < 256 ? 2 * chunk : 256;
        CHECK(look == b);
        look = hand_next(look);
    }
    CHECK(b >= 10000);  // the default iteration limit of a step's solves
}

// while starts fail, tries get rare; one that succeeds brings every solve back
static void starts()
{
    TeamStarts s;
    for (int i = 0; i < 5; ++i) {
        CHECK(s.now());
        s.ended(true);
    }
    int tries = 0;
    for (int i = 0; i < 1000; ++i)
        if (s.now()) {
            ++tries;
            s.ended(false);
        }
    CHECK(tries <= 25);  // 6 on the way to one in 64, then one in 64
    CHECK(tries >= 15);
    while (!s.now()) {
    }
    s.ended(true);
    for (int i = 0; i < 5; ++i) {
        CHECK(s.now());
        s.ended(true);
    }
    CHECK(TEAM_WAIT <= 2000);  // polls of about a microsecond: no longer than a short solve
}

// a launch needs all of its waiting workgroups resident at once
static void fits()
{
    CHECK(team_fits(256, false, 256) && !team_fits(257, false, 512) && !team_fits(257, true, 256));
    // a partition of 32 compute units
    CHECK(team_fits(32, false, 32) && !team_fits(33, false, 32) && team_fits(33, true, 32));
    CHECK(!team_fits(1, false, 0) && team_fits(1, true, 0));
}

// every byte offset of the longest vector fits 32 bits
static void addresses()
{
    CHECK(team_addresses(32768) && team_addresses(89478485));
    CHECK(48ll * 89478485 <= 0xffffffffll && 48ll * 89478486 > 0xffffffffll);
    CHECK(!team_addresses(89478486) && !team_addresses(0x7fffffff));
}

int main()
{
    fits();
    addresses();
    looks();
    starts();
    std::puts("ok");
    return 0;
}
