// The numbers by which the workgroups of a team meet (torsh_amd/csrc/hipq_team_words.h), on the CPU.
#include <cstdio>
#include <initializer_list>

#include "hipq_team_words.h"

using namespace hipq;

static int failures = 0;
static void check(bool ok, const char *what, unsigned long long a, unsigned long long b) {
    if (!ok) {
        std::printf("FAIL %s: %llu, %llu\n", what, a, b);
        ++failures;
    }
}

int main() {
    // (the number of a launch is a count of arrivals / 32 and goes round after 2^27)
    for (uint32_t first : {0u, 1u, (1u << 19) - 2, (1u << 20) - 3, (1u << 27) - 4})
        for (uint32_t i = 0; i < 8; ++i) {
            const uint32_t launch = (first + i) % (1u << 27), before = (launch + (1u << 27) - 1) % (1u << 27);
            for (uint32_t xcc : {0u, 15u})
                for (uint32_t left : {0u, 1u, 119u, kTeamPhases - 1})  // where the launch before left the flag
                    check(!team_flag_reached(team_flag(before, left) | xcc, team_flag(launch, 1)), "a flag of the launch before", launch, left);
            for (uint32_t at = 1; at < kTeamPhases; ++at)
                for (uint32_t seen : {at - 1, at, at + 1})
                    if (seen < kTeamPhases)
                        check(team_flag_reached(team_flag(launch, seen) | 7u, team_flag(launch, at)) == (seen >= at), "meetings of a launch", seen, at);
        }
    // Launches that a team does not go through together, one after the other: what the first one finds that it does go through.
    for (uint32_t alone : {1u, 1000u, (1u << 19) - 1, 1u << 19, (1u << 19) + 1, (1u << 20) - 1, 1u << 20, (1u << 20) + 1}) {
        uint32_t flag = team_flag(0, 100);  // launch 0, together
        for (uint32_t launch = 1; launch <= alone; ++launch) flag = team_flag(launch, 0);
        check(!team_flag_reached(flag, team_flag(alone + 1, 1)), "launches of one workgroup before", alone, flag);
    }
    check(team_flag_reached(team_flag(0, 100), team_flag((1u << 19) + 1, 1)), "a flag that nobody refreshed would pass", 0, 0);
    return failures != 0;
}
