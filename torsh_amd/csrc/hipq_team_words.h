// Numbers by which the workgroups of a team meet (hipq_stack_team.hip).  Plain C++, so that they can be checked without a device.
#pragma once

#include <cstdint>

#if defined(__HIPCC__)
#define HIPQ_TEAM_HD __host__ __device__
#else
#define HIPQ_TEAM_HD
#endif

namespace hipq {

constexpr uint32_t kTeamPhases = 256;  // meetings that a launch may hold

// What a workgroup's flag says once it has come to meeting `meeting` (1, 2, ...) of the team's launch `launch`; the low four bits are
// free to name its XCD.  Numbers go round after 2^20 launches, so flags are compared by their distance, and a flag must not be
// older than that can tell: EVERY launch that a team takes part in leaves its number in all of the team's flags, also one that the team
// does not go through together (meeting 0, where nobody has come to anything).
HIPQ_TEAM_HD constexpr uint32_t team_flag(uint32_t launch, uint32_t meeting) { return (launch * kTeamPhases + meeting) * 16u; }

// Whether a workgroup whose flag is `seen` has come to the meeting that `flag` stands for.
HIPQ_TEAM_HD constexpr bool team_flag_reached(uint32_t seen, uint32_t flag) { return static_cast<int32_t>(seen - flag) >= 0; }

}  // namespace hipq
