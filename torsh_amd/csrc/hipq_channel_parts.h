// How the per-channel quantizer over a middle axis reads its input once (channel_parts_kernel): a group's elements stay in the
// registers of the `parts` workgroups that share it while those agree on its range.  Plain C++, so that the rules can be
// checked without a device.
#pragma once

#include <cstddef>
#include <cstdint>

#if defined(__HIPCC__)
#define HIPQ_HOST_DEVICE __host__ __device__
#else
#define HIPQ_HOST_DEVICE
#endif

namespace hipq {

constexpr int kPartThreads = 256;
constexpr int kPartVec = 16;          // float4 a lane: what four workgroups per compute unit hold
constexpr uint32_t kMostParts = 128;  // 64 x 32 x 12544 49 parts 40.4 -> 32.9 us, 256 x 16 x 6000 94 40.7 -> 34.8, 512 x 16 x 6000 188 72.5 -> 71.4
constexpr int kPartLooks = 1 << 13;   // some twelve milliseconds; a part is microseconds behind

// How often a workgroup looks for the range of a part it shares a group with before it reads the group's range itself.  In full
// until that has happened once: parts are microseconds behind each other, unless other work keeps them from starting, and then
// it does so at the workgroup's next items as well.  After that no longer than the reading takes (a look is a microsecond and
// a half; a workgroup reads a part of 64 KiB in two or three at best), so that it loses the full wait once, not once per item.
struct PartPatience {
    int most;
    bool lost;
    HIPQ_HOST_DEVICE explicit PartPatience(int looks) : most(looks), lost(false) {}
    HIPQ_HOST_DEVICE int looks(uint32_t parts) const {
        const int few = 2 * static_cast<int>(parts);
        return lost && few < most ? few : most;
    }
};

}  // namespace hipq
