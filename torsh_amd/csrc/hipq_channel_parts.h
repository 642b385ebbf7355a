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

struct ChannelPartsPlan {
    size_t run, vecs;     // floats of a group's run in a row; float4s of a group
    size_t parts, items;  // workgroups that share a group; parts of all groups
    size_t words;         // 64-bit words through which the parts of a group agree
};

// Whether a dense [outer, channels, inner] view with groups of `group` channels, its rows a whole number of aligned float4s, is read
// once, from its shape alone.  `resident`: workgroups that run at once.  `room`: bytes of scratch for the words that every
// context has from its creation on, so that neither the choice nor a call under capture depends on what the context did before.
//
// Read once where the device's registers hold the tensor at once, or where runs are long enough that parts share few lines and
// the parts fill a third of the registers.  us, two passes / once: [500,30,300] 31.0 / 14.2, [64,40,1000] 21.6 / 14.2,
// [100,1000,128] 21.5 / 16.6; several rounds: [2,4096,4096] 58.9 / 37.8, [32,2048,768] 75.8 / 60.0, [2,8000,3000] (0.37 of the
// registers) 84 / 70, [4,8192,1024] (0.25) 54.4 / 55.2, [2,8192,1024] (0.12) 34.8 / 44.0, [128,1024,196] 39.4 / 40.8,
// [8,8192,400] 42 / 61.  Few parts too, where two passes have eight workgroups per compute unit: [64,4,1024] (16 parts) 10.4 / 9.0,
// [2,2,65536] (16) 11.0 / 9.0, [8,64,512] (64) 8.8 / 6.3, [2,100,4096] (100) 9.7 / 7.0.
inline bool plan_channel_parts(size_t outer, size_t channels, size_t inner, size_t group, size_t resident, size_t room,
                               ChannelPartsPlan *p) {
    constexpr size_t kPartVecs = size_t(kPartVec) * kPartThreads;
    if (channels % group != 0) return false;
    p->run = group * inner;
    p->vecs = outer * p->run / 4;
    p->parts = (p->vecs + kPartVecs - 1) / kPartVecs;
    p->items = p->parts * (channels / group);
    p->words = p->parts > 1 ? 2 * p->items : 0;
    if (p->run < 128 || p->parts > kMostParts || p->parts > resident || outer * channels * inner / 4 >= size_t(1) << 31) return false;
    if (p->words * sizeof(uint64_t) > room) return false;
    return p->items <= resident || (p->run >= 512 && p->vecs >= p->parts * (kPartVecs * 5 / 16));
}

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
