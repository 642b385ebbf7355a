// The rules of the per-channel quantizer that reads its input once (torsh_amd/csrc/hipq_channel_parts.h), on the CPU.
#include <cstdio>
#include <initializer_list>

#include "hipq_channel_parts.h"

using namespace hipq;

static int failures = 0;
static void check(bool ok, const char *what, long long a, long long b) {
    if (!ok) {
        std::printf("FAIL %s: %lld, %lld\n", what, a, b);
        ++failures;
    }
}

// A workgroup whose partners never start: looks over `items` items, as channel_parts_kernel takes them.
static long long looks_in_vain(int most, uint32_t parts, int items) {
    PartPatience patience(most);
    long long sum = 0;
    for (int i = 0; i < items; ++i) {
        sum += patience.looks(parts) + 1;
        patience.lost = true;
    }
    return sum;
}

static void check_patience() {
    for (uint32_t parts : {2u, 13u, kMostParts}) {
        for (int items : {1, 2, 5, 100}) {
            const long long got = looks_in_vain(kPartLooks, parts, items), most = kPartLooks + 1 + (items - 1) * (2ll * parts + 1);
            check(got <= most, "looks of a workgroup that has given up once", got, most);
        }
        check(PartPatience(kPartLooks).looks(parts) == kPartLooks, "full patience before that", parts, 0);
        check(looks_in_vain(0, parts, 7) == 7, "a limit of 0 is one look an item", parts, 0);
    }
}

// Which views are read once, on a device of 256 compute units: from the shape alone, in scratch that every context has.
static void check_plan() {
    constexpr size_t kResident = 1024, kRoom = (size_t(8) << 20) - 4096;
    struct View {
        size_t outer, channels, inner, group, resident;
        bool once;
    };
    const View views[] = {
        {64, 4, 1024, 1, kResident, true},    {2, 100, 4096, 1, kResident, true},  {64, 256, 3136, 1, kResident, true},
        {500, 30, 300, 1, kResident, true},   {2, 4096, 4096, 1, kResident, true}, {32, 1040, 768, 1, kResident, true},
        {40, 60, 200, 5, kResident, true},    {2, 8000, 3000, 1, kResident, true},
        {40, 61, 200, 5, kResident, false},                                                     // a last group that is shorter
        {40, 60, 124, 1, kResident, false},                                                     // short runs
        {2, 8192, 1024, 1, kResident, false},                                                   // parts that are nearly empty
        {512, 16, 6000, 1, kResident, false},                                                   // more parts than a group may have
        {64, 256, 3136, 1, 8, false},         {64, 4, 1024, 1, 0, false},                       // a small or no share of the device
        {1, 2, size_t(1) << 32, 1, kResident, false},                                           // offsets beyond 32 bits
        {2, 99900, 21504, 1, kResident, true}, {2, 174000, 21504, 1, kResident, true}, {2, 176000, 21504, 1, kResident, false},  // the room
    };
    for (const View &v : views) {
        ChannelPartsPlan p;
        const bool once = plan_channel_parts(v.outer, v.channels, v.inner, v.group, v.resident, kRoom, &p);
        check(once == v.once, "read once", v.channels, v.inner);
        if (!once) continue;
        check(p.words * 8 <= kRoom, "words in scratch that every context has", p.words * 8, kRoom);
        check(p.items == p.parts * (v.channels / v.group) && p.parts <= v.resident, "parts", p.parts, p.items);
        const size_t per_part = (p.vecs + p.parts - 1) / p.parts;
        check(per_part <= size_t(kPartVec) * kPartThreads && (p.parts - 1) * per_part < p.vecs, "every part holds something",
              per_part, p.vecs);
    }
}

int main() {
    check_patience();
    check_plan();
    if (!failures) std::printf("ok\n");
    return failures != 0;
}
