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

int main() {
    check_patience();
    if (!failures) std::printf("ok\n");
    return failures != 0;
}
