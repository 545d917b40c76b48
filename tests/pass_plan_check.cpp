// Checks pass_plan.hpp: workgroup counts are the ceilings they stand for, and
// a launch fits exactly while its work-items count in 32 bits.  Prints "ok"
// and exits 0.
#include <cstdio>
#include <initializer_list>

#include "pass_plan.hpp"

using namespace fgl;

#define CHECK(x)                                            \
    if (!(x)) {                                             \
        std::printf("line %d: %s\n", __LINE__, #x);         \
        return 1;                                           \
    }

int main()
{
    CHECK(launch_fits((1 << 24) - 1) && !launch_fits(1 << 24));
    CHECK(kMaxBlocks * 256 <= 0xffffffffLL && (kMaxBlocks + 1) * 256 > 0xffffffffLL);
    for (int lanes : {1, 4, 16})
        for (int n : {0, 1, 15, 16, 17, 63, 64, 65, 255, 256, 257, 100001, 0x3fffffff, 0x7fffffff}) {
            const long long per = 256 / lanes, g = direct_groups(n, lanes);
            CHECK(g * per >= n && (g - 1) * per < n);
            const long long v = vertex_blocks(n);
            CHECK(v * 256 >= n && (v - 1) * 256 < n);
        }
    for (long long k : {1LL, 2047LL, 2048LL, 2049LL, 1LL << 28, 1LL << 34}) {
        const long long c = clear_blocks(k);
        CHECK(c * 256 * kClearKeys >= k && (c - 1) * 256 * kClearKeys < k);
    }
    // many small draws beside a large one: what the draws hold, not the
    // number of draws times the largest
    const long long nt = 8192 + 131072;
    const int lanes = 4;
    CHECK(launch_fits(8192 * direct_groups(1, lanes) + direct_groups(131072, lanes)));
    CHECK(!launch_fits(8193 * direct_groups(131072, lanes)));
    // lanes by pixels a face, all of them where triangles are few
    CHECK(direct_lanes(32768, 32768, 1, false) == 16 && direct_lanes(32769, 32769, 1, false) == 1);
    CHECK(direct_lanes(1 << 20, 1000, 24000, false) == 16 && direct_lanes(1 << 20, 1000, 23999, false) == 4);
    CHECK(direct_lanes(1 << 20, 1000, 2500, false) == 4 && direct_lanes(1 << 20, 1000, 2499, false) == 1);
    CHECK(direct_lanes(1 << 20, 1000, 72000, true) == 16 && direct_lanes(1 << 20, 1000, 71998, true) == 4);
    CHECK(direct_lanes(1 << 20, 0, 1, false) == 16);   // a draw of none: no groups whatever its lanes
    CHECK(direct_lanes(0x7fffffff, 0x7fffffff, 1LL << 34, false) == 4);
    CHECK(lanes_slot(1) == 0 && lanes_slot(4) == 1 && lanes_slot(16) == 2);
    // every face of the largest pass, 16 lanes each, does not fit
    CHECK(!launch_fits(direct_groups(0x7fffffff, 16)) && launch_fits(direct_groups(0x7fffffff, 1)));
    // 64 shadow maps of 8192 x 8192 in 64 x 4 blocks do not, 63 do
    CHECK(!launch_fits(64LL * 128 * 2048) && launch_fits(63LL * 128 * 2048));
    std::puts("ok");
    return 0;
}
