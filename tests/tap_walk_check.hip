// Host-side check of the sparse convs' tap lists (tap_walk.h): for every list
// length, group count and steps per tap, a loader's walk (prepare, then issue
// and prepare again after each step, as sparse_conv_kernel does) may read only
// written list entries, and the groups together walk the list once, in order.
// Prints "ok" and exits 0, or names the first failure.
#include "tap_walk.h"

#include <cstdio>

int main() {
    constexpr int kTaps = 27;
    for (int listed = 0; listed <= kTaps; ++listed)
        for (int groups = 1; groups <= 4; ++groups)
            for (int kc : {1, 2, 4}) {
                int expect = 0;  // next list position the groups should walk
                for (int g = 0; g < groups; ++g) {
                    bfhip::TapWalk walk(listed, groups, g);
                    const int steps = (walk.end - walk.next) * kc;
                    int read = -1;
                    const auto prepare = [&]() {
                        if (!walk.starts_tap()) return true;
                        read = walk.next;
                        return read >= 0 && read < listed;
                    };
                    bool ok = steps >= 0 && prepare();
                    for (int k = 0; ok && k < steps; ++k) {
                        ok = read == expect + k / kc;
                        walk.step(kc);
                        ok = ok && prepare();
                    }
                    if (!ok) {
                        std::printf("list of %d, group %d of %d, %d steps a tap: reads position %d\n", listed, g,
                                    groups, kc, read);
                        return 1;
                    }
                    expect += steps / kc;
                }
                if (expect != listed) {
                    std::printf("list of %d, %d groups: %d walked\n", listed, groups, expect);
                    return 1;
                }
            }
    std::printf("ok\n");
    return 0;
}
