// A tap group's walk over its row block's list of active taps (lidar.hip).
// The list holds `listed` taps; entries past them are unwritten, or left over
// from an earlier row block, so a position is read only where starts_tap()
// says that a tap begins there (tests/tap_walk_check.hip walks every list
// length, group and step count on the host).
#pragma once

#include <hip/hip_runtime.h>

namespace bfhip {

struct TapWalk {
    int next, end;  // list positions of this group still to walk
    int c = 0;      // 32-channel step within the tap at `next`

    __host__ __device__ TapWalk(int listed, int groups, int group) {
        const int per = (listed + groups - 1) / groups;
        next = listed < group * per ? listed : group * per;
        end = listed < next + per ? listed : next + per;
    }
    __host__ __device__ bool starts_tap() const { return c == 0 && next < end; }
    __host__ __device__ void step(int steps_per_tap) {
        if (++c == steps_per_tap) {
            c = 0;
            ++next;
        }
    }
};

}  // namespace bfhip
