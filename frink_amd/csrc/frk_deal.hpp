// How the workgroups of a launch take the entries of a work list so that every XCD has an equal share (plain C++: the
// host side counts with the same functions).
#pragma once

#if defined(__HIPCC__)
#define FRK_HOST_DEVICE __host__ __device__
#else
#define FRK_HOST_DEVICE
#endif

namespace frk {

// Workgroups go to the 8 XCDs in turn (block id mod 8).  Each XCD takes one run of the list, neighbouring entries together
// in its L2, and the runs differ by one entry at most: a list of at most 32 entries an XCD is one round of its CUs.
FRK_HOST_DEVICE inline int deal_grid(int entries) { return (entries + 7) / 8 * 8; }
// the entry of workgroup `block`, or -1 where its XCD's run has ended
FRK_HOST_DEVICE inline int deal_entry(int block, int entries) {
    const int xcd = block & 7, place = block >> 3, each = entries >> 3, rest = entries & 7;
    if (place >= each + (xcd < rest ? 1 : 0)) return -1;
    return xcd * each + (xcd < rest ? xcd : rest) + place;
}

}  // namespace frk
