// How the blocks of a launch of few segments are dealt to the eight XCDs.  Plain C++, for the kernel and for a host compiler alike.
#pragma once

namespace come {

// Of a list of `items`, each XCD takes a contiguous range, items / 8 long or one longer.  The items that are left over go to the XCDs
// one after another, and the next list goes on where the one before ended (`dealt`: left over in all lists in front), so that the sums
// over all lists differ by one at most.  (With the same XCDs first in every list they add up: 3 segments of 801 keys, 12 heads, have 252 blocks
// of 128 queries, and half of the XCDs would get 33 where 32 fit at a time.)
// of `n` items dealt one after another from XCD 0 on, those of `xcd`
constexpr int dealt_to(int n, int xcd) { return (n + 7 - xcd) >> 3; }

// Items of `xcd` from lists of `items` together, of which those numbered `dealt` to `dealt_after` - 1 were left over.
constexpr int items_to(int items, int dealt, int dealt_after, int xcd) {
    return ((items - (dealt_after - dealt)) >> 3) + dealt_to(dealt_after, xcd) - dealt_to(dealt, xcd);
}

// The range of one list.
struct XcdShare {
    int first, count;
};
constexpr XcdShare share_of(int items, int dealt, int xcd) {
    const int whole = items >> 3, from = dealt & 7, to = from + (items & 7), wrapped = to > 8 ? to - 8 : 0;      // one more: XCDs from .. to - 1, modulo 8
    const int below = (xcd < to ? xcd : to) - (xcd < from ? xcd : from) + (xcd < wrapped ? xcd : wrapped);           // of them in front of `xcd`
    return {xcd * whole + below, items_to(items, dealt, dealt + (items & 7), xcd)};
}

}  // namespace come
