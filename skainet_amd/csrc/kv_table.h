// What a device's copy of a page table holds, entry by entry (plain C++, so that a host program can play it through).
#pragma once
#include <cstddef>
#include <cstdint>
#include <vector>

struct skn_device_table {
    std::vector<int32_t> held;      // what the device holds; kUnknown: anything
    std::vector<uint8_t> recorded;  // an upload of the entry is part of a graph, and every launch of that repeats it
    static constexpr int32_t kUnknown = -2;

    void assign(size_t entries) { held.assign(entries, -1), recorded.assign(entries, 0); }

    // First and last of the `need` entries from `at` on that the device lacks of row[0 .. need - 1]; false: none.
    bool lacks(size_t at, const int32_t* row, int need, int& first, int& last) const {
        first = 0, last = need - 1;
        while (first < need && held[at + first] == row[first]) first++;
        while (last > first && held[at + last] == row[last]) last--;
        return first < need;
    }

    // Entries first .. last have been uploaded from `row` -- or, in a capture, will be whenever the graph is launched, if ever.
    void uploaded(size_t at, const int32_t* row, int first, int last, bool capture) {
        for (int p = first; p <= last; p++) {
            held[at + p] = capture ? kUnknown : row[p];
            if (capture) recorded[at + p] = 1;
        }
    }

    // The entry's page is given back: the device keeps what it holds, but for an entry that a graph uploads, which a launch from now on may
    // write over with the host's row as it then is.
    void given_back(size_t entry) {
        if (recorded[entry]) held[entry] = kUnknown;
    }
};
