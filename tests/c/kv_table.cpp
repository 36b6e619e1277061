// Plays a page table's uploads through with a device and graphs in memory: sequences grow and start again, directly and in captures, whose
// uploads are repeated at any later time with the host's row as it then is.  After a direct call the device holds every entry of its
// sequence.  Prints the number of direct calls and how many of them uploaded something.
#include <cstdio>
#include <cstdlib>
#include <random>

#include "kv_table.h"

constexpr int kSeqs = 3, kPages = 6;

struct Host {
    std::vector<int32_t> table = std::vector<int32_t>(kSeqs * kPages, -1), device = table, free_pages;
    skn_device_table on_device;
    struct Copy {
        int at, count;
    };
    std::vector<Copy> graph;
    Host() {
        on_device.assign(table.size());
        for (int p = kSeqs * kPages - 1; p >= 0; p--) free_pages.push_back(p);
    }
    void copy(const Copy& c) {
        for (int i = c.at; i < c.at + c.count; i++) device[i] = table[i];
    }
    bool reserve(int seq, int need, bool capture) {  // (true: uploads)
        const int at = seq * kPages;
        for (int p = 0; p < need; p++)
            if (table[at + p] < 0) table[at + p] = free_pages.back(), free_pages.pop_back();
        int first, last;
        if (!on_device.lacks(at, &table[at], need, first, last)) return false;
        const Copy c = {at + first, last - first + 1};
        if (capture) graph.push_back(c);
        else copy(c);
        on_device.uploaded(at, &table[at], first, last, capture);
        return true;
    }
    void release(int seq) {
        for (int p = kPages - 1; p >= 0; p--) {
            int32_t& e = table[seq * kPages + p];
            if (e >= 0) free_pages.push_back(e), on_device.given_back(seq * kPages + p), e = -1;
        }
    }
    void replay() {
        for (const Copy& c : graph) copy(c);
    }
    void check(int seq, int need, const char* what) {
        for (int p = 0; p < need; p++)
            if (device[seq * kPages + p] != table[seq * kPages + p]) {
                std::printf("%s: entry %d of sequence %d is %d, not %d\n", what, p, seq, device[seq * kPages + p], table[seq * kPages + p]);
                std::exit(1);
            }
    }
};

int main() {
    {  // a sequence that is started again gets the pages it had: nothing to upload up to where it ended
        Host h;
        for (int turn = 0; turn < 3; turn++) {
            const int uploads = h.reserve(0, 2, false) + h.reserve(0, 2, false) + h.reserve(0, 4, false);
            if (uploads != (turn == 0 ? 2 : 0)) return std::printf("turn %d: %d uploads\n", turn, uploads), 1;
            h.release(0);
        }
        if (!h.reserve(0, 5, false)) return std::printf("nothing uploaded for a page that was never mapped\n"), 1;
        h.check(0, 5, "one page more");
    }
    {  // the upload of a capture is repeated after the sequence's pages have been given back
        Host h;
        h.reserve(0, 2, true), h.reserve(0, 2, false), h.check(0, 2, "direct after a capture");
        h.release(0), h.replay(), h.reserve(0, 2, false), h.check(0, 2, "mapped again after a replay");
    }
    std::mt19937 rng(7);
    long long calls = 0, uploads = 0;
    for (int round = 0; round < 2000; round++) {
        Host h;
        for (int step = 0; step < 60; step++) {
            const int seq = (int)(rng() % kSeqs), need = 1 + (int)(rng() % kPages), what = (int)(rng() % 10);
            if (what < 5) calls++, uploads += h.reserve(seq, need, false), h.check(seq, need, "direct");
            else if (what < 6) h.reserve(seq, need, true);
            else if (what < 8) h.release(seq);
            else h.replay();
        }
    }
    std::printf("%lld calls, %lld with an upload\n", calls, uploads);
    return uploads < calls ? 0 : 1;
}
