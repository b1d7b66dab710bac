// CPU test of the rule by which resident launches of a device run at the same
// time (csrc/vti_res_gate.h), on mocked streams and events driven by a
// discrete-event simulation (test infrastructure; tests/test_res_gate.py builds
// and runs it).
//
// Launches of random sizes come in a random order of streams.  A launch starts
// when its stream's previous one and all it waits for are done, and takes a
// random time.  Checked at every start:
//   - the workgroups of the launches that run, each number a multiple of 8, are
//     no more than the least per_cu among them times the CUs;
// and in all:
//   - every launch runs;
//   - launches of one stream alone wait for nothing;
//   - some run at the same time, in particular every two that fit together and
//     come from two streams with nothing before them.
// `./res_gate open` leaves the waits out and counts the violations (the test
// expects some, so the check can fail).
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#include "vti_res_gate.h"

namespace {

struct Launch {
    int tiles, per_cu, stream;
    double start = -1, end = -1, length;
    std::vector<int> after;
};

struct World {
    std::vector<Launch> l;
    std::vector<int> event;      // event -> launch it was last recorded behind
    std::vector<int> pending;    // waits of the launch being entered
    double now = 0;              // the host's clock
    bool open = false;
    // start and end of every launch so far, in submission order (waits only look back)
    void place(int k)
    {
        Launch &x = l[k];
        x.start = now;
        for (int j = 0; j < k; ++j)
            if (l[j].stream == x.stream) x.start = std::max(x.start, l[j].end);
        for (int j : x.after) x.start = std::max(x.start, l[j].end);
        x.end = x.start + x.length;
    }
} *W;

struct RT {
    using Stream = int;
    using Event = int;
    static bool make(Event *e)
    {
        *e = (int)W->event.size();
        W->event.push_back(-1);
        return true;
    }
    static bool record(Event e, Stream)
    {
        W->event[e] = (int)W->l.size() - 1;
        return true;
    }
    static bool wait(Stream, Event e)
    {
        W->pending.push_back(W->event[e]);
        return true;
    }
    static bool done(Event e) { return W->l[W->event[e]].end <= W->now; }
};

int rounded(const Launch &x) { return (x.tiles + 7) / 8 * 8; }

}  // namespace

int main(int argc, char **argv)
{
    const bool open = argc > 1 && !std::strcmp(argv[1], "open");
    long long violations = 0, together = 0, needless = 0, launches = 0;
    for (int seed = 0; seed < 400; ++seed) {
        std::mt19937 rng(seed);
        World w;
        W = &w;
        vti::ResGate<RT> gate;
        const int cus = seed % 3 ? 256 : 32, streams = 1 + seed % 7;
        for (int k = 0; k < 120; ++k) {
            Launch x;
            x.per_cu = 1 + (int)(rng() % 4);
            const int cap = cus * x.per_cu;
            x.tiles = 1 + (int)(rng() % (rng() % 3 ? std::max(1, cap / 6) : cap));
            x.stream = (int)(rng() % streams);
            x.length = 1 + rng() % 50;
            if (rng() % 4 == 0) w.now += rng() % 60;
            w.pending.clear();
            if (!gate.enter(x.tiles, x.per_cu, cus, x.stream)) return 2;
            if (streams == 1) needless += (long long)w.pending.size();
            if (!open) x.after = w.pending;
            w.l.push_back(x);
            w.place(k);
            if (!gate.leave()) return 2;
            ++launches;
        }
        for (const Launch &x : w.l) {
            int total = 0, least = 99, n = 0;
            for (const Launch &y : w.l)
                if (y.start <= x.start && x.start < y.end) {
                    total += rounded(y);
                    least = std::min(least, y.per_cu);
                    ++n;
                }
            violations += total > least * cus;
            together += n > 1;
            if (x.start < 0 || x.end < x.start) return 2;
        }
    }
    // two that fit together, and two of which one fills the chip
    for (int full = 0; full < 2; ++full) {
        World w;
        W = &w;
        vti::ResGate<RT> gate;
        for (int k = 0; k < 2; ++k) {
            Launch x;
            x.tiles = full && k ? 768 : 304;
            x.per_cu = 3;
            x.stream = k;
            x.length = 10;
            w.pending.clear();
            if (!gate.enter(x.tiles, x.per_cu, 256, x.stream)) return 2;
            x.after = w.pending;
            w.l.push_back(x);
            w.place(k);
            if (!gate.leave()) return 2;
        }
        if (w.l[1].start != (full ? 10 : 0)) ++violations;
    }
    std::printf("launches %lld violations %lld together %lld waits of a single stream %lld\n", launches, violations,
                together, needless);
    return needless || (!open && violations) ? 1 : 0;
}
