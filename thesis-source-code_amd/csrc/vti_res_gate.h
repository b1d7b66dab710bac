// Which resident launches of a device may run at the same time
// (vti2d_res.h), written against a runtime policy so that the same code runs
// on HIP and on a mocked stream / event layer in the CPU tests
// (tests/test_res_gate.py).
//
// The workgroups of a resident launch wait for one another, so all of them have
// to find a place while it runs.  Launches that together could leave one of
// each without a place must not run together: both would wait until their
// bounded waits run out.
//
// Rule: a CU that holds at most k-1 workgroups takes another one when none of
// them needs more than 1/(2k-1) of it (per_cu counts on the same), so launches
// may run together while their workgroups number no more than k on every CU, k
// being the least per_cu among them.  Workgroups go to the 8 XCDs in turn, from
// the first one in every launch, hence each launch counts as a multiple of 8.
//
// A launch goes behind every earlier one of the device that would be too much
// beside it and the ones after that: the newest of the runs not known to be done
// are kept while they and the new one fit, the new launch's stream waits for
// the rest.  In any set of launches that run at once, the newest did not wait for the
// others, so they were all among those it was counted with.  Of a stream's runs only
// one is on the chip at a time, the largest is counted; the launch's own stream's
// earlier ones are done before it.
//
// What it is for: one launch after the other, the calls of a process's several
// contexts wait for each other's passes, which fill a part of the chip where
// the shots are small.  Calls a second of 4 and of 8 threads, each with its own
// context, shots of 340 x 200 points, 401 levels -- on the per-level kernels /
// resident one after the other / by this rule: modelling 1441, 1796 / 1143, 1147 /
// 1504, 2052; RTM 816, 861 / 577, 577 / 1033, 1149; a plan's run 1079, 1058 / 612,
// 607 / 1258, 997.  Shots that fill over half of the chip still take turns: a plan's
// run at 640 x 440 points 552, 560 / 498, 500 / 497, 481.
#pragma once

#include <algorithm>
#include <deque>
#include <mutex>
#include <utility>
#include <vector>

namespace vti {

template <class RT>
class ResGate {
public:
    using Stream = typename RT::Stream;
    using Event = typename RT::Event;

    // Makes s wait for what must be done before `tiles` workgroups, per_cu of
    // which find a place on each of the device's cus for certain, are
    // launched on it.  From here to leave() the caller holds mu.
    std::mutex mu;
    bool enter(int tiles, int per_cu, int cus, Stream s)
    {
        for (size_t k = 0; k < runs_.size();) {
            if (RT::done(runs_[k].ev)) {
                spare_.push_back(runs_[k].ev);
                runs_.erase(runs_.begin() + (long)k);
            } else {
                ++k;
            }
        }
        const int need = (tiles + 7) / 8 * 8;
        next_ = Run{need, per_cu, s, Event{}};
        std::vector<std::pair<Stream, int>> most;  // the largest run of each other stream
        int total = need, least = per_cu;
        size_t k = runs_.size();
        for (; k > 0; --k) {
            const Run &r = runs_[k - 1];
            if (r.s == s) continue;
            auto at = std::find_if(most.begin(), most.end(), [&](const auto &m) { return m.first == r.s; });
            const int more = std::max(0, r.need - (at == most.end() ? 0 : at->second)), k1 = std::min(least, r.per_cu);
            if (total + more > k1 * cus) break;
            total += more;
            least = k1;
            if (at == most.end()) most.emplace_back(r.s, r.need);
            else at->second += more;
        }
        std::vector<Stream> waited;  // (a stream's last run stands for those before it)
        for (; k > 0; --k) {
            const Run &r = runs_[k - 1];
            if (r.s == s || std::find(waited.begin(), waited.end(), r.s) != waited.end()) continue;
            if (!RT::wait(s, r.ev)) return false;
            waited.push_back(r.s);
        }
        return true;
    }
    // after the launch
    bool leave()
    {
        if (spare_.empty()) {
            if (!RT::make(&next_.ev)) return false;
        } else {
            next_.ev = spare_.back();
            spare_.pop_back();
        }
        if (!RT::record(next_.ev, next_.s)) return false;
        runs_.push_back(next_);
        return true;
    }

private:
    struct Run {
        int need, per_cu;
        Stream s;
        Event ev;
    };
    Run next_{};
    std::deque<Run> runs_;       // those not known to be done, oldest first
    std::vector<Event> spare_;
};

}  // namespace vti
