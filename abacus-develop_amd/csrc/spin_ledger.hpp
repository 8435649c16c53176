// Which reductions may run at the same time (host code; Api: the stream and event calls).
#pragma once

#include <algorithm>
#include <deque>
#include <mutex>
#include <vector>

namespace apw {

// Launches of the multi-workgroup reductions, whose workgroups wait on each other's ring values,
// may run at the same time on several streams only while all their workgroups fit on the GPU
// together (each workgroup fits one CU): then none can wait on a workgroup that cannot start, and
// ordinary kernels beside them always finish and free their CUs.  A device-wide ledger keeps the
// reductions not known to have finished, in launch order, with the CUs they need on each XCD: a
// device-wide form an eighth of its workgroups on every XCD, a one-XCD form all of its workgroups
// on one, the least loaded.  A new one that would not fit first makes its stream wait for the
// oldest of the other streams' (its own stream's are over before it starts), as many as needed.
// Every set of reductions that can run together then fits: a later one overlaps an earlier one
// only if it did not wait for it, and then the earlier one was counted.
//
// Api has the types Stream and Event and the static functions finished(Event), running(Event) (an
// event that cannot be asked is neither), wait(Stream, Event), create(), record(Event, Stream) and
// destroy(Event).
template <class Api>
struct SpinLedger {
    using Stream = typename Api::Stream;
    using Event = typename Api::Event;
    static constexpr int NXCD = 8;
    struct Entry {
        Event ev;      // completion
        Stream s;
        int w, xcd;    // workgroups; the XCD they run on, or -1: all
    };
    std::mutex m;
    std::deque<Entry> live;
    std::vector<Entry> pool;   // finished

    // go(at) launches a reduction of w workgroups on s: xcd: all of them on XCD at; else (at = 0) an
    // eighth of them on every XCD.  m is held.
    template <class F>
    void launch(Stream s, int w, bool xcd, int num_cu, F&& go) {
        while (!live.empty() && Api::finished(live.front().ev)) {
            pool.push_back(live.front());
            live.pop_front();
        }
        // load[x]: eighths of CUs, a device-wide width rounded up to the same share of every XCD
        int load[NXCD] = {};
        auto add = [&](const Entry& g, int sign) {
            for (int x = 0; x < NXCD; ++x)
                if (g.xcd < 0 || g.xcd == x) load[x] += sign * (g.xcd < 0 ? (g.w + NXCD - 1) / NXCD * NXCD : NXCD * g.w);
        };
        for (const auto& g : live)
            if (g.s != s) add(g, 1);
        auto place = [&]() {   // the XCD to run on (0 for a device-wide form), -1 if it does not fit yet
            if (xcd) {
                const int x = (int)(std::min_element(load, load + NXCD) - load);
                return load[x] + NXCD * w <= num_cu ? x : -1;
            }
            return *std::max_element(load, load + NXCD) + (w + NXCD - 1) / NXCD * NXCD <= num_cu ? 0 : -1;
        };
        int at = place();
        for (auto it = live.begin(); at < 0 && it != live.end(); ++it) {
            if (it->s == s) continue;
            Api::wait(s, it->ev);
            add(*it, -1);
            at = place();
        }
        go(at);
        Event ev;
        if (!pool.empty()) {
            ev = pool.back().ev;
            pool.pop_back();
        } else {
            ev = Api::create();
        }
        Api::record(ev, s);
        live.push_back(Entry{ev, s, w, xcd ? at : -1});
    }

    // A context on s ends; s has been synchronised and may be destroyed next.  An event may outlive
    // the stream it was last recorded on, but not be queried then: a query that looked at a freed
    // stream has failed as if that stream were being captured.  What still runs was queued after
    // the synchronisation by another context on the same stream and stays until that one ends.
    // m is held.
    void forget(Stream s) {
        auto drop = [&](auto& list) {
            for (auto it = list.begin(); it != list.end();) {
                if (it->s == s && !Api::running(it->ev)) {
                    Api::destroy(it->ev);
                    it = list.erase(it);
                } else {
                    ++it;
                }
            }
        };
        drop(live);
        drop(pool);
    }
};

}  // namespace apw
