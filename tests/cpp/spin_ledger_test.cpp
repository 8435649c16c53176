// The ledger of reductions in flight with streams and events that the test steps by hand.
#include <cstdio>
#include <utility>
#include <vector>

#include "spin_ledger.hpp"

struct Fake {
    using Stream = int;
    using Event = int;
    static std::vector<int> state;                       // of an event: 0 running, 1 finished, 2 destroyed
    static std::vector<std::pair<Stream, Event>> waits;
    static bool finished(Event e) { return state[e] == 1; }
    static bool running(Event e) { return state[e] == 0; }
    static void wait(Stream s, Event e) { waits.emplace_back(s, e); }
    static Event create() {
        state.push_back(0);
        return (Event)state.size() - 1;
    }
    static void record(Event e, Stream) { state[e] = 0; }
    static void destroy(Event e) { state[e] = 2; }
};
std::vector<int> Fake::state;
std::vector<std::pair<int, int>> Fake::waits;

#define EXPECT(c)                                                     \
    do {                                                              \
        if (!(c)) {                                                   \
            std::printf("line %d: %s\n", __LINE__, #c);               \
            return 1;                                                 \
        }                                                             \
    } while (0)

int main() {
    apw::SpinLedger<Fake> L;
    int at = -2;
    auto go = [&](int x) { at = x; };
    // two contexts on stream 1: the second one's reduction runs when the first one ends
    L.launch(1, 200, false, 256, go);                    // event 0
    L.forget(1);
    EXPECT(L.live.size() == 1 && Fake::state[0] == 0);
    L.launch(2, 200, false, 256, go);                    // event 1: 400 workgroups do not fit together
    EXPECT(Fake::waits.size() == 1 && Fake::waits[0] == std::make_pair(2, 0));
    // the last one ends: finished reductions go, with their events
    Fake::state[0] = 1;
    L.forget(1);
    EXPECT(Fake::state[0] == 2 && L.live.size() == 1);
    Fake::state[1] = 1;
    // one-XCD forms take the least loaded XCD, and wait where none has room
    L.launch(3, 20, true, 256, go);                      // event 1 again
    EXPECT(at == 0 && Fake::waits.size() == 1);
    L.launch(4, 20, true, 256, go);
    EXPECT(at == 1 && Fake::waits.size() == 1);
    for (int s = 5; s <= 10; ++s) L.launch(s, 20, true, 256, go);
    EXPECT(at == 7 && Fake::waits.size() == 1);
    L.launch(11, 20, true, 256, go);                     // the ninth, after the oldest
    EXPECT(at == 0 && Fake::waits.size() == 2 && Fake::waits[1] == std::make_pair(11, 1));
    // a reduction after one of its own stream does not count that one
    apw::SpinLedger<Fake> M;
    M.launch(1, 256, false, 256, go);
    M.launch(1, 256, false, 256, go);
    EXPECT(Fake::waits.size() == 2);
    std::printf("ok\n");
    return 0;
}
