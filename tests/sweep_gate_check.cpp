// Checks of csrc/sweep_gate.hpp, built and run by test_sweep_gate.py.
#include "../multiregionfoam_amd/csrc/sweep_gate.hpp"

#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <thread>

using namespace mrfg;

static void check(bool ok, const char *what)
{
    if (!ok) {
        std::printf("failed: %s\n", what);
        std::exit(1);
    }
}

// whether a further holder of `more` gets in beside `held`, as `expected`
static bool together(int slots, std::vector<int> held, int more, bool expected)
{
    auto *gate = new SweepGate(slots);   // (kept: a waiting thread may outlive this call)
    for (int t : held) gate->acquire(t);
    auto *in = new std::atomic<bool>(false);
    std::thread th([=] {
        gate->acquire(more);
        *in = true;
    });
    for (int k = 0; k < (expected ? 10000 : 100) && !*in; ++k) std::this_thread::sleep_for(std::chrono::milliseconds(2));
    const bool yes = *in;
    if (yes) gate->release(more);
    // everyone gets in once the others are done
    for (int t : held) gate->release(t);
    th.join();
    return yes == expected;
}

int main()
{
    check(together(96, {}, 5000, true), "the first always");
    check(together(96, {5000}, 95, true), "beside a larger one, with a slot left");
    check(together(96, {5000}, 96, false), "no slot left");
    check(together(96, {38, 38}, 38, true), "three of 300 tiles");
    check(together(96, {38, 38, 38}, 38, false), "four of 300 tiles");
    check(together(96, {38, 38}, 5000, true), "a large one beside small ones");
    check(together(96, {48, 48}, 5000, false), "small ones that fill an XCD");
    check(together(96, {5000, 20}, 0, true), "no box tiles");
    // many threads: the rule holds at all times and all get through
    SweepGate gate(96);
    std::mutex m;
    std::vector<int> in;
    std::atomic<bool> ok{true};
    std::vector<std::thread> th;
    for (int k = 0; k < 16; ++k)
        th.emplace_back([&, k] {
            for (int i = 0; i < 200; ++i) {
                const int t = 1 + (k * 37 + i * 13) % 130;
                SweepHold hold(gate, t);
                {
                    std::lock_guard<std::mutex> lk(m);
                    in.push_back(t);
                    int sum = 0, most = 0;
                    for (int x : in) sum += x, most = std::max(most, x);
                    if (sum - most >= 96) ok = false;
                }
                std::this_thread::yield();
                std::lock_guard<std::mutex> lk(m);
                in.erase(std::find(in.begin(), in.end(), t));
            }
        });
    for (auto &t : th) t.join();
    check(ok, "the rule with many threads");
    std::printf("ok\n");
    return 0;
}
