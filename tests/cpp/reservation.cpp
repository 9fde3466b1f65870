// Threads that each want 3/5 of the device, or 2/5, round after round: some
// request of every round is granted, and no more than fit at once.
#include "ekx_reservation.hpp"

#include <atomic>
#include <cstdio>
#include <thread>
#include <vector>

int main()
{
    constexpr int kThreads = 3, kRounds = 100000, kCapacity = 100;
    const int want[kThreads] = {60, 60, 40};
    std::atomic<int> taken{0}, arrived{0}, granted{0}, refusedRounds{0},
        overfull{0};
    std::atomic<int> round{0};
    auto barrier = [&](int &phase)
    {
        ++phase;
        if (arrived.fetch_add(1) + 1 == kThreads)
        {
            arrived = 0;
            round = phase;
        }
        else { while (round < phase) { std::this_thread::yield(); } }
    };
    std::vector<std::thread> threads;
    for (int t = 0; t < kThreads; ++t)
    {
        threads.emplace_back([&, t]()
        {
            int phase = 0;
            for (int k = 0; k < kRounds; ++k)
            {
                ekx::FlowReservation r;
                if (r.take(taken, want[t], kCapacity)) { granted += 1; }
                if (taken > kCapacity) { overfull += 1; }
                barrier(phase);
                if (t == 0)
                {
                    if (granted == 0) { refusedRounds += 1; }
                    granted = 0;
                }
                r.release();
                barrier(phase);
            }
        });
    }
    for (std::thread &t : threads) { t.join(); }
    std::printf("rounds refused %d, overfull %d, left %d\n",
                refusedRounds.load(), overfull.load(), taken.load());
    return refusedRounds == 0 && overfull == 0 && taken == 0 ? 0 : 1;
}
