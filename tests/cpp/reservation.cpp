// Threads that want parts of a device's waves.  Without waiting: some request
// of every round is granted, and no more than fit at once.  Waiting: every
// request is granted, in the order it came where all want the same.  A wait
// past its end is refused, and holds nobody up.
#include "ekx_reservation.hpp"

#include <atomic>
#include <cstdio>
#include <thread>
#include <vector>

namespace
{
constexpr int kThreads = 3, kCapacity = 100;
const int kWant[kThreads] = {60, 60, 40};
using Seconds = std::chrono::duration<double>;

int rounds_without_waiting()
{
    constexpr int kRounds = 20000;
    ekx::FlowWaves waves;
    std::atomic<int> arrived{0}, granted{0}, refused{0}, overfull{0}, round{0};
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
                if (r.take(waves, kWant[t], kCapacity, Seconds(0)))
                {
                    granted += 1;
                }
                if (waves.in_use() > kCapacity) { overfull += 1; }
                barrier(phase);
                if (t == 0)
                {
                    if (granted == 0) { refused += 1; }
                    granted = 0;
                }
                r.release();
                barrier(phase);
            }
        });
    }
    for (std::thread &t : threads) { t.join(); }
    std::printf("without waiting: rounds refused %d, overfull %d, left %d\n",
                refused.load(), overfull.load(), waves.in_use());
    return refused + overfull + waves.in_use();
}

int all_granted_waiting()
{
    constexpr int kRounds = 3000;
    ekx::FlowWaves waves;
    std::atomic<int> refused{0}, overfull{0};
    std::vector<std::thread> threads;
    for (int t = 0; t < kThreads; ++t)
    {
        threads.emplace_back([&, t]()
        {
            for (int k = 0; k < kRounds; ++k)
            {
                ekx::FlowReservation r;
                if (!r.take(waves, kWant[t], kCapacity, Seconds(60)))
                {
                    refused += 1;
                }
                if (waves.in_use() > kCapacity) { overfull += 1; }
            }
        });
    }
    for (std::thread &t : threads) { t.join(); }
    std::printf("waiting: refused %d, overfull %d, left %d\n", refused.load(),
                overfull.load(), waves.in_use());
    return refused + overfull + waves.in_use();
}

int refused_in_time()
{
    ekx::FlowWaves waves;
    ekx::FlowReservation all;
    int bad = all.take(waves, kCapacity, kCapacity, Seconds(0)) ? 0 : 1;
    // one waits for more than it gets; the small one after it, once the first
    // has given up and the device is free, is granted
    std::atomic<bool> late{true}, after{false};
    const auto t0 = std::chrono::steady_clock::now();
    std::thread a([&]()
    {
        ekx::FlowReservation r;
        late = r.take(waves, kCapacity, kCapacity, Seconds(0.05));
    });
    a.join();
    const Seconds waited = std::chrono::steady_clock::now() - t0;
    std::thread b([&]()
    {
        ekx::FlowReservation r;
        after = r.take(waves, 10, kCapacity, Seconds(60));
    });
    all.release();
    b.join();
    ekx::FlowReservation more;
    bad += late ? 1 : 0;
    bad += after ? 0 : 1;
    bad += waited.count() >= 0.05 && waited.count() < 10 ? 0 : 1;
    // more than the device has is never granted
    bad += more.take(waves, kCapacity + 1, kCapacity, Seconds(0.01)) ? 1 : 0;
    std::printf("refused in time: wrong %d, waited %.3f s, left %d\n", bad,
                waited.count(), waves.in_use());
    return bad + waves.in_use();
}
} // namespace

int main()
{
    return rounds_without_waiting() + all_granted_waiting() +
                   refused_in_time() == 0 ? 0 : 1;
}
