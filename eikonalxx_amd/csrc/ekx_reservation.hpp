// ekx_reservation.hpp -- waves of flow launches in progress, per device.
#pragma once
#include <chrono>
#include <condition_variable>
#include <cstdint>
#include <deque>
#include <mutex>

namespace ekx
{

// The resident waves of one device, as flow launches of the process's threads
// take them.  Requests are served in the order they come.
class FlowWaves
{
public:
    // n waves out of `capacity`, waiting up to maxWait for others' to be
    // given back; false: not granted.
    bool take(int n, int capacity, std::chrono::duration<double> maxWait)
    {
        std::unique_lock<std::mutex> lock(mutex);
        const uint64_t me = ++last;
        waiting.push_back(me);
        const bool granted = changed.wait_for(lock, maxWait, [&]()
        {
            return waiting.front() == me && n <= capacity - taken;
        });
        for (auto it = waiting.begin(); it != waiting.end(); ++it)
        {
            if (*it == me)
            {
                waiting.erase(it);
                break;
            }
        }
        if (granted) { taken += n; }
        // (the next in line may fit beside, or was held up by this one)
        changed.notify_all();
        return granted;
    }
    void give(int n)
    {
        {
            std::lock_guard<std::mutex> lock(mutex);
            taken -= n;
        }
        changed.notify_all();
    }
    int in_use()
    {
        std::lock_guard<std::mutex> lock(mutex);
        return taken;
    }

private:
    std::mutex mutex;
    std::condition_variable changed;
    std::deque<uint64_t> waiting;
    uint64_t last = 0;
    int taken = 0;
};

// A flow launch needs the waves of a problem resident together, so it takes
// place only if its waves fit beside those of the other flow launches of the
// process (other threads' solvers).
class FlowReservation
{
public:
    FlowReservation() = default;
    FlowReservation(const FlowReservation &) = delete;
    FlowReservation &operator=(const FlowReservation &) = delete;
    ~FlowReservation() { release(); }
    bool take(FlowWaves &from_, int n, int capacity,
              std::chrono::duration<double> maxWait)
    {
        release();
        if (!from_.take(n, capacity, maxWait)) { return false; }
        from = &from_;
        waves = n;
        return true;
    }
    void release()
    {
        if (from) { from->give(waves); }
        from = nullptr;
    }

private:
    FlowWaves *from = nullptr;
    int waves = 0;
};

} // namespace ekx
