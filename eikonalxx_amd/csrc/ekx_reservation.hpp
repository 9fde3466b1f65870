// ekx_reservation.hpp -- waves of flow launches in progress, per device.
#pragma once
#include <atomic>

namespace ekx
{

// A flow launch needs the waves of a problem resident together, so it takes
// place only if its waves fit beside those of the other flow launches of the
// process (other threads' solvers); otherwise the solve uses the launches
// per diagonal.
class FlowReservation
{
public:
    FlowReservation() = default;
    FlowReservation(const FlowReservation &) = delete;
    FlowReservation &operator=(const FlowReservation &) = delete;
    ~FlowReservation() { release(); }
    // n waves out of `capacity`, of which `taken` are in use.  Refused only
    // if they do not fit: nothing is added before it is known to.
    bool take(std::atomic<int> &taken, int n, int capacity)
    {
        release();
        int now = taken.load();
        do
        {
            if (n > capacity - now) { return false; }
        } while (!taken.compare_exchange_weak(now, now + n));
        from = &taken;
        waves = n;
        return true;
    }
    void release()
    {
        if (from) { from->fetch_sub(waves); }
        from = nullptr;
    }

private:
    std::atomic<int> *from = nullptr;
    int waves = 0;
};

} // namespace ekx
