// ekx_reads.hpp -- the stream that large fields are read back on.
#pragma once
#include <hip/hip_runtime.h>

#include <mutex>

namespace ekx
{

// Reads up to this size share the stream of the work: they go through the
// runtime's own buffers.
constexpr size_t kSmallRead = (size_t) 1 << 20;

// The stream of larger reads, one for every device and, like the default
// stream, for all handles and threads and the life of the process; null if it
// cannot be made.  On the default stream a read fails while another thread's
// solver captures its graph.  On the stream of the work the next upload pays
// for it: the runtime lets go of the host pages of a stream's last copy with
// the next one (a new solver's set_slowness after the first read of a 257 x
// 257 x 193 field: 19 ms, 8 so).  A stream for every handle costs as much
// when it is made and destroyed (129^3: 0.7 ms at the first read, 1.9 at the
// end).
inline hipStream_t read_stream()
{
    constexpr int kDevices = 64;
    static std::mutex mutex;
    static hipStream_t streams[kDevices] = {};
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess || device < 0 ||
        device >= kDevices)
    {
        return nullptr;
    }
    std::lock_guard<std::mutex> lock(mutex);
    hipStream_t &s = streams[device];
    if (!s && hipStreamCreateWithFlags(&s, hipStreamNonBlocking) != hipSuccess)
    {
        s = nullptr;
        (void) hipGetLastError();
    }
    return s;
}

// Device to host after the work on `work`, done when it returns.
inline hipError_t read_back(void *dst, const void *src, size_t bytes,
                            hipStream_t work)
{
    hipStream_t s = bytes > kSmallRead ? read_stream() : work;
    if (!s) { s = work; }
    if (s != work)
    {
        const hipError_t e = hipStreamSynchronize(work);
        if (e != hipSuccess) { return e; }
    }
    const hipError_t e = hipMemcpyAsync(dst, src, bytes,
                                        hipMemcpyDeviceToHost, s);
    return e == hipSuccess ? hipStreamSynchronize(s) : e;
}

} // namespace ekx
