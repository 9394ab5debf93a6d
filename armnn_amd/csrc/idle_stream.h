// A stream without a user, kept for the next one.
#pragma once

#include <mutex>
#include <utility>

namespace mi355x
{

// At most one stream waits here, whichever thread brought it.  A stream belongs to the device that was current when it was
// created, and threads of one process select devices of their own: it is only handed to a thread on that device.
template <typename Stream>
class IdleStream
{
public:
    // The waiting stream if it is `device`'s, else null (another device's stays).
    Stream Take(int device)
    {
        std::lock_guard<std::mutex> lock(m_mutex);
        return m_stream && m_device == device ? std::exchange(m_stream, nullptr) : nullptr;
    }

    // `stream` of `device` waits from now on.  Returns what waited before, the caller's to destroy.
    Stream Put(int device, Stream stream)
    {
        std::lock_guard<std::mutex> lock(m_mutex);
        m_device = device;
        return std::exchange(m_stream, stream);
    }

    // Whatever waits.
    Stream TakeAny()
    {
        std::lock_guard<std::mutex> lock(m_mutex);
        return std::exchange(m_stream, nullptr);
    }

private:
    std::mutex m_mutex;
    Stream m_stream = nullptr;
    int m_device = 0;
};

} // namespace mi355x
