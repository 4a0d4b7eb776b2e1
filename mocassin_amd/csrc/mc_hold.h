// mc_hold.h - a lock on memory that kernels of a stream work in.
#pragma once
#include <mutex>

namespace mcl {

// Taken without waiting.  It is let go when the stream is done with the
// memory, also where a call in between fails and the caller returns: `wait`
// (which waits for the stream) runs before the mutex is free again if work
// has begun and not been seen to end.
template <class Wait>
class Hold {
public:
    explicit Hold(Wait wait) : wait_(wait) {}
    Hold(const Hold &) = delete;
    Hold &operator=(const Hold &) = delete;
    ~Hold() { drop(); }
    bool take(std::mutex &m)
    {
        lock_ = std::unique_lock<std::mutex>(m, std::try_to_lock);
        return lock_.owns_lock();
    }
    void drop()
    {
        if (busy_) wait_();
        busy_ = false;
        if (lock_.owns_lock()) lock_.unlock();
    }
    void began() { busy_ = true; }
    void ended() { busy_ = false; }

private:
    std::unique_lock<std::mutex> lock_;
    Wait wait_;
    bool busy_ = false;
};

}  // namespace mcl
