// What the device writes into host memory in parts, each followed by an event, and threads that need some of it.  Host code,
// tried on the host.
#pragma once

#include <condition_variable>
#include <cstdint>
#include <exception>
#include <mutex>
#include <utility>
#include <vector>

// Event: synchronize() returns when the work in front of it is done, or throws.  Threads that need what lies before some place wait
// for the part that holds it: one of them for the event, the others asleep until that one has it.  (Region growing waits about 200 us
// for its rows with up to 16 threads, on cores that a data loader may want.  Three rooms of 100000 points take 762 - 776 us, and took
// 741 - 774 with the others asking again and again.)
template <typename Event>
class Arrivals
{
public:
    // All before `end` is there when `event` has happened.  (Every part before the first wait.)
    void part(int64_t end, Event&& event)
    {
        ends_.push_back(end);
        events_.push_back(std::move(event));
    }
    // Waits for all before `end`.  False: a wait failed, here or in another thread (rethrow() has the error).
    bool wait(int64_t end)
    {
        std::unique_lock<std::mutex> lock(state_);
        while (there_ < end)
        {
            if (error_)
                return false;
            if (one_waits_)
            {
                more_.wait(lock);
                continue;
            }
            one_waits_ = true;
            lock.unlock();
            std::exception_ptr error;
            try
            {
                events_.at(next_).synchronize(); // (events_ and next_ are this thread's as long as one_waits_)
            }
            catch (...)
            {
                error = std::current_exception();
            }
            lock.lock();
            one_waits_ = false;
            if (error)
                error_ = error;
            else
                there_ = ends_[next_++];
            lock.unlock(); // (those that wake find it free)
            more_.notify_all();
            lock.lock();
        }
        return true;
    }
    void rethrow()
    {
        if (error_)
            std::rethrow_exception(error_);
    }

private:
    std::vector<Event> events_;
    std::vector<int64_t> ends_;
    size_t next_ = 0;
    int64_t there_ = 0;
    bool one_waits_ = false;
    std::exception_ptr error_;
    std::mutex state_;
    std::condition_variable more_;
};
