// What the device writes into host memory in parts, each followed by an event, and threads that need some of it.  Host code,
// tried on the host.
#pragma once

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdint>
#include <exception>
#include <mutex>
#include <thread>
#include <utility>
#include <vector>

// Event: synchronize() returns when the work in front of it is done, or throws.  Threads that need what lies before some place wait
// for the part that holds it: one of them for the event, the others for that one - awake for a millisecond, which is what the rows of
// region growing mostly take, then asleep, since the stream may have other work in front and their cores other users.
// (400000 points of four pieces: 1770 us, and 2300 where they sleep at once: a core that was asleep wakes late and walks slowly.)
template <typename Event>
class Arrivals
{
public:
    static constexpr std::chrono::microseconds AWAKE{1000};

    // All before `end` is there when `event` has happened.  (Every part before the first wait.)
    void part(int64_t end, Event&& event)
    {
        ends_.push_back(end);
        events_.push_back(std::move(event));
    }
    // Waits for all before `end`.  False: a wait failed, here or in another thread (rethrow() has the error).
    bool wait(int64_t end)
    {
        const auto awake_until = std::chrono::steady_clock::now() + AWAKE;
        while (there_.load(std::memory_order_acquire) < end)
        {
            if (failed_.load(std::memory_order_acquire))
                return false;
            if (!one_waits_.exchange(true, std::memory_order_acquire))
            {
                wait_for_next(end);
                one_waits_.store(false, std::memory_order_release);
                {
                    std::lock_guard<std::mutex> lock(state_); // (a thread about to sleep has looked before, or sees it now)
                }
                more_.notify_all();
            }
            else if (std::chrono::steady_clock::now() < awake_until)
                std::this_thread::yield();
            else
            {
                std::unique_lock<std::mutex> lock(state_);
                more_.wait(lock, [&] {
                    return there_.load(std::memory_order_acquire) >= end || failed_.load(std::memory_order_acquire) ||
                           !one_waits_.load(std::memory_order_acquire);
                });
            }
        }
        return true;
    }
    void rethrow()
    {
        if (error_)
            std::rethrow_exception(error_);
    }

private:
    // (events_ and next_ are the thread's that has set one_waits_)
    void wait_for_next(int64_t end)
    {
        if (there_.load(std::memory_order_relaxed) >= end || failed_.load(std::memory_order_relaxed))
            return;
        try
        {
            events_.at(next_).synchronize();
            there_.store(ends_[next_++], std::memory_order_release);
        }
        catch (...)
        {
            error_ = std::current_exception();
            failed_.store(true, std::memory_order_release);
        }
    }

    std::vector<Event> events_;
    std::vector<int64_t> ends_;
    size_t next_ = 0;
    std::atomic<int64_t> there_{0};
    std::atomic<bool> one_waits_{false}, failed_{false};
    std::exception_ptr error_;
    std::mutex state_;
    std::condition_variable more_;
};
