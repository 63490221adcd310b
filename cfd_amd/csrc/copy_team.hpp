// Helper threads of the result copies, and the ring of slots that a copy's pieces pass through. Host
// code only: staging.cpp gives it the device's side.
#pragma once

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <mutex>
#include <thread>

namespace cfdg {

// Threads that run work beside a caller, asleep between calls; a call that finds them busy with others
// goes on alone, as does one in a process that was refused the threads. (OpenMP teams instead: a team
// of another size than the last region's is rebuilt, and a call took up to milliseconds longer.) The
// threads are detached and use the object for as long as the process lives: it is never destroyed.
class CopyTeam {
public:
    static constexpr int k_helpers = 3; // beside the caller: seven gain nothing

    // The process's team. Its threads start once the object is complete; those that the system refuses
    // are done without.
    static CopyTeam& get() noexcept {
        alignas(CopyTeam) static unsigned char storage[sizeof(CopyTeam)];
        static CopyTeam* const team = [] {
            auto* t = new (storage) CopyTeam;
            t->start();
            return t;
        }();
        return *team;
    }

    [[nodiscard]] int helpers() const noexcept { return helpers_; }

    // Runs work() on the caller and on the helpers that wake in time; returns when every one of them
    // has returned from it. work() does not throw.
    template <class F>
    void run(F& work) noexcept {
        Job job;
        job.call = [](void* f) noexcept { (*static_cast<F*>(f))(); };
        job.work = &work;
        {
            std::lock_guard<std::mutex> lock(m_);
            job.next = jobs_;
            jobs_ = &job;
        }
        wake_.notify_all();
        work();
        std::unique_lock<std::mutex> lock(m_);
        Job** at = &jobs_;
        while (*at != &job) {
            at = &(*at)->next;
        }
        *at = job.next;
        done_.wait(lock, [&] { return job.users == 0; });
    }

private:
    struct Job { // on the caller's stack while it is listed
        void (*call)(void*) = nullptr;
        void* work = nullptr;
        Job* next = nullptr;
        int users = 0;
        bool taken[k_helpers] = {};
    };

    CopyTeam() = default;

    void start() noexcept {
        for (int k = 0; k < k_helpers; ++k) {
            try {
                std::thread([this, k] { loop(k); }).detach();
            } catch (...) { // a limit on threads or memory
                return;
            }
            ++helpers_;
        }
    }

    void loop(int k) noexcept {
        std::unique_lock<std::mutex> lock(m_);
        for (;;) {
            Job* job = nullptr;
            wake_.wait(lock, [&] {
                for (Job* j = jobs_; j != nullptr && job == nullptr; j = j->next) {
                    job = j->taken[k] ? nullptr : j;
                }
                return job != nullptr;
            });
            job->taken[k] = true;
            ++job->users;
            lock.unlock();
            job->call(job->work);
            lock.lock();
            if (--job->users == 0) {
                done_.notify_all();
            }
        }
    }

    std::mutex m_;
    std::condition_variable wake_;
    std::condition_variable done_;
    Job* jobs_ = nullptr;
    int helpers_ = 0;
};

// Pieces 0 .. count - 1 of a copy through Ring slots, piece i through slot i mod Ring: queued on the
// device as soon as the slot's previous piece has been copied out, then copied out by the thread that
// took it when it has arrived. A thread takes pieces in order, so a piece that another one waits for is
// always already taken. Device (its functions don't throw; 0 is success): int enter() in every thread,
// int queue(piece, slot), int arrived(slot, bool& yes) for the slot's last queued piece,
// void copy_out(piece, slot).
template <int Ring, class Device>
class RingCopy {
public:
    RingCopy(Device& device, int count) noexcept : d_(device), count_(count) {
        for (auto& q : queued_) {
            q.store(-1);
        }
    }

    // Queues the first pieces; the team (or the caller alone) then runs the object. The first error, or 0.
    int run(CopyTeam* team) noexcept {
        for (int i = 0; i < std::min(count_, Ring) && !failed(); ++i) {
            queue(i);
        }
        if (team != nullptr) {
            team->run(*this);
        } else {
            (*this)();
        }
        return error_.load();
    }

    void operator()() noexcept {
        check(d_.enter());
        for (int i = next_.fetch_add(1); i < count_ && !failed(); i = next_.fetch_add(1)) {
            wait(i);
            if (!failed()) {
                d_.copy_out(i, i % Ring);
            }
            if (i + Ring < count_ && !failed()) {
                queue(i + Ring);
            }
        }
    }

private:
    [[nodiscard]] bool failed() const noexcept { return error_.load(std::memory_order_relaxed) != 0; }
    bool check(int e) noexcept {
        int none = 0;
        if (e != 0) {
            error_.compare_exchange_strong(none, e);
        }
        return e == 0;
    }
    void queue(int i) noexcept {
        const int slot = i % Ring;
        check(d_.queue(i, slot));
        queued_[slot].store(i, std::memory_order_release);
    }
    void wait(int i) noexcept { // until piece i, queued by whichever thread, has arrived
        const int slot = i % Ring;
        while (queued_[slot].load(std::memory_order_acquire) < i && !failed()) {
        }
        bool yes = false;
        while (!failed() && check(d_.arrived(slot, yes)) && !yes) {
        }
    }

    Device& d_;
    int count_;
    std::atomic<int> next_{0};
    std::atomic<int> error_{0};
    std::atomic<int> queued_[Ring]; // the piece last queued through the slot
};

} // namespace cfdg
