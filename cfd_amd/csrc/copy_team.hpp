// Helper threads of the result copies, and the ring of slots that a copy's pieces pass through. Host
// code only: staging.cpp gives it the device's side.
//
// Made for a machine whose CPUs are all taken: the workers of a BLAS spin for 100 ms after a norm of the
// right-hand side, and a thread that shares a CPU with one of them, or gives its CPU up by sleeping on a
// lock or by a yield, has it back a scheduler's slice (3 to 4 ms) later. So the caller never sleeps or
// yields, and waits for no helper that is not in the middle of a piece; helpers make no device calls (their
// locks would be waited for), a thread takes a piece only once it has arrived, and a helper goes when the
// caller has stopped asking for arrivals. Copies of 16 MiB near such a norm that took over 1.5 ms: 1 of
// 288; with the caller asleep until three helpers had returned, each waiting for pieces of its own, 24 of
// 288 (through the runtime 5 of 288, at twice the time).
#pragma once

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <mutex>
#include <thread>

namespace cfdg {

// Threads that help with a job, asleep between jobs; they come as they wake, and a job is done without
// those that don't, or that the system refused to start. (OpenMP teams instead: a team of another size
// than the last region's is rebuilt, and a call took up to milliseconds longer.) The threads are detached
// and use the object for as long as the process lives: it is never destroyed.
class CopyTeam {
public:
    static constexpr int k_helpers = 3; // beside the caller: seven gain nothing

    struct Job {
        void (*help)(Job&) = nullptr;  // a helper's part; does not throw
        void (*leave)(Job&) = nullptr; // called once when nobody uses the job any more; does not throw

    private:
        friend class CopyTeam;
        Job* next = nullptr;
        int users = 0;
        int wanted = 0;
        bool open = false;
        bool taken[k_helpers] = {};
    };

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

    // Offers the job to `wanted` of the helpers until it is closed.
    void open(Job& job, int wanted) noexcept {
        spin_lock();
        job.users = 0;
        job.wanted = wanted;
        job.open = true;
        for (bool& t : job.taken) {
            t = false;
        }
        job.next = jobs_;
        jobs_ = &job;
        m_.unlock();
        wake_.notify_all();
    }

    // No helper begins the job any more. Its leave() is called when the last one has returned from it,
    // here if none is in it.
    void close(Job& job) noexcept {
        spin_lock();
        Job** at = &jobs_;
        while (*at != &job) {
            at = &(*at)->next;
        }
        *at = job.next;
        job.open = false;
        const bool last = job.users == 0;
        m_.unlock();
        if (last) {
            job.leave(job);
        }
    }

    static void pause() noexcept { __builtin_ia32_pause(); }

private:
    CopyTeam() = default;

    void spin_lock() noexcept { // held for a few instructions only
        while (!m_.try_lock()) {
            pause();
        }
    }

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
                    job = j->taken[k] || k >= j->wanted ? nullptr : j;
                }
                return job != nullptr;
            });
            job->taken[k] = true;
            ++job->users;
            lock.unlock();
            job->help(*job);
            lock.lock();
            if (--job->users == 0 && !job->open) {
                lock.unlock();
                job->leave(*job);
                lock.lock();
            }
        }
    }

    std::mutex m_;
    std::condition_variable wake_;
    Job* jobs_ = nullptr;
    int helpers_ = 0;
};

// Pieces 0 .. count - 1 of a copy through Ring slots, piece i through slot i mod Ring. The caller queues a
// piece on the device as soon as the slot's previous one has been copied out and asks for its arrival;
// whoever is free, the caller among them, copies out the next piece that has arrived. Device (its
// functions don't throw; 0 is success; all but copy_out are called by the caller only): int queue(piece,
// slot), int arrived(slot, bool& yes) for the slot's last queued piece, bool copy_out(piece, slot, part) for the
// part-th part of a piece, true if there are more, void drain() after an error until no queued piece is in flight, void leave() when nobody uses this object any
// more.
template <int Ring, class Device>
class RingCopy : private CopyTeam::Job {
public:
    RingCopy(const Device& device, int count) noexcept : d_(device), count_(count) {
        help = [](CopyTeam::Job& j) { static_cast<RingCopy&>(j).assist(); };
        leave = [](CopyTeam::Job& j) {
            Device d = static_cast<RingCopy&>(j).d_;
            d.leave();
        };
        for (auto& o : out_) {
            o.store(-1);
        }
    }
    RingCopy(const RingCopy&) = delete;
    RingCopy& operator=(const RingCopy&) = delete;

    // The copy, on the caller and `helpers` of the team (which may be null). The first error, or 0. No piece
    // is touched after it returns; the object may be until leave().
    int run(CopyTeam* team, int helpers) noexcept {
        if (team != nullptr) {
            team->open(*this, helpers);
        }
        int error = 0;
        while (error == 0 && copied_.load(std::memory_order_acquire) < count_) {
            error = advance();
            const int i = claim();
            if (i < 0) {
                CopyTeam::pause();
                continue;
            }
            for (int part = 0; d_.copy_out(i, i % Ring, part); ++part) {
                error = error != 0 ? error : advance(); // the device and the helpers don't wait for the piece's end
            }
            finish(i);
        }
        const int claimed = next_.exchange(count_); // after an error: no new pieces, those begun are ended
        while (copied_.load(std::memory_order_acquire) < claimed) {
            CopyTeam::pause();
        }
        if (error != 0) {
            d_.drain();
        }
        if (team != nullptr) {
            team->close(*this);
        } else {
            leave(*this);
        }
        return error;
    }

private:
    int advance() noexcept {
        beat_.store(beat_.load(std::memory_order_relaxed) + 1, std::memory_order_relaxed);
        int e = 0;
        if (queued_ < count_ && (queued_ < Ring || out_[queued_ % Ring].load(std::memory_order_acquire) == queued_ - Ring)) {
            e = d_.queue(queued_, queued_ % Ring);
            queued_ += e == 0 ? 1 : 0;
        }
        int a = arrived_.load(std::memory_order_relaxed);
        for (bool yes = true; e == 0 && yes && a < queued_;) {
            e = d_.arrived(a % Ring, yes);
            if (e == 0 && yes) {
                arrived_.store(++a, std::memory_order_release);
            }
        }
        return e;
    }
    int claim() noexcept { // the next piece that has arrived, or -1
        int i = next_.load(std::memory_order_relaxed);
        do {
            if (i >= arrived_.load(std::memory_order_acquire)) {
                return -1;
            }
        } while (!next_.compare_exchange_weak(i, i + 1));
        return i;
    }
    void finish(int i) noexcept {
        out_[i % Ring].store(i, std::memory_order_release);
        copied_.fetch_add(1, std::memory_order_release);
    }
    // A helper goes when the caller has stopped to ask for pieces: it has lost its CPU, perhaps to the helper.
    void assist() noexcept {
        using clock = std::chrono::steady_clock;
        unsigned seen = beat_.load(std::memory_order_relaxed);
        auto since = clock::now();
        while (next_.load(std::memory_order_relaxed) < count_) {
            const int i = claim();
            if (i >= 0) {
                for (int part = 0; d_.copy_out(i, i % Ring, part); ++part) {
                }
                finish(i);
                since = clock::now();
                continue;
            }
            CopyTeam::pause();
            const unsigned beat = beat_.load(std::memory_order_relaxed);
            const auto now = clock::now();
            if (beat != seen) {
                seen = beat;
                since = now;
            } else if (now - since > k_silent) {
                return;
            }
        }
    }

    static constexpr std::chrono::microseconds k_silent{200}; // it asks every 20 to 60, between the parts of a piece
    Device d_;
    const int count_;
    int queued_ = 0;                    // pieces queued; the caller's
    std::atomic<unsigned> beat_{0};     // the caller's questions for arrivals
    std::atomic<int> arrived_{0};       // pieces that have arrived, in order
    std::atomic<int> next_{0};          // the next piece to be copied out
    std::atomic<int> copied_{0};        // pieces copied out
    std::atomic<int> out_[Ring];        // the piece last copied out of the slot
};

} // namespace cfdg
