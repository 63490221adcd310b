// Large host <-> device copies through pinned staging memory. A copy from or to pageable memory
// runs at a fraction of the PCIe rate; here the pageable side is copied by the host threads into
// (or out of) pinned chunks while the DMA engine moves the previous chunk. Staging areas come
// from a process-wide free list (one per concurrent caller, kept until the process ends).
//
// The results of solves and finite-volume calls (d2h_copies) take a finer pipeline with threads of
// its own. The set-up's copies keep the OpenMP team that runs the loops around them: more threads
// beside its spinning workers exceed a CPU quota of the team's size, and the process is stopped for
// the rest of the scheduler's period (set-up 4% slower, the first solve after it up to 5 ms).
#include "hip_util.hpp"

#include <omp.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>

namespace cfdg {

namespace {

// The host threads of the library's OpenMP regions (LLVM libomp) sleep 1 ms after a region
// instead of the runtime's default 200 ms of spinning, unless the process set KMP_BLOCKTIME or
// OMP_WAIT_POLICY itself. With a CPU quota equal to the worker count (a cgroup cpu.max of 16
// CPUs for 16 threads) the spinning workers and the thread that polls the GPU exceed the quota
// after every host-side setup, the process is throttled for the rest of the scheduler period, and
// solves queued meanwhile stall for milliseconds between two kernels. Runs when the library is
// loaded: kmp_set_blocktime covers the loading thread, kmp_set_defaults threads that start
// OpenMP regions later.
__attribute__((constructor)) void short_omp_blocktime() {
    if (std::getenv("KMP_BLOCKTIME") != nullptr || std::getenv("OMP_WAIT_POLICY") != nullptr) {
        return;
    }
    kmp_set_defaults("KMP_BLOCKTIME=1");
    kmp_set_blocktime(1);
}

constexpr std::size_t k_chunk = std::size_t(16) << 20; // bytes per chunk; two chunks per area

constexpr std::size_t k_slot = std::size_t(4) << 20; // d2h_copies' share of a chunk
constexpr int k_slots_per_chunk = static_cast<int>(k_chunk / k_slot);
constexpr int k_ring = 2 * k_slots_per_chunk;        // its slots per area
constexpr int k_helpers = 3;                         // its threads beside the caller: seven gain nothing

// Bytes per piece of d2h_copies: small enough that a copy's first and last pieces, which nothing
// overlaps, are a small part of it, large enough for the 10 us that each costs. Measured with 1, 2
// and 4 MiB (us): 4 MiB 221, 201, 259; 17 MiB 642, 555, 565 (1025 through the runtime, whose one
// thread copies while the link waits); 64 MiB 2610, 2640, 2336 (6773).
constexpr std::size_t piece_bytes(std::size_t total) {
    return total > (std::size_t(32) << 20) ? k_slot : std::size_t(2) << 20;
}

struct Area {
    char* buf[2] = {nullptr, nullptr};
    hipEvent_t done[2] = {nullptr, nullptr};
    hipEvent_t slot_done[k_ring] = {};
    int device = -1;
    [[nodiscard]] char* slot(int i) const {
        return buf[i / k_slots_per_chunk] + static_cast<std::size_t>(i % k_slots_per_chunk) * k_slot;
    }
};

thread_local bool t_host_parallel = true;

std::mutex g_mutex;
std::vector<Area*> g_free;

Area* acquire(int device) {
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        for (std::size_t i = 0; i < g_free.size(); ++i) {
            if (g_free[i]->device == device) {
                Area* a = g_free[i];
                g_free.erase(g_free.begin() + static_cast<std::ptrdiff_t>(i));
                return a;
            }
        }
    }
    auto* a = new Area;
    a->device = device;
    for (int k = 0; k < 2; ++k) {
        hip_check(hipHostMalloc(reinterpret_cast<void**>(&a->buf[k]), k_chunk, hipHostMallocDefault),
                  "hipHostMalloc staging");
        hip_check(hipEventCreateWithFlags(&a->done[k], hipEventDisableTiming), "staging event");
    }
    for (hipEvent_t& e : a->slot_done) {
        hip_check(hipEventCreateWithFlags(&e, hipEventDisableTiming), "staging event");
    }
    return a;
}

void release(Area* a) {
    std::lock_guard<std::mutex> lock(g_mutex);
    g_free.push_back(a);
}

// Host memcpy split over the host threads for large blocks.
void host_copy(char* dst, const char* src, std::size_t n) {
    constexpr std::size_t piece = std::size_t(1) << 20;
    const long long pieces = static_cast<long long>((n + piece - 1) / piece);
    if (pieces <= 1 || !t_host_parallel) {
        std::memcpy(dst, src, n);
        return;
    }
#pragma omp parallel for schedule(static)
    for (long long i = 0; i < pieces; ++i) {
        const std::size_t o = static_cast<std::size_t>(i) * piece;
        std::memcpy(dst + o, src + o, n - o < piece ? n - o : piece);
    }
}

// Helper threads of the copies, started with the first one and asleep between copies; a copy that
// finds them busy with others goes on alone. (OpenMP teams instead: a team of another size than the
// last region's is rebuilt, and a call took up to milliseconds longer.) Never destroyed: the threads
// may outlive static objects.
class Helpers {
public:
    static Helpers& get() {
        static Helpers* h = new Helpers;
        return *h;
    }
    // Runs work() on the caller and on the helpers that wake in time; returns when every one of them
    // has returned from it.
    void run(const std::function<void()>& work) {
        Job job{&work, 0};
        {
            std::lock_guard<std::mutex> lock(m_);
            jobs_.push_back(&job);
        }
        wake_.notify_all();
        work();
        std::unique_lock<std::mutex> lock(m_);
        jobs_.erase(std::find(jobs_.begin(), jobs_.end(), &job));
        done_.wait(lock, [&] { return job.users == 0; });
    }

private:
    struct Job {
        const std::function<void()>* work;
        int users;
        bool taken[k_helpers] = {};
    };
    Helpers() {
        for (int k = 0; k < k_helpers; ++k) {
            std::thread([this, k] { loop(k); }).detach();
        }
    }
    void loop(int k) {
        std::unique_lock<std::mutex> lock(m_);
        for (;;) {
            Job* job = nullptr;
            wake_.wait(lock, [&] {
                for (Job* j : jobs_) {
                    if (!j->taken[k]) {
                        job = j;
                        return true;
                    }
                }
                return false;
            });
            job->taken[k] = true;
            ++job->users;
            lock.unlock();
            (*job->work)();
            lock.lock();
            if (--job->users == 0) {
                done_.notify_all();
            }
        }
    }
    std::mutex m_;
    std::condition_variable wake_;
    std::condition_variable done_;
    std::vector<Job*> jobs_;
};

} // namespace

bool host_parallel() { return t_host_parallel; }

void set_host_parallel(bool on) { t_host_parallel = on; }

void parallel_copy(void* dst, const void* src, std::size_t bytes) {
    host_copy(static_cast<char*>(dst), static_cast<const char*>(src), bytes);
}

void h2d_staged(void* dst, const void* src, std::size_t bytes, hipStream_t s) {
    if (bytes < k_staged_min_bytes) {
        if (bytes > 0) {
            hip_check(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s), "H2D copy");
            hip_check(hipStreamSynchronize(s), "H2D copy sync");
        }
        return;
    }
    int device = 0;
    hip_check(hipGetDevice(&device), "hipGetDevice");
    Area* a = acquire(device);
    try {
        const char* in = static_cast<const char*>(src);
        char* out = static_cast<char*>(dst);
        bool used[2] = {false, false};
        int k = 0;
        for (std::size_t o = 0; o < bytes; o += k_chunk, k ^= 1) {
            const std::size_t n = bytes - o < k_chunk ? bytes - o : k_chunk;
            if (used[k]) { // the chunk's previous DMA must be done before it is refilled
                hip_check(hipEventSynchronize(a->done[k]), "staging wait");
            }
            host_copy(a->buf[k], in + o, n);
            hip_check(hipMemcpyAsync(out + o, a->buf[k], n, hipMemcpyHostToDevice, s), "staged H2D");
            hip_check(hipEventRecord(a->done[k], s), "staging record");
            used[k] = true;
        }
        hip_check(hipStreamSynchronize(s), "staged H2D sync");
    } catch (...) {
        (void)hipStreamSynchronize(s);
        release(a);
        throw;
    }
    release(a);
}

void d2h_staged(void* dst, const void* src, std::size_t bytes, hipStream_t s) {
    if (bytes < k_staged_min_bytes) {
        if (bytes > 0) {
            hip_check(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s), "D2H copy");
            hip_check(hipStreamSynchronize(s), "D2H copy sync");
        }
        return;
    }
    int device = 0;
    hip_check(hipGetDevice(&device), "hipGetDevice");
    Area* a = acquire(device);
    try {
        const char* in = static_cast<const char*>(src);
        char* out = static_cast<char*>(dst);
        // chunk i goes to buffer i % 2; it is copied out on the host while chunk i + 1 moves
        std::size_t prev_o = 0;
        std::size_t prev_n = 0;
        int k = 0;
        for (std::size_t o = 0; o < bytes; o += k_chunk, k ^= 1) {
            const std::size_t n = bytes - o < k_chunk ? bytes - o : k_chunk;
            hip_check(hipMemcpyAsync(a->buf[k], in + o, n, hipMemcpyDeviceToHost, s), "staged D2H");
            hip_check(hipEventRecord(a->done[k], s), "staging record");
            if (prev_n > 0) {
                hip_check(hipEventSynchronize(a->done[k ^ 1]), "staging wait");
                host_copy(out + prev_o, a->buf[k ^ 1], prev_n);
            }
            prev_o = o;
            prev_n = n;
        }
        if (prev_n > 0) {
            hip_check(hipEventSynchronize(a->done[k ^ 1]), "staging wait");
            host_copy(out + prev_o, a->buf[k ^ 1], prev_n);
        }
    } catch (...) {
        (void)hipStreamSynchronize(s);
        release(a);
        throw;
    }
    release(a);
}

namespace {

// Copies the pieces of a list from the device through the ring of one area, piece i through slot
// i mod k_ring: queued on s as soon as the slot's previous piece has been copied out, then copied out
// by the thread that took it when it has arrived. A thread takes pieces in order, so a piece that
// another one waits for is always already taken; queued[slot] is the number of the piece that was
// last queued through the slot.
hipError_t copy_pieces(const HostCopy* list, int n, Area& a, hipStream_t s, std::size_t piece) {
    struct Piece {
        const char* dev;
        char* host;
        std::size_t bytes;
    };
    std::vector<Piece> pieces;
    for (int k = 0; k < n; ++k) {
        for (std::size_t o = 0; o < list[k].bytes; o += piece) {
            pieces.push_back({static_cast<const char*>(list[k].dev) + o, static_cast<char*>(list[k].host) + o,
                              std::min(piece, list[k].bytes - o)});
        }
    }
    const int count = static_cast<int>(pieces.size());
    std::atomic<int> next{0};
    std::atomic<int> error{static_cast<int>(hipSuccess)};
    std::atomic<int> queued[k_ring];
    for (auto& q : queued) {
        q.store(-1);
    }
    auto failed = [&] { return error.load(std::memory_order_relaxed) != static_cast<int>(hipSuccess); };
    auto check = [&](hipError_t e) {
        if (e != hipSuccess) {
            error.store(static_cast<int>(e));
        }
        return e == hipSuccess;
    };
    auto queue = [&](int i) {
        const Piece& p = pieces[static_cast<std::size_t>(i)];
        const int slot = i % k_ring;
        (void)(check(hipMemcpyAsync(a.slot(slot), p.dev, p.bytes, hipMemcpyDeviceToHost, s)) &&
               check(hipEventRecord(a.slot_done[slot], s)));
        queued[slot].store(i, std::memory_order_release);
    };
    auto wait = [&](int i) { // until piece i, queued by whichever thread, has arrived
        const int slot = i % k_ring;
        while (queued[slot].load(std::memory_order_acquire) < i && !failed()) {
        }
        while (!failed()) {
            const hipError_t e = hipEventQuery(a.slot_done[slot]);
            if (e == hipSuccess) {
                return;
            }
            if (e != hipErrorNotReady) {
                check(e);
            }
        }
    };
    for (int i = 0; i < std::min(count, k_ring) && !failed(); ++i) {
        queue(i);
    }
    const std::function<void()> work = [&] {
        check(hipSetDevice(a.device));
        for (int i = next.fetch_add(1); i < count && !failed(); i = next.fetch_add(1)) {
            const Piece& p = pieces[static_cast<std::size_t>(i)];
            wait(i);
            if (!failed()) {
                std::memcpy(p.host, a.slot(i % k_ring), p.bytes);
            }
            if (i + k_ring < count) {
                queue(i + k_ring);
            }
        }
    };
    if (t_host_parallel) {
        Helpers::get().run(work);
    } else {
        work();
    }
    return static_cast<hipError_t>(error.load());
}

} // namespace

void d2h_copies(const HostCopy* list, int n, hipStream_t s) {
    std::size_t total = 0;
    for (int k = 0; k < n; ++k) {
        total += list[k].bytes;
    }
    if (total < k_pieces_min_bytes) {
        for (int k = 0; k < n; ++k) {
            if (list[k].bytes > 0) {
                hip_check(hipMemcpyAsync(list[k].host, list[k].dev, list[k].bytes, hipMemcpyDeviceToHost, s), "D2H copy");
            }
        }
        hip_check(hipStreamSynchronize(s), "D2H copy sync");
        return;
    }
    int device = 0;
    hip_check(hipGetDevice(&device), "hipGetDevice");
    Area* a = acquire(device);
    const hipError_t e = copy_pieces(list, n, *a, s, piece_bytes(total));
    const hipError_t w = hipStreamSynchronize(s); // the area is free again
    release(a);
    hip_check(e, "D2H copy");
    hip_check(w, "D2H copy sync");
}

} // namespace cfdg
