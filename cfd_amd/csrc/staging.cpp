// Large host <-> device copies through pinned staging memory. A copy from or to pageable memory
// runs at a fraction of the PCIe rate; here the pageable side is copied by the host threads into
// (or out of) pinned chunks while the DMA engine moves the previous chunk. Staging areas come
// from a process-wide free list: at most k_kept_areas are kept, until cfdg_release_cached_memory, and
// result copies that would need more go through the runtime.
//
// The results of solves and finite-volume calls (d2h_copies) take a finer pipeline, by the caller and, if
// they are large, helper threads of its own (copy_team.hpp). The set-up's copies keep the OpenMP team that
// runs the loops around them: more threads beside its spinning workers exceed a CPU quota of the team's
// size, and the process is stopped for the rest of the scheduler's period (set-up 4% slower, the first
// solve after it up to 5 ms).
#include "copy_team.hpp"
#include "hip_util.hpp"

#include <omp.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <type_traits>

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

// Helper threads of d2h_copies: one, with which the caller keeps up with the link (16 MiB 0.48 ms, alone
// 0.52, with three 0.49, through the runtime 0.95); from k_large_copy on, where malloc hands out fresh pages
// each time and the copy waits for their zeroing, all of them (32 MiB 1.05 ms, with one 1.8, alone 2.0).
constexpr std::size_t k_large_copy = std::size_t(24) << 20;
constexpr int helpers_of(std::size_t total) { return total >= k_large_copy ? CopyTeam::k_helpers : 1; }

constexpr std::size_t k_slot = std::size_t(4) << 20; // d2h_copies' share of a chunk
constexpr int k_slots_per_chunk = static_cast<int>(k_chunk / k_slot);
constexpr int k_ring = 2 * k_slots_per_chunk;        // its slots per area

// Bytes per piece of d2h_copies: small enough that a copy's first and last pieces, which nothing
// overlaps, are a small part of it, large enough for the 10 us that each costs. 2 and 4 MiB at 200 MiB: 6.9
// and 5.6 ms; 1, 2 and 4 MiB at 17 MiB: 642, 555 and 565 us.
constexpr std::size_t piece_bytes(std::size_t total) {
    return total > (std::size_t(32) << 20) ? k_slot : std::size_t(2) << 20;
}

struct Area {
    char* buf[2] = {nullptr, nullptr};
    hipEvent_t done[2] = {nullptr, nullptr};
    hipEvent_t slot_done[k_ring] = {};
    int device = -1;
    Area* next = nullptr; // in the free list
    alignas(64) unsigned char copy[512]; // d2h_copies' state, used by a late helper after the call returned
    Area() = default;
    Area(const Area&) = delete;
    Area& operator=(const Area&) = delete;
    ~Area() {
        for (char* b : buf) {
            if (b != nullptr) {
                (void)hipHostFree(b);
            }
        }
        for (hipEvent_t e : done) {
            if (e != nullptr) {
                (void)hipEventDestroy(e);
            }
        }
        for (hipEvent_t e : slot_done) {
            if (e != nullptr) {
                (void)hipEventDestroy(e);
            }
        }
    }
    [[nodiscard]] char* slot(int i) const {
        return buf[i / k_slots_per_chunk] + static_cast<std::size_t>(i % k_slots_per_chunk) * k_slot;
    }
};

thread_local bool t_host_parallel = true;

constexpr int k_kept_areas = 8; // 32 MiB each

std::mutex g_mutex;
Area* g_free = nullptr;
int g_areas = 0; // in use or free

// An idle area of the device, or null.
Area* take_free(int device) {
    for (Area** at = &g_free; *at != nullptr; at = &(*at)->next) {
        if ((*at)->device == device) {
            Area* a = *at;
            *at = a->next;
            return a;
        }
    }
    return nullptr;
}

Area* acquire(int device) {
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        if (Area* a = take_free(device)) {
            return a;
        }
    }
    auto a = std::make_unique<Area>();
    a->device = device;
    for (int k = 0; k < 2; ++k) {
        hip_check(hipHostMalloc(reinterpret_cast<void**>(&a->buf[k]), k_chunk, hipHostMallocDefault),
                  "hipHostMalloc staging");
        hip_check(hipEventCreateWithFlags(&a->done[k], hipEventDisableTiming), "staging event");
    }
    for (hipEvent_t& e : a->slot_done) {
        hip_check(hipEventCreateWithFlags(&e, hipEventDisableTiming), "staging event");
    }
    std::lock_guard<std::mutex> lock(g_mutex);
    ++g_areas;
    return a.release();
}

// As acquire; null where the area would be one too many or cannot be had.
Area* try_acquire(int device) noexcept {
    try {
        {
            std::lock_guard<std::mutex> lock(g_mutex);
            if (Area* a = take_free(device)) {
                return a;
            }
            if (g_areas >= k_kept_areas) {
                return nullptr;
            }
        }
        return acquire(device);
    } catch (...) { // no pinned memory to be had
        (void)hipGetLastError();
        return nullptr;
    }
}

void release(Area* a) noexcept {
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        if (g_areas <= k_kept_areas) {
            a->next = g_free;
            g_free = a;
            return;
        }
        --g_areas;
    }
    delete a;
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

} // namespace

bool host_parallel() { return t_host_parallel; }

void set_host_parallel(bool on) { t_host_parallel = on; }

void release_staging() noexcept {
    for (;;) {
        Area* a = nullptr;
        {
            std::lock_guard<std::mutex> lock(g_mutex);
            a = g_free;
            if (a == nullptr) {
                return;
            }
            g_free = a->next;
            --g_areas;
        }
        delete a;
    }
}

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

// The device's side of d2h_copies: the pieces of a list of copies, through the slots of one area.
struct PieceCopy {
    const HostCopy* list; // the caller's
    int n;
    std::size_t piece;
    Area* a;
    hipStream_t s;

    struct Part {
        const char* dev;
        char* host;
        std::size_t bytes;
    };
    [[nodiscard]] int count() const {
        std::size_t c = 0;
        for (int k = 0; k < n; ++k) {
            c += pieces(list[k].bytes);
        }
        return static_cast<int>(c);
    }
    [[nodiscard]] std::size_t pieces(std::size_t bytes) const { return (bytes + piece - 1) / piece; }
    [[nodiscard]] Part part(int i) const {
        std::size_t j = static_cast<std::size_t>(i);
        const HostCopy* c = list;
        for (; j >= pieces(c->bytes); ++c) {
            j -= pieces(c->bytes);
        }
        const std::size_t o = j * piece;
        return {static_cast<const char*>(c->dev) + o, static_cast<char*>(c->host) + o, std::min(piece, c->bytes - o)};
    }
    [[nodiscard]] int queue(int i, int slot) const {
        const Part p = part(i);
        const hipError_t e = hipMemcpyAsync(a->slot(slot), p.dev, p.bytes, hipMemcpyDeviceToHost, s);
        return e != hipSuccess ? e : hipEventRecord(a->slot_done[slot], s);
    }
    [[nodiscard]] int arrived(int slot, bool& yes) const {
        const hipError_t e = hipEventQuery(a->slot_done[slot]);
        yes = e == hipSuccess;
        return e == hipErrorNotReady ? hipSuccess : e;
    }
    [[nodiscard]] bool copy_out(int i, int slot, int k) const {
        constexpr std::size_t step = std::size_t(256) << 10; // 20 us
        const Part p = part(i);
        const std::size_t o = static_cast<std::size_t>(k) * step;
        std::memcpy(p.host + o, a->slot(slot) + o, std::min(step, p.bytes - o));
        return o + step < p.bytes;
    }
    void drain() const { (void)hipStreamSynchronize(s); }
    void leave() const { release(a); }
};

using Copy = RingCopy<k_ring, PieceCopy>;
static_assert(sizeof(Copy) <= sizeof(Area::copy) && alignof(Copy) <= 64 && std::is_trivially_destructible_v<Copy>,
              "a copy lives in its area until the area is used again");

} // namespace

void d2h_copies(const HostCopy* list, int n, hipStream_t s) {
    std::size_t total = 0;
    for (int k = 0; k < n; ++k) {
        total += list[k].bytes;
    }
    int device = 0;
    hip_check(hipGetDevice(&device), "hipGetDevice");
    Area* a = total < k_pieces_min_bytes ? nullptr : try_acquire(device);
    if (a == nullptr) { // small, or the runtime's way
        for (int k = 0; k < n; ++k) {
            if (list[k].bytes > 0) {
                hip_check(hipMemcpyAsync(list[k].host, list[k].dev, list[k].bytes, hipMemcpyDeviceToHost, s), "D2H copy");
            }
        }
        hip_check(hipStreamSynchronize(s), "D2H copy sync");
        return;
    }
    const PieceCopy pieces{list, n, piece_bytes(total), a, s};
    Copy* copy = new (a->copy) Copy(pieces, pieces.count());
    const int e = copy->run(t_host_parallel ? &CopyTeam::get() : nullptr, helpers_of(total));
    hip_check(static_cast<hipError_t>(e), "D2H copy");
}

} // namespace cfdg
