#include "host_copy.hpp"

#include <pthread.h>
#include <sched.h>
#include <signal.h>
#include <unistd.h>

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <deque>
#include <map>
#include <mutex>
#include <thread>

#include "runtime.hpp"

namespace mdp {
namespace {

// Up to 7 threads that move bytes beside the calling one; started by the first large copy, joined when the library goes.
// A process without them (a fork's child, a refused thread) copies with the calling thread alone.
class CopyThreads {
public:
    ~CopyThreads() {
        {
            std::lock_guard<std::mutex> lk(m);
            stop = true;
        }
        work.notify_all();
        for (std::thread& t : threads) t.join();
    }
    using Group = HostCopies::Group;
    // src_pages: src is written to later on, its pages are made before it is read.
    // src null: only has the pages of dst made, ahead of the copy that will fill them
    void post(Group& g, void* dst, const void* src, size_t bytes, bool src_pages = false) {
        std::lock_guard<std::mutex> lk(m);
        start();
        if (!src && threads.empty()) return;
        for (size_t o = 0; o < bytes; o += GRAIN) {
            queue.push_back({static_cast<char*>(dst) + o, src ? static_cast<const char*>(src) + o : nullptr,
                             std::min(GRAIN, bytes - o), src_pages, &g});
            ++g.left;
        }
        work.notify_all();
    }
    // helps until the group's work is done
    void wait(Group& g) {
        std::unique_lock<std::mutex> lk(m);
        while (g.left > 0)
            if (!queue.empty())
                one(lk);
            else
                done.wait(lk, [&] { return g.left == 0 || !queue.empty(); });
    }

private:
    static constexpr size_t GRAIN = size_t(128) << 10;
    struct Piece {
        char* dst;
        const char* src;
        size_t bytes;
        bool src_pages;
        Group* group;
    };
    std::mutex m;
    std::condition_variable work, done;
    std::deque<Piece> queue;
    bool stop = false, started = false;
    std::vector<std::thread> threads;

    // A freshly allocated array's pages, by a write to each that changes nothing.  A read first would map the shared zero
    // page and have the later write replace it under every thread (4.5 MB: 7 ms against 0.4); asking for them in bulk
    // (MADV_POPULATE_WRITE) serialises the threads (0.7 ms).
    static void make_pages(char* p, size_t bytes) {
        static const size_t page = static_cast<size_t>(sysconf(_SC_PAGESIZE));
        static volatile char nothing = 0;   // not a constant: an `or` with a known 0 would become a read
        const char z = nothing;
        for (size_t o = 0; o < bytes; o += page) __atomic_fetch_or(p + o, z, __ATOMIC_RELAXED);
        if (bytes) __atomic_fetch_or(p + bytes - 1, z, __ATOMIC_RELAXED);
    }
    void one(std::unique_lock<std::mutex>& lk) {
        const Piece p = queue.front();
        queue.pop_front();
        lk.unlock();
        if (p.src_pages) make_pages(const_cast<char*>(p.src), p.bytes);
        if (p.src)
            std::memcpy(p.dst, p.src, p.bytes);
        else
            make_pages(p.dst, p.bytes);
        lk.lock();
        if (--p.group->left == 0) done.notify_all();
    }
    void start() {
        if (started) return;
        started = true;
        cpu_set_t set;
        const int cpus = sched_getaffinity(0, sizeof(set), &set) == 0 ? CPU_COUNT(&set) : 1;
        sigset_t all, old;   // signals stay with the program's own threads
        sigfillset(&all);
        pthread_sigmask(SIG_SETMASK, &all, &old);
        try {
            for (int k = 1; k < std::min(cpus, 8); ++k)
                threads.emplace_back([this] {
                    std::unique_lock<std::mutex> lk(m);
                    for (;;) {
                        work.wait(lk, [&] { return stop || !queue.empty(); });
                        if (queue.empty()) return;
                        one(lk);
                    }
                });
        } catch (const std::exception&) {   // as many as there are
        }
        pthread_sigmask(SIG_SETMASK, &old, nullptr);
    }
};

CopyThreads& copy_threads() {
    struct Owner {
        CopyThreads* t = new CopyThreads;
        pid_t pid = getpid();
        ~Owner() {
            if (getpid() == pid) delete t;   // a fork's child has the object but not the threads to join
        }
    };
    static Owner o;
    return *o.t;
}

int device_of(hipStream_t st) {
    hipDevice_t d = 0;
    MDP_HIP(hipStreamGetDevice(st, &d));
    return d;
}

// The stream's device as the current one: pinned memory and events belong to the device that is current when they are made,
// and an event can only be recorded on that device's streams.
class OnDeviceOf {
public:
    explicit OnDeviceOf(hipStream_t st) {
        const int device = device_of(st);
        MDP_HIP(hipGetDevice(&before));
        if (before == device)
            before = -1;
        else
            MDP_HIP(hipSetDevice(device));
    }
    ~OnDeviceOf() {
        if (before >= 0) (void)hipSetDevice(before);
    }

private:
    int before = -1;
};

// below this a thread's wake-up costs more than its share of the copy
constexpr size_t SHARED = size_t(192) << 10;

}  // namespace

HostCopies::~HostCopies() {
    for (Chunk& c : chunks) {
        for (hipEvent_t e : c.ev)
            if (e) (void)hipEventDestroy(e);
        if (c.p) (void)hipHostFree(c.p);
    }
}

// room for at most PIECE bytes; *ev is the event that belongs to it
char* HostCopies::take(size_t bytes, hipStream_t st, hipEvent_t** ev) {
    bytes = (bytes + 63) / 64 * 64;
    if (at % PIECE + bytes > PIECE) at = (at / PIECE + 1) * PIECE;   // a piece does not straddle
    if (at >= CHUNK * MAX_CHUNKS) finish(st);
    const size_t k = at / CHUNK, o = at % CHUNK;
    if (k >= chunks.size()) {
        Chunk c;
        const OnDeviceOf on(st);
        MDP_HIP(hipHostMalloc(reinterpret_cast<void**>(&c.p), CHUNK, hipHostMallocDefault));
        chunks.push_back(c);
    }
    at += bytes;
    *ev = &chunks[k].ev[o / PIECE];
    return chunks[k].p + o;
}

void HostCopies::put(void* dst, const void* src, size_t bytes, hipStream_t st, bool get_follows) {
    hipEvent_t* ev;
    char* const d = static_cast<char*>(dst);
    const char* const s = static_cast<const char*>(src);
    if (bytes < SHARED) {
        if (!bytes) return;
        char* p = take(bytes, st, &ev);
        std::memcpy(p, s, bytes);
        MDP_HIP(hipMemcpyAsync(d, p, bytes, hipMemcpyHostToDevice, st));
        return;
    }
    // a batch of pieces at a time: all are given to the threads, each goes to the device when it is in place
    constexpr size_t BATCH = CHUNK * MAX_CHUNKS / PIECE / 2;
    CopyThreads::Group group[BATCH];
    char* at_pinned[BATCH];
    for (size_t o = 0; o < bytes;) {
        size_t k = 0;
        hipError_t e = hipSuccess;
        const size_t pieces = std::min(BATCH, (bytes - o + PIECE - 1) / PIECE);
        if ((at + PIECE - 1) / PIECE + pieces > CHUNK * MAX_CHUNKS / PIECE) finish(st);
        for (size_t q = o; k < pieces; ++k, q += PIECE) at_pinned[k] = take(std::min(PIECE, bytes - q), st, &ev);
        for (size_t i = 0; i < k; ++i)
            copy_threads().post(group[i], at_pinned[i], s + o + i * PIECE, std::min(PIECE, bytes - o - i * PIECE), get_follows);
        for (size_t i = 0; i < k; ++i) {
            copy_threads().wait(group[i]);
            const size_t n = std::min(PIECE, bytes - o - i * PIECE);
            if (e == hipSuccess) e = hipMemcpyAsync(d + o + i * PIECE, at_pinned[i], n, hipMemcpyHostToDevice, st);
        }
        MDP_HIP(e);
        o += k * PIECE;
    }
}

void HostCopies::get(void* dst, const void* src, size_t bytes, hipStream_t st) {
    if (bytes) get_parts({{dst, 0, bytes}}, src, bytes, st);
}

void HostCopies::get_parts(const std::vector<Part>& parts, const void* src, size_t bytes, hipStream_t st) {
    const size_t before = pending.size();
    try {
        // while the device works on what was asked of it before
        for (const Part& t : parts)
            if (t.bytes >= SHARED) copy_threads().post(moving, t.dst, nullptr, t.bytes);
        issue(parts, src, bytes, st);
    } catch (...) {   // the caller may free what the threads make pages of as it unwinds
        copy_threads().wait(moving);
        if (pending.size() > before) pending.erase(pending.begin() + static_cast<long>(before), pending.end());
        throw;
    }
}

// the copies of get_parts into the pinned chunks, and what is to be moved on from there
void HostCopies::issue(const std::vector<Part>& parts, const void* src, size_t bytes, hipStream_t st) {
    hipEvent_t* ev;
    size_t k = 0;
    for (size_t o = 0; o < bytes; o += PIECE) {
        const size_t n = std::min(PIECE, bytes - o);
        char* p = take(n, st, &ev);
        MDP_HIP(hipMemcpyAsync(p, static_cast<const char*>(src) + o, n, hipMemcpyDeviceToHost, st));
        Pending q{p, nullptr, {}};
        if (n >= SHARED) {   // its bytes are moved on while the next piece is under way
            if (!*ev) {
                const OnDeviceOf on(st);
                MDP_HIP(hipEventCreateWithFlags(ev, hipEventDisableTiming));
            }
            MDP_HIP(hipEventRecord(*ev, st));
            q.ready = *ev;
        }
        for (; k < parts.size() && parts[k].from < o + n; ++k) {
            const size_t a = std::max(parts[k].from, o), b = std::min(parts[k].from + parts[k].bytes, o + n);
            q.parts.push_back({static_cast<char*>(parts[k].dst) + (a - parts[k].from), a - o, b - a});
            if (parts[k].from + parts[k].bytes > o + n) break;   // goes on in the next piece
        }
        pending.push_back(std::move(q));
    }
}

void HostCopies::finish(hipStream_t st) {
    // the large pieces first, each when it has arrived; the others with the end of the stream
    for (const Pending& q : pending)
        if (q.ready) {
            if (const hipError_t e = hipEventSynchronize(q.ready); e != hipSuccess) {
                copy_threads().wait(moving);
                pending.clear();
                MDP_HIP(e);
            }
            for (const Part& t : q.parts)
                if (t.bytes >= SHARED / 4)
                    copy_threads().post(moving, t.dst, q.pinned + t.from, t.bytes);
                else
                    std::memcpy(t.dst, q.pinned + t.from, t.bytes);
        }
    const hipError_t e = hipStreamSynchronize(st);
    if (e == hipSuccess)
        for (const Pending& q : pending)
            if (!q.ready)
                for (const Part& t : q.parts) std::memcpy(t.dst, q.pinned + t.from, t.bytes);
    copy_threads().wait(moving);
    pending.clear();
    at = 0;
    MDP_HIP(e);
}

void HostCopies::abandon(hipStream_t st) noexcept {
    if (st) (void)hipStreamSynchronize(st);
    copy_threads().wait(moving);
    pending.clear();
    at = 0;
}

namespace {
// The sets that no engine's copies use at the moment, by device.  Four of a device (of at most 32 MB of pinned memory each)
// are kept for the next copies, more are given back: as many engines as a program runs on different threads copy without
// allocating.
struct IdleSets {
    static constexpr size_t KEPT = 4;
    std::mutex m;
    std::map<int, std::vector<std::unique_ptr<HostCopies>>> of_device;
};
IdleSets& idle_sets() {
    static IdleSets s;
    return s;
}
}  // namespace

EngineCopies::EngineCopies(hipStream_t s) : st(s), device(device_of(s)) {
    IdleSets& idle = idle_sets();
    {
        std::lock_guard<std::mutex> lk(idle.m);
        auto& sets = idle.of_device[device];
        sets.reserve(IdleSets::KEPT);
        if (!sets.empty()) {
            set = std::move(sets.back());
            sets.pop_back();
        }
    }
    if (!set) set = std::make_unique<HostCopies>();
}
EngineCopies::~EngineCopies() {
    if (open) set->abandon(st);
    IdleSets& idle = idle_sets();
    std::lock_guard<std::mutex> lk(idle.m);
    auto& sets = idle.of_device[device];
    if (sets.size() < IdleSets::KEPT) sets.push_back(std::move(set));
}
void EngineCopies::put(void* dst, const void* src, size_t bytes) {
    open = true;
    set->put(dst, src, bytes, st);
}
void EngineCopies::get(void* dst, const void* src, size_t bytes) {
    open = true;
    set->get(dst, src, bytes, st);
}
void EngineCopies::finish() {
    set->finish(st);
    open = false;
}

}  // namespace mdp
