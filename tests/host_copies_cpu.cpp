// The copies between host arrays and the device (mdp_amd/csrc/host_copy.cpp) on the CPU: the few HIP calls they make
// are played here.  A stream is a queue of copies that run when it, or an event behind them, is waited for, so a chunk
// that is filled again too early, or a byte that is handed on too early, shows as wrong data.
//   host_copies_cpu bytes | unwind | two_engines | two_devices
#include <sys/mman.h>
#include <unistd.h>

#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <random>
#include <set>
#include <string>
#include <thread>
#include <vector>

#include "../mdp_amd/csrc/host_copy.hpp"
#include "../mdp_amd/csrc/runtime.hpp"

namespace {

struct Stream {
    int device = 0;
    std::vector<std::function<void()>> queue;
    size_t done = 0;
    std::function<void()> work;   // what the stream is busy with before its copies
    void run(size_t upto) {
        if (work) work();
        for (; done < upto; ++done) queue[done]();
    }
};
struct Event {
    int device;
    Stream* stream = nullptr;
    size_t upto = 0;
};
thread_local int current_device = 0;
struct Pinned {
    size_t bytes;
    int device;
    std::set<int> used_by;
};
std::mutex pinned_lock;
std::map<char*, Pinned> pinned_blocks;
void used(const void* p, int device) {
    std::lock_guard<std::mutex> lk(pinned_lock);
    char* q = static_cast<char*>(const_cast<void*>(p));
    auto b = pinned_blocks.upper_bound(q);
    if (b == pinned_blocks.begin()) return;
    --b;
    if (q < b->first + b->second.bytes) b->second.used_by.insert(device);
}
bool refuse_copies = false;

Stream* of(hipStream_t s) { return reinterpret_cast<Stream*>(s); }
hipStream_t handle(Stream& s) { return reinterpret_cast<hipStream_t>(&s); }

}  // namespace

extern "C" {
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    std::lock_guard<std::mutex> lk(pinned_lock);
    if (!(*p = std::malloc(n))) return hipErrorOutOfMemory;
    pinned_blocks[static_cast<char*>(*p)] = Pinned{n, current_device, {}};
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    std::lock_guard<std::mutex> lk(pinned_lock);
    pinned_blocks.erase(static_cast<char*>(p));
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
    if (refuse_copies) return hipErrorUnknown;
    used(d, of(st)->device);
    used(s, of(st)->device);
    of(st)->queue.push_back([=] { std::memcpy(d, s, n); });
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t st) {
    of(st)->run(of(st)->queue.size());
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = reinterpret_cast<hipEvent_t>(new Event{current_device});
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    delete reinterpret_cast<Event*>(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t st) {
    Event* v = reinterpret_cast<Event*>(e);
    if (v->device != of(st)->device) return hipErrorInvalidHandle;
    v->stream = of(st);
    v->upto = of(st)->queue.size();
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    Event* v = reinterpret_cast<Event*>(e);
    v->stream->run(v->upto);
    return hipSuccess;
}
hipError_t hipStreamGetDevice(hipStream_t st, hipDevice_t* device) {
    *device = of(st)->device;
    return hipSuccess;
}
hipError_t hipGetDevice(int* device) {
    *device = current_device;
    return hipSuccess;
}
hipError_t hipSetDevice(int device) {
    current_device = device;
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "an error of the test"; }
}

namespace {

void expect(bool ok, const std::string& what) {
    if (ok) return;
    std::printf("FAILED: %s\n", what.c_str());
    std::exit(1);
}

// Every size on both sides of the limits: shared among threads or not (192 KB), one piece or more (2 MB), one batch of
// pieces or more (16 MB), all chunks in use (32 MB); several copies before a finish; parts with gaps between them.
void bytes() {
    std::mt19937_64 rng(1);
    mdp::HostCopies c;
    Stream st;
    const size_t KB = 1 << 10, MB = 1 << 20;
    const std::vector<std::vector<size_t>> groups = {
        {1, 63, 64, 65}, {192 * KB - 1, 192 * KB, 5}, {2 * MB - 1, 2 * MB, 2 * MB + 1}, {16 * MB - 3, 16 * MB + 3},
        {30 * MB, 3 * MB, 7}, {32 * MB, 64}, {40 * MB + 5, 2 * MB + 11, 192 * KB, 100}};
    for (const auto& sizes : groups) {
        std::vector<std::vector<unsigned char>> src, dev, back, kept;
        for (size_t n : sizes) {
            src.emplace_back(n);
            for (size_t i = 0; i < n; i += 8) {
                const unsigned long long r = rng();
                std::memcpy(&src.back()[i], &r, std::min<size_t>(8, n - i));
            }
            dev.emplace_back(n, 0);
            back.emplace_back(n, 0xAA);
        }
        kept = src;
        for (size_t k = 0; k < sizes.size(); ++k) {
            c.put(dev[k].data(), src[k].data(), sizes[k], handle(st), k % 2);
            std::memset(src[k].data(), 0x55, sizes[k]);   // the call has read it
        }
        for (size_t k = 0; k < sizes.size(); ++k) {
            if (k % 2 && sizes[k] > 10) {   // in three parts, a byte left out between them
                const size_t a = sizes[k] / 3, b = sizes[k] / 2;
                unsigned char* d = back[k].data();
                c.get_parts({{d, 0, a}, {d + a + 1, a + 1, b - a - 1}, {d + b + 1, b + 1, sizes[k] - b - 1}}, dev[k].data(),
                            sizes[k], handle(st));
                kept[k][a] = kept[k][b] = 0xAA;
            } else {
                c.get(back[k].data(), dev[k].data(), sizes[k], handle(st));
            }
        }
        c.finish(handle(st));
        for (size_t k = 0; k < sizes.size(); ++k)
            expect(back[k] == kept[k], "bytes of " + std::to_string(sizes[k]) + " as they were");
        std::printf("%zu copies from %zu bytes on: ok\n", sizes.size(), sizes[0]);
    }
}

size_t resident(void* p, size_t n) {
    std::vector<unsigned char> v(n / 4096);
    expect(mincore(p, n, v.data()) == 0, "mincore");
    size_t k = 0;
    for (unsigned char b : v) k += b & 1;
    return k;
}

// A copy that fails leaves nothing behind that still writes to its destination: the caller may free it as it unwinds.
void unwind() {
    const size_t n = size_t(512) << 20;
    void* p = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
    expect(p != MAP_FAILED, "mmap");
    madvise(p, n, MADV_NOHUGEPAGE);
    mdp::HostCopies c;
    Stream st;
    std::vector<char> src(1 << 20);
    refuse_copies = true;
    bool thrown = false;
    try {
        c.get(p, src.data(), n, handle(st));
    } catch (const mdp::Error&) {
        thrown = true;
    }
    const size_t at_throw = resident(p, n);
    usleep(300000);
    const size_t later = resident(p, n);
    std::printf("pages when the call failed %zu, 0.3 s later %zu\n", at_throw, later);
    expect(thrown, "the failed copy is reported");
    expect(at_throw == later, "no page of the destination is written after the call has failed");
    refuse_copies = false;
    c.finish(handle(st));   // and nothing of it is left to be delivered
}

// An engine whose stream is busy keeps no other engine's copies waiting.  The first engine's stream is done only when the
// second one has its bytes, or after 10 s.
void two_engines() {
    std::mutex m;
    std::condition_variable cv;
    bool waiting = false, second_done = false, in_time = false;
    Stream busy, idle;
    busy.work = [&] {
        std::unique_lock<std::mutex> lk(m);
        waiting = true;
        cv.notify_all();
        in_time = cv.wait_for(lk, std::chrono::seconds(10), [&] { return second_done; });
    };
    std::vector<char> a(100, 1), b(100, 2), got_a(100), got_b(100);
    std::thread first([&] {
        mdp::EngineCopies c(handle(busy));
        c.get(got_a.data(), a.data(), a.size());
        c.finish();
    });
    {
        std::unique_lock<std::mutex> lk(m);
        cv.wait(lk, [&] { return waiting; });
    }
    {
        mdp::EngineCopies c(handle(idle));
        c.get(got_b.data(), b.data(), b.size());
        c.finish();
    }
    {
        std::lock_guard<std::mutex> lk(m);
        second_done = true;
        cv.notify_all();
    }
    first.join();
    expect(got_a == a && got_b == b, "bytes as they were");
    expect(in_time, "the second engine's copies do not wait for the first engine's stream");
}

// Engines on two devices of one process, one after another and in turn, whichever device is the current one: an event
// can only be recorded on a stream of the device it was made on, and pinned memory belongs to the device that allocated it.
void two_devices() {
    const size_t n = size_t(3) << 20;   // two pieces, each with an event
    for (int k = 0; k < 8; ++k) {
        Stream st;
        st.device = k / 2 % 2;
        current_device = k % 2;
        std::vector<char> src(n, static_cast<char>(k)), back(n, 99);
        mdp::EngineCopies c(handle(st));
        c.get(back.data(), src.data(), n);
        c.finish();
        expect(back == src, "bytes as they were");
        expect(current_device == k % 2, "the current device is left as it was");
    }
    for (const auto& b : pinned_blocks)
        for (int d : b.second.used_by)
            expect(d == b.second.device, "pinned memory is used by the device it was allocated for");
}

}  // namespace

int main(int argc, char** argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "bytes")
        bytes();
    else if (what == "unwind")
        unwind();
    else if (what == "two_engines")
        two_engines();
    else if (what == "two_devices")
        two_devices();
    else
        return 2;
    std::printf("ok\n");
    return 0;
}
