// Copies between a caller's ordinary (pageable) host arrays and the device, through pinned chunks that several threads
// fill and empty.
//
// Why: the runtime's own pageable copies of 20 MB run at 27 GB/s to the device and 15 from it, 4 into freshly allocated
// memory (one host thread moves the bytes and takes the page faults), and cost 35 us at 64 KB; the link carries 55.  These:
// 38 and 35 GB/s, 9 into fresh memory, 10 us.  Pieces of 2 MB: half of that costs 15 % at 20 MB, twice it gains nothing.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <memory>
#include <vector>

namespace mdp {

// One set of pinned chunks, for streams of one device.  Not thread-safe: its owner serialises the use.
class HostCopies {
public:
    HostCopies() = default;
    HostCopies(const HostCopies&) = delete;
    HostCopies& operator=(const HostCopies&) = delete;
    ~HostCopies();
    // src is read before the call returns; the device sees the bytes in stream order.  get_follows: src is also where
    // results go (it is writable)
    void put(void* dst, const void* src, size_t bytes, hipStream_t st, bool get_follows = false);
    // a part of a device array and where it goes
    struct Part {
        void* dst;
        size_t from, bytes;
    };
    // dst is written by the next finish() on the same stream
    void get(void* dst, const void* src, size_t bytes, hipStream_t st);
    // the parts (ascending, disjoint) of src[0..bytes).  Where it throws, nothing writes to this call's parts any more
    void get_parts(const std::vector<Part>& parts, const void* src, size_t bytes, hipStream_t st);
    // waits for the stream and for every byte of the gets
    void finish(hipStream_t st);
    // forgets what is pending, after an error; waits for the stream first
    void abandon(hipStream_t st) noexcept;
    // a part of the threads' work that can be waited for by itself (its count is theirs)
    struct Group {
        int left = 0;
    };

private:
    static constexpr size_t CHUNK = size_t(4) << 20, MAX_CHUNKS = 8, PIECE = size_t(2) << 20;
    struct Chunk {
        char* p = nullptr;
        hipEvent_t ev[CHUNK / PIECE] = {};
    };
    struct Pending {
        const char* pinned;
        hipEvent_t ready;   // null: with the end of the stream
        std::vector<Part> parts;   // `from` within the piece
    };
    std::vector<Chunk> chunks;
    std::vector<Pending> pending;
    Group moving;    // what the threads still do for the gets
    size_t at = 0;   // first free byte over all chunks
    char* take(size_t bytes, hipStream_t st, hipEvent_t** ev);
    void issue(const std::vector<Part>& parts, const void* src, size_t bytes, hipStream_t st);
};

// Copies of the engines' own calls, through a set of chunks that nobody else uses while this object lives: engines on
// different threads don't wait for one another's streams.  Every copy is complete after finish().
class EngineCopies {
public:
    explicit EngineCopies(hipStream_t st);
    ~EngineCopies();
    EngineCopies(const EngineCopies&) = delete;
    EngineCopies& operator=(const EngineCopies&) = delete;
    void put(void* dst, const void* src, size_t bytes);
    void get(void* dst, const void* src, size_t bytes);
    void finish();

private:
    hipStream_t st;
    int device;   // of the stream: what the set belongs to
    std::unique_ptr<HostCopies> set;
    bool open = false;   // something was asked for since the last finish()
};

}  // namespace mdp
