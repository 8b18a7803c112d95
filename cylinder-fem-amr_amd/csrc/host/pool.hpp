// Reuse of freed device blocks by the host layer's arrays. A run, a solver object or a remesh allocates
// and frees hundreds of arrays, and each hipFree waits for the device and unmaps (54-90 us on average),
// each hipMalloc maps (13-42 us): 46 of 323 ms of an adaptive run of 62 steps, 34 of 58 ms of a solve of
// a stored pressure system.
#pragma once

#include <cstddef>
#include <functional>
#include <map>
#include <mutex>
#include <unordered_map>

namespace cfa {

// Freed blocks are kept by size, at most `bound` bytes of them (a block beyond that is freed at once),
// and given out again for requests they fit within 1.5 times. hipFree returns only when the device has
// finished everything submitted before; here that wait moves to the reuse: a block given out again was
// freed before the last full device synchronisation, or one is made first. So a block may be freed while
// kernels of any stream still use it, as with hipFree. When the device cannot be synchronised (another
// thread may be capturing a stream), a new block is allocated instead. Safe from several threads.
class BlockPool {
public:
    std::function<int(void**, size_t)> alloc;   // 0 on success
    std::function<int(void*)> free;
    std::function<int()> sync;                  // waits for the whole device
    size_t bound = (size_t)2 << 30;

    // a block of at least `bytes`; on failure everything kept is given back and the request repeated
    int get(void** ptr, size_t bytes);
    void put(void* ptr);
    void trim();   // gives every kept block back
    size_t kept_bytes();

    static size_t class_of(size_t bytes);   // size a request is rounded to: eight steps per octave

private:
    struct Block {
        void* ptr;
        unsigned long long freed;   // value of clock_ when it was freed
    };
    std::mutex m_;
    std::multimap<size_t, Block> kept_;
    std::unordered_map<void*, size_t> size_of_;   // blocks given out
    size_t kept_bytes_ = 0;
    unsigned long long clock_ = 1, synced_ = 0;   // blocks with freed <= synced_ are idle
    void trim_locked();
};

// The pool of the host layer's device arrays (cfa_malloc, cfa_free, cfa_device_sync): one for the process,
// whose host layer works on device 0 (every entry point selects it)
BlockPool& device_pool();

}  // namespace cfa
