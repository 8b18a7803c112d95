#include "pool.hpp"

#include "../../../include/cfa_hip.h"
#include "../../../include/cfa_host.h"

namespace cfa {

size_t BlockPool::class_of(size_t bytes) {
    size_t step = 512;
    while (step * 16 < bytes) step *= 2;   // sizes 8 step .. 16 step in steps of `step`
    return (bytes + step - 1) / step * step;
}

int BlockPool::get(void** ptr, size_t bytes) {
    const size_t want = class_of(bytes > 0 ? bytes : 1);
    std::lock_guard<std::mutex> lock(m_);
    auto pick = kept_.end();
    for (auto it = kept_.lower_bound(want); it != kept_.end() && it->first <= want + want / 2; ++it) {
        if (it->second.freed <= synced_) { pick = it; break; }   // idle: no wait
        if (pick == kept_.end()) pick = it;
    }
    if (pick != kept_.end() && pick->second.freed > synced_) {
        if (sync() == 0) synced_ = clock_++;
        else pick = kept_.end();   // not known to be idle: it stays kept
    }
    if (pick != kept_.end()) {
        *ptr = pick->second.ptr;
        size_of_[*ptr] = pick->first;
        kept_bytes_ -= pick->first;
        kept_.erase(pick);
        return 0;
    }
    int rc = alloc(ptr, want);
    if (rc != 0 && !kept_.empty()) {
        trim_locked();
        rc = alloc(ptr, want);
    }
    if (rc == 0) size_of_[*ptr] = want;
    return rc;
}

void BlockPool::put(void* ptr) {
    if (!ptr) return;
    std::lock_guard<std::mutex> lock(m_);
    const auto it = size_of_.find(ptr);
    if (it == size_of_.end()) return;
    const size_t size = it->second;
    size_of_.erase(it);
    if (size > bound || kept_bytes_ > bound - size) {
        (void)free(ptr);
        return;
    }
    kept_bytes_ += size;
    kept_.insert({size, Block{ptr, clock_}});
}

void BlockPool::trim_locked() {
    for (const auto& b : kept_) (void)free(b.second.ptr);
    kept_.clear();
    kept_bytes_ = 0;
}

void BlockPool::trim() {
    std::lock_guard<std::mutex> lock(m_);
    trim_locked();
}

size_t BlockPool::kept_bytes() {
    std::lock_guard<std::mutex> lock(m_);
    return kept_bytes_;
}

BlockPool& device_pool() {
    // never destroyed: arrays of static objects may be freed after any static pool's destructor, and the
    // memory goes back to the system with the process
    static BlockPool* pool = [] {
        auto* p = new BlockPool();
        p->alloc = [](void** ptr, size_t bytes) { return cfa_malloc(ptr, bytes); };
        p->free = [](void* ptr) { return cfa_free(ptr); };
        p->sync = [] { return cfa_device_sync(); };
        return p;
    }();
    return *pool;
}

}  // namespace cfa

extern "C" {

void cfa_pool_trim(void) { cfa::device_pool().trim(); }

long long cfa_pool_bytes(void) { return (long long)cfa::device_pool().kept_bytes(); }

}  // extern "C"
