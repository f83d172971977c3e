// devbuf.h -- owning device buffers and HIP error checks shared by the
// host-side implementation files of libleo2d.  Internal.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>
#include <cstdlib>
#include <iterator>
#include <map>
#include <mutex>
#include <set>
#include <stdexcept>
#include <string>

#include "../../include/leo2d.h"

namespace leo2d {

// Device buffers a handle has given back, kept for its next allocations.  A call
// allocates and frees a dozen small buffers, each some 10-30 us with the device-wide
// wait of a free; on a 230-orbital deck that was half of the time.  Buffers of GBs cost
// more: a conductivity call that allocated and freed 3 GB of vector sets took 21 ms in
// one process and 50 to 90 ms in the next, and 20 ms in each with the sets kept.
// Everything a handle queues runs on its one stream, so a buffer taken again is
// written only by work queued after its last use.
// Bounded: buffers of at most kPoolMost bytes, at most kPoolKeep in all handles of the
// process (a handle's longest unused go first); all of every handle are freed when an
// allocation fails, a handle's own with it, and leo2d_batch_clear leaves its handle at most
// kPoolCleared.  A pool serves its handle alone; the lock
// is for the handle whose allocation failed.
class DevPool {
public:
    static constexpr size_t kPoolMost = size_t(2) << 30;
    static constexpr size_t kPoolKeep = size_t(4) << 30;
    static constexpr size_t kPoolCleared = size_t(256) << 20;   // the buffers of small calls
    DevPool()
    {
        std::lock_guard<std::mutex> g(all().lock);
        all().pools.insert(this);
    }
    DevPool(const DevPool&) = delete;
    DevPool& operator=(const DevPool&) = delete;
    ~DevPool()
    {
        {
            std::lock_guard<std::mutex> g(all().lock);
            all().pools.erase(this);
        }
        clear();
    }
    // a kept buffer of at least `bytes` (and less than twice that), or nullptr; cap: its size
    void* take(size_t bytes, size_t& cap)
    {
        std::lock_guard<std::mutex> g(lock_);
        auto it = free_.lower_bound(bytes);
        if (it == free_.end() || it->first / 2 > bytes) return nullptr;
        cap = it->first;
        return drop(it);
    }
    void give(void* p, size_t cap)
    {
        std::lock_guard<std::mutex> g(lock_);
        if (cap <= kPoolMost) {
            // reserve first: two handles must not both take the last room
            size_t was = all().kept.fetch_add(cap);
            while (was + cap > kPoolKeep && !free_.empty()) {
                auto old = free_.begin();
                for (auto it = free_.begin(); it != free_.end(); ++it)
                    if (it->second.given < old->second.given) old = it;
                was -= old->first;
                (void)hipFree(drop(old));
            }
            if (was + cap <= kPoolKeep) {
                free_.emplace(cap, Kept{p, ++given_});
                return;
            }
            all().kept -= cap;
        }
        (void)hipFree(p);
    }
    void clear() { trim(0); }
    // frees the largest kept buffers until at most `most` bytes are left
    void trim(size_t most)
    {
        std::lock_guard<std::mutex> g(lock_);
        size_t kept = 0;
        for (const auto& f : free_) kept += f.first;
        while (kept > most) {
            const auto it = std::prev(free_.end());
            kept -= it->first;
            (void)hipFree(drop(it));
        }
    }
    // every handle's kept buffers (a free waits for the work that may still use them)
    static void clear_all()
    {
        std::lock_guard<std::mutex> g(all().lock);
        for (DevPool* p : all().pools) p->clear();
    }
    // the pool of the handle whose entry point this thread is in
    static DevPool*& current()
    {
        static thread_local DevPool* pool = nullptr;
        return pool;
    }
    struct Use {   // makes `pool` current for a scope
        DevPool* was;
        explicit Use(DevPool* pool) : was(current()) { current() = pool; }
        ~Use() { current() = was; }
    };

private:
    struct Kept {
        void* p;
        uint64_t given;   // order of return
    };
    using Free = std::multimap<size_t, Kept>;   // by size
    struct All {
        std::mutex lock;
        std::set<DevPool*> pools;
        std::atomic<size_t> kept{0};
    };
    static All& all()
    {
        static All* const a = new All;   // outlives every handle
        return *a;
    }
    void* drop(Free::iterator it)
    {
        void* p = it->second.p;
        all().kept -= it->first;
        free_.erase(it);
        return p;
    }
    std::mutex lock_;
    Free free_;
    uint64_t given_ = 0;
};

// owning device allocation (given back on release() or destruction; movable, not copyable)
struct DevBuf {
    void* p = nullptr;
    size_t bytes = 0;          // as asked for
    size_t cap = 0;            // as allocated
    DevPool* pool = nullptr;   // where it goes back to (nullptr: freed)
    DevBuf() = default;
    DevBuf(const DevBuf&) = delete;
    DevBuf& operator=(const DevBuf&) = delete;
    DevBuf(DevBuf&& o) noexcept : p(o.p), bytes(o.bytes), cap(o.cap), pool(o.pool)
    {
        o.p = nullptr;
        o.bytes = 0;
    }
    DevBuf& operator=(DevBuf&& o) noexcept
    {
        if (this != &o) {
            release();
            p = o.p;
            bytes = o.bytes;
            cap = o.cap;
            pool = o.pool;
            o.p = nullptr;
            o.bytes = 0;
        }
        return *this;
    }
    ~DevBuf() { release(); }
    void release()
    {
        if (p) {
            if (pool) pool->give(p, cap);
            else (void)hipFree(p);
        }
        p = nullptr;
        bytes = 0;
    }
};

struct HipError : std::runtime_error {
    int code;
    HipError(const std::string& m, int c) : std::runtime_error(m), code(c) {}
};

inline void check(hipError_t e, const char* what)
{
    if (e != hipSuccess) {
        const int code = (e == hipErrorOutOfMemory || e == hipErrorMemoryAllocation) ? LEO2D_ERR_ALLOC : LEO2D_ERR_HIP;
        throw HipError(std::string(what) + ": " + hipGetErrorString(e), code);
    }
}

// LEO2D_ALLOC_LIMIT: bytes above which an allocation fails as on a full device, so that what
// a call leaves behind after a failed allocation can be tested on an empty one
inline size_t alloc_limit()
{
    const char* e = std::getenv("LEO2D_ALLOC_LIMIT");
    return e ? (size_t)std::strtoull(e, nullptr, 10) : SIZE_MAX;
}

// The old buffer goes first: where the allocation fails b is empty, so what describes b's
// contents is cleared before the call, or the new buffer is a local one moved in when whole.
inline void dalloc(DevBuf& b, size_t bytes, const char* what)
{
    b.release();
    if (bytes == 0) bytes = 16;
    if (bytes > alloc_limit()) check(hipErrorOutOfMemory, what);
    DevPool* const pool = DevPool::current();
    // a pooled buffer's size is rounded up (to an eighth of its power of two), so that calls on
    // slightly different sizes find each other's buffers
    size_t cap = bytes;
    if (pool && bytes <= DevPool::kPoolMost) {
        size_t step = 256;
        while (step * 16 < bytes) step *= 2;
        cap = (bytes + step - 1) / step * step;
        size_t got = 0;
        if (void* p = pool->take(cap, got)) {
            b.p = p;
            b.bytes = bytes;
            b.cap = got;
            b.pool = pool;
            return;
        }
    }
    hipError_t e = hipMalloc(&b.p, cap);
    if (e != hipSuccess) {
        // what the pools keep may be what is missing
        (void)hipGetLastError();
        DevPool::clear_all();
        e = hipMalloc(&b.p, cap);
    }
    if (e != hipSuccess) {
        // a failed allocation is not sticky, but it stays the runtime's last error:
        // clear it, or the next launch check (hipGetLastError) would report it
        (void)hipGetLastError();
        b.p = nullptr;
        check(e, what);
    }
    b.bytes = bytes;
    b.cap = cap;
    b.pool = pool;
}

}  // namespace leo2d
