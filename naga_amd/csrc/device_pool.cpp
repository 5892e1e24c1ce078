// Device memory blocks kept between allocations.
//
// A scene's set-up and its end allocate and free about a hundred buffers.
// hipMalloc and hipFree map and unmap their pages each time and hipFree waits
// for the device: closing a 132,651-node D3Q27 scene took 4.5 ms and its
// set-up's temporaries as much again, where the set-up's kernels take 5.
// Released blocks are kept for later allocations of about their size, up to
// kPoolBytes in all: past that the oldest are freed, so that sizes that no
// longer come do not hold the room.  device_trim gives them back, and all are
// freed when the device runs out of memory.  A block is handed out again only
// after the device has been synchronised since its release (one wait covers
// every block released before it), which is what freeing it waited for.  The
// wait is the one that hipFree performs, on a small block of its own:
// hipDeviceSynchronize would invalidate a stream capture in progress on another
// thread.
//
// Idle blocks are found by size, then age: a search passes at most the sizes
// within an eighth of the request's, however many blocks are idle (a closed
// batch of 256 scenes leaves thousands).
#include <map>
#include <mutex>
#include <tuple>
#include <unordered_map>
#include <vector>

#include "device_buffer.hpp"

namespace naga_amd {

namespace {

constexpr size_t kPoolBytes = size_t(4) << 30;

struct Block {
    void* p;
    size_t bytes;
    int device;
};

using Key = std::tuple<int, size_t, uint64_t>;  // device, bytes, release

struct Pool {
    std::mutex mu;
    std::map<Key, void*> idle;
    std::map<uint64_t, Key> by_age;  // the same blocks by release
    std::unordered_map<void*, Block> live;
    size_t idle_bytes = 0;
    uint64_t releases = 0;
    std::unordered_map<int, uint64_t> synced;  // per device: releases it has synchronised since

    // The smallest idle block for a request: at most an eighth larger.
    // ready: among those that no work can still use.
    std::map<Key, void*>::iterator find(size_t bytes, int device, bool ready) {
        const uint64_t upto = synced[device];
        auto it = idle.lower_bound(Key{device, bytes, 0});
        while (it != idle.end() && std::get<0>(it->first) == device &&
               std::get<1>(it->first) <= bytes + bytes / 8) {
            // the first of its size is the one released first
            if (!ready || std::get<2>(it->first) <= upto) return it;
            it = idle.lower_bound(Key{device, std::get<1>(it->first) + 1, 0});
        }
        return idle.end();
    }
    void* remove(std::map<Key, void*>::iterator it) {
        void* p = it->second;
        idle_bytes -= std::get<1>(it->first);
        by_age.erase(std::get<2>(it->first));
        idle.erase(it);
        return p;
    }
    void* take(std::map<Key, void*>::iterator it) {
        live.emplace(it->second, Block{it->second, std::get<1>(it->first), std::get<0>(it->first)});
        return remove(it);
    }
    // Takes the oldest idle blocks out until at most `keep` bytes are idle.
    void oldest_past(size_t keep, std::vector<void*>& out) {
        while (idle_bytes > keep) {
            out.push_back(nullptr);  // the room first: it may throw
            out.back() = remove(idle.find(by_age.begin()->second));
        }
    }
};

// never destroyed: buffers with static storage may outlive any other object
Pool& pool() {
    static Pool* p = new Pool;
    return *p;
}

void free_all(const std::vector<void*>& blocks) {
    for (void* p : blocks)
        if (p) (void)hipFree(p);  // waits for their work
}

}  // namespace

void* device_allocate(size_t bytes) {
    // whole units, so that equal scenes find each other's blocks
    const size_t unit = bytes >= (size_t(1) << 20) ? size_t(64) << 10 : 256;
    bytes = (bytes + unit - 1) / unit * unit;
    int device = 0;
    NAGA_HIP(hipGetDevice(&device));
    Pool& P = pool();
    {
        std::unique_lock<std::mutex> lk(P.mu);
        auto it = P.find(bytes, device, true);
        if (it != P.idle.end()) return P.take(it);
        if (P.find(bytes, device, false) != P.idle.end()) {
            const uint64_t upto = P.releases;
            lk.unlock();  // other threads go on while this one waits
            void* token = nullptr;
            const bool ok =
                hipMalloc(&token, 256) == hipSuccess && hipFree(token) == hipSuccess;
            if (!ok) (void)hipGetLastError();
            lk.lock();
            if (ok && P.synced[device] < upto) P.synced[device] = upto;
            it = P.find(bytes, device, true);
            if (it != P.idle.end()) return P.take(it);
        }
    }
    void* p = nullptr;
    hipError_t e = hipMalloc(&p, bytes);
    if (e == hipErrorOutOfMemory || e == hipErrorMemoryAllocation) {
        (void)hipGetLastError();
        device_trim(0);
        e = hipMalloc(&p, bytes);
    }
    NAGA_HIP(e);
    std::lock_guard<std::mutex> lk(P.mu);
    P.live.emplace(p, Block{p, bytes, device});
    return p;
}

void device_release(void* p) noexcept {
    Pool& P = pool();
    std::vector<void*> old;
    try {
        std::lock_guard<std::mutex> lk(P.mu);
        const auto it = P.live.find(p);
        if (it != P.live.end()) {
            const Block b = it->second;
            P.live.erase(it);
            if (b.bytes <= kPoolBytes) {
                P.oldest_past(kPoolBytes - b.bytes, old);
                const Key key{b.device, b.bytes, P.releases + 1};
                const auto aged = P.by_age.emplace(P.releases + 1, key).first;
                try {
                    P.idle.emplace(key, p);
                } catch (...) {
                    P.by_age.erase(aged);
                    throw;
                }
                ++P.releases;
                P.idle_bytes += b.bytes;
                p = nullptr;
            }
        }
    } catch (...) {  // no memory to keep it: free it
    }
    if (p) (void)hipFree(p);
    free_all(old);
}

size_t device_trim(size_t keep) {
    Pool& P = pool();
    std::vector<void*> old;
    size_t kept;
    {
        std::lock_guard<std::mutex> lk(P.mu);
        P.oldest_past(keep, old);
        kept = P.idle_bytes;
    }
    free_all(old);
    return kept;
}

}  // namespace naga_amd
