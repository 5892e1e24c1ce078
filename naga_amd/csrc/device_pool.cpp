// Device memory blocks kept between allocations.
//
// A scene's set-up and its end allocate and free about a hundred buffers.
// hipMalloc and hipFree map and unmap their pages each time and hipFree waits
// for the device: closing a 132,651-node D3Q27 scene took 4.5 ms and its
// set-up's temporaries as much again, where the set-up's kernels take 5.
// Released blocks of up to kPoolBytes in all are kept for later allocations
// of about their size; the rest is freed at once, and all of it when the
// device runs out of memory.  A block is handed out again only after the
// device has been synchronised since its release (one wait covers every block
// released before it), which is what freeing it waited for.  The wait is the
// one that hipFree performs, on a small block of its own: hipDeviceSynchronize
// would invalidate a stream capture in progress on another thread.
#include <mutex>
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
    uint64_t released;  // position among all releases
};

struct Pool {
    std::mutex mu;
    std::vector<Block> idle;
    std::unordered_map<void*, Block> live;
    size_t idle_bytes = 0;
    uint64_t releases = 0;
    std::unordered_map<int, uint64_t> synced;  // per device: releases it has synchronised since

    // The smallest idle block for a request: at most an eighth larger.
    // ready: among those that no work can still use.
    int find(size_t bytes, int device, bool ready) {
        const uint64_t upto = synced[device];
        int best = -1;
        for (size_t i = 0; i < idle.size(); ++i) {
            const Block& b = idle[i];
            if (b.device != device || b.bytes < bytes || b.bytes > bytes + bytes / 8) continue;
            if (ready && b.released > upto) continue;
            if (best < 0 || b.bytes < idle[size_t(best)].bytes) best = int(i);
        }
        return best;
    }
    void* take(int i) {
        const Block b = idle[size_t(i)];
        idle[size_t(i)] = idle.back();
        idle.pop_back();
        idle_bytes -= b.bytes;
        live.emplace(b.p, b);
        return b.p;
    }
};

// never destroyed: buffers with static storage may outlive any other object
Pool& pool() {
    static Pool* p = new Pool;
    return *p;
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
        int i = P.find(bytes, device, true);
        if (i >= 0) return P.take(i);
        if (P.find(bytes, device, false) >= 0) {
            const uint64_t upto = P.releases;
            lk.unlock();  // other threads go on while this one waits
            void* token = nullptr;
            const bool ok =
                hipMalloc(&token, 256) == hipSuccess && hipFree(token) == hipSuccess;
            if (!ok) (void)hipGetLastError();
            lk.lock();
            if (ok && P.synced[device] < upto) P.synced[device] = upto;
            i = P.find(bytes, device, true);
            if (i >= 0) return P.take(i);
        }
    }
    void* p = nullptr;
    hipError_t e = hipMalloc(&p, bytes);
    if (e == hipErrorOutOfMemory || e == hipErrorMemoryAllocation) {
        (void)hipGetLastError();
        std::vector<Block> all;
        {
            std::lock_guard<std::mutex> lk(P.mu);
            all.swap(P.idle);
            P.idle_bytes = 0;
        }
        for (const Block& b : all) (void)hipFree(b.p);  // waits for their work
        e = hipMalloc(&p, bytes);
    }
    NAGA_HIP(e);
    std::lock_guard<std::mutex> lk(P.mu);
    P.live.emplace(p, Block{p, bytes, device, 0});
    return p;
}

void device_release(void* p) noexcept {
    Pool& P = pool();
    try {
        std::lock_guard<std::mutex> lk(P.mu);
        const auto it = P.live.find(p);
        if (it != P.live.end()) {
            Block b = it->second;
            P.live.erase(it);
            if (P.idle_bytes + b.bytes <= kPoolBytes) {
                b.released = ++P.releases;
                P.idle.push_back(b);
                P.idle_bytes += b.bytes;
                return;
            }
        }
    } catch (...) {  // no memory to keep it: free it
    }
    (void)hipFree(p);
}

}  // namespace naga_amd
