// The kept device blocks (naga_amd/csrc/device_pool.cpp) against a counting
// allocator in place of the device's: pool_main <check>.
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <set>
#include <thread>
#include <vector>

#include "device_buffer.hpp"

using naga_amd::device_allocate;
using naga_amd::device_release;
using naga_amd::device_trim;

namespace {
std::mutex mu;
std::map<void*, size_t> held;  // what the fake device has given out
size_t in_use = 0, capacity = size_t(64) << 30;
int mallocs = 0, frees = 0;
std::atomic<uint64_t> waits{0};  // hipFree calls: each waits for the device
uintptr_t next = 1 << 20;

#define CHECK(x)                                                  \
    do {                                                          \
        if (!(x)) {                                               \
            std::printf("%s:%d: %s\n", __FILE__, __LINE__, #x);   \
            std::exit(1);                                         \
        }                                                         \
    } while (0)
constexpr size_t MiB = size_t(1) << 20, GiB = size_t(1) << 30;
}  // namespace

hipError_t hipMalloc(void** p, size_t bytes) {
    std::lock_guard<std::mutex> lk(mu);
    if (in_use + bytes > capacity) return hipErrorOutOfMemory;
    *p = reinterpret_cast<void*>(next);
    next += (bytes + 255) / 256 * 256;
    held[*p] = bytes;
    in_use += bytes;
    ++mallocs;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    std::lock_guard<std::mutex> lk(mu);
    const auto it = held.find(p);
    CHECK(it != held.end());
    in_use -= it->second;
    held.erase(it);
    ++frees;
    ++waits;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) {
    return hipSuccess;
}

// Sizes that do not come back make room for those that do.
void eviction() {
    std::vector<void*> v;
    for (int i = 0; i < 80; ++i) v.push_back(device_allocate((64 + 9 * size_t(i)) * MiB));
    for (int i = 0; i < 4096; ++i) v.push_back(device_allocate(MiB));
    for (void* p : v) device_release(p);  // 37 GiB in 81 sizes
    CHECK(in_use <= 4 * GiB);
    void* a = device_allocate(3 * MiB);
    device_release(a);
    const int before = mallocs;
    void* b = device_allocate(3 * MiB);  // kept, though 4 GiB were idle
    CHECK(b == a && mallocs <= before + 1);  // (one small block to wait on)
    device_release(b);
    CHECK(in_use <= 4 * GiB);
    void* big = device_allocate(5 * GiB);  // more than is ever kept
    device_release(big);
    CHECK(in_use <= 4 * GiB);
}

// Blocks are handed out again only after a wait, and one wait serves all.
void waiting() {
    std::vector<void*> v;
    for (int i = 0; i < 10; ++i) v.push_back(device_allocate(2 * MiB));
    for (void* p : v) device_release(p);
    const uint64_t w = waits;
    std::set<void*> again;
    for (int i = 0; i < 10; ++i) again.insert(device_allocate(2 * MiB));
    CHECK(again == std::set<void*>(v.begin(), v.end()));
    CHECK(waits == w + 1);
}

void trimming() {
    std::vector<void*> v;
    for (int i = 0; i < 8; ++i) v.push_back(device_allocate(128 * MiB));
    void* live = device_allocate(MiB);
    for (void* p : v) device_release(p);
    CHECK(device_trim(2 * GiB) == GiB);
    CHECK(device_trim(300 * MiB) == 256 * MiB && in_use == 257 * MiB);
    CHECK(held.count(v[7]) && held.count(v[6]));  // the oldest went first
    CHECK(device_trim(0) == 0 && in_use == MiB && held.count(live));
    device_release(live);
}

// When the device has no more, what is idle is given back first.
void exhaustion() {
    capacity = GiB;
    device_release(device_allocate(600 * MiB));
    void* p = device_allocate(900 * MiB);
    CHECK(p && in_use == 900 * MiB);
    bool failed = false;
    try {
        device_allocate(200 * MiB);
    } catch (const naga_amd::Error& e) {
        failed = e.status == naga_amd::kOutOfMemory;
    }
    CHECK(failed);
    device_release(p);
}

// Opening again what was closed takes time in proportion to its blocks.
double reopen(int n) {
    std::vector<void*> v(static_cast<size_t>(n));
    auto size = [](int i) { return size_t(1 + i * 37 % 400) * 256; };
    for (int i = 0; i < n; ++i) v[size_t(i)] = device_allocate(size(i));
    for (void* p : v) device_release(p);
    const auto t0 = std::chrono::steady_clock::now();
    for (int i = 0; i < n; ++i) v[size_t(i)] = device_allocate(size(i));
    const double t =
        std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    for (void* p : v) device_release(p);
    device_trim(0);
    return t;
}
void many_blocks() {
    reopen(2000);
    const double few = reopen(2000), many = reopen(60000);
    std::printf("%g %g\n", few, many);
    CHECK(many < 250 * few);  // 30 times the blocks; by scans of them all 900
}

// No block has two holders, whatever threads do.
void threads() {
    std::mutex m;
    std::set<void*> mine;
    auto drop = [&](std::vector<void*>& v) {
        {
            std::lock_guard<std::mutex> lk(m);
            mine.erase(v.back());
        }
        device_release(v.back());
        v.pop_back();
    };
    auto work = [&](int seed) {
        unsigned r = unsigned(seed);
        std::vector<void*> v;
        for (int i = 0; i < 20000; ++i) {
            r = r * 1664525u + 1013904223u;
            if (v.size() < 20 && (r >> 8) % 2) {
                void* p = device_allocate(size_t(1 + (r >> 16) % 64) * MiB);
                std::lock_guard<std::mutex> lk(m);
                CHECK(mine.insert(p).second);
                v.push_back(p);
            } else if (!v.empty()) {
                drop(v);
            }
            if ((r >> 20) % 512 == 0) device_trim(GiB);
        }
        while (!v.empty()) drop(v);
    };
    std::vector<std::thread> t;
    for (int i = 0; i < 8; ++i) t.emplace_back(work, i);
    for (auto& x : t) x.join();
    CHECK(in_use <= 4 * GiB);
    device_trim(0);
    CHECK(in_use == 0 && held.empty());
}

int main(int argc, char** argv) {
    const std::map<std::string, void (*)()> checks = {
        {"eviction", eviction},     {"waiting", waiting},         {"trimming", trimming},
        {"exhaustion", exhaustion}, {"many_blocks", many_blocks}, {"threads", threads}};
    checks.at(argv[1])();
    std::puts("ok");
}
