// The library's memory code (bsx_mem.hip) over an allocator of 1,000 MB that hands
// out addresses only: kept workspaces, their bounds, and their return where
// memory runs out. Prints "ok" and returns 0, or names the check that failed.
#include <atomic>
#include <cstdio>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

#include "bsx_internal.h"

static std::mutex mu;
static std::map<void*, size_t> live[2];   // device, pinned
static size_t used[2], calls;
static std::atomic<int> waits{0};   // for the device
static char* next_address = (char*)0x1000;
static const size_t MB = 1u << 20, CAPACITY = 1000 * MB;

static hipError_t take(int kind, void** p, size_t bytes) {
    std::lock_guard<std::mutex> g(mu);
    ++calls;
    if (used[kind] + bytes > CAPACITY) return hipErrorOutOfMemory;
    used[kind] += bytes;
    *p = next_address;
    next_address += 4096;
    live[kind][*p] = bytes;
    return hipSuccess;
}
static hipError_t give(int kind, void* p) {
    std::lock_guard<std::mutex> g(mu);
    auto it = live[kind].find(p);
    if (it == live[kind].end()) {
        printf("freed twice or never allocated\n");
        exit(1);
    }
    used[kind] -= it->second;
    live[kind].erase(it);
    return hipSuccess;
}
extern "C" {
hipError_t hipMalloc(void** p, size_t bytes) { return take(0, p, bytes); }
hipError_t hipFree(void* p) { return give(0, p); }
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) { return take(1, p, bytes); }
hipError_t hipHostFree(void* p) { return give(1, p); }
hipError_t hipGetDevice(int* dev) { *dev = 0; return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { ++waits; return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return ""; }
}
namespace bsx {
void set_error(const char*, ...) {}
}

#define CHECK(c)                                        \
    do {                                                \
        if (!(c)) {                                     \
            printf("line %d: %s\n", __LINE__, #c);      \
            return 1;                                   \
        }                                               \
    } while (0)

using bsx::Scratch;

int main() {
    void* first = nullptr;
    for (int pinned = 0; pinned < 2; ++pinned) {
        {
            Scratch a(pinned);
            CHECK(a.get(100 * MB) == hipSuccess);
            first = a.as<void>();
            a.release();
        }
        const size_t before = calls;
        {
            Scratch a(pinned);   // the kept one again
            CHECK(a.get(90 * MB) == hipSuccess && a.as<void>() == first && calls == before);
            a.release();
        }
        {
            Scratch a(pinned);   // far too large for this: another
            CHECK(a.get(1 * MB) == hipSuccess && a.as<void>() != first);
        }                        // not released: freed
        CHECK(used[pinned] == 100 * MB);
        // a buffer that its call has not released may be in use by the device
        const int seen = waits;
        {
            Scratch a(pinned);
            CHECK(a.get(600 * MB) == hipSuccess);
        }
        CHECK(waits == seen + 1);
        {
            Scratch a(pinned);   // released, but too large to keep
            CHECK(a.get(600 * MB) == hipSuccess);
            a.release();
        }
        CHECK(waits == seen + 1 && used[pinned] == 100 * MB);
    }
    // an allocation that does not fit beside the kept buffers takes their place
    void* p = nullptr;
    CHECK(bsx::device_malloc(&p, 950 * MB) == hipSuccess && p && used[0] == 950 * MB && used[1] == 0);
    void* q = (void*)1;
    CHECK(bsx::device_malloc(&q, 100 * MB) == hipErrorOutOfMemory && q == nullptr);
    {
        Scratch a;
        CHECK(a.get(100 * MB) == hipErrorOutOfMemory && a.as<void>() == nullptr);
    }
    hipFree(p);
    {
        Scratch a(true);
        CHECK(a.get(400 * MB) == hipSuccess);
        a.release();
    }
    CHECK(bsx::pinned_malloc(&p, 900 * MB) == hipSuccess && used[1] == 900 * MB);
    hipHostFree(p);
    // bounds: 16 buffers, 512 MB, none larger
    {
        std::vector<Scratch*> v;
        for (int i = 0; i < 40; ++i) {
            v.push_back(new Scratch);
            CHECK(v.back()->get(MB + i) == hipSuccess);
        }
        for (Scratch* s : v) {
            s->release();
            delete s;
        }
        CHECK(live[0].size() == 16);
    }
    for (int i = 0; i < 5; ++i) {
        Scratch a, b;
        CHECK(a.get((200 + 10 * i) * MB) == hipSuccess && b.get(150 * MB) == hipSuccess);
        a.release();
        b.release();
        CHECK(used[0] <= 512 * MB);
    }
    {
        Scratch a;
        CHECK(a.get(600 * MB) == hipSuccess);
        a.release();
    }
    CHECK(used[0] <= 512 * MB && used[0] > 0);
    CHECK(bsx_release_workspaces() == BSX_OK && used[0] == 0 && used[1] == 0);
    // threads that share the store
    std::atomic<int> bad{0};
    std::mutex held_mu;
    std::map<void*, int> held;
    std::vector<std::thread> ts;
    for (int t = 0; t < 8; ++t)
        ts.emplace_back([&, t] {
            for (int i = 0; i < 2000; ++i) {
                Scratch a(i & 1);
                if (a.get(MB * (1 + (t * 7 + i) % 40)) != hipSuccess) continue;
                {
                    std::lock_guard<std::mutex> g(held_mu);
                    if (held[a.as<void>()]++) ++bad;   // in use by two calls
                }
                if (i % 50 == 0) bsx_release_workspaces();
                {
                    std::lock_guard<std::mutex> g(held_mu);
                    held[a.as<void>()]--;
                }
                if (i % 3) a.release();
            }
        });
    for (auto& t : ts) t.join();
    CHECK(bad == 0);
    bsx_release_workspaces();
    CHECK(live[0].empty() && live[1].empty());
    printf("ok\n");
    return 0;
}
