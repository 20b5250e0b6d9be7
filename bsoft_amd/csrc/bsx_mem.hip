// bsx_mem.hip — every allocation of the library, and the workspaces that calls
// without a handle keep between them (host code only).
#include <mutex>

#include "bsx_internal.h"

namespace bsx {

namespace {
constexpr size_t MOST = 512u << 20;   // bytes kept of a kind (device, pinned host)
constexpr int COUNT = 16;             // buffers kept of a kind

struct Kept {
    void* p;
    size_t bytes;
    int dev;
    bool pinned;
    uint64_t used;
};
// a fixed table: release() cannot fail, whatever the state of the heap
std::mutex kept_mu;
Kept kept[2 * COUNT + 1];
int nkept = 0;
uint64_t kept_clock = 0;

void buffer_free(void* p, bool pinned) {
    if (pinned) (void)hipHostFree(p);
    else (void)hipFree(p);
}

hipError_t allocate(void** p, size_t bytes, bool pinned) {
    *p = nullptr;
    return pinned ? hipHostMalloc(p, bytes, hipHostMallocDefault) : hipMalloc(p, bytes);
}

hipError_t allocate_or_empty(void** p, size_t bytes, bool pinned) {
    hipError_t e = allocate(p, bytes, pinned);
    if (e == hipErrorOutOfMemory && release_workspaces() > 0) {
        (void)hipGetLastError();
        e = allocate(p, bytes, pinned);
    }
    if (e != hipSuccess) *p = nullptr;
    return e;
}
}  // namespace

hipError_t device_malloc(void** p, size_t bytes) { return allocate_or_empty(p, bytes, false); }
hipError_t pinned_malloc(void** p, size_t bytes) { return allocate_or_empty(p, bytes, true); }

int release_workspaces() {
    Kept all[2 * COUNT + 1];
    int n;
    {
        std::lock_guard<std::mutex> g(kept_mu);
        n = nkept;
        for (int i = 0; i < n; ++i) all[i] = kept[i];
        nkept = 0;
    }
    for (int i = 0; i < n; ++i) buffer_free(all[i].p, all[i].pinned);
    return n;
}

hipError_t Scratch::get(size_t bytes) {
    const hipError_t e = hipGetDevice(&dev_);
    if (e != hipSuccess) return e;
    bytes = (bytes + 255) / 256 * 256;
    {
        // the smallest kept buffer that fits and is not far too large
        std::lock_guard<std::mutex> g(kept_mu);
        int at = -1;
        for (int i = 0; i < nkept; ++i)
            if (kept[i].dev == dev_ && kept[i].pinned == pinned_ && kept[i].bytes >= bytes &&
                kept[i].bytes <= 4 * bytes + (1 << 20) && (at < 0 || kept[i].bytes < kept[at].bytes))
                at = i;
        if (at >= 0) {
            p_ = kept[at].p;
            bytes_ = kept[at].bytes;
            kept[at] = kept[--nkept];
            return hipSuccess;
        }
    }
    bytes_ = bytes;
    return allocate_or_empty(&p_, bytes, pinned_);
}

void Scratch::release() {
    idle_ = true;
    if (!p_ || bytes_ > MOST) return;   // freed by the destructor
    Kept out[COUNT + 1];
    int nout = 0;
    {
        std::lock_guard<std::mutex> g(kept_mu);
        kept[nkept++] = Kept{p_, bytes_, dev_, pinned_, ++kept_clock};
        p_ = nullptr;
        for (;;) {
            size_t sum = 0;
            int n = 0, at = -1;
            for (int i = 0; i < nkept; ++i) {
                if (kept[i].pinned != pinned_) continue;
                sum += kept[i].bytes;
                ++n;
                if (at < 0 || kept[i].used < kept[at].used) at = i;
            }
            if (sum <= MOST && n <= COUNT) break;
            out[nout++] = kept[at];
            kept[at] = kept[--nkept];
        }
    }
    for (int i = 0; i < nout; ++i) buffer_free(out[i].p, out[i].pinned);
}

Scratch::~Scratch() {
    if (!p_) return;
    if (!idle_) (void)hipDeviceSynchronize();   // freeing pinned memory need not wait for copies from it
    buffer_free(p_, pinned_);
}

}  // namespace bsx

extern "C" int bsx_release_workspaces(void) {
    bsx::release_workspaces();
    return BSX_OK;
}
