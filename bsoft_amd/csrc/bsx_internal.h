// bsx_internal.h — shared declarations of libbsx (HIP, gfx950).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>
#include <string>

#include "../../include/bsx.h"

namespace bsx {

// ---- error handling: thread-local last error, status codes, no throws ----
void set_error(const char* fmt, ...);
const char* last_error();

#define BSX_HIP(call)                                                                   \
    do {                                                                                \
        hipError_t _e = (call);                                                         \
        if (_e != hipSuccess) {                                                         \
            ::bsx::set_error("%s:%d %s: %s", __FILE__, __LINE__, #call,                 \
                             hipGetErrorString(_e));                                    \
            return BSX_ERR_DEVICE;                                                      \
        }                                                                               \
    } while (0)

#define BSX_REQUIRE(cond, code, ...)                                                    \
    do {                                                                                \
        if (!(cond)) {                                                                  \
            ::bsx::set_error(__VA_ARGS__);                                              \
            return (code);                                                              \
        }                                                                               \
    } while (0)

// ---- memory (bsx_mem.hip) ----
// Every device and pinned allocation of the library: where memory has run out, the
// workspaces below are given back before it fails.
hipError_t device_malloc(void** p, size_t bytes);
hipError_t pinned_malloc(void** p, size_t bytes);
template <class T> hipError_t device_malloc(T** p, size_t bytes) {
    return device_malloc((void**)p, bytes);
}
template <class T> hipError_t pinned_malloc(T** p, size_t bytes) {
    return pinned_malloc((void**)p, bytes);
}
// Frees the workspaces that no call is using; returns their number.
int release_workspaces();

// Workspaces of calls without a handle: a device (or pinned host) buffer for one
// call. Allocating and freeing on every call cost more than the kernels of small
// calls and stalled large ones for milliseconds, so a buffer that its call has
// finished with is kept for the next one: at most 16 buffers and 512 MB of each
// kind, the least recently used going first, all of them given back when an
// allocation of the library fails and by bsx_release_workspaces. release() says that the
// call's stream has been waited for, i.e. that nothing uses the buffer any more, so
// any thread may take it for any stream; a buffer that is destroyed without it
// (an error return) is freed once the device is idle.
class Scratch {
public:
    explicit Scratch(bool pinned = false) : pinned_(pinned) {}
    Scratch(const Scratch&) = delete;
    Scratch& operator=(const Scratch&) = delete;
    ~Scratch();
    hipError_t get(size_t bytes);
    void release();
    template <class T> T* as() const { return static_cast<T*>(p_); }

private:
    void* p_ = nullptr;
    size_t bytes_ = 0;
    int dev_ = 0;
    bool pinned_;
    bool idle_ = false;   // released
};

// ---- FFT launchers (bsx_fft.hip) ----
// Batched in-place C2C transform along one axis of a (nz, ny, nx) complex
// array, `batch` arrays of nx*ny*nz each. axis 0 = x, 1 = y, 2 = z.
// sign -1 forward, +1 backward. scale multiplies every output.
int fft_axis(float2* data, int nx, int ny, int nz, int64_t batch, int axis, int sign,
             float scale, hipStream_t s);
int fft_axis_ex(float2* data, float* real_out, int nx, int ny, int nz, int64_t batch, int axis,
                int sign, float scale, hipStream_t s);
int fft_real_x(const float* in, float2* out, int nx, long long nlines, int keep, hipStream_t s);
int fft_z_to_origin(float2* data, int n, float scale, const double origin[3], hipStream_t s);
bool fft_length_supported(int n);

// Per-particle transform stages (bsx_recon.hip).
struct PartRec;   // device record of one particle (see bsx_recon.hip)

// Twiddle table for length n, sign-independent: tw[a] = (cos 2pi a/n, sin 2pi a/n).
const float2* twiddles(int n, hipStream_t s);

}  // namespace bsx
