// bsx_fft.hip — batched C2C transforms along one axis (x, y or z) of complex
// arrays, built from the in-LDS Stockham line FFT in bsx_fft_dev.h.
//
// Replaces fft_setup_plan / fftw (src/util/fft.cpp:31-114) for the volume
// transforms of the finish (fft_back, Bimage.h:903-908) and of the map
// transform used for projection (Bimage_project.cpp:373).
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <map>
#include <mutex>
#include <vector>

#include "bsx_fft_dev.h"
#include "bsx_internal.h"

namespace bsx {

// ------------------------------------------------------------------ errors
static thread_local char g_err[1024] = "no error";

void set_error(const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
}
const char* last_error() { return g_err; }

// ---------------------------------------------------------------- twiddles
const float2* twiddles(int n, hipStream_t s) {
    static std::mutex mu;
    static std::map<std::pair<int, int>, float2*> cache;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    std::lock_guard<std::mutex> g(mu);
    auto key = std::make_pair(dev, n);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
    std::vector<float2> h(n);
    for (int a = 0; a < n; ++a) {
        double ang = 2.0 * M_PI * (double)a / (double)n;
        h[a] = make_float2((float)cos(ang), (float)sin(ang));
    }
    float2* d = nullptr;
    if (device_malloc(&d, sizeof(float2) * n) != hipSuccess) return nullptr;
    if (hipMemcpyAsync(d, h.data(), sizeof(float2) * n, hipMemcpyHostToDevice, s) != hipSuccess)
        return nullptr;
    if (hipStreamSynchronize(s) != hipSuccess) return nullptr;
    cache[key] = d;
    return d;
}

bool fft_length_supported(int n) {
    switch (n) {
        case 16: case 32: case 64: case 128: case 256: case 512:
        case 24: case 48: case 96: case 192: case 384:
            return true;
        default:
            return false;
    }
}

// ------------------------------------------------------------ axis kernels
// Both kernels hold B lines in padded LDS lines, one value further apart than
// their size, so that neither the passes nor the transposed accesses of the
// strided axes meet in one bank. They are bound by memory: a 256^3 pass takes
// 45 us (x) and 43 us (y, z), 6 TB/s; with plain lines and a 64-bit division per
// element it took 56 and 78 us.
template <int L> constexpr int fft_pitch = line_size<L> + 1;

// x axis: a workgroup's lines are contiguous in memory. RIN: the input is real
// (`real_in`, the same lines); the first `keep` values of a line (L: all) go to
// `data`, lines `keep` apart (in place unless RIN or keep < L).
template <int L, int S, int B, bool RIN>
__global__ __launch_bounds__(256) void k_fft_x(const float* __restrict__ real_in, float2* data,
                                               float* __restrict__ real_out, long long nlines, int keep,
                                               float scale, const float2* __restrict__ twg) {
    constexpr int T = FftThreads<L>::value, G = 256 / T, NT = G * T, LP = fft_pitch<L>;
    constexpr int E = B * L / NT;   // values per thread
    static_assert(B % G == 0 && E * NT == B * L, "whole lines per group, whole values per thread");
    __shared__ float2 lds[B * LP + L];
    float2* tw = lds + B * LP;
    const int tid = threadIdx.x;
    for (int i = tid; i < L; i += NT) tw[i] = twg[i];
    const long long line0 = (long long)blockIdx.x * B, left = (nlines - line0) * L;
    float2 v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int idx = tid + e * NT;
        v[e] = make_float2(0.f, 0.f);
        if (idx < left) {
            if (RIN) v[e].x = real_in[line0 * L + idx];
            else v[e] = data[line0 * L + idx];
        }
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int idx = tid + e * NT, l = idx / L, i = idx - l * L;
        lds[l * LP + line_at<true>(i)] = v[e];
    }
    __syncthreads();
    const int g = tid / T, t = tid % T;
#pragma unroll 1
    for (int r0 = 0; r0 < B; r0 += G) FftLine<L, S, T, true>::run(lds + (r0 + g) * LP, tw, t);
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int idx = tid + e * NT, l = idx / L, i = idx - l * L;
        if (idx >= left || i >= keep) continue;
        const float2 z = lds[l * LP + line_at<true>(i)];
        const long long at = (line0 + l) * keep + i;
        if (real_out) real_out[at] = z.x * scale;
        else data[at] = make_float2(z.x * scale, z.y * scale);
    }
}

// phase_shift_to_origin (Bimage_complex.cpp:490-543) of a cubic map's
// transform: x e^{i phi}, phi = h sx + (l sz + k sy), s = origin / size 2 pi.
struct FftPhase {
    double sx, sy, sz;
};

// y or z axis: element i of line q at (q / inner) outer + q % inner + i stride;
// consecutive lanes take consecutive lines. If real_out is set, the real part
// goes there instead of updating `data`. PH (z axis of a cube): the phase shift.
template <int L, int S, int B, bool PH>
__global__ __launch_bounds__(256) void k_fft_s(float2* __restrict__ data, float* __restrict__ real_out,
                                               long long nlines, long long inner, long long outer,
                                               long long stride, float scale,
                                               const float2* __restrict__ twg, FftPhase ph) {
    constexpr int T = FftThreads<L>::value, G = 256 / T, NT = G * T, LP = fft_pitch<L>;
    static_assert(B % G == 0 && NT % B == 0, "whole lines per group, one line per thread");
    constexpr int D = NT / B, E = L / D;   // elements a step, values per thread
    static_assert(E * D == L, "whole values per thread");
    __shared__ float2 lds[B * LP + L];
    float2* tw = lds + B * LP;
    const int tid = threadIdx.x;
    for (int i = tid; i < L; i += NT) tw[i] = twg[i];
    const int l = tid % B, i0 = tid / B;
    const long long line = (long long)blockIdx.x * B + l;
    const bool ok = line < nlines;
    const long long hi = ok ? line / inner : 0, lo = ok ? line - hi * inner : 0;
    float2* src = data + hi * outer + lo;
    float2 v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = ok ? src[(i0 + e * D) * stride] : make_float2(0.f, 0.f);
#pragma unroll
    for (int e = 0; e < E; ++e) lds[l * LP + line_at<true>(i0 + e * D)] = v[e];
    __syncthreads();
    const int g = tid / T, t = tid % T;
#pragma unroll 1
    for (int r0 = 0; r0 < B; r0 += G) FftLine<L, S, T, true>::run(lds + (r0 + g) * LP, tw, t);
    if (!ok) return;
    double pxy = 0, ky = 0;
    if (PH) {
        const int x = (int)(lo % L), y = (int)(lo / L);
        pxy = (x > (L - 1) / 2 ? x - L : x) * ph.sx;
        ky = (y > (L - 1) / 2 ? y - L : y) * ph.sy;
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int i = i0 + e * D;
        float2 z = lds[l * LP + line_at<true>(i)];
        z.x *= scale;
        z.y *= scale;
        if (PH) {
            const double phi = pxy + ((i > (L - 1) / 2 ? i - L : i) * ph.sz + ky);
            double sn, cs;
            sincos(phi, &sn, &cs);
            z = make_float2((float)(z.x * cs - z.y * sn), (float)(z.x * sn + z.y * cs));
        }
        if (real_out) real_out[hi * outer + lo + i * stride] = z.x;
        else src[i * stride] = z;
    }
}

// Lines per workgroup of a strided axis: a multiple of the line groups that
// divides the threads, at least 16 (128-byte runs).
template <int L> constexpr int strided_lines() {
    constexpr int G = 256 / FftThreads<L>::value, NT = G * FftThreads<L>::value;
    int b = G;
    while (b < 16 || NT % b) b += G;
    return b;
}

template <int L, int S>
static int launch_axis(const float* real_in, float2* data, float* real_out, long long nlines,
                       long long inner, long long outer, long long stride, int keep, float scale,
                       const FftPhase* ph, hipStream_t s) {
    constexpr int T = FftThreads<L>::value;
    constexpr int G = 256 / T;
    constexpr int NT = G * T;
    const float2* tw = twiddles(L, s);
    BSX_REQUIRE(tw != nullptr, BSX_ERR_DEVICE, "twiddle table allocation failed for L=%d", L);
    constexpr int B = strided_lines<L>();
    const dim3 gx((unsigned)((nlines + G - 1) / G)), gs((unsigned)((nlines + B - 1) / B));
    if (stride == 1 && real_in)
        hipLaunchKernelGGL((k_fft_x<L, S, G, true>), gx, dim3(NT), 0, s, real_in, data, real_out, nlines,
                           keep, scale, tw);
    else if (stride == 1)
        hipLaunchKernelGGL((k_fft_x<L, S, G, false>), gx, dim3(NT), 0, s, (const float*)nullptr, data,
                           real_out, nlines, L, scale, tw);
    else if (ph)
        hipLaunchKernelGGL((k_fft_s<L, S, B, true>), gs, dim3(NT), 0, s, data, real_out, nlines, inner,
                           outer, stride, scale, tw, *ph);
    else
        hipLaunchKernelGGL((k_fft_s<L, S, B, false>), gs, dim3(NT), 0, s, data, real_out, nlines, inner,
                           outer, stride, scale, tw, FftPhase{0, 0, 0});
    BSX_HIP(hipGetLastError());
    return BSX_OK;
}

template <int S>
static int dispatch_axis(int L, const float* real_in, float2* data, float* real_out, long long nlines,
                         long long inner, long long outer, long long stride, int keep, float scale,
                         const FftPhase* ph, hipStream_t s) {
    switch (L) {
#define BSX_AXIS(LEN) case LEN: return launch_axis<LEN, S>(real_in, data, real_out, nlines, inner, outer, \
                                                           stride, keep, scale, ph, s);
        BSX_AXIS(16) BSX_AXIS(32) BSX_AXIS(64) BSX_AXIS(128) BSX_AXIS(256) BSX_AXIS(512)
        BSX_AXIS(24) BSX_AXIS(48) BSX_AXIS(96) BSX_AXIS(192) BSX_AXIS(384)
#undef BSX_AXIS
        default:
            set_error("FFT length %d not supported (16..512 powers of 2, 3*2^k to 384)", L);
            return BSX_ERR_ARG;
    }
}

static int axis_any(float2* data, float* real_out, int nx, int ny, int nz, int64_t batch, int axis,
                    int sign, float scale, const FftPhase* ph, hipStream_t s) {
    long long nxy = (long long)nx * ny, n3 = nxy * nz;
    long long L, nlines, inner, outer, stride;
    if (axis == 0) { L = nx; nlines = n3 / nx * batch; inner = 1; outer = nx; stride = 1; }
    else if (axis == 1) { L = ny; nlines = (long long)nx * nz * batch; inner = nx; outer = nxy; stride = nx; }
    else { L = nz; nlines = nxy * batch; inner = nxy; outer = n3; stride = nxy; }
    if (L == 1) return BSX_OK;
    // a strided axis of a one-wide array is contiguous
    auto go = sign < 0 ? dispatch_axis<-1> : dispatch_axis<+1>;
    return go((int)L, nullptr, data, real_out, nlines, inner, outer, stride, (int)L, scale, ph, s);
}

// Public launcher used by the finish and map-transform paths.
int fft_axis_ex(float2* data, float* real_out, int nx, int ny, int nz, int64_t batch, int axis,
                int sign, float scale, hipStream_t s) {
    return axis_any(data, real_out, nx, ny, nz, batch, axis, sign, scale, nullptr, s);
}

// Forward transform of the `nlines` real lines of nx values at `in`; the first
// `keep` frequencies of each go to `out`, lines `keep` apart.
int fft_real_x(const float* in, float2* out, int nx, long long nlines, int keep, hipStream_t s) {
    return dispatch_axis<-1>(nx, in, out, nullptr, nlines, 1, nx, 1, keep, 1.0f, nullptr, s);
}

// Forward transform of an n^3 map along z, x scale, moved to `origin` (voxels).
int fft_z_to_origin(float2* data, int n, float scale, const double origin[3], hipStream_t s) {
    const FftPhase ph{origin[0] / n * 2 * M_PI, origin[1] / n * 2 * M_PI, origin[2] / n * 2 * M_PI};
    return axis_any(data, nullptr, n, n, n, 1, 2, -1, scale, &ph, s);
}

int fft_axis(float2* data, int nx, int ny, int nz, int64_t batch, int axis, int sign, float scale,
             hipStream_t s) {
    return fft_axis_ex(data, nullptr, nx, ny, nz, batch, axis, sign, scale, s);
}

}  // namespace bsx

using namespace bsx;

extern "C" int bsx_fft(float* data_dev, int nx, int ny, int nz, int64_t batch, int dir, int norm,
                       void* stream) {
    BSX_REQUIRE(data_dev != nullptr, BSX_ERR_ARG, "bsx_fft: null data");
    BSX_REQUIRE(nx >= 1 && ny >= 1 && nz >= 1 && batch >= 1, BSX_ERR_ARG, "bsx_fft: bad sizes");
    BSX_REQUIRE((nx == 1 || fft_length_supported(nx)) && (ny == 1 || fft_length_supported(ny)) &&
                    (nz == 1 || fft_length_supported(nz)),
                BSX_ERR_ARG, "bsx_fft: unsupported length %dx%dx%d", nx, ny, nz);
    BSX_REQUIRE(dir == -1 || dir == 1, BSX_ERR_ARG, "bsx_fft: dir must be -1 or +1");
    hipStream_t s = (hipStream_t)stream;
    double n = (double)nx * ny * nz;
    double sc = norm == 1 ? 1.0 / sqrt(n) : norm == 2 ? 1.0 / n : 1.0;
    float2* d = (float2*)data_dev;
    int axes[3] = {0, 1, 2};
    int last = nz > 1 ? 2 : ny > 1 ? 1 : 0;
    for (int a : axes) {
        int L = a == 0 ? nx : a == 1 ? ny : nz;
        if (L == 1) continue;
        int r = fft_axis(d, nx, ny, nz, batch, a, dir, a == last ? (float)sc : 1.0f, s);
        if (r != BSX_OK) return r;
    }
    return BSX_OK;
}

extern "C" const char* bsx_last_error(void) { return bsx::last_error(); }
