// bsx_extract.hip — the mirror of insertion and the quality measures:
//   3 axis FFTs (real input, phase shift with the last) : map transform
//       (Bimage::project prologue, src/img/Bimage_project.cpp:373-375)
//   k_extract        : central sections by FSI-kernel gather interpolation
//       (Bimage::central_section, Bimage_project.cpp:288-338;
//        Bimage::fspace_interpolate, Bimage_fspace.cpp:85-147;
//        FSI_Kernel, include/FSI_Kernel.h:28-68), centre shift as project()
//   k_fsc            : FP64 shell sums of Bimage::fsc (Bimage_resolution.cpp:330-406)
//   k_frc_pairs      : img_recip_space_fom, fom_type 0 (src/mg/mg_refine.cpp:660-781)
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <mutex>
#include <vector>

#include "bsx_common.h"

using namespace bsx;

// ------------------------------------------------------------- extraction
// 8 x 8 pixel tiles of a section, WPT wavefronts each. The tile samples a patch of
// a plane, so the taps of its 64 samples lie in a small box of the transform. A
// lane's taps are scattered over many cache lines, and a load instruction costs
// the texture path about a cycle per line it touches; with W^3 = 512 taps a
// sample, each voxel of the box is used about 10 times.
// WPT > 0: the box is loaded into LDS once (rows of 16 or 32 lanes), the taps are
// read from there in the order and precision of fsi_sample, and the wavefronts
// share the tap planes, whose sums are added in order. Where a box is beyond `cap`
// voxels (matrices that are no rotations) they read their planes from memory: 200
// sections of 128^2 by a matrix that stretches the plane twofold at W = 10 take 3.6 ms
// (3.7 with one thread a pixel, 16.1 with the tile sampled by one wavefront alone).
// WPT 0: narrow kernels (at W = 4 a voxel is used about twice) take the taps from
// memory, four tiles a workgroup with the kernel table in LDS.
// Whole calls with the map transform, 200 sections of 128^2, before (one thread a
// pixel of a row, taps from memory) and now: W = 3 322 / 183 us, 4 520 / 317,
// 5 803 / 337, 6 1,016 / 414, 8 1,989 / 699; 50 sections of 256^2: 589 / 282,
// 869 / 414, 1,234 / 415, 1,502 / 499, 2,845 / 830. LDS reads bound it at W = 8 (busy
// 71 %, 61 % of that conflicts: the lanes' taps start anywhere and meet in banks); when whole calls took
// 967 us with four wavefronts a tile there, they took 1,100 with one and 1,025 with two.
struct __attribute__((packed, aligned(4))) Float4u {
    float v[4];
};

// Row of the kernel table for a fraction, in 16-byte loads (each lane has a row of
// its own, so a load instruction costs one cache line per lane whatever its
// width).
template <int WD>
__device__ __forceinline__ void table_row(const float* __restrict__ ktab, double frac, float (&w)[WD]) {
    const float* r = ktab + ((int)(frac * FSI_NDIV + 0.5)) * WD;
#pragma unroll
    for (int q = 0; q + 4 <= WD; q += 4) {
        const Float4u f = *(const Float4u*)(r + q);
#pragma unroll
        for (int e = 0; e < 4; ++e) w[q + e] = f.v[e];
    }
#pragma unroll
    for (int q = WD / 4 * 4; q < WD; ++q) w[q] = r[q];
}

template <int WD, int WPT>
__global__ __launch_bounds__(WPT ? 64 * WPT : 256) __attribute__((amdgpu_waves_per_eu(WPT ? 4 : 1))) void k_extract(const float2* __restrict__ ft, int N,
                                                const double* __restrict__ mats, double inv,
                                                double rs, double maxs2, int center, int tiles,
                                                int nviews, int nblk, int cap, const float* __restrict__ ktab,
                                                float2* __restrict__ out) {
    constexpr int HW = (WD - 1) / 2;
    constexpr bool LDSBOX = WPT > 0;
    constexpr int PW = WPT ? (WD + WPT - 1) / WPT : WD;   // tap planes per wavefront
    extern __shared__ float2 box[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // hardware block b runs on XCD b % 8: each XCD takes a contiguous range of
    // (view, tile), so that the tiles of a section meet in one L2
    const int per_xcd = (nblk + 7) / 8;
    const int blk = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    if (blk >= nblk) return;
    // without LDS boxes a workgroup takes four tiles and holds the kernel table
    const float* K = ktab;
    if (!LDSBOX) {
        float* t = (float*)box;
        for (int i = threadIdx.x; i < (FSI_NDIV + 1) * WD; i += 256) t[i] = ktab[i];
        __syncthreads();
        K = t;
    }
    const int task = LDSBOX ? blk : blk * 4 + wave;
    const int v = task / (tiles * tiles), tile = task - v * tiles * tiles;
    if (v >= nviews) return;
    // tiles of the centred frequency plane (from -N/2 on), so that the 64
    // samples of a tile are one patch of the plane
    const int h = tile % tiles * 8 + (lane & 7) - N / 2;
    const int k = tile / tiles * 8 + (lane >> 3) - N / 2;
    const bool inside = h <= (N - 1) / 2 && k <= (N - 1) / 2;
    const double* M = mats + 9 * v;
    const double ivy = (double)k * inv, ivx = (double)h * inv;
    const double s2 = ivx * ivx + ivy * ivy;
    const bool band = inside && s2 <= maxs2;
    double m[3] = {0, 0, 0};
    for (int c = 0; c < 3; ++c) m[c] = (ivx * M[3 * c] + ivy * M[3 * c + 1] + 0.0 * M[3 * c + 2]) * rs;
    double vr = 0, vi = 0;
    if (LDSBOX) {
        if (__ballot(band)) {   // wavefront-uniform
            const double fl[3] = {floor(m[0]), floor(m[1]), floor(m[2])};
            // the coordinates are monotone in h and in k, so the tile's corners
            // (lanes 0, 7, 56, 63) bound the box; uniform values
            int lo[3], n[3];
            bool fits = true;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const int f = (int)fl[c] - HW;
                const int c0 = __builtin_amdgcn_readlane(f, 0), c1 = __builtin_amdgcn_readlane(f, 7);
                const int c2 = __builtin_amdgcn_readlane(f, 56), c3 = __builtin_amdgcn_readlane(f, 63);
                lo[c] = min(min(c0, c1), min(c2, c3));
                n[c] = max(max(c0, c1), max(c2, c3)) + WD - lo[c];
                fits = fits && n[c] <= 32 && lo[c] >= -N && lo[c] + n[c] <= N;   // one periodic wrap
            }
            const int sx = n[0] | 1;   // odd row stride: rows start in different banks
            fits = fits && sx * n[1] * n[2] <= cap;
            float pr[PW], pi[PW];   // sums over this wavefront's tap planes
#pragma unroll
            for (int q = 0; q < PW; ++q) pr[q] = pi[q] = 0.f;
            if (fits) {
                // this lane's kernel weights, in flight together with the box
                float wx[WD], wy[WD], wz[PW];
                table_row<WD>(ktab, m[0] - fl[0], wx);
                table_row<WD>(ktab, m[1] - fl[1], wy);
                const float* kz = ktab + ((int)((m[2] - fl[2]) * FSI_NDIV + 0.5)) * WD;
#pragma unroll
                for (int q = 0; q < PW; ++q) wz[q] = kz[min(wave * PW + q, WD - 1)];
                // lanes per row and rows per step; a lane keeps its RY row offsets
                // of a plane, the planes are uniform; two planes of loads in flight
                const int rl = n[0] <= 16 ? 16 : 32, per = 64 * WPT / rl;
                const int lx = threadIdx.x & (rl - 1), ly = threadIdx.x / rl;
                const bool on = lx < n[0];
                int jx = lo[0] + min(lx, n[0] - 1);
                jx += jx < 0 ? N : 0;
                constexpr int RY = WPT >= 4 ? 3 : 5;
                for (int y0 = 0; y0 < n[1]; y0 += RY * per) {
                    int off[RY];
#pragma unroll
                    for (int u = 0; u < RY; ++u) {
                        int jy = lo[1] + min(y0 + u * per + ly, n[1] - 1);   // past the end: reread
                        jy += jy < 0 ? N : 0;
                        off[u] = jy * N + jx;
                    }
                    for (int z = 0; z < n[2]; z += 2) {
                        int ja = lo[2] + z, jb = lo[2] + min(z + 1, n[2] - 1);
                        ja += ja < 0 ? N : 0;
                        jb += jb < 0 ? N : 0;
                        const float2* pa = ft + (size_t)ja * N * N;
                        const float2* pb = ft + (size_t)jb * N * N;
                        float2 va[RY], vb[RY];
#pragma unroll
                        for (int u = 0; u < RY; ++u) {
                            va[u] = pa[off[u]];
                            vb[u] = pb[off[u]];
                        }
                        float2* d = box + (z * n[1] + y0 + ly) * sx + lx;
#pragma unroll
                        for (int u = 0; u < RY; ++u)
                            if (on && y0 + u * per + ly < n[1]) {
                                d[u * per * sx] = va[u];
                                if (z + 1 < n[2]) d[(n[1] + u * per) * sx] = vb[u];
                            }
                    }
                }
                __syncthreads();
                if (band) {
                    const float2* t = box + (((int)fl[2] - HW - lo[2] + wave * PW) * n[1] + (int)fl[1] - HW - lo[1]) * sx +
                                      (int)fl[0] - HW - lo[0];
#pragma unroll
                    for (int q = 0; q < PW; ++q, t += n[1] * sx) {
                        if (wave * PW + q >= WD) break;
                        const float kzz = wz[q];
#pragma unroll
                        for (int y2 = 0; y2 < WD; ++y2) {
                            const float w = wy[y2] * kzz;
                            const float2* row = t + y2 * sx;
#pragma unroll
                            for (int e = 0; e < WD; ++e) {
                                const float kw = wx[e] * w;
                                const float2 a = row[e];
                                pr[q] = fmaf(a.x, kw, pr[q]);
                                pi[q] = fmaf(a.y, kw, pi[q]);
                            }
                        }
                    }
                }
            } else if (band) {
                // from memory, with one periodic wrap or more
                const float* kx = ktab + ((int)((m[0] - fl[0]) * FSI_NDIV + 0.5)) * WD;
                const float* ky = ktab + ((int)((m[1] - fl[1]) * FSI_NDIV + 0.5)) * WD;
                const float* kz = ktab + ((int)((m[2] - fl[2]) * FSI_NDIV + 0.5)) * WD;
                int jx[WD];
#pragma unroll
                for (int e = 0; e < WD; ++e) jx[e] = wrap_index((int)fl[0] - HW + e, N);
#pragma unroll
                for (int q = 0; q < PW; ++q) {
                    const int z2 = wave * PW + q;
                    if (z2 >= WD) break;
                    const float2* plane = ft + (size_t)wrap_index((int)fl[2] - HW + z2, N) * N * N;
                    const float kzz = kz[z2];
#pragma unroll 1
                    for (int y2 = 0; y2 < WD; ++y2) {
                        const float2* row = plane + (size_t)wrap_index((int)fl[1] - HW + y2, N) * N;
                        const float w = ky[y2] * kzz;
#pragma unroll
                        for (int e = 0; e < WD; ++e) {
                            const float kw = kx[e] * w;
                            const float2 a = row[jx[e]];
                            pr[q] = fmaf(a.x, kw, pr[q]);
                            pi[q] = fmaf(a.y, kw, pi[q]);
                        }
                    }
                }
            }
            // plane sums of every wavefront, added in the order of the planes
            __syncthreads();
            if (wave)
#pragma unroll
                for (int q = 0; q < PW; ++q) box[((wave - 1) * PW + q) * 64 + lane] = make_float2(pr[q], pi[q]);
            __syncthreads();
            if (wave) return;
#pragma unroll
            for (int q = 0; q < PW; ++q) {
                vr += pr[q];
                vi += pi[q];
            }
            for (int q = 0; q < WD - PW; ++q) {
                const float2 p = box[q * 64 + lane];
                vr += p.x;
                vi += p.y;
            }
        }
        if (wave) return;
    } else if (band) {
        fsi_sample<WD>(ft, N, m, K, vr, vi);
    }
    if (!inside) return;
    if (center) {
        // phase_shift_to_center of a 2D section: x (-1)^(h+k) for even N
        if ((N & 1) == 0) {
            if ((h + k) & 1) { vr = -vr; vi = -vi; }
        } else {
            const double t = -2 * M_PI * (double)(N / 2) / N;
            double sn, cs;
            sincos(h * t + k * t, &sn, &cs);
            const double a = vr, b = vi;
            vr = a * cs - b * sn;
            vi = a * sn + b * cs;
        }
    }
    out[((long long)v * N + (k < 0 ? k + N : k)) * N + (h < 0 ? h + N : h)] = make_float2((float)vr, (float)vi);
}

// -------------------------------------------------------------------- FSC
__global__ __launch_bounds__(256) void k_fsc(const float2* __restrict__ a,
                                             const float2* __restrict__ b, int N, long maxrad,
                                             double* __restrict__ sums) {
    extern __shared__ double sh[];   // 3 * maxrad
    for (long i = threadIdx.x; i < 3 * maxrad; i += blockDim.x) sh[i] = 0;
    __syncthreads();
    const long long n3 = (long long)N * N * N;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n3;
         i += (long long)gridDim.x * blockDim.x) {
        const long long xx = i % N, yy = (i / N) % N, zz = i / ((long long)N * N);
        const double h = xx > (N - 1) / 2 ? (double)(xx - N) : (double)xx;
        const double k = yy > (N - 1) / 2 ? (double)(yy - N) : (double)yy;
        const double l = zz > (N - 1) / 2 ? (double)(zz - N) : (double)zz;
        // radius = rad_scale*sqrt(rx^2+ry^2+rz^2), rx = h/(N pix): voxel units
        const double radius = sqrt(h * h + k * k + l * l);
        const long ir = (long)radius;
        if (ir >= maxrad) continue;
        const double f = radius - ir, f1 = 1 - f;
        const float2 u = a[i], v = b[i];
        const double p1 = (double)u.x * u.x + (double)u.y * u.y;
        const double p2 = (double)v.x * v.x + (double)v.y * v.y;
        const double re = (double)u.x * v.x + (double)u.y * v.y;
        atomicAdd(&sh[ir], f1 * p1);
        atomicAdd(&sh[maxrad + ir], f1 * p2);
        atomicAdd(&sh[2 * maxrad + ir], f1 * re);
        if (ir + 1 < maxrad) {
            atomicAdd(&sh[ir + 1], f * p1);
            atomicAdd(&sh[maxrad + ir + 1], f * p2);
            atomicAdd(&sh[2 * maxrad + ir + 1], f * re);
        }
    }
    __syncthreads();
    for (long i = threadIdx.x; i < 3 * maxrad; i += blockDim.x)
        if (sh[i] != 0) atomicAdd(&sums[i], sh[i]);
}

// FP64 shell sums of Bimage::fsc_dpr (Bimage_resolution.cpp:93-181) for two
// real maps transformed separately (the same F1, F2 as unpacking the packed
// transform): over x < N/2 (all that a and b hold), linear interpolation between
// shells i and i+1 (both must exist), sums[c * maxrad + i] for c = |F1|^2,
// |F2|^2, Re F1 conj F2, (|F1|^2 + |F2|^2) dphi^2 (the sum of the first two
// weighs the last). The phase difference is the angle of F2 conj F1; where one
// value is zero, that of the other. The LDS adds bound it (neighbouring lanes
// share shells): 103 us at 256^3 (131 us with five sums, two phase angles and
// whole transforms).
__global__ __launch_bounds__(256) void k_fsc_dpr(const float2* __restrict__ a,
                                                 const float2* __restrict__ b, int N, int nz,
                                                 double inv_ratio, int maxrad,
                                                 double* __restrict__ sums) {
    extern __shared__ double sh[];   // 4 * maxrad
    for (int i = threadIdx.x; i < 4 * maxrad; i += blockDim.x) sh[i] = 0;
    __syncthreads();
    const unsigned hx = N / 2;
    const long long nv = (long long)hx * N * nz;   // nz = 1: a 2D image
    for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < nv;
         t += (long long)gridDim.x * blockDim.x) {
        const unsigned yz = (unsigned)(t / hx);
        const int xx = (int)(t - (long long)yz * hx), yy = (int)(yz % (unsigned)N), zz = (int)(yz / (unsigned)N);
        const double h = xx;
        const double k = yy > (N - 1) / 2 ? (double)(yy - N) : (double)yy;
        const double l = zz > (nz - 1) / 2 ? (double)(zz - nz) : (double)zz;
        const double radius = inv_ratio * sqrt(h * h + k * k + l * l);
        if (!(radius < maxrad - 1)) continue;
        const int ir = (int)radius;
        const double f = radius - ir, f1 = 1 - f;
        const float2 u = a[t], v = b[t];
        const double I1 = (double)u.x * u.x + (double)u.y * u.y;
        const double I2 = (double)v.x * v.x + (double)v.y * v.y;
        const double re = (double)u.x * v.x + (double)u.y * v.y;
        double dphi;
        if (I1 > 0 && I2 > 0) {
            dphi = atan2((double)u.y * v.x - (double)u.x * v.y, re);
        } else {
            dphi = atan2((double)u.y, (double)u.x) - atan2((double)v.y, (double)v.x);
        }
        const double val[4] = {I1, I2, re, (I1 + I2) * (dphi * dphi)};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            atomicAdd(&sh[c * maxrad + ir], f1 * val[c]);
            atomicAdd(&sh[c * maxrad + ir + 1], f * val[c]);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 4 * maxrad; i += blockDim.x)
        if (sh[i] != 0) atomicAdd(&sums[i], sh[i]);
}

// ------------------------------------------------------------ FRC scoring
// One workgroup per (particle, reference) pair. Ring sums in LDS (FP64).
__global__ __launch_bounds__(256) void k_frc_pairs(const float2* __restrict__ part,
                                                   const float2* __restrict__ ref, int N,
                                                   const int* __restrict__ pairs,
                                                   double min_rad_sq, double max_rad_cv_sq,
                                                   double max_rad, double max_rad_cv,
                                                   double* __restrict__ out,
                                                   double* __restrict__ out_cv) {
    extern __shared__ double rs[];   // 3 * N
    double* fom = rs;
    double* dsum = rs + N;
    double* msum = rs + 2 * N;
    for (int i = threadIdx.x; i < 3 * N; i += blockDim.x) rs[i] = 0;
    __syncthreads();
    const int ip = pairs[2 * blockIdx.x], ir = pairs[2 * blockIdx.x + 1];
    const long long np = (long long)N * N;
    const float2* P = part + (long long)ip * np;
    const float2* R = ref + (long long)ir * np;
    const int hx = (N - 1) / 2;
    for (long long i = threadIdx.x; i < np; i += blockDim.x) {
        const int xx = (int)(i % N), yy = (int)(i / N);
        const double ix = xx > hx ? (double)xx - N : (double)xx;
        const double iy = yy > hx ? (double)yy - N : (double)yy;
        const double d2 = ix * ix + iy * iy;
        if (d2 >= min_rad_sq && d2 <= max_rad_cv_sq) {
            const int j = (int)sqrt(d2);
            if (j >= N) continue;
            const float2 d = P[i], r = R[i];
            atomicAdd(&fom[j], (double)d.x * r.x + (double)d.y * r.y);
            atomicAdd(&msum[j], (double)r.x * r.x + (double)r.y * r.y);
            atomicAdd(&dsum[j], (double)d.x * d.x + (double)d.y * d.y);
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double f = 0, wsum = 0, cv = 0;
        for (int j = 0; j < max_rad && j < N; ++j) {
            wsum += 1;
            const double den = dsum[j] * msum[j];
            if (den > 0) f += fom[j] / sqrt(den);
        }
        f = wsum > 0 ? f / wsum : 0;
        wsum = 0;
        for (int j = (int)max_rad; j < max_rad_cv && j < N; ++j) {
            wsum += 1;
            const double den = dsum[j] * msum[j];
            if (den > 0) cv += fom[j] / sqrt(den);
        }
        out[blockIdx.x] = f;
        if (out_cv) out_cv[blockIdx.x] = wsum > 0 ? cv / wsum : 0;
    }
}

// ================================================================ C-ABI
static double check_res(double res, int n, double sampling, int ndim) {
    if (res > n * sampling) return n * sampling;
    double rm = 2 / sqrt(ndim / (sampling * sampling));
    return res < rm ? rm : res;
}

extern "C" {

int bsx_map_transform(const float* map_dev, int n, const double origin[3], float* ft_dev,
                      void* stream) {
    BSX_REQUIRE(map_dev && ft_dev && origin, BSX_ERR_ARG, "bsx_map_transform: null argument");
    BSX_REQUIRE(fft_length_supported(n), BSX_ERR_ARG, "bsx_map_transform: size %d unsupported", n);
    hipStream_t s = (hipStream_t)stream;
    const long long n3 = (long long)n * n * n;
    float2* v = (float2*)ft_dev;
    const float sc = (float)(1.0 / sqrt((double)n3));
    int r = fft_real_x(map_dev, v, n, (long long)n * n, n, s);
    if (r == BSX_OK) r = fft_axis_ex(v, nullptr, n, n, n, 1, 1, -1, 1.0f, s);
    if (r == BSX_OK) r = fft_z_to_origin(v, n, sc, origin, s);
    return r;
}

// Argument checks shared by bsx_extract and bsx_extract_noalloc; normalises
// width, sampling and resolution as the reference's defaults do.
static int extract_args(const float* ft_dev, int n, double& sampling, const double* mats,
                        int64_t nviews, double& resolution, int& kernel_width, int kernel_power,
                        const float* out_dev, const char* who) {
    BSX_REQUIRE(ft_dev && mats && out_dev, BSX_ERR_ARG, "%s: null argument", who);
    BSX_REQUIRE(n >= 2 && nviews >= 0 && nviews < 65536, BSX_ERR_ARG,
                "%s: n %d / nviews %lld out of range", who, n, (long long)nviews);
    if (kernel_power < 0) kernel_width = 1;
    BSX_REQUIRE(kernel_width >= 1 && kernel_width <= 10, BSX_ERR_ARG,
                "%s: kernel width %d out of range 1..10", who, kernel_width);
    if (sampling < 1e-10) sampling = 1;
    if (resolution < 1e-10) resolution = sampling;
    for (int64_t i = 0; i < 9 * nviews; ++i)
        BSX_REQUIRE(std::isfinite(mats[i]) && fabs(mats[i]) <= 1.0 + 1e-9, BSX_ERR_ARG,
                    "%s: matrix %lld is not a rotation", who, (long long)(i / 9));
    return BSX_OK;
}

// Launches k_extract<width> over nviews sections; dtab / dmats are device
// copies of the kernel table and the view matrices.
static int extract_launch(const float* ft_dev, int n, double sampling, const double* dmats,
                          int64_t nviews, double resolution, int kernel_width, int center,
                          const float* dtab, float* out_dev, hipStream_t s) {
    const double inv = 1.0 / (n * sampling), rs = n * sampling;
    const double maxs2 = 1.0 / (resolution * resolution);
    const int tiles = (n + 7) / 8;
    const float2* ft = (const float2*)ft_dev;
    // a launch takes fewer than 2^32 threads; at most 2^23 tiles of up to 256 each
    // go into one, so that any number of views is accepted
    const int64_t per = std::max<int64_t>(1, (1ll << 23) / ((int64_t)tiles * tiles));
    for (int64_t v0 = 0; v0 < nviews; v0 += per) {
        const int nv = (int)std::min(per, nviews - v0);
        const int ntile = tiles * tiles * nv;
        const double* m = dmats + 9 * v0;
        float2* out = (float2*)out_dev + v0 * n * n;
        switch (kernel_width) {
// LDS boxes from width 5 on (see k_extract); cap holds the boxes of 8 x 8 patches of
// rotations: the largest of 10^7 random ones at W = 8 had 4,590 voxels, cap is 4,654
// (37 KB, four workgroups per CU); 1 to 2 % above the largest at the other widths
#define BSX_EXT(W) case W: { \
            constexpr int WPT = W >= 8 ? 4 : W >= 5 ? 2 : 0; \
            constexpr int cap = WPT ? (W + 10) * (W + 9) * (W + 7) + 64 : 0; \
            constexpr size_t lds = WPT ? sizeof(float2) * cap : sizeof(float) * (FSI_NDIV + 1) * W; \
            const int nblk = WPT ? ntile : (ntile + 3) / 4; \
            hipLaunchKernelGGL((k_extract<W, WPT>), dim3((unsigned)((nblk + 7) / 8 * 8)), dim3(WPT ? 64 * WPT : 256), \
                               lds, s, ft, n, m, inv, rs, maxs2, center, tiles, nv, nblk, cap, dtab, out); \
            break; }
            BSX_EXT(1) BSX_EXT(2) BSX_EXT(3) BSX_EXT(4) BSX_EXT(5)
            BSX_EXT(6) BSX_EXT(7) BSX_EXT(8) BSX_EXT(9) BSX_EXT(10)
#undef BSX_EXT
        }
        BSX_HIP(hipGetLastError());
    }
    return BSX_OK;
}

int bsx_extract(const float* ft_dev, int n, double sampling, const double* mats, int64_t nviews,
                double resolution, int kernel_width, int kernel_power, int center, float* out_dev,
                void* stream) {
    int r = extract_args(ft_dev, n, sampling, mats, nviews, resolution, kernel_width,
                         kernel_power, out_dev, "bsx_extract");
    if (r != BSX_OK || nviews == 0) return r;
    hipStream_t s = (hipStream_t)stream;
    const std::vector<float>& tab = fsi_table_kept(kernel_width, kernel_power);
    // matrices, then the kernel table: one copy from pinned memory
    const size_t nm = sizeof(double) * 9 * nviews, nt = sizeof(float) * tab.size();
    Scratch dev, pin(true);
    BSX_HIP(dev.get(nm + nt));
    BSX_HIP(pin.get(nm + nt));
    memcpy(pin.as<char>(), mats, nm);
    memcpy(pin.as<char>() + nm, tab.data(), nt);
    BSX_HIP(hipMemcpyAsync(dev.as<char>(), pin.as<char>(), nm + nt, hipMemcpyHostToDevice, s));
    r = extract_launch(ft_dev, n, sampling, dev.as<double>(), nviews, resolution, kernel_width, center,
                       (const float*)(dev.as<char>() + nm), out_dev, s);
    BSX_HIP(hipStreamSynchronize(s));
    dev.release();
    pin.release();
    return r;
}

// ---------------------------------------------- allocation-free extraction
// Scratch of bsx_extract_noalloc: the view matrices (FP64, at most
// BSX_NOALLOC_MAX_VIEWS) followed by the FSI kernel table (at most width 10).
// One copy per GPU, held until the process ends. In host code `scratch` is
// only a symbol: its device address comes from hipGetSymbolAddress, once per
// device, and only that address is handed to copies and kernels.
constexpr size_t kScratchMats = sizeof(double) * 9 * BSX_NOALLOC_MAX_VIEWS;
constexpr size_t kScratchTab = sizeof(float) * (FSI_NDIV + 1) * 10;
static __device__ __align__(256) unsigned char scratch[kScratchMats + kScratchTab];

constexpr int kMaxDevices = 64;
static std::mutex scratch_mu;
static void* scratch_ptr[kMaxDevices];

// Device address of the current device's scratch (looked up on the first
// call on that device).
static int scratch_address(void** out) {
    int dev = 0;
    BSX_HIP(hipGetDevice(&dev));
    BSX_REQUIRE(dev >= 0 && dev < kMaxDevices, BSX_ERR_DEVICE, "device %d out of range", dev);
    std::lock_guard<std::mutex> g(scratch_mu);
    if (!scratch_ptr[dev]) {
        void* p = nullptr;
        BSX_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        scratch_ptr[dev] = p;
    }
    *out = scratch_ptr[dev];
    return BSX_OK;
}

int bsx_extract_noalloc(const float* ft_dev, int n, double sampling, const double* mats,
                        int64_t nviews, double resolution, int kernel_width, int kernel_power,
                        int center, float* out_dev, void* stream) {
    int r = extract_args(ft_dev, n, sampling, mats, nviews, resolution, kernel_width,
                         kernel_power, out_dev, "bsx_extract_noalloc");
    if (r != BSX_OK) return r;
    BSX_REQUIRE(nviews <= BSX_NOALLOC_MAX_VIEWS, BSX_ERR_ARG,
                "bsx_extract_noalloc: %lld views exceed the scratch capacity of %d",
                (long long)nviews, BSX_NOALLOC_MAX_VIEWS);
    if (nviews == 0) return BSX_OK;
    void* base = nullptr;
    r = scratch_address(&base);
    if (r != BSX_OK) return r;
    double* dmats = (double*)base;
    float* dtab = (float*)((unsigned char*)base + kScratchMats);
    // the kernel table on the host stack (no heap), then both into scratch
    float tab[(FSI_NDIV + 1) * 10];
    fsi_table_into(tab, kernel_width, kernel_power);
    const size_t ntab = (size_t)(FSI_NDIV + 1) * (kernel_power < 0 ? 1 : kernel_width);
    hipStream_t s = (hipStream_t)stream;
    BSX_HIP(hipMemcpyAsync(dtab, tab, sizeof(float) * ntab, hipMemcpyHostToDevice, s));
    BSX_HIP(hipMemcpyAsync(dmats, mats, sizeof(double) * 9 * nviews, hipMemcpyHostToDevice, s));
    r = extract_launch(ft_dev, n, sampling, dmats, nviews, resolution, kernel_width, center, dtab,
                       out_dev, s);
    if (r != BSX_OK) return r;
    // the host copies above read `tab` and `mats`: wait before returning
    BSX_HIP(hipStreamSynchronize(s));
    return BSX_OK;
}

int bsx_fsc(const float* a_dev, const float* b_dev, int n, double sampling, double hi_res,
            double* fsc, int* nshell, void* stream) {
    BSX_REQUIRE(a_dev && b_dev && fsc && nshell, BSX_ERR_ARG, "bsx_fsc: null argument");
    BSX_REQUIRE(n >= 2 && sampling > 0, BSX_ERR_ARG, "bsx_fsc: bad size/sampling");
    hipStream_t s = (hipStream_t)stream;
    hi_res = check_res(hi_res, n, sampling, 3);
    long maxrad = (long)(n * sampling / hi_res);
    BSX_REQUIRE(maxrad <= *nshell, BSX_ERR_ARG, "bsx_fsc: %ld shells exceed capacity %d", maxrad,
                *nshell);
    Scratch buf;
    BSX_HIP(buf.get(sizeof(double) * 3 * (maxrad + 1)));
    double* d = buf.as<double>();
    BSX_HIP(hipMemsetAsync(d, 0, sizeof(double) * 3 * (maxrad + 1), s));
    hipLaunchKernelGGL(k_fsc, dim3(1024), dim3(256), sizeof(double) * 3 * maxrad, s,
                       (const float2*)a_dev, (const float2*)b_dev, n, maxrad, d);
    hipError_t le = hipGetLastError();
    std::vector<double> h(3 * maxrad);
    if (maxrad > 0)
        BSX_HIP(hipMemcpyAsync(h.data(), d, sizeof(double) * 3 * maxrad, hipMemcpyDeviceToHost, s));
    BSX_HIP(hipStreamSynchronize(s));
    buf.release();
    BSX_HIP(le);
    for (long i = 0; i < maxrad; ++i) {
        double den = h[i] * h[maxrad + i];
        fsc[i] = den > 0 ? h[2 * maxrad + i] / sqrt(den) : 0;
    }
    if (maxrad > 0) fsc[0] = 1;
    *nshell = (int)maxrad;
    return BSX_OK;
}

// n x n x nz maps, nz = n (3D) or 1 (2D images).
static int fsc_dpr_impl(const float* map1_dev, const float* map2_dev, int n, int nz,
                        double sampling, double hi_res, double sampling_ratio, double* curves,
                        int* nrows, void* stream) {
    BSX_REQUIRE(map1_dev && map2_dev && curves && nrows, BSX_ERR_ARG, "bsx_fsc_dpr: null argument");
    BSX_REQUIRE(n >= 2 && n % 2 == 0 && sampling > 0, BSX_ERR_ARG, "bsx_fsc_dpr: bad size/sampling");
    if (sampling_ratio <= 0) sampling_ratio = 1;
    hipStream_t s = (hipStream_t)stream;
    hi_res = check_res(hi_res, n, sampling, nz > 1 ? 3 : 2);
    const double rad_scale = n * sampling / sampling_ratio;
    const long maxrad = (long)(2 + rad_scale / hi_res);
    BSX_REQUIRE(maxrad <= *nrows, BSX_ERR_ARG, "bsx_fsc_dpr: %ld rows exceed capacity %d", maxrad,
                *nrows);
    const long long n3 = (long long)(n / 2) * n * nz;   // a transform's kept half
    Scratch vols, sums;
    if (vols.get(sizeof(float2) * 2 * n3) != hipSuccess || sums.get(sizeof(double) * 4 * maxrad) != hipSuccess) {
        set_error("bsx_fsc_dpr: allocation failed");
        return BSX_ERR_NOMEM;
    }
    float2* v = vols.as<float2>();
    double* d = sums.as<double>();
    int r = BSX_OK;
    // the sums read x < n / 2 only: the x pass keeps that half, the other passes
    // transform both halves' columns in one launch each
    for (int m = 0; m < 2 && r == BSX_OK; ++m)
        r = fft_real_x(m ? map2_dev : map1_dev, v + m * n3, n, (long long)n * nz, n / 2, s);
    for (int axis = 1; axis < (nz > 1 ? 3 : 2) && r == BSX_OK; ++axis)
        r = fft_axis_ex(v, nullptr, n / 2, n, nz, 2, axis, -1, 1.0f, s);
    if (r == BSX_OK) {
        (void)hipMemsetAsync(d, 0, sizeof(double) * 4 * maxrad, s);
        hipLaunchKernelGGL(k_fsc_dpr, dim3(1024), dim3(256), sizeof(double) * 4 * maxrad, s, v,
                           v + n3, n, nz, 1.0 / sampling_ratio, (int)maxrad, d);
        if (hipGetLastError() != hipSuccess) r = BSX_ERR_DEVICE;
    }
    std::vector<double> h(4 * maxrad);
    if (r == BSX_OK &&
        (hipMemcpyAsync(h.data(), d, sizeof(double) * 4 * maxrad, hipMemcpyDeviceToHost, s) !=
             hipSuccess ||
         hipStreamSynchronize(s) != hipSuccess))
        r = BSX_ERR_DEVICE;
    if (r) {
        set_error("bsx_fsc_dpr: device error");
        return r;
    }
    vols.release();
    sums.release();
    // curves: (s, FSC, DPR in degrees) per row (Bimage_resolution.cpp:225-239)
    for (long i = 0; i < maxrad; ++i) {
        double fsc = h[2 * maxrad + i], dpr = 0;
        if (i == 0) {
            fsc = 1;
        } else {
            const double f12 = h[i] * h[maxrad + i];
            if (f12 > 1e-30) fsc /= sqrt(f12);
            fsc = std::min(1.0, std::max(-1.0, fsc));
            const double fs = h[i] + h[maxrad + i];
            dpr = fs > 1e-30 ? sqrt(h[3 * maxrad + i] / fs) * 180.0 / M_PI : 0;
        }
        curves[3 * i] = i / rad_scale;
        curves[3 * i + 1] = fsc;
        curves[3 * i + 2] = dpr;
    }
    *nrows = (int)maxrad;
    return BSX_OK;
}

int bsx_fsc_dpr(const float* map1_dev, const float* map2_dev, int n, double sampling,
                double hi_res, double sampling_ratio, double* curves, int* nrows, void* stream) {
    return fsc_dpr_impl(map1_dev, map2_dev, n, n, sampling, hi_res, sampling_ratio, curves, nrows,
                        stream);
}

int bsx_fsc_dpr_2d(const float* img1_dev, const float* img2_dev, int n, double sampling,
                   double hi_res, double sampling_ratio, double* curves, int* nrows,
                   void* stream) {
    return fsc_dpr_impl(img1_dev, img2_dev, n, 1, sampling, hi_res, sampling_ratio, curves, nrows,
                        stream);
}

int bsx_score_frc(const float* part_dev, int64_t nparts, const float* ref_dev, int64_t nrefs,
                  int n, double sampling, double hi_res, double lo_res, const int32_t* pairs,
                  int64_t npairs, double* out, void* stream) {
    BSX_REQUIRE(part_dev && ref_dev && pairs && out, BSX_ERR_ARG, "bsx_score_frc: null argument");
    BSX_REQUIRE(n >= 2 && npairs >= 0, BSX_ERR_ARG, "bsx_score_frc: bad sizes");
    if (npairs == 0) return BSX_OK;
    for (int64_t i = 0; i < npairs; ++i)
        BSX_REQUIRE(pairs[2 * i] >= 0 && pairs[2 * i] < nparts && pairs[2 * i + 1] >= 0 &&
                        pairs[2 * i + 1] < nrefs,
                    BSX_ERR_ARG, "bsx_score_frc: pair %lld (%d, %d) out of range", (long long)i,
                    pairs[2 * i], pairs[2 * i + 1]);
    hipStream_t s = (hipStream_t)stream;
    if (lo_res > 0 && hi_res > lo_res) std::swap(hi_res, lo_res);
    hi_res = check_res(hi_res, n, sampling, 2);
    double max_rad = n * sampling / hi_res;
    double max_rad_cv = 1.1 * max_rad;
    if (max_rad_cv <= max_rad) max_rad_cv = max_rad + 1;
    double min_rad_sq = 0;
    if (lo_res > 0) { min_rad_sq = n * sampling / lo_res; min_rad_sq *= min_rad_sq; }
    Scratch bp, bo;
    BSX_HIP(bp.get(sizeof(int) * 2 * npairs));
    BSX_HIP(bo.get(sizeof(double) * npairs));
    int* dp = bp.as<int>();
    double* dout = bo.as<double>();
    BSX_HIP(hipMemcpyAsync(dp, pairs, sizeof(int) * 2 * npairs, hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(k_frc_pairs, dim3((unsigned)npairs), dim3(256), sizeof(double) * 3 * n, s,
                       (const float2*)part_dev, (const float2*)ref_dev, n, dp, min_rad_sq,
                       max_rad_cv * max_rad_cv, max_rad, max_rad_cv, dout, (double*)nullptr);
    hipError_t le = hipGetLastError();
    BSX_HIP(hipMemcpyAsync(out, dout, sizeof(double) * npairs, hipMemcpyDeviceToHost, s));
    BSX_HIP(hipStreamSynchronize(s));
    bp.release();
    bo.release();
    BSX_HIP(le);
    return BSX_OK;
}

}  // extern "C"
