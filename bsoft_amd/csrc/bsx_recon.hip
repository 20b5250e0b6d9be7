// bsx_recon.hip — Fourier-space reconstruction on gfx950.
//
// Per batch of particles (the per-particle loop of particle_reconstruct,
// src/mg/mg_reconstruct.cpp:143-229):
//   K1 k_background  background mean outside the inscribed ellipse
//                    (Bimage::calculate_background, Bimage_background.cpp:27-89)
//   K2 k_rows        pad with the background + x-direction FFT of the padded
//                    ft x ft image (Bimage::pad, Bimage_resize.cpp:347 and the
//                    first half of Bimage::fft, Bimage_fft.cpp:176-234). Two
//                    real rows share one complex FFT; only the half spectrum
//                    x = 0..ft/2 is kept, written transposed (x-major).
//   K3 k_cols_insert y-direction FFT of each kept column, x 1/ft, DC background
//                    term, phase shift to origin (Bimage_complex.cpp:490-543),
//                    CTF (mg_ctf.cpp:46-110, 661-676) and insertion of the
//                    column and of its Friedel mate into the FP32 volume
//                    accumulators (Bimage::fspace_pack_2D and
//                    fspace_2D_interpolate, Bimage_reconstruct.cpp:25-174).
// Finish (img_reconstruction_sum_weigh, mg_reconstruct.cpp:266-361):
//   K4 k_weigh_pairs sum of half sets, FP64 weighing, SNR FOM, centre shift
//   K5 3 axis FFTs   inverse 3D transform, x 1/sqrt(N^3), real part.
#include <cmath>
#include <algorithm>
#include <cstring>
#include <vector>
#include <cctype>
#include <climits>
#include <string>

#include "bsx_insert.h"

// ------------------------------------------------------------------- K1
// Block-wide sums of 256 threads (FP64 and int).
__device__ __forceinline__ void block_sum256(double& a, double& b, int& c, int& d) {
    __shared__ double sa[256], sb[256];
    __shared__ int sc[256], sd[256];
    sa[threadIdx.x] = a;
    sb[threadIdx.x] = b;
    sc[threadIdx.x] = c;
    sd[threadIdx.x] = d;
    __syncthreads();
    for (int o = blockDim.x / 2; o > 0; o >>= 1) {
        if (threadIdx.x < o) {
            sa[threadIdx.x] += sa[threadIdx.x + o];
            sb[threadIdx.x] += sb[threadIdx.x + o];
            sc[threadIdx.x] += sc[threadIdx.x + o];
            sd[threadIdx.x] |= sd[threadIdx.x + o];
        }
        __syncthreads();
    }
    a = sa[0];
    b = sb[0];
    c = sc[0];
    d = sd[0];
    __syncthreads();
}

// One workgroup per particle record: the background (mean of the pixels
// outside the inscribed ellipse about the image-header origin,
// Bimage::calculate_background, Bimage_background.cpp:27-89). With `resc`
// (breconstruct -rescale, flags bit 1) the image is first rescaled to
// average 0 and standard deviation 1 (rescale_to_avg_std(0, 1),
// mg_reconstruct.cpp:160; statistics as Bimage::statistics,
// Bimage_stats.cpp:104-148: FP64 sums, population deviation): the
// (scale, shift) pair is stored in resc[p] and the background is that of
// the rescaled FP32 pixels.
__global__ __launch_bounds__(256) void k_background(const float* __restrict__ imgs,
                                                    const PartDev* __restrict__ recs, int box,
                                                    float* __restrict__ bkg,
                                                    int* __restrict__ nonfinite,
                                                    double2* __restrict__ resc) {
    const int p = blockIdx.x;
    const float* img = imgs + (size_t)recs[p].src * box * box;
    const double ox = recs[p].hox, oy = recs[p].hoy;
    const long hx = box / 2, hy = box / 2;
    const int npix = box * box;
    // squared normalised distances per column and per row (the same FP64
    // operations as a per-pixel evaluation, computed once)
    __shared__ double cx2[1024], ry2[1024];
    for (int i = threadIdx.x; i < box; i += blockDim.x) {
        double x2 = (i - ox) / hx;
        cx2[i] = x2 * x2;
        double y2 = (i - oy) / hy;
        ry2[i] = y2 * y2;
    }
    double2 r = make_double2(1.0, 0.0);
    int bad = 0;
    // boxes of a multiple of 4 pixels: each thread reads 4 fixed columns
    // of every R-th row with one 16-byte load
    const int q = box / 4;
    const bool vec = (box & 3) == 0 && q <= (int)blockDim.x && ((uintptr_t)img & 15) == 0;
    const int R = vec ? (int)blockDim.x / q : 0;
    const int xq = vec ? (int)threadIdx.x % q : 0, yr = vec ? (int)threadIdx.x / q : 0;
    if (resc) {
        double s1 = 0, s2 = 0;
        int unused = 0;
        if (vec) {
            for (int y = yr; yr < R && y < box; y += R) {
                const float4 v4 = *reinterpret_cast<const float4*>(img + (size_t)y * box + 4 * xq);
                const float vv[4] = {v4.x, v4.y, v4.z, v4.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const double v = vv[e];
                    if (!isfinite(v)) bad = 1;
                    s1 += v;
                    s2 += v * v;
                }
            }
        } else {
            for (int i = threadIdx.x; i < npix; i += blockDim.x) {
                const double v = img[i];
                if (!isfinite(v)) bad = 1;
                s1 += v;
                s2 += v * v;
            }
        }
        block_sum256(s1, s2, unused, bad);
        const double avg = s1 / npix;
        double var = s2 / npix - avg * avg;
        const double sd = var > 0 ? sqrt(var) : 0.0;
        r.x = sd > 1e-30 ? 1.0 / sd : 1.0;
        r.y = 0.0 - avg * r.x;
        if (threadIdx.x == 0) resc[p] = r;
    }
    __syncthreads();
    double sum = 0, dummy = 0;
    int cnt = 0;
    if (vec) {
        const double c[4] = {cx2[4 * xq], cx2[4 * xq + 1], cx2[4 * xq + 2], cx2[4 * xq + 3]};
        for (int y = yr; yr < R && y < box; y += R) {
            const float4 v4 = *reinterpret_cast<const float4*>(img + (size_t)y * box + 4 * xq);
            const float vv[4] = {v4.x, v4.y, v4.z, v4.w};
            const double ry = ry2[y];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float v = vv[e];
                if (!isfinite(v)) bad = 1;
                if (resc) v = rescaled(v, r);
                if (c[e] + ry - 1 > 0) { sum += v; ++cnt; }
            }
        }
    } else {
        int yy = (int)threadIdx.x / box, xx = (int)threadIdx.x - yy * box;
        const int step_y = (int)blockDim.x / box, step_x = (int)blockDim.x - step_y * box;
        for (int i = threadIdx.x; i < npix; i += blockDim.x) {
            float v = img[i];
            if (!isfinite(v)) bad = 1;
            if (resc) v = rescaled(v, r);
            if (cx2[xx] + ry2[yy] - 1 > 0) { sum += v; ++cnt; }
            xx += step_x;
            yy += step_y;
            if (xx >= box) { xx -= box; ++yy; }
        }
    }
    block_sum256(sum, dummy, cnt, bad);
    if (threadIdx.x == 0) {
        bkg[p] = cnt ? (float)(sum / cnt) : 0.0f;
        if (bad && nonfinite) atomicOr(nonfinite, 1);
    }
}

// Per-bin piece offsets (one workgroup): poff[b] = sum over bins below b of
// ceil(binned / PIECE), poff[nbins] = all pieces, pbin[piece] = its bin (at
// most maxpieces pieces are listed); `total` accumulates the entries binned
// since the last reset. Positions past the chunk table (maxc chunks) went to
// the atomic fallback and are not binned.
__global__ __launch_bounds__(1024) void k_piece_scan(const int* __restrict__ fill, int nbins,
                                                     int maxc, int piece, int* __restrict__ poff,
                                                     int* __restrict__ pbin, int maxpieces,
                                                     unsigned long long* __restrict__ total) {
    __shared__ int ppart[1024];
    __shared__ unsigned long long epart[1024];
    const int tid = threadIdx.x;
    const int per = (nbins + 1023) / 1024;   // bins per thread
    const int b0 = tid * per, b1 = min(nbins, b0 + per);
    const int cap = maxc * BSX_CHUNK;
    int psum = 0;
    unsigned long long esum = 0;
    for (int i = b0; i < b1; ++i) {
        const int f = min(fill[i], cap);
        psum += (f + piece - 1) / piece;
        esum += (unsigned)f;
    }
    ppart[tid] = psum;
    epart[tid] = esum;
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {
        const int pv = tid >= o ? ppart[tid - o] : 0;
        __syncthreads();
        ppart[tid] += pv;
        __syncthreads();
    }
    int prun = ppart[tid] - psum;
    for (int i = b0; i < b1; ++i) {
        poff[i] = prun;
        const int np = (min(fill[i], cap) + piece - 1) / piece;
        for (int q = 0; q < np && prun + q < maxpieces; ++q) pbin[prun + q] = i;
        prun += np;
    }
    for (int o = 512; o > 0; o >>= 1) {
        if (tid < o) epart[tid] += epart[tid + o];
        __syncthreads();
    }
    if (tid == 1023) poff[nbins] = ppart[1023];
    if (tid == 0) *total += epart[0];
}

// Fills n 32-bit words with v; a kernel rather than a memset so that the
// clears of a group run sit in its captured graph. vec: p is 16-byte aligned.
__global__ void k_set32(unsigned* __restrict__ p, long long n, unsigned v, int vec) {
    const long long stride = (long long)gridDim.x * blockDim.x;
    const long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    const long long n4 = vec ? n >> 2 : 0;
    uint4* q = reinterpret_cast<uint4*>(p);
    for (long long i = t; i < n4; i += stride) q[i] = make_uint4(v, v, v, v);
    for (long long i = 4 * n4 + t; i < n; i += stride) p[i] = v;
}

// One launch for the clears of a reset: the volume records a (na words), and
// where they are not clean already the binned accumulator x (nx words), the bin
// counters f (nf) and the chunk table c (nc, to -1); pool: the free-chunk
// counter and the fallback flags. a, x: 16-byte aligned.
__global__ __launch_bounds__(256) void k_reset(unsigned* __restrict__ a, long long na,
                                               unsigned* __restrict__ x, long long nx,
                                               unsigned* __restrict__ f, long long nf,
                                               unsigned* __restrict__ c, long long nc,
                                               unsigned* __restrict__ pool) {
    const long long stride = (long long)gridDim.x * 256, t = blockIdx.x * 256LL + threadIdx.x;
    uint4* a4 = reinterpret_cast<uint4*>(a);
    for (long long i = t; i < na / 4; i += stride) a4[i] = make_uint4(0, 0, 0, 0);
    for (long long i = na / 4 * 4 + t; i < na; i += stride) a[i] = 0;
    uint4* x4 = reinterpret_cast<uint4*>(x);
    for (long long i = t; i < nx / 4; i += stride) x4[i] = make_uint4(0, 0, 0, 0);
    for (long long i = nx / 4 * 4 + t; i < nx; i += stride) x[i] = 0;
    for (long long i = t; i < nf; i += stride) f[i] = 0;
    for (long long i = t; i < nc; i += stride) c[i] = 0xFFFFFFFFu;
    if (t < 2 && pool) pool[t] = 0;
}

// Clears the bin counters and the used chunk-table entries for the next
// batch (kernels, not memsets, so that the batch can be captured in a graph).
__global__ void k_bin_reset(int* __restrict__ fill, int* __restrict__ chunks, int maxc, int nbins,
                            int* __restrict__ pool) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b == 0) pool[0] = 0;
    if (b >= nbins) return;
    const int n = min(maxc, (fill[b] + BSX_CHUNK - 1) / BSX_CHUNK);
    int* c = chunks + (size_t)b * maxc;
    for (int i = 0; i < n; ++i) c[i] = -1;
    fill[b] = 0;
}

// Float add into LDS through an integer compare-and-swap loop: one IEEE
// rounding per add like an atomic float add, but measured about 3x faster
// here than ds_add_f32 for the tile sums (integer LDS atomics are cheap,
// float ones are not).
__device__ __forceinline__ void lds_fadd(float* p, float x) {
    unsigned* u = reinterpret_cast<unsigned*>(p);
    unsigned old = *reinterpret_cast<volatile unsigned*>(u);
    while (true) {
        const unsigned assumed = old;
        old = atomicCAS(u, assumed, __float_as_uint(__uint_as_float(assumed) + x));
        if (old == assumed) break;
    }
}

// Two float adds to one 8-byte LDS word by a 64-bit compare-and-swap loop:
// the real and imaginary sums of a record move together.
__device__ __forceinline__ void lds_fadd2(float2* p, float x, float y) {
    unsigned long long* u = reinterpret_cast<unsigned long long*>(p);
    unsigned long long old = *reinterpret_cast<volatile unsigned long long*>(u);
    while (true) {
        const unsigned long long assumed = old;
        const float ax = __uint_as_float((unsigned)assumed) + x;
        const float ay = __uint_as_float((unsigned)(assumed >> 32)) + y;
        const unsigned long long next =
            (unsigned long long)__float_as_uint(ax) | ((unsigned long long)__float_as_uint(ay) << 32);
        old = atomicCAS(u, assumed, next);
        if (old == assumed) break;
    }
}

// One workgroup per piece of a (half, tile) bin: sum its entries in LDS, then
// add the tile partial to the volume — a plain read-modify-write when the bin
// is a single piece, float atomics per touched record for multi-piece bins.
// Each thread keeps 8 entry loads in flight before its LDS adds. FOM: the
// entries' (sum w|F|^2, sum w^2) come from bins2 and the records hold 5 floats,
// 80 KB of LDS, so that one workgroup fits a CU: 1024 threads of 4 loads
// (674 -> 648 us a batch
// of 2,048 particles against 512 threads of 8).
template <bool FOM>
__global__ __launch_bounds__(FOM ? 1024 : 512) void k_tile_accum(const int* __restrict__ fill,
                                                    const int* __restrict__ chunks, int maxc,
                                                    int piece_len, const int* __restrict__ poff,
                                                    const int* __restrict__ pbin, int nbins,
                                                    const float4* __restrict__ bins,
                                                    const float2* __restrict__ bins2,
                                                    float* __restrict__ acc) {
    constexpr int RS = FOM ? 5 : 3;                 // floats per record
    constexpr int TN = FOM ? 1024 : 512;            // threads
    constexpr int PC = BSX_PIECE_MAX / BSX_CHUNK;   // chunks per piece, at most
    const int pcn = piece_len / BSX_CHUNK;
    const int piece = blockIdx.x;
    if (piece >= poff[nbins]) return;
    const int bin = pbin[piece];
    const int j = piece - poff[bin];
    const bool single = poff[bin + 1] - poff[bin] == 1;
    const int beg = j * piece_len;
    const int end = min(min(fill[bin], maxc * BSX_CHUNK), beg + piece_len);
    if (beg >= end) return;
    __shared__ float2 sri[4096];   // (sum re, sum im) per record
    __shared__ float sw[4096];
    __shared__ float2 spw[FOM ? 4096 : 1];   // (sum w|F|^2, sum w^2) per record
    __shared__ int pc[PC];
    if (threadIdx.x < PC && (int)threadIdx.x < pcn) {
        const int ci = beg / BSX_CHUNK + threadIdx.x;
        pc[threadIdx.x] = (ci < maxc && ci * BSX_CHUNK < end) ? chunks[(size_t)bin * maxc + ci] : -1;
    }
    float* g = acc + (size_t)bin * 4096 * RS;
    for (int i = threadIdx.x; i < 4096; i += blockDim.x) {
        sri[i] = make_float2(0.f, 0.f);
        sw[i] = 0.f;
        if (FOM) spw[i] = make_float2(0.f, 0.f);
    }
    __syncthreads();
    constexpr int U = FOM ? 4 : 8;
    const int stride = blockDim.x;
    for (int e0 = beg + threadIdx.x; e0 < end; e0 += U * stride) {
        float4 v[U];
        float2 v2[FOM ? U : 1];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int e = e0 + u * stride;
            const int c = e < end ? pc[(e - beg) / BSX_CHUNK] : -1;
            const size_t at = (size_t)c * BSX_CHUNK + (e & (BSX_CHUNK - 1));
            v[u] = c >= 0 ? bins[at] : make_float4(0.f, 0.f, 0.f, __int_as_float(-1));
            if (FOM) v2[u] = c >= 0 ? bins2[at] : make_float2(0.f, 0.f);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int li = __float_as_int(v[u].w);
            if (li >= 0 && li < 4096) {
                lds_fadd2(&sri[li], v[u].x, v[u].y);
                lds_fadd(&sw[li], v[u].z);
                if (FOM) lds_fadd2(&spw[li], v2[FOM ? u : 0].x, v2[FOM ? u : 0].y);
            }
        }
    }
    __syncthreads();
    if (single) {
        // the tile's 4096 RS floats as float4: all loads, then all stores
        float4* g4 = reinterpret_cast<float4*>(g);
        constexpr int NV = 1024 * RS / TN;
        float4 cur[NV];
#pragma unroll
        for (int u = 0; u < NV; ++u) cur[u] = g4[threadIdx.x + u * TN];
#pragma unroll
        for (int u = 0; u < NV; ++u) {
            const int f = 4 * (threadIdx.x + u * TN);
            float add[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int li = (f + q) / RS, c = (f + q) - li * RS;
                add[q] = c == 0 ? sri[li].x : c == 1 ? sri[li].y : c == 2 ? sw[li]
                         : c == 3 ? spw[FOM ? li : 0].x : spw[FOM ? li : 0].y;
            }
            cur[u].x += add[0];
            cur[u].y += add[1];
            cur[u].z += add[2];
            cur[u].w += add[3];
            g4[threadIdx.x + u * TN] = cur[u];
        }
    } else {
        for (int li = threadIdx.x; li < 4096; li += blockDim.x) {
            const float2 ri = sri[li];
            const float2 pw = FOM ? spw[FOM ? li : 0] : make_float2(0.f, 0.f);
            if (sw[li] != 0.f || ri.x != 0.f || ri.y != 0.f || pw.x != 0.f || pw.y != 0.f) {
                unsafeAtomicAdd(g + RS * li + 0, ri.x);
                unsafeAtomicAdd(g + RS * li + 1, ri.y);
                unsafeAtomicAdd(g + RS * li + 2, sw[li]);
                if (FOM) {
                    unsafeAtomicAdd(g + RS * li + 3, pw.x);
                    unsafeAtomicAdd(g + RS * li + 4, pw.y);
                }
            }
        }
    }
}

// ------------------------------------------------------------------- K4
// FP64 values added over a workgroup of 16 wavefronts, then atomically to
// dst[q] by one thread.
template <int Q>
__device__ __forceinline__ void block_add(double (&v)[Q], double* __restrict__ dst) {
    __shared__ double sh[16][Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v[q] += __shfl_xor(v[q], o, 64);
        if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6][q] = v[q];
    }
    __syncthreads();
    if (threadIdx.x < Q) {
        double t = 0;
        for (int w = 0; w < (int)blockDim.x / 64; ++w) t += sh[w][threadIdx.x];
        atomicAdd(dst + threadIdx.x, t);
    }
}

// Sum of half sets, weighing (fspace_reconstruction_weigh,
// Bimage_reconstruct.cpp:486-515) in FP64, SNR FOM (:610-634), centre shift
// (phase_shift_to_center: x (-1)^(h+k+l), N being even) and the Friedel
// residual sums (Bimage::friedel_check, Bimage_fspace.cpp:2024-2074). With FOLD the binned accumulator X is first
// brought into the records S and cleared, as k_fold does.
//
// One thread takes a voxel v and its Friedel mate u = -v: the fold needs both
// X records, the residual both weighed values, so each record is read once and
// nothing is read back. fin: coverage, sum w, and the residual's sums of w,
// w dre^2, w dim^2 over the half space x < N / 2 (on the plane x = 0
// both voxels of a pair count).
// Bound by memory at large maps; at small ones by the workgroups' five
// atomics, so at most 512 workgroups of 1024 threads run. The three separate
// passes this replaces (fold, weigh, residual; 2,048 workgroups each, the fold
// repeated for every map): 96 -> 8 us at 32^3, 603 -> 164 us for the three maps
// of two 128^3 halves with FOM sums.
template <bool FOM, bool FOLD>
__global__ __launch_bounds__(1024) void k_weigh_pairs(float* __restrict__ S, float* __restrict__ X,
                                                      int N, int nz, int NT, long long nrec, int hmask,
                                                      int nhalves, float2* __restrict__ out,
                                                      float* __restrict__ fom_out,
                                                      double* __restrict__ fin, int* __restrict__ flags) {
    constexpr int RS = FOM ? 5 : 3;
    const unsigned nxh = N / 2 + 1, total = nxh * (unsigned)N * (unsigned)nz;
    double sums[5] = {0, 0, 0, 0, 0};
    for (unsigned i = blockIdx.x * 1024u + threadIdx.x; i < total; i += gridDim.x * 1024u) {
        const int x = (int)(i % nxh);
        const unsigned yz = i / nxh;
        const int y = (int)(yz % (unsigned)N), z = (int)(yz / (unsigned)N);
        const int mx = x ? N - x : 0, my = y ? N - y : 0, mz = z ? nz - z : 0;
        // planes that hold their own mates: the lower (y, z) takes the pair
        if (mx == x && mz * N + my < z * N + y) continue;
        const bool self = mx == x && my == y && mz == z;
        const size_t rv = (size_t)rec_index(x, y, z, NT) * RS;
        const size_t ru = (size_t)rec_index(mx, my, mz, NT) * RS;
        double av[5] = {0, 0, 0, 0, 0}, au[5] = {0, 0, 0, 0, 0};
        for (int hh = 0; hh < nhalves; ++hh) {
            const bool want = (hmask >> hh) & 1;
            if (!FOLD && !want) continue;
            float* s = S + (size_t)hh * nrec * RS;
            float sv[RS], su[RS];
#pragma unroll
            for (int c = 0; c < RS; ++c) {
                sv[c] = s[rv + c];
                su[c] = s[ru + c];
            }
            if (FOLD) {
                float* xa = X + (size_t)hh * nrec * RS;
                float xv[RS], xu[RS];
#pragma unroll
                for (int c = 0; c < RS; ++c) {
                    xv[c] = xa[rv + c];
                    xu[c] = xa[ru + c];
                }
#pragma unroll
                for (int c = 0; c < RS; ++c) {
                    // a pair entry stands for its value at v and the conjugate
                    // at -v; the weights and FOM sums are those of both
                    const float m = c == 1 ? -xu[c] : xu[c];
                    sv[c] += xv[c] + m;
                    su[c] += c == 1 ? xu[c] - xv[c] : xu[c] + xv[c];
                    s[rv + c] = sv[c];
                    xa[rv + c] = 0.f;
                    if (!self) {
                        s[ru + c] = su[c];
                        xa[ru + c] = 0.f;
                    }
                }
            }
            if (want)
#pragma unroll
                for (int c = 0; c < RS; ++c) {
                    av[c] += sv[c];
                    au[c] += su[c];
                }
        }
        const bool odd = (x + y + z) & 1;
        float2 val[2];
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            if (m == 1 && self) {
                val[1] = val[0];
                continue;
            }
            const double* a = m ? au : av;
            double W = a[2], P = FOM ? a[3] : 0;
            sums[1] += W;
            float ofr = 0.f, ofi = 0.f;
            if (W > 1e-30) {
                ofr = (float)(a[0] / W);
                ofi = (float)(a[1] / W);
                if (FOM) {
                    const double w2 = W - a[4] / W;
                    if (w2 > 1) P /= w2;
                    else if (W > 1) P /= W;
                    if (P < 0) P = 0;
                }
                sums[0] += 1;
            } else {
                P = 0;
                W = 1e-30;
            }
            const size_t at = m ? ((size_t)mz * N + my) * N + mx : ((size_t)z * N + y) * N + x;
            if (fom_out) {
                if (at == 0) P = 1;
                const double signal = (double)ofr * ofr + (double)ofi * ofi;
                double noise = P - signal;
                if (noise < signal) noise = signal;
                float oP = 0.f;
                if (W > 1 && signal > 1e-30 && noise > 1e-30) oP = (float)((W * signal - P) / noise);
                if (at == 0) oP = 1.f;
                fom_out[at] = oP;
            }
            val[m] = odd ? make_float2(-ofr, -ofi) : make_float2(ofr, ofi);
            out[at] = val[m];
        }
        if (x < N / 2) {
            const float2 a = val[0], b = val[1];
            const double n = (x == 0 && !self) ? 2 : 1;
            const double w = n * ((double)a.x * a.x + (double)a.y * a.y + (double)b.x * b.x + (double)b.y * b.y) / 2;
            double d = (double)a.x - b.x;
            sums[3] += d * d * w;
            d = (double)a.y + b.y;
            sums[4] += d * d * w;
            sums[2] += w;
        }
    }
    block_add(sums, fin);
    if (flags && blockIdx.x == 0 && threadIdx.x == 0) {
        *(int*)(fin + 5) = *flags;
        *flags = 0;
    }
}

// Shell sums of fspace_reconstruction_stats (Bimage_reconstruct.cpp:526-599).
// Per voxel the values fspace_reconstruction_weigh (:486-515) leaves in the
// four accumulator images (F / sum w, the weighed power, sum w, and
// w - sum w^2 / w; empty voxels 0, 0, 1e-30, 1e-30; power[0] = 1), each held
// in FP32 as the reference's images are; then
//  - |F|^2 over the shells of fspace_radial_power (Bimage_fspace.cpp:
//    848-925): radius = rad_scale |s|, split between the two nearest shells
//    (sums 0: counts, 1: |F|^2), nr1 shells;
//  - the power, weight and weight2 over the shells of Bimage::radial
//    (Bimage_polar.cpp:79-170, origin 0, wrap): radius |(dx, dy, dz)|
//    (sums 2: counts, 3: power, 4: weight, 5: weight2), nr2 <= nr1 shells.
// FP64 sums in LDS per block; block partials to part[block][6][nr1].
__global__ __launch_bounds__(256) void k_recon_stats(const float* __restrict__ acc, long long n3,
                                                     int N, int nz, int NT, long long nrec, int stride,
                                                     int hmask, int nhalves, double rad_scale,
                                                     double freq_scale, int nr1, int nr2,
                                                     double* __restrict__ part) {
    extern __shared__ double sh[];
    for (int i = threadIdx.x; i < 6 * nr1; i += blockDim.x) sh[i] = 0;
    __syncthreads();
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n3;
         i += (long long)gridDim.x * blockDim.x) {
        double fr = 0, fi = 0, W = 0, P = 0, W2 = 0;
        const long long xx = i % N, yy = (i / N) % N, zz = i / ((long long)N * N);
        const long long ri = rec_index(xx, yy, zz, NT);
        for (int hh = 0; hh < nhalves; ++hh) {
            if (!((hmask >> hh) & 1)) continue;
            const float* r = acc + ((size_t)hh * nrec + ri) * stride;
            fr += r[0];
            fi += r[1];
            W += r[2];
            P += r[3];
            W2 += r[4];
        }
        float ofr = 0.f, ofi = 0.f;
        double w2 = 1e-30;
        if (W > 1e-30) {
            w2 = W - W2 / W;
            ofr = (float)(fr / W);
            ofi = (float)(fi / W);
            if (w2 > 1) P /= w2;
            else if (W > 1) P /= W;
            if (P < 0) P = 0;
        } else {
            P = 0;
            W = 1e-30;
        }
        if (i == 0) P = 1;
        const double Pf = (float)P, Wf = (float)W, W2f = (float)w2;
        const double pw = (double)ofr * ofr + (double)ofi * ofi;
        // fspace_radial_power: wrap above (N - 1) / 2
        const long hx = xx > (N - 1) / 2 ? xx - N : xx;
        const long hy = yy > (N - 1) / 2 ? yy - N : yy;
        const long hz = zz > (nz - 1) / 2 ? zz - nz : zz;
        double rx = hx * freq_scale, ry = hy * freq_scale, rz = hz * freq_scale;
        rx *= rx;
        ry *= ry;
        rz *= rz;
        const double radius = rad_scale * sqrt(rx + ry + rz);
        const long ir = (long)radius;
        if (ir < nr1) {
            const double f = radius - ir, f1 = 1 - f;
            atomicAdd(&sh[ir], f1);
            atomicAdd(&sh[nr1 + ir], f1 * pw);
            if (ir + 1 < nr1) {
                atomicAdd(&sh[ir + 1], f);
                atomicAdd(&sh[nr1 + ir + 1], f * pw);
            }
        }
        // Bimage::radial, origin 0 with wrap: d = x for x <= N/2, else x - N
        const long dx = xx > N / 2 ? xx - N : xx;
        const long dy = yy > N / 2 ? yy - N : yy;
        const long dz = zz > nz / 2 ? zz - nz : zz;
        const double r2 = sqrt((double)(dx * dx) + (double)(dy * dy) + (double)(dz * dz));
        const long jr = (long)r2;
        if (jr < nr2) {
            const double f = r2 - jr, f1 = 1 - f;
            atomicAdd(&sh[2 * nr1 + jr], f1);
            atomicAdd(&sh[3 * nr1 + jr], f1 * Pf);
            atomicAdd(&sh[4 * nr1 + jr], f1 * Wf);
            atomicAdd(&sh[5 * nr1 + jr], f1 * W2f);
            if (jr + 1 < nr2) {
                atomicAdd(&sh[2 * nr1 + jr + 1], f);
                atomicAdd(&sh[3 * nr1 + jr + 1], f * Pf);
                atomicAdd(&sh[4 * nr1 + jr + 1], f * Wf);
                atomicAdd(&sh[5 * nr1 + jr + 1], f * W2f);
            }
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 6 * nr1; i += blockDim.x)
        part[(size_t)blockIdx.x * 6 * nr1 + i] = sh[i];
}

// Sum of the block partials in block order: one thread per (sum, shell).
__global__ void k_stats_sum(const double* __restrict__ part, int nblocks, int m,
                            double* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    double s = 0;
    for (int b = 0; b < nblocks; ++b) s += part[(size_t)b * m + i];
    out[i] = s;
}

// Folds the binned accumulator X into the volume records S (3 floats per
// record, both in the tiled layout, `nrec` records per half) and clears X.
// A binned entry stands for a sample and its Friedel mate: an X record at v for
// the same sums at v and their conjugates at -v (mod N), so
// S(v) += X(v) + conj(X(-v)) and the weight W(v) += Xw(v) + Xw(-v). One
// thread per voxel pair {v, -v}; linear order decides which voxel of the
// pair handles it.
__global__ void k_fold(float* __restrict__ S, float* __restrict__ X, long long n3, int N, int NT,
                       long long nrec, int nhalves, int rs) {
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n3 * nhalves;
         i += (long long)gridDim.x * blockDim.x) {
        const int half = (int)(i / n3);
        const long long j = i - (long long)half * n3;
        const long x = j % N, y = (j / N) % N, z = j / ((long long)N * N);
        float* s = S + (size_t)half * nrec * rs;
        float* xa = X + (size_t)half * nrec * rs;
        const size_t rv = (size_t)rec_index(x, y, z, NT) * rs;
        const long mx = x ? N - x : 0, my = y ? N - y : 0, mz = z ? N - z : 0;
        const long long jm = mx + (long long)N * (my + (long long)N * mz);
        if (jm < j) continue;
        const size_t ru = (size_t)rec_index(mx, my, mz, NT) * rs;
        const float vr = xa[rv], vi = xa[rv + 1], vw = xa[rv + 2];
        // the FOM sums (w|F|^2, w^2) of a pair entry are those of both mates
        if (jm == j) {
            s[rv] += 2.f * vr;
            s[rv + 2] += 2.f * vw;
            for (int c = 3; c < rs; ++c) s[rv + c] += 2.f * xa[rv + c];
            for (int c = 0; c < rs; ++c) xa[rv + c] = 0.f;
            continue;
        }
        const float ur = xa[ru], ui = xa[ru + 1], uw = xa[ru + 2];
        s[rv] += vr + ur;
        s[rv + 1] += vi - ui;
        s[rv + 2] += vw + uw;
        s[ru] += ur + vr;
        s[ru + 1] += ui - vi;
        s[ru + 2] += uw + vw;
        for (int c = 3; c < rs; ++c) {
            const float a = xa[rv + c], b = xa[ru + c];
            s[rv + c] += a + b;
            s[ru + c] += b + a;
        }
        for (int c = 0; c < rs; ++c) xa[rv + c] = xa[ru + c] = 0.f;
    }
}

// Raw accumulator planes of one half set in (z, y, x) order.
__global__ void k_planes(const float* __restrict__ acc, long long n3, int N, int NT, int stride,
                         int fom, float* __restrict__ out) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n3;
         i += (long long)gridDim.x * blockDim.x) {
        const long long ri = rec_index(i % N, (i / N) % N, i / ((long long)N * N), NT);
        for (int q = 0; q < 5; ++q)
            out[q * n3 + i] = (q < 3 || fom) ? acc[ri * stride + q] : 0.f;
    }
}

// The inverse of k_planes: planes (z, y, x order) into the tiled records.
__global__ void k_set_planes(float* __restrict__ acc, long long n3, int N, int NT, int stride,
                             const float* __restrict__ in) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n3;
         i += (long long)gridDim.x * blockDim.x) {
        const long long ri = rec_index(i % N, (i / N) % N, i / ((long long)N * N), NT);
        for (int q = 0; q < stride; ++q) acc[ri * stride + q] = in[q * n3 + i];
    }
}

// ================================================================== host side
// Drops every captured insert graph (their kernels hold the record buffers'
// addresses and the record count).
static void clear_graphs(bsx_recon* h) {
    for (auto& e : h->graphs)
        if (e.exec) (void)hipGraphExecDestroy(e.exec);
    h->graphs.clear();
}

// Timing marks: an event after each kernel, labelled with the kernel it closes.
static int tmark(bsx_recon* h, hipStream_t s, int label) {
    if (!h->timing) return BSX_OK;
    if (h->nev >= h->evs.size()) {
        hipEvent_t e;
        BSX_HIP(hipEventCreate(&e));
        h->evs.push_back(e);
        h->evlab.push_back(0);
    }
    h->evlab[h->nev] = label;
    BSX_HIP(hipEventRecord(h->evs[h->nev], s));
    ++h->nev;
    return BSX_OK;
}

static double check_resolution(double res, int n, double sampling, int ndim = 3) {
    // Bimage::check_resolution (Bimage.cpp:633-648): a square or cubic map
    // with ndim axes longer than one voxel
    if (res > n * sampling) return n * sampling;
    double rm = 2 / sqrt(ndim / (sampling * sampling));
    return res < rm ? rm : res;
}

static void make_rec(const bsx_recon* h, const bsx_particle& q, PartDev& r) {
    const int ft = h->p.ft_size, box = h->p.box;
    view_matrix(q.view, r.R);
    double scale = q.mag > 0 ? 1.0 / q.mag : 1.0;
    r.invscale = scale / (ft * q.pixel_size);
    r.phx = q.ori[0] / ft * 2 * M_PI;
    r.phy = q.ori[1] / ft * 2 * M_PI;
    const int T = ft / 8;
    r.rot[0] = cos(T * r.phy);
    r.rot[1] = sin(T * r.phy);
    r.rot[2] = cos((T - ft) * r.phy);
    r.rot[3] = sin((T - ft) * r.phy);
    r.nyq[0] = cos(-ft * r.phy);
    r.nyq[1] = sin(-ft * r.phy);
    double wl = lambda_of(q.volt);
    double t1 = M_PI_2 * wl * wl * wl, t2 = -M_PI * wl, dev = fabs(q.def_dev);
    r.c0 = -q.amp_shift;
    r.c20 = t2 * q.def_avg;
    r.c22 = t2 * dev * cos(2 * q.ast_angle);
    r.c2m2 = t2 * dev * sin(2 * q.ast_angle);
    r.c40 = t1 * q.cs;
    r.fscale = 1.0 / (ft * q.pixel_size);
    r.ew = (h->p.flags & BSX_FLAG_EWALD) ? wl / 2 : 0;
    r.hox = q.hdr_ori[0];
    r.hoy = q.hdr_ori[1];
    double w = (h->p.flags & BSX_FLAG_BOOTSTRAP) ? q.sel : 1.0;
    double pad_ratio = (double)ft / box;
    if (pad_ratio > 1) { pad_ratio *= pad_ratio * 0.6; w /= pad_ratio; }
    r.wp = (float)w;
    r.half = h->p.nhalves > 1 ? (q.half & 1) : 0;
}

// ------------------------------------------------------------- symmetry
// Point-group operators (axis, order) of Bsymmetry::Bsymmetry
// (src/util/symmetry.cpp:42-122, labels cleaned as Bsymmetry::clean_symstring,
// include/symmetry.h:73-99); helical symmetry is not a point group and is
// rejected.
struct SymOp {
    double ax[3];
    int order;
};

static int parse_symmetry(const char* label, std::vector<SymOp>& ops) {
    ops.clear();
    std::string l;
    for (const char* c = label ? label : ""; *c; ++c)
        if (!isspace((unsigned char)*c)) l += *c;
    if (l.empty()) l = "C1";
    if (isdigit((unsigned char)l[0])) {
        const int j = atoi(l.c_str());
        if (l.find("532") != std::string::npos && l.find("90") != std::string::npos) l = "I90";
        else if (l.find("532") != std::string::npos) l = "I";
        else if (l.find("432") != std::string::npos) l = "O";
        else if (l.find("23") != std::string::npos) l = "T";
        else if (j > 0) l = "C" + std::to_string(j);
        else l = "C1";
    }
    l[0] = (char)toupper((unsigned char)l[0]);
    auto has = [&](const char* t) { return l.find(t) != std::string::npos; };
    auto add = [&](double x, double y, double z, int order) {
        const double n = sqrt(x * x + y * y + z * z);
        ops.push_back(SymOp{{x / n, y / n, z / n}, order});
    };
    const double G = 1.61803398874989484820458683436563811772;   // golden ratio
    if (l[0] == 'C') {
        const int n = (l == "Cs" || l == "CS") ? 1 : atoi(l.c_str() + 1);
        BSX_REQUIRE(n >= 1 && n <= 1000, BSX_ERR_ARG, "symmetry %s: bad order", l.c_str());
        add(0, 0, 1, n);
    } else if (l[0] == 'D') {
        const int n = atoi(l.c_str() + 1);
        BSX_REQUIRE(n >= 1 && n <= 1000, BSX_ERR_ARG, "symmetry %s: bad order", l.c_str());
        add(0, 0, 1, n);
        add(1, 0, 0, 2);
    } else if (l[0] == 'T') {
        if (!has("-3")) add(1, 1, 1, 3);
        add(0, 0, 1, 2);
        add(1, 0, 0, 2);
    } else if (l[0] == 'O') {
        if (!has("-3")) add(1, 1, 1, 3);
        if (has("-4")) {
            add(1, -1, 0, 2);
        } else if (has("-2")) {
            add(0, 0, 1, 4);
        } else {
            add(0, 0, 1, 4);
            add(1, 0, 0, 2);
        }
    } else if (l[0] == 'I') {
        if (!has("-3")) add(1, 1, 1, 3);
        if (has("-5")) add(1, 0, 0, 2);
        else if (has("-2")) add(1, -1, 0, 2);
        else add(1, 1.0 / G, G, 2);
        if (!has("-5")) add(1.0 / G, 1, 0, 5);
        if (!has("-2")) add(0, 0, 1, 2);
        if (has("90"))   // axes rotated by 90 degrees about z
            for (SymOp& o : ops) {
                const double x = o.ax[0], y = o.ax[1];
                o.ax[0] = -y;
                o.ax[1] = x;
            }
    } else {
        set_error("symmetry %s: not a point group (C, D, T, O, I)", l.c_str());
        return BSX_ERR_ARG;
    }
    return BSX_OK;
}

// View::normalize / check (include/View.h:32-36, 110-116): unit view vector,
// tiny components zeroed, angle in [-pi, pi].
static void view_normalize(double v[4]) {
    const double size = sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
    if (size < 1e-30) { v[0] = v[1] = 0; v[2] = 1; }
    else { v[0] /= size; v[1] /= size; v[2] /= size; }
    for (int i = 0; i < 3; ++i)
        if (fabs(v[i]) < 1e-30) v[i] = 0;
    v[3] = remainder(v[3], 2 * M_PI);
    if (fabs(v[3]) < 1e-30) v[3] = 0;
}

// Quaternion::check (include/Quaternion.h:28-32)
static void quat_check(double q[4]) {
    for (int i = 0; i < 4; ++i)
        if (fabs(q[i]) < 1e-30) q[i] = 0;
}

// View::quaternion (include/View.h:131-153)
static void view_quaternion(double v[4], double q[4]) {
    view_normalize(v);
    const double ang = v[3] / 2.0L, ca = cos(ang), sa = sin(ang);
    const double z1 = v[2] + 1;
    q[0] = ca; q[1] = 0; q[2] = 0; q[3] = sa;
    if (v[2] < 1.0L - 1e-30) {
        if (v[2] <= 1e-30 - 1.0L) {
            q[0] = 0; q[1] = sa; q[2] = ca; q[3] = 0;
        } else {
            const double f1 = sqrt(z1 / 2.0), f2 = sqrt(1.0 / (2 * z1));
            q[0] = f1 * ca;
            q[1] = f2 * (v[0] * sa - v[1] * ca);
            q[2] = f2 * (v[0] * ca + v[1] * sa);
            q[3] = f1 * sa;
        }
    }
    quat_check(q);
}

// View(Quaternion&) (include/View.h:52-63)
static void quaternion_view(const double q[4], double v[4]) {
    double ang = atan2(q[3], q[0]);
    const double ca = cos(ang), sa = sin(ang);
    const double q2 = q[0] * q[0] + q[3] * q[3];
    const double f2 = 2 * sqrt(q2);
    if (q2 < 1e-30) ang = atan2(q[1], q[2]);
    v[0] = f2 * (q[2] * ca + q[1] * sa);
    v[1] = f2 * (q[2] * sa - q[1] * ca);
    v[2] = 2 * q2 - 1;
    v[3] = 2 * ang;
    view_normalize(v);
}

// symmetry_get_all_views (src/util/symmetry.cpp:277-319): the view first,
// then for each operator and each multiple j of its angle the rotated copies
// of all views so far (Quaternion(axis, angle) * view quaternion).
static void symmetry_views(const std::vector<SymOp>& ops, const double view[4],
                           std::vector<double>& out) {
    out.assign(view, view + 4);
    view_normalize(out.data());
    size_t nview = 1;
    for (const SymOp& o : ops) {
        for (int j = 1; j < o.order; ++j) {
            const double angle = j * (2 * M_PI) * 1.0L / o.order;
            const double a = angle / 2.0L;
            double q[4] = {cos(a), o.ax[0] * sin(a), o.ax[1] * sin(a), o.ax[2] * sin(a)};
            quat_check(q);
            for (size_t k = 0; k < nview; ++k) {
                double v[4] = {out[4 * k], out[4 * k + 1], out[4 * k + 2], out[4 * k + 3]};
                double p[4];
                view_quaternion(v, p);
                const double r[4] = {
                    q[0] * p[0] - (q[1] * p[1] + q[2] * p[2] + q[3] * p[3]),
                    q[0] * p[1] + q[1] * p[0] + q[2] * p[3] - q[3] * p[2],
                    q[0] * p[2] + q[2] * p[0] + q[3] * p[1] - q[1] * p[3],
                    q[0] * p[3] + q[3] * p[0] + q[1] * p[2] - q[2] * p[1]};
                double nv[4];
                quaternion_view(r, nv);
                out.insert(out.end(), nv, nv + 4);
            }
        }
        nview *= (size_t)o.order;
    }
}

// ------------------------------------------------ real-space symmetrization
// Bimage::symmetrize (src/img/Bimage_symmetry.cpp:31-100) of a real N^3 map:
// for each operator (axis, order m) the map becomes the sum of itself and
// its m - 1 rotations about the origin, each rotation
// Bimage::transform (src/img/Bimage_transform.cpp:138-214) with
// Bimage::interpolate (src/img/Bimage.cpp:1436-1484) and the background as
// the fill; after the last operator the map is multiplied by 1 / order.

// Rotation matrix of Matrix3(axis, angle): Quaternion::from_axis_angle
// (include/Quaternion.h:34-41, check() zeroes components below 1e-30), then
// Matrix3::from_quaternion and check() (include/Matrix3.h:21-42).
static void axis_angle_matrix(const double ax[3], double angle, double M[9]) {
    const double n = sqrt(ax[0] * ax[0] + ax[1] * ax[1] + ax[2] * ax[2]);
    const double a = angle / 2;
    double q[4] = {cos(a), ax[0] / n * sin(a), ax[1] / n * sin(a), ax[2] / n * sin(a)};
    for (int i = 1; i < 4; ++i)
        if (fabs(q[i]) < 1e-30) q[i] = 0;
    M[0] = q[0] * q[0] + q[1] * q[1] - q[2] * q[2] - q[3] * q[3];
    M[1] = 2 * q[1] * q[2] - 2 * q[0] * q[3];
    M[2] = 2 * q[1] * q[3] + 2 * q[0] * q[2];
    M[3] = 2 * q[1] * q[2] + 2 * q[0] * q[3];
    M[4] = q[0] * q[0] - q[1] * q[1] + q[2] * q[2] - q[3] * q[3];
    M[5] = 2 * q[2] * q[3] - 2 * q[0] * q[1];
    M[6] = 2 * q[1] * q[3] - 2 * q[0] * q[2];
    M[7] = 2 * q[2] * q[3] + 2 * q[0] * q[1];
    M[8] = q[0] * q[0] - q[1] * q[1] - q[2] * q[2] + q[3] * q[3];
    for (int i = 0; i < 9; ++i) {
        if (fabs(M[i]) < 1e-12) M[i] = 0;
        if (M[i] > 1) M[i] = 1;
        if (M[i] < -1) M[i] = -1;
    }
}

// Bimage::interpolate: trilinear over the (up to) 2 x 2 x 2 neighbours inside
// the map, weights toggled as the reference's loops toggle them (an edge
// neighbour missing in one axis leaves that axis's weight alternating),
// normalised by their sum; outside the map: fill.
__device__ inline double interp_fill(const float* __restrict__ a, int n, int zn, double xx,
                                     double yy, double zz, double fill) {
    if (xx < 0 || xx >= n || yy < 0 || yy >= n || zz < 0 || zz >= zn) return fill;
    const long ix = (long)xx, iy = (long)yy, iz = (long)zz;
    const int nx = (n < ix + 2) ? 1 : 2, ny = (n < iy + 2) ? 1 : 2, nz = (zn < iz + 2) ? 1 : 2;
    double fx = xx - ix, fy = yy - iy, fz = zz - iz;
    double value = 0, ws = 0;
    for (int zk = 0; zk < nz; ++zk) {
        fz = 1.0 - fz;
        for (int yk = 0; yk < ny; ++yk) {
            fy = 1.0 - fy;
            const double wyz = fy * fz;
            const size_t row = ((size_t)(iz + zk) * n + (iy + yk)) * n;
            for (int xk = 0; xk < nx; ++xk) {
                fx = 1.0 - fx;
                const double w = fx * wyz;
                ws += w;
                value += (double)a[row + ix + xk] * w;
            }
        }
    }
    return ws != 0 ? value / ws : fill;
}

// Background of Bimage::calculate_background (flag 0,
// src/img/Bimage_background.cpp:27-80): mean of the voxels outside the
// ellipsoid ((x - o) / (N/2))^2 + ... = 1. Per-block FP64 partial sums, then
// one block adds them in a fixed order.
__global__ __launch_bounds__(256) void k_bkg_partial(const float* __restrict__ a, int n, int zn, double o0,
                                                     double o1, double o2,
                                                     double* __restrict__ part) {
    __shared__ double ss[256], sc[256];
    const int64_t total = (int64_t)n * n * zn;
    const double h = (double)(n / 2);
    double s = 0, c = 0;
    for (int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x; v < total;
         v += (int64_t)gridDim.x * 256) {
        const int x = (int)(v % n), y = (int)((v / n) % n), z = (int)(v / ((int64_t)n * n));
        double x2 = (x - o0) / h, y2 = (y - o1) / h, z2 = zn > 1 ? (z - o2) / (double)(zn / 2) : 0;
        x2 *= x2;
        y2 *= y2;
        z2 *= z2;
        if (x2 + y2 + z2 - 1 > 0) {
            s += a[v];
            c += 1;
        }
    }
    ss[threadIdx.x] = s;
    sc[threadIdx.x] = c;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) {
            ss[threadIdx.x] += ss[threadIdx.x + o];
            sc[threadIdx.x] += sc[threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = ss[0];
        part[2 * blockIdx.x + 1] = sc[0];
    }
}

__global__ void k_bkg_final(const double* __restrict__ part, int nblocks, double* __restrict__ bkg) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    double s = 0, c = 0;
    for (int b = 0; b < nblocks; ++b) {
        s += part[2 * b];
        c += part[2 * b + 1];
    }
    bkg[0] = c > 0 ? s / c : 0;
}

// One operator: out = in + sum over j of in rotated by mats[j] (m - 1
// matrices, the image rotated by R samples the input at R^T (x - o) + o),
// each term rounded to FP32 and added in FP32 as Bimage::sum does; the last
// operator also multiplies by `scale` (1 / order).
__global__ __launch_bounds__(256) void k_sym_op(const float* __restrict__ in,
                                                float* __restrict__ out, int n, int zn, double o0,
                                                double o1, double o2,
                                                const double* __restrict__ mats, int nm,
                                                const double* __restrict__ bkg, double scale) {
    const int64_t total = (int64_t)n * n * zn;
    const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (v >= total) return;
    const int x = (int)(v % n), y = (int)((v / n) % n), z = (int)(v / ((int64_t)n * n));
    const double u0 = x - o0, u1 = y - o1, u2 = z - o2;
    const double fill = bkg[0];
    float acc = in[v];
    for (int j = 0; j < nm; ++j) {
        const double* M = mats + 9 * j;
        const double a0 = M[0] * u0 + M[3] * u1 + M[6] * u2 + o0;
        const double a1 = M[1] * u0 + M[4] * u1 + M[7] * u2 + o1;
        const double a2 = M[2] * u0 + M[5] * u1 + M[8] * u2 + o2;
        const float pj = (float)interp_fill(in, n, zn, a0, a1, a2, fill);
        acc = (float)((double)acc + (double)pj);
    }
    if (scale != 1) acc = (float)((double)acc * scale);
    out[v] = acc;
}

// Whether calls on the stream are being recorded into a graph. The legacy default
// stream cannot be recorded, so that calls on it do not pay for the question (2 us).
static bool recording(hipStream_t s) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (!s) return false;
    if (hipStreamIsCapturing(s, &st) == hipSuccess) return st != hipStreamCaptureStatusNone;
    (void)hipGetLastError();
    return true;
}

// Insertion of one batch: rows and fill, then for binned entries the piece
// table, the tile pass and the clearing of the bins.
static int run_batch(bsx_recon* h, const float* imgs, int64_t p0, int nb, hipStream_t s) {
    int r;
    switch (h->p.ft_size) {
        case 32: r = insert_batch<32>(h, imgs, p0, nb, s, tmark); break;
        case 64: r = insert_batch<64>(h, imgs, p0, nb, s, tmark); break;
        case 128: r = insert_batch<128>(h, imgs, p0, nb, s, tmark); break;
        case 256: r = insert_batch<256>(h, imgs, p0, nb, s, tmark); break;
        case 512: r = insert_batch<512>(h, imgs, p0, nb, s, tmark); break;
        default:
            set_error("ft_size %d not supported (32..512, power of 2)", h->p.ft_size);
            return BSX_ERR_ARG;
    }
    if (r || !h->binned) return r;
    const unsigned maxpieces = (unsigned)(h->nbins + (size_t)h->npool * BSX_CHUNK / h->piece + 1);
    hipLaunchKernelGGL(k_piece_scan, dim3(1), dim3(1024), 0, s, h->fill, h->nbins, h->maxc,
                       h->piece, h->poff, h->pbin, (int)maxpieces, h->entries);
    BSX_HIP(hipGetLastError());
    if ((r = tmark(h, s, KT_SCAN))) return r;
    if (h->K.fom)
        hipLaunchKernelGGL(k_tile_accum<true>, dim3(maxpieces), dim3(1024), 0, s, h->fill,
                           h->chunks, h->maxc, h->piece, h->poff, h->pbin, h->nbins, h->bins,
                           h->bins2, h->xacc);
    else
        hipLaunchKernelGGL(k_tile_accum<false>, dim3(maxpieces), dim3(512), 0, s, h->fill,
                           h->chunks, h->maxc, h->piece, h->poff, h->pbin, h->nbins, h->bins,
                           nullptr, h->xacc);
    BSX_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_bin_reset, dim3((h->nbins + 255) / 256), dim3(256), 0, s, h->fill,
                       h->chunks, h->maxc, h->nbins, h->pool);
    BSX_HIP(hipGetLastError());
    return tmark(h, s, KT_TILE);
}

extern "C" {

int bsx_version(int* major, int* minor) {
    if (major) *major = 0;
    if (minor) *minor = 1;
    return BSX_OK;
}

int bsx_device_info(char* name, int name_len, int* cu_count, int64_t* hbm_bytes) {
    int dev = 0;
    BSX_HIP(hipGetDevice(&dev));
    hipDeviceProp_t pr;
    BSX_HIP(hipGetDeviceProperties(&pr, dev));
    if (name && name_len > 0) {
        strncpy(name, pr.gcnArchName, name_len - 1);
        name[name_len - 1] = 0;
    }
    if (cu_count) *cu_count = pr.multiProcessorCount;
    if (hbm_bytes) *hbm_bytes = (int64_t)pr.totalGlobalMem;
    return BSX_OK;
}

// part_ft_size, src/mg/mg_reconstruct.cpp:38-64
int bsx_part_ft_size(int xsize, double scale, int pad_factor) {
    if (xsize <= 0) {
        set_error("part_ft_size: size not set");
        return 0;
    }
    auto next_pow2 = [](int start) { int r = 2; while (r < start) r *= 2; return r; };
    int ft = xsize;
    if (scale > 1) ft = (int)(xsize * scale);
    if (pad_factor < 1) return ft;
    if (pad_factor > 8) pad_factor = 8;
    ft = next_pow2((int)(pad_factor * xsize * scale));
    if (ft < xsize) ft = next_pow2(xsize);
    return ft;
}

int bsx_recon_create(bsx_recon** out, const bsx_recon_params* p) {
    BSX_REQUIRE(out && p, BSX_ERR_ARG, "bsx_recon_create: null argument");
    *out = nullptr;
    BSX_REQUIRE(p->size >= 2 && p->size <= 512, BSX_ERR_ARG, "size %d out of range 2..512",
                p->size);
    BSX_REQUIRE(fft_length_supported(p->size), BSX_ERR_ARG,
                "map size %d: inverse FFT length not supported", p->size);
    BSX_REQUIRE(p->box >= 2 && p->ft_size >= p->box, BSX_ERR_ARG, "box %d / ft_size %d invalid",
                p->box, p->ft_size);
    BSX_REQUIRE(p->ft_size >= 32 && p->ft_size <= 512 && (p->ft_size & (p->ft_size - 1)) == 0,
                BSX_ERR_ARG, "ft_size %d not supported (32..512, power of 2)", p->ft_size);
    BSX_REQUIRE(p->interp >= 0 && p->interp <= 2, BSX_ERR_ARG, "interp %d invalid", p->interp);
    BSX_REQUIRE(p->nhalves == 1 || p->nhalves == 2, BSX_ERR_ARG, "nhalves must be 1 or 2");
    BSX_REQUIRE(p->sampling > 0, BSX_ERR_ARG, "sampling must be positive");
    BSX_REQUIRE(p->method == 0 || p->method == 1, BSX_ERR_ARG,
                "method must be 0 (binned) or 1 (direct atomics)");
    BSX_REQUIRE(p->order >= 0 && p->order <= 2, BSX_ERR_ARG, "order must be 0, 1 or 2");
    BSX_REQUIRE(p->merge >= 0 && p->merge <= 2, BSX_ERR_ARG, "merge must be 0, 1 or 2");
    bsx_recon* h = new bsx_recon();
    h->p = *p;
    BSX_HIP(hipGetDevice(&h->dev));
    h->hi_res = check_resolution(p->hi_res > 0 ? p->hi_res : p->sampling, p->size, p->sampling,
                                 (p->flags & BSX_FLAG_2D) ? 2 : 3);
    ReconConst& K = h->K;
    K.N = p->size;
    K.ft = p->ft_size;
    K.box = p->box;
    K.fom = (p->flags & BSX_FLAG_FOM) ? 1 : 0;
    K.stride = K.fom ? 5 : 3;
    K.NT = (p->size + 15) / 16;
    // tile-binned insertion (method 0; the FOM sums ride in a second pool
    // array) or direct atomics (method 1)
    h->binned = p->method == 0;
    K.interp = p->interp;
    K.nhalves = p->nhalves;
    // img_ctf_calculate (mg_ctf.cpp:100-107) as particle_reconstruct calls it
    // (flip = action 1): any other action is a Wiener filter when the factor is
    // positive, else the CTF is applied
    K.ctf_mode = p->ctf_action == 0 ? 0 : p->ctf_action == 1 ? 1 : p->wiener > 0 ? 3 : 2;
    K.wiener = p->ctf_action >= 2 ? p->wiener : 0;
    double hi = h->hi_res < 0.5 ? 0.5 : h->hi_res;   // fspace_pack_2D limit (:116)
    K.mins2 = p->lo_res > 0 ? 1.0 / (p->lo_res * p->lo_res) : 0;
    K.maxs2 = 1.0 / (hi * hi);
    K.mscale = p->size * p->sampling;
    K.mscz = (p->flags & BSX_FLAG_2D) ? 1.0 : K.mscale;
    K.nz = (p->flags & BSX_FLAG_2D) ? 1 : p->size;
    K.shi2 = 1.0 / (h->hi_res * h->hi_res);          // img_ctf_calculate hires
    K.ewald = (p->flags & BSX_FLAG_EWALD) ? 1 : 0;
    K.merge = 0;
    const size_t ntile = (size_t)K.NT * K.NT * K.NT;
    const size_t nrec = ntile * 4096;   // records incl. tile padding
    h->acc_elems = nrec * K.stride * p->nhalves;
    h->nbins = (int)(ntile * p->nhalves);
    const size_t ft2 = (size_t)p->ft_size * p->ft_size;
    const int mult = (K.ewald ? 2 : 1) * (p->interp == 2 ? 8 : 1);
    const size_t inter_pp = (size_t)(p->ft_size / 2 + 1) * p->box * sizeof(float2);
    const size_t bins_pp = h->binned ? ft2 * mult * sizeof(float4) : 0;
    int batch = p->batch;
    if (batch <= 0) {
        // intermediate half-spectra within 512 MB and bin entries within 2 GB
        size_t b = (512u << 20) / inter_pp;
        if (bins_pp) b = std::min(b, (size_t)(2ull << 30) / bins_pp);
        batch = (int)std::max<size_t>(1, std::min<size_t>(4096, b));
    }
    h->batch = batch;
    h->batch_cap = batch;
    const size_t inter_bytes = (size_t)batch * inter_pp;
    h->bins_cap = (size_t)batch * ft2 * mult;
    BSX_REQUIRE(!h->binned || h->bins_cap < (1ull << 31), BSX_ERR_ARG,
                "batch %d too large for 32-bit bin offsets", batch);
    // pool: every entry of a batch plus a partly filled chunk per bin; chunk
    // table: 256 chunks (1 M entries) per bin and batch share of 2048 entries
    // per particle and bin, whichever is more (beyond it entries take the
    // atomic fallback)
    const size_t cap_chunks = (h->bins_cap + BSX_CHUNK - 1) / BSX_CHUNK;
    h->npool = (int)(cap_chunks + std::min<size_t>(h->nbins, cap_chunks) + 1);
    h->maxc = (int)std::min<size_t>(cap_chunks + 1,
                                    std::max<size_t>(256, ((size_t)batch * 2048 * mult +
                                                           BSX_CHUNK - 1) / BSX_CHUNK + 1));
    const size_t bins_bytes = h->binned ? (size_t)h->npool * BSX_CHUNK * sizeof(float4) : 0;
    const size_t bins2_bytes = h->binned && K.fom ? (size_t)h->npool * BSX_CHUNK * sizeof(float2) : 0;
    const size_t bin_idx_bytes =
        h->binned ? ((size_t)h->nbins * (h->maxc + 3) + (size_t)h->npool * BSX_CHUNK / BSX_PIECE_MIN +
                     4) * sizeof(int) + 8
                  : 0;
    h->bytes = h->acc_elems * sizeof(float) * (h->binned ? 2 : 1) + inter_bytes + bins_bytes +
               bins2_bytes + bin_idx_bytes;
    if (p->mem_cap > 0 && (int64_t)h->bytes > p->mem_cap) {
        set_error("device memory %zu bytes exceeds the cap %lld", h->bytes, (long long)p->mem_cap);
        delete h;
        return BSX_ERR_NOMEM;
    }
    bool ok = device_malloc(&h->acc, h->acc_elems * sizeof(float)) == hipSuccess &&
              device_malloc(&h->inter, inter_bytes) == hipSuccess &&
              device_malloc(&h->nonfinite, sizeof(int)) == hipSuccess;
    if (ok && bins2_bytes) ok = device_malloc(&h->bins2, bins2_bytes) == hipSuccess;
    if (ok && h->binned)
        ok = device_malloc(&h->bins, bins_bytes) == hipSuccess &&
             device_malloc(&h->xacc, h->acc_elems * sizeof(float)) == hipSuccess &&
             device_malloc(&h->fill, sizeof(int) * h->nbins) == hipSuccess &&
             device_malloc(&h->chunks, sizeof(int) * (size_t)h->nbins * h->maxc) == hipSuccess &&
             device_malloc(&h->pool, sizeof(int) * 2) == hipSuccess &&
             device_malloc(&h->poff, sizeof(int) * (h->nbins + 1)) == hipSuccess &&
             device_malloc(&h->pbin, sizeof(int) * ((size_t)h->nbins +
                                                (size_t)h->npool * BSX_CHUNK / BSX_PIECE_MIN + 1)) ==
                 hipSuccess &&
             device_malloc(&h->entries, sizeof(unsigned long long)) == hipSuccess;
    if (!ok) {
        set_error("device allocation of %zu bytes failed", h->bytes);
        bsx_recon_destroy(h);
        return BSX_ERR_NOMEM;
    }
    if (h->binned) {
        BSX_HIP(hipMemset(h->xacc, 0, h->acc_elems * sizeof(float)));
        BSX_HIP(hipMemset(h->fill, 0, sizeof(int) * h->nbins));
        BSX_HIP(hipMemset(h->chunks, 0xFF, sizeof(int) * (size_t)h->nbins * h->maxc));
        BSX_HIP(hipMemset(h->pool, 0, sizeof(int) * 2));
        BSX_HIP(hipMemset(h->entries, 0, sizeof(unsigned long long)));
    }
    BSX_HIP(hipMemset(h->acc, 0, h->acc_elems * sizeof(float)));
    BSX_HIP(hipDeviceSynchronize());
    *out = h;
    return BSX_OK;
}

int bsx_recon_destroy(bsx_recon* h) {
    if (!h) return BSX_OK;
    if (h->acc) (void)hipFree(h->acc);
    if (h->xacc) (void)hipFree(h->xacc);
    if (h->inter) (void)hipFree(h->inter);
    if (h->bkg) (void)hipFree(h->bkg);
    if (h->resc) (void)hipFree(h->resc);
    if (h->recs) (void)hipFree(h->recs);
    if (h->nonfinite) (void)hipFree(h->nonfinite);
    if (h->bins) (void)hipFree(h->bins);
    if (h->bins2) (void)hipFree(h->bins2);
    if (h->fill) (void)hipFree(h->fill);
    if (h->chunks) (void)hipFree(h->chunks);
    if (h->pool) (void)hipFree(h->pool);
    if (h->poff) (void)hipFree(h->poff);
    if (h->pbin) (void)hipFree(h->pbin);
    if (h->entries) (void)hipFree(h->entries);
    for (auto e : h->evs) (void)hipEventDestroy(e);
    if (h->copied) {
        (void)hipEventSynchronize(h->copied);
        (void)hipEventDestroy(h->copied);
    }
    if (h->hrecs) (void)hipHostFree(h->hrecs);
    if (h->gvol) (void)hipFree(h->gvol);
    if (h->gfin) (void)hipFree(h->gfin);
    clear_graphs(h);
    if (h->cap_stream) (void)hipStreamDestroy(h->cap_stream);
    delete h;
    return BSX_OK;
}

int bsx_recon_reset(bsx_recon* h, void* stream) {
    BSX_REQUIRE(h, BSX_ERR_ARG, "null handle");
    const long long n = (long long)h->acc_elems;
    // a recorded reset clears everything: what is clean now need not be when the
    // graph is replayed, and nothing is cleared before
    const bool rec = recording((hipStream_t)stream);
    const bool x = h->binned && (rec || h->xdirty), b = h->binned && (rec || h->bins_dirty);
    hipLaunchKernelGGL(k_reset, dim3((unsigned)std::min(2048LL, (n / 4 + 255) / 256)), dim3(256), 0,
                       (hipStream_t)stream, (unsigned*)h->acc, n, (unsigned*)h->xacc, x ? n : 0,
                       (unsigned*)h->fill, b ? (long long)h->nbins : 0, (unsigned*)h->chunks,
                       b ? (long long)h->nbins * h->maxc : 0, (unsigned*)h->pool);
    BSX_HIP(hipGetLastError());
    if (!rec) h->xdirty = h->bins_dirty = false;
    h->inserted[0] = h->inserted[1] = 0;
    return BSX_OK;
}

int bsx_recon_device_bytes(const bsx_recon* h, int64_t* bytes) {
    BSX_REQUIRE(h && bytes, BSX_ERR_ARG, "null argument");
    *bytes = (int64_t)h->bytes + h->recs_cap * (int64_t)(sizeof(PartDev) + sizeof(float));
    return BSX_OK;
}

// Host side of an insert: validation, symmetry expansion, and the particle
// records (insertion order, run-merge decision) uploaded to h->recs on
// stream s. *nrec is the number of records; add[q] counts the particles of
// half q, for the caller to add once the kernels are launched.
static int insert_prepare(bsx_recon* h, const bsx_particle* parts, int64_t n, hipStream_t s,
                          int64_t* nrec, int64_t add[2]) {
    {
        // validation on host threads; the lowest failing particle is reported
        std::vector<int64_t> bad(16, INT64_MAX);
        std::vector<int> why(16, 0);
        host_parallel(n, 8192, [&](int64_t b, int64_t e, unsigned t) {
            for (int64_t i = b; i < e; ++i) {
                const bsx_particle& q = parts[i];
                int w = 0;
                if (!(q.pixel_size > 0)) w = 1;
                const double vals[] = {q.view[0], q.view[1], q.view[2], q.view[3], q.ori[0],
                                       q.ori[1], q.hdr_ori[0], q.hdr_ori[1], q.mag, q.volt, q.cs,
                                       q.amp_shift, q.def_avg, q.def_dev, q.ast_angle, q.sel};
                for (double v : vals)
                    if (!w && !std::isfinite(v)) w = 2;
                if (!w && h->p.nhalves > 1 && q.half != 0 && q.half != 1) w = 3;
                if (w) {
                    bad[t] = i;
                    why[t] = w;
                    return;
                }
            }
        });
        int64_t first = INT64_MAX;
        int w = 0;
        for (int t = 0; t < 16; ++t)
            if (bad[t] < first) { first = bad[t]; w = why[t]; }
        BSX_REQUIRE(w != 1, BSX_ERR_ARG, "particle %lld: pixel size not set", (long long)first);
        BSX_REQUIRE(w != 2, BSX_ERR_ARG, "particle %lld: non-finite parameter", (long long)first);
        BSX_REQUIRE(w != 3, BSX_ERR_ARG, "particle %lld: half must be 0 or 1", (long long)first);
    }
    // point-group symmetry: one record per symmetry-related view, all reading
    // the particle's image (fspace_pack_2D over symmetry_get_all_views)
    const int64_t n_parts = n;
    std::vector<bsx_particle> expanded;
    std::vector<int64_t> image_of;
    if (!h->sym_order.empty()) {
        std::vector<SymOp> ops;
        for (size_t o = 0; o < h->sym_order.size(); ++o)
            ops.push_back(SymOp{{h->sym_axis[3 * o], h->sym_axis[3 * o + 1], h->sym_axis[3 * o + 2]},
                                h->sym_order[o]});
        std::vector<double> sv;
        for (int64_t i = 0; i < n_parts; ++i) {
            symmetry_views(ops, parts[i].view, sv);
            for (size_t k = 0; k < sv.size() / 4; ++k) {
                bsx_particle q = parts[i];
                for (int c = 0; c < 4; ++c) q.view[c] = sv[4 * k + c];
                expanded.push_back(q);
                image_of.push_back(i);
            }
        }
        parts = expanded.data();
        n = (int64_t)expanded.size();
    }
    const bool rescale = h->p.flags & BSX_FLAG_RESCALE;
    if (n > h->recs_cap) {
        // captured inserts read the old record buffers
        BSX_HIP(hipStreamSynchronize(s));
        clear_graphs(h);
        if (h->recs) (void)hipFree(h->recs);
        if (h->bkg) (void)hipFree(h->bkg);
        if (h->resc) (void)hipFree(h->resc);
        h->recs = nullptr;
        h->bkg = nullptr;
        h->resc = nullptr;
        int64_t extra = n * (int64_t)(sizeof(PartDev) + sizeof(float) +
                                      (rescale ? sizeof(double2) : 0));
        if (h->p.mem_cap > 0 && (int64_t)h->bytes + extra > h->p.mem_cap) {
            h->recs_cap = 0;
            set_error("particle records (%lld bytes) exceed the device-memory cap", (long long)extra);
            return BSX_ERR_NOMEM;
        }
        if (device_malloc(&h->recs, sizeof(PartDev) * n) != hipSuccess ||
            device_malloc(&h->bkg, sizeof(float) * n) != hipSuccess ||
            (rescale && device_malloc(&h->resc, sizeof(double2) * n) != hipSuccess)) {
            h->recs_cap = 0;
            set_error("allocation of %lld particle records failed", (long long)n);
            return BSX_ERR_NOMEM;
        }
        h->recs_cap = n;
    }
    if (h->copied) BSX_HIP(hipEventSynchronize(h->copied));
    else BSX_HIP(hipEventCreateWithFlags(&h->copied, hipEventDisableTiming));
    if (n > h->hrecs_cap) {
        if (h->hrecs) BSX_HIP(hipHostFree(h->hrecs));
        h->hrecs = nullptr;
        h->hrecs_cap = 0;
        BSX_HIP(pinned_malloc(&h->hrecs, sizeof(PartDev) * n));
        h->hrecs_cap = n;
    }
    // Insertion order: by plane orientation (normal folded to one hemisphere,
    // 2-degree polar bands, snake order in azimuth) so that particles in flight
    // together touch the same voxel lines; the result differs only by FP32
    // summation order.
    std::vector<int64_t> perm(n);
    for (int64_t i = 0; i < n; ++i) perm[i] = i;
    // auto: input order for the binned path (sorted orders concentrate the
    // bin-counter increments of a batch on fewer counters), sorted for the
    // direct path (neighbouring planes share cache lines)
    const int order = h->p.order ? h->p.order : (h->binned ? 1 : 2);
    if (order == 2 && n > 1) {
        std::vector<double> key(n);
        for (int64_t i = 0; i < n; ++i) {
            double v0 = parts[i].view[0], v1 = parts[i].view[1], v2 = parts[i].view[2];
            double nn = sqrt(v0 * v0 + v1 * v1 + v2 * v2);
            if (nn < 1e-30) { v0 = v1 = 0; v2 = 1; nn = 1; }
            v0 /= nn; v1 /= nn; v2 /= nn;
            if (v2 < 0) { v0 = -v0; v1 = -v1; v2 = -v2; }
            const double th = acos(std::min(1.0, v2)), ph = atan2(v1, v0);
            const int band = (int)(th / (2 * M_PI / 180));
            const double az = (band & 1) ? -ph : ph;
            key[i] = band * 10.0 + (az + M_PI);
        }
        std::stable_sort(perm.begin(), perm.end(),
                         [&](int64_t a, int64_t b) { return key[a] < key[b]; });
    }
    double max_step = 0;
    int max_run = 0;
    {
        std::vector<double> tmax(16, 0.0);
        std::vector<int> trun(16, 0);
        // a record takes 0.13 us and a thread some 15 us to start, or milliseconds
        // when other threads of the process have used up the CPU share, so that
        // smaller sets stay on this thread (3,001 records: 390 us, 160 us on 8
        // threads, at times 3 ms); 10,000 records 700 us on 2 threads, 350 us on 16
        host_parallel(n, 8192, [&](int64_t b, int64_t e, unsigned t) {
            double m = 0;
            int run = 0;
            for (int64_t i = b; i < e; ++i) {
                PartDev& q = h->hrecs[i];
                make_rec(h, parts[perm[i]], q);
                q.src = image_of.empty() ? perm[i] : image_of[perm[i]];
                m = std::max(m, q.invscale * h->K.mscale);
                // a run of one voxel along a column: one coordinate moves by
                // a >= the largest step per sample row, so it spans at most
                // floor(1 / a) + 1 rows
                const double a = q.invscale * std::max(std::max(fabs(q.R[1]), fabs(q.R[4])) *
                                                           h->K.mscale,
                                                       fabs(q.R[7]) * h->K.mscz);
                run = std::max(run, a > 1e-3 ? (int)std::floor(1.0 / a + 1e-6) + 1 : 1 << 20);
            }
            tmax[t] = m;
            trun[t] = run;
        }, 640);
        for (double m : tmax) max_step = std::max(max_step, m);
        for (int r : trun) max_run = std::max(max_run, r);
    }
    // run merge: equal voxels are contiguous within a merge group of up to 16
    // consecutive samples when 15 steps stay shorter than N - 1 voxels; runs
    // of at most 4 samples need only the first two merge steps
    {
        const int T = h->p.ft_size / 8, MG = T < 16 ? T : 16;
        const bool safe = !h->K.ewald && (MG - 1) * max_step < h->K.N - 1;
        h->K.merge = (h->p.merge != 2) && safe ? (max_run <= 4 ? 2 : 1) : 0;
    }
    BSX_HIP(hipMemcpyAsync(h->recs, h->hrecs, sizeof(PartDev) * n, hipMemcpyHostToDevice, s));
    BSX_HIP(hipEventRecord(h->copied, s));
    add[0] = add[1] = 0;
    for (int64_t i = 0; i < n; ++i)
        if (image_of.empty() || i == 0 || image_of[i] != image_of[i - 1])
            add[h->p.nhalves > 1 ? (parts[i].half & 1) : 0]++;
    *nrec = n;
    return BSX_OK;
}

int bsx_recon_insert(bsx_recon* h, const float* imgs_dev, const bsx_particle* parts, int64_t n,
                     void* stream) {
    BSX_REQUIRE(h, BSX_ERR_ARG, "null handle");
    if (n == 0) return BSX_OK;
    BSX_REQUIRE(n > 0 && imgs_dev && parts, BSX_ERR_ARG, "bsx_recon_insert: bad arguments");
    hipStream_t s = (hipStream_t)stream;
    BSX_HIP(hipSetDevice(h->dev));
    int64_t add[2] = {0, 0};
    {
        const int rp = insert_prepare(h, parts, n, s, &n, add);
        if (rp) return rp;
    }
    const bool rescale = h->p.flags & BSX_FLAG_RESCALE;
    const bool check_nan = h->p.flags & BSX_FLAG_CHECK_NAN;
    if (check_nan) BSX_HIP(hipMemsetAsync(h->nonfinite, 0, sizeof(int), s));
    h->timing = h->p.flags & BSX_FLAG_TIMING;
    h->nev = 0;
    // (the entry count is read with the timing only)
    if (h->binned && h->timing) BSX_HIP(hipMemsetAsync(h->entries, 0, sizeof(unsigned long long), s));
    int r = tmark(h, s, -1);
    if (r) return r;
    hipLaunchKernelGGL(k_background, dim3((unsigned)n), dim3(256), 0, s, imgs_dev, h->recs,
                       h->p.box, h->bkg, check_nan ? h->nonfinite : nullptr,
                       rescale ? h->resc : nullptr);
    BSX_HIP(hipGetLastError());
    if ((r = tmark(h, s, KT_BG))) return r;
    if (check_nan) {
        int bad = 0;
        BSX_HIP(hipMemcpyAsync(&bad, h->nonfinite, sizeof(int), hipMemcpyDeviceToHost, s));
        BSX_HIP(hipStreamSynchronize(s));
        BSX_REQUIRE(!bad, BSX_ERR_NONFINITE, "non-finite values in the particle images");
    }
    h->xdirty = h->bins_dirty = h->binned;
    const int64_t nbatches = (n + h->batch - 1) / h->batch;
    auto batch_loop = [&](hipStream_t st) -> int {
        for (int64_t b = 0; b < nbatches; ++b) {
            const int64_t p0 = b * h->batch;
            const int nb = (int)std::min<int64_t>(h->batch, n - p0);
            const int rr = run_batch(h, imgs_dev, p0, nb, st);
            if (rr) return rr;
        }
        return BSX_OK;
    };
    const bool graph = (h->p.flags & BSX_FLAG_GRAPH) && !h->timing;
    bsx_recon::GraphEntry* ge = nullptr;
    if (graph)
        for (auto& e : h->graphs)
            if (e.imgs == imgs_dev && e.n == n && e.batch == h->batch && e.merge == h->K.merge &&
                e.piece == h->piece) {
                ge = &e;
                ge->used = ++h->graph_clock;
                break;
            }
    if (ge && ge->exec) {
        BSX_HIP(hipGraphLaunch(ge->exec, s));
        h->graph_launches++;
    } else if (ge && ge->seen >= 1) {
        // second identical call: every lazily created resource (twiddles)
        // exists, so the loop can be captured and replayed from now on
        hipGraph_t g = nullptr;
        if (!h->cap_stream) BSX_HIP(hipStreamCreateWithFlags(&h->cap_stream, hipStreamNonBlocking));
        BSX_HIP(hipStreamBeginCapture(h->cap_stream, hipStreamCaptureModeThreadLocal));
        r = batch_loop(h->cap_stream);
        hipError_t ce = hipStreamEndCapture(h->cap_stream, &g);
        if (r) {
            if (g) (void)hipGraphDestroy(g);
            return r;
        }
        BSX_HIP(ce);
        hipError_t ie = hipGraphInstantiate(&ge->exec, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (ie != hipSuccess) ge->exec = nullptr;
        BSX_HIP(ie);
        BSX_HIP(hipGraphLaunch(ge->exec, s));
        h->graph_launches++;
    } else {
        if ((r = batch_loop(s))) return r;
        if (ge) {
            ge->seen++;
        } else if (graph) {
            if (h->graphs.size() >= 8) {
                auto lru = h->graphs.begin();
                for (auto it = h->graphs.begin(); it != h->graphs.end(); ++it)
                    if (it->used < lru->used) lru = it;
                if (lru->exec) (void)hipGraphExecDestroy(lru->exec);
                h->graphs.erase(lru);
            }
            h->graphs.push_back(bsx_recon::GraphEntry{imgs_dev, n, h->batch, h->K.merge, h->piece, 1,
                                                      nullptr, ++h->graph_clock});
        }
    }
    h->bins_dirty = false;   // every batch cleared its bins
    h->inserted[0] += add[0];
    h->inserted[1] += add[1];
    h->last_launches = nbatches;
    if (h->timing) {
        BSX_HIP(hipStreamSynchronize(s));
        for (int q = 0; q < KT_END; ++q) h->ktime[q] = 0;
        for (size_t i = 1; i < h->nev; ++i) {
            float ms = 0;
            BSX_HIP(hipEventElapsedTime(&ms, h->evs[i - 1], h->evs[i]));
            h->ktime[h->evlab[i]] += ms;
        }
        unsigned long long ne = 0;
        if (h->binned) {
            BSX_HIP(hipMemcpy(&ne, h->entries, sizeof(ne), hipMemcpyDeviceToHost));
            int flags = 0;
            BSX_HIP(hipMemcpy(&flags, h->pool + 1, sizeof(int), hipMemcpyDeviceToHost));
            BSX_HIP(hipMemset(h->pool + 1, 0, sizeof(int)));
            h->ktime[KT_FALLBACK] = flags;
            h->fallback_flags |= flags;
        }
        h->last_entries = (double)ne;
    }
    return BSX_OK;
}

// Batch-size autotuner: inserts the sample at each candidate batch (the
// allocated batch and its halvings down to 1/8, at least 32) and keeps the
// fastest. The handle must be empty; it is left empty (accumulators reset).
int bsx_recon_autotune(bsx_recon* h, const float* imgs_dev, const bsx_particle* parts, int64_t n,
                       int32_t* chosen_batch, double* best_ms, void* stream) {
    BSX_REQUIRE(h && imgs_dev && parts && n > 0, BSX_ERR_ARG, "bsx_recon_autotune: bad arguments");
    BSX_REQUIRE(h->inserted[0] == 0 && h->inserted[1] == 0, BSX_ERR_STATE,
                "bsx_recon_autotune: call it before inserting particles");
    hipStream_t s = (hipStream_t)stream;
    const int cap = h->batch_cap;
    const int saved_flags = h->p.flags;
    h->p.flags &= ~(BSX_FLAG_TIMING | BSX_FLAG_GRAPH);
    hipEvent_t e0, e1;
    BSX_HIP(hipEventCreate(&e0));
    BSX_HIP(hipEventCreate(&e1));
    int best = cap, rc = BSX_OK;
    double bms = 1e300;
    for (int div = 8; div >= 1 && rc == BSX_OK; div /= 2) {
        const int b = std::max(32, cap / div);
        if (b > cap || (div > 1 && b == std::max(32, cap / (div / 2)))) continue;
        h->batch = b;
        rc = bsx_recon_insert(h, imgs_dev, parts, n, stream);      // warm-up
        if (rc) break;
        float ms = 0;
        if (hipEventRecord(e0, s) != hipSuccess) { rc = BSX_ERR_DEVICE; break; }
        rc = bsx_recon_insert(h, imgs_dev, parts, n, stream);
        if (rc) break;
        if (hipEventRecord(e1, s) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
            hipEventElapsedTime(&ms, e0, e1) != hipSuccess) {
            set_error("bsx_recon_autotune: timing failed");
            rc = BSX_ERR_DEVICE;
            break;
        }
        if (ms < bms) { bms = ms; best = b; }
    }
    // then the piece length of the tile pass at that batch
    h->batch = best;
    int best_piece = h->piece;
    if (h->binned) {
        for (int pl = BSX_PIECE_MIN; pl <= BSX_PIECE_MAX && rc == BSX_OK; pl *= 2) {
            if (pl == h->piece) continue;   // measured above
            const int saved = h->piece;
            h->piece = pl;
            rc = bsx_recon_insert(h, imgs_dev, parts, n, stream);
            if (rc) break;
            float ms = 0;
            if (hipEventRecord(e0, s) != hipSuccess) { rc = BSX_ERR_DEVICE; break; }
            rc = bsx_recon_insert(h, imgs_dev, parts, n, stream);
            if (rc) break;
            if (hipEventRecord(e1, s) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
                hipEventElapsedTime(&ms, e0, e1) != hipSuccess) {
                set_error("bsx_recon_autotune: timing failed");
                rc = BSX_ERR_DEVICE;
                break;
            }
            if (ms < bms) { bms = ms; best_piece = pl; }
            h->piece = saved;
        }
        h->piece = best_piece;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    h->p.flags = saved_flags;
    h->batch = best;
    h->inserted[0] = h->inserted[1] = 0;
    const int r2 = bsx_recon_reset(h, stream);
    if (rc) return rc;
    if (chosen_batch) *chosen_batch = best;
    if (best_ms) *best_ms = bms;
    return r2;
}

int bsx_recon_tuning(const bsx_recon* h, int32_t* batch, int32_t* piece) {
    BSX_REQUIRE(h, BSX_ERR_ARG, "bsx_recon_tuning: null handle");
    if (batch) *batch = h->batch;
    if (piece) *piece = h->piece;
    return BSX_OK;
}

int bsx_recon_set_tuning(bsx_recon* h, int32_t batch, int32_t piece) {
    BSX_REQUIRE(h, BSX_ERR_ARG, "bsx_recon_set_tuning: null handle");
    BSX_REQUIRE(batch <= h->batch_cap, BSX_ERR_ARG,
                "bsx_recon_set_tuning: batch %d above the allocated %d", batch, h->batch_cap);
    BSX_REQUIRE(piece <= 0 || (piece >= BSX_PIECE_MIN && piece <= BSX_PIECE_MAX &&
                               piece % BSX_CHUNK == 0),
                BSX_ERR_ARG, "bsx_recon_set_tuning: piece %d not a multiple of %d in [%d, %d]",
                piece, BSX_CHUNK, BSX_PIECE_MIN, BSX_PIECE_MAX);
    if (batch > 0) h->batch = batch;
    if (piece > 0) h->piece = piece;
    return BSX_OK;
}

int bsx_recon_set_symmetry(bsx_recon* h, const char* sym) {
    BSX_REQUIRE(h, BSX_ERR_ARG, "bsx_recon_set_symmetry: null handle");
    std::vector<SymOp> ops;
    const int rc = parse_symmetry(sym, ops);
    if (rc) return rc;
    h->sym_order.clear();
    h->sym_axis.clear();
    size_t total = 1;
    for (const SymOp& o : ops) total *= (size_t)o.order;
    if (total <= 1) return BSX_OK;   // C1
    for (const SymOp& o : ops) {
        h->sym_order.push_back(o.order);
        h->sym_axis.insert(h->sym_axis.end(), o.ax, o.ax + 3);
    }
    // the graphs of earlier inserts hold the record counts of those inserts
    clear_graphs(h);
    return BSX_OK;
}

int bsx_symmetry_views(const char* sym, const double* views, int64_t n, double* out, int64_t cap,
                       int64_t* count) {
    BSX_REQUIRE(count && (n == 0 || views) && n >= 0, BSX_ERR_ARG,
                "bsx_symmetry_views: bad arguments");
    std::vector<SymOp> ops;
    const int rc = parse_symmetry(sym, ops);
    if (rc) return rc;
    int64_t order = 1;
    for (const SymOp& o : ops) order *= o.order;
    *count = n * order;
    if (!out) return BSX_OK;
    BSX_REQUIRE(cap >= n * order, BSX_ERR_ARG, "bsx_symmetry_views: room for %lld views, need %lld",
                (long long)cap, (long long)(n * order));
    std::vector<double> sv;
    for (int64_t i = 0; i < n; ++i) {
        for (int c = 0; c < 4; ++c)
            BSX_REQUIRE(std::isfinite(views[4 * i + c]), BSX_ERR_ARG,
                        "bsx_symmetry_views: view %lld is not finite", (long long)i);
        symmetry_views(ops, views + 4 * i, sv);
        std::copy(sv.begin(), sv.end(), out + 4 * i * order);
    }
    return BSX_OK;
}

// n x n x zn maps: zn = n (3D) or 1 (2D images, cyclic groups only).
static int symmetrize_impl(const float* in_dev, float* out_dev, int32_t n, int32_t zn,
                           const double* origin, const char* sym, void* stream) {
    BSX_REQUIRE(in_dev && out_dev && origin && n >= 1 && n <= 2048, BSX_ERR_ARG,
                "bsx_symmetrize: bad arguments");
    BSX_REQUIRE(in_dev != out_dev, BSX_ERR_ARG, "bsx_symmetrize: input and output must differ");
    for (int c = 0; c < 3; ++c)
        BSX_REQUIRE(std::isfinite(origin[c]), BSX_ERR_ARG, "bsx_symmetrize: origin not finite");
    std::vector<SymOp> all, ops;
    const int rc = parse_symmetry(sym, all);
    if (rc) return rc;
    if (zn == 1)   // Bimage::symmetrize on a 2D image (Bimage_symmetry.cpp:40-46)
        for (const SymOp& o : all)
            BSX_REQUIRE(o.ax[0] == 0 && o.ax[1] == 0, BSX_ERR_ARG,
                        "bsx_symmetrize_2d: only cyclic point groups apply to 2D images");
    int64_t order = 1;
    for (const SymOp& o : all) {
        order *= o.order;
        if (o.order > 1) ops.push_back(o);
    }
    hipStream_t s = (hipStream_t)stream;
    const int64_t total = (int64_t)n * n * zn;
    if (ops.empty()) {   // C1 and Cs: Bimage::symmetrize leaves the map unchanged
        BSX_HIP(hipMemcpyAsync(out_dev, in_dev, sizeof(float) * total, hipMemcpyDeviceToDevice, s));
        return BSX_OK;
    }
    // matrices of every operator, j = 1 .. m - 1 (angle j 2 pi / m)
    std::vector<double> mats;
    std::vector<int> first;
    for (const SymOp& o : ops) {
        first.push_back((int)(mats.size() / 9));
        for (int j = 1; j < o.order; ++j) {
            double M[9];
            axis_angle_matrix(o.ax, j * M_PI * 2.0 / o.order, M);
            mats.insert(mats.end(), M, M + 9);
        }
    }
    const int nblk = 1024;
    float* tmp = nullptr;
    double* dm = nullptr;
    double* part = nullptr;
    auto release = [&]() {
        if (tmp) (void)hipFree(tmp);
        if (dm) (void)hipFree(dm);
        if (part) (void)hipFree(part);
    };
    hipError_t e = device_malloc(&dm, sizeof(double) * mats.size());
    if (e == hipSuccess) e = device_malloc(&part, sizeof(double) * (2 * nblk + 1));
    if (e == hipSuccess && ops.size() > 1) e = device_malloc(&tmp, sizeof(float) * total);
    if (e != hipSuccess) {
        release();
        BSX_REQUIRE(false, BSX_ERR_DEVICE, "bsx_symmetrize: device allocation failed (%s)",
                    hipGetErrorString(e));
    }
    e = hipMemcpyAsync(dm, mats.data(), sizeof(double) * mats.size(), hipMemcpyHostToDevice, s);
    double* bkg = part + 2 * nblk;
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_bkg_partial, dim3(nblk), dim3(256), 0, s, in_dev, n, zn, origin[0],
                           origin[1], origin[2], part);
        hipLaunchKernelGGL(k_bkg_final, dim3(1), dim3(64), 0, s, part, nblk, bkg);
        e = hipGetLastError();
    }
    const int K = (int)ops.size();
    const float* src = in_dev;
    for (int k = 0; k < K && e == hipSuccess; ++k) {
        float* dst = ((K - 1 - k) % 2 == 0) ? out_dev : tmp;
        const double scale = k == K - 1 ? 1.0 / (double)order : 1.0;
        hipLaunchKernelGGL(k_sym_op, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, src,
                           dst, n, zn, origin[0], origin[1], origin[2], dm + 9 * first[k],
                           ops[k].order - 1, (const double*)bkg, scale);
        e = hipGetLastError();
        src = dst;
    }
    if (e == hipSuccess) e = hipStreamSynchronize(s);   // the buffers are released below
    release();
    BSX_HIP(e);
    return BSX_OK;
}

int bsx_symmetrize(const float* in_dev, float* out_dev, int32_t n, const double* origin,
                   const char* sym, void* stream) {
    return symmetrize_impl(in_dev, out_dev, n, n, origin, sym, stream);
}

int bsx_symmetrize_2d(const float* in_dev, float* out_dev, int32_t n, const double* origin,
                      const char* sym, void* stream) {
    BSX_REQUIRE(origin, BSX_ERR_ARG, "bsx_symmetrize_2d: null origin");
    const double o3[3] = {origin[0], origin[1], 0.0};
    return symmetrize_impl(in_dev, out_dev, n, 1, o3, sym, stream);
}

// ------------------------------------------------ output map post-processing
// FP64 sum and sum of squares of a float array, per workgroup.
__global__ __launch_bounds__(256) void k_moments(const float* __restrict__ d, long long n,
                                                 double2* __restrict__ part) {
    double s1 = 0, s2 = 0;
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        const double v = d[i];
        s1 += v;
        s2 += v * v;
    }
    __shared__ double a[256], b[256];
    a[threadIdx.x] = s1;
    b[threadIdx.x] = s2;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) {
            a[threadIdx.x] += a[threadIdx.x + o];
            b[threadIdx.x] += b[threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = make_double2(a[0], b[0]);
}

// Scale and shift of Bimage::rescale_to_avg_std (Bimage_rescale.cpp:163-183)
// from the partial moments: average and population standard deviation as
// Bimage::statistics (Bimage_stats.cpp:140-148).
__global__ void k_rescale_coef(const double2* __restrict__ part, int nblk, long long n,
                               double nuavg, double nustd, double2* __restrict__ coef) {
    __shared__ double a[256], b[256];
    double s1 = 0, s2 = 0;
    for (int i = threadIdx.x; i < nblk; i += 256) {
        s1 += part[i].x;
        s2 += part[i].y;
    }
    a[threadIdx.x] = s1;
    b[threadIdx.x] = s2;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) {
            a[threadIdx.x] += a[threadIdx.x + o];
            b[threadIdx.x] += b[threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double avg = a[0] / n;
        const double var = b[0] / n - avg * avg;
        const double sd = var > 0 ? sqrt(var) : 0.0;
        const double sc = sd > 1e-30 ? nustd / sd : 1.0;
        coef[0] = make_double2(sc, nuavg - avg * sc);
    }
}

__global__ __launch_bounds__(256) void k_rescale_apply(float* __restrict__ d, long long n,
                                                       const double2* __restrict__ coef) {
    const double2 c = coef[0];
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256)
        d[i] = (float)((double)d[i] * c.x + c.y);
}

// Bimage::filter_sinc (Bimage_filter.cpp:484-509): every voxel times
// (r / sin r)^2, r = pi |d|, d = (voxel - origin) / size per axis; the
// origin voxel (r = 0) is left as is.
__global__ __launch_bounds__(256) void k_filter_sinc(float* __restrict__ d, int nx, int ny, int nz,
                                                     double ox, double oy, double oz) {
    const long long n = (long long)nx * ny * nz;
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        const int x = (int)(i % nx);
        const long long t = i / nx;
        const int y = (int)(t % ny), z = (int)(t / ny);
        const double dx = (x - ox) / nx, dy = (y - oy) / ny, dz = (z - oz) / nz;
        const double r = M_PI * sqrt(dx * dx + dy * dy + dz * dz);
        if (r != 0) {
            const double w = r / sin(r);
            d[i] = (float)(w * w * (double)d[i]);
        }
    }
}

int bsx_rescale_to_avg_std(float* data_dev, int64_t n, double avg, double std, void* stream) {
    BSX_REQUIRE(data_dev && n > 0, BSX_ERR_ARG, "bsx_rescale_to_avg_std: bad arguments");
    BSX_REQUIRE(std::isfinite(avg) && std::isfinite(std), BSX_ERR_ARG,
                "bsx_rescale_to_avg_std: average and deviation must be finite");
    BSX_REQUIRE(std >= 0, BSX_ERR_ARG,
                "bsx_rescale_to_avg_std: cannot use a negative standard deviation (%g)", std);
    hipStream_t s = (hipStream_t)stream;
    const int nblk = (int)std::min<int64_t>(1024, (n + 255) / 256);
    Scratch buf;
    BSX_HIP(buf.get(sizeof(double2) * (nblk + 1)));
    double2* part = buf.as<double2>();
    hipLaunchKernelGGL(k_moments, dim3(nblk), dim3(256), 0, s, data_dev, (long long)n, part);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_rescale_coef, dim3(1), dim3(256), 0, s, part, nblk, (long long)n, avg,
                           std, part + nblk);
        e = hipGetLastError();
    }
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_rescale_apply, dim3(nblk), dim3(256), 0, s, data_dev, (long long)n,
                           part + nblk);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    BSX_HIP(e);
    buf.release();
    return BSX_OK;
}

int bsx_filter_sinc(float* data_dev, int32_t nx, int32_t ny, int32_t nz, const double* origin,
                    void* stream) {
    BSX_REQUIRE(data_dev && origin && nx > 0 && ny > 0 && nz > 0, BSX_ERR_ARG,
                "bsx_filter_sinc: bad arguments");
    BSX_REQUIRE(std::isfinite(origin[0]) && std::isfinite(origin[1]) && std::isfinite(origin[2]),
                BSX_ERR_ARG, "bsx_filter_sinc: origin not finite");
    const long long n = (long long)nx * ny * nz;
    const int nblk = (int)std::min<long long>(4096, (n + 255) / 256);
    hipLaunchKernelGGL(k_filter_sinc, dim3(nblk), dim3(256), 0, (hipStream_t)stream, data_dev, nx,
                       ny, nz, origin[0], origin[1], origin[2]);
    BSX_HIP(hipGetLastError());
    return BSX_OK;
}

int bsx_recon_fallbacks(const bsx_recon* h, int32_t* flags) {
    BSX_REQUIRE(h && flags, BSX_ERR_ARG, "null argument");
    *flags = h->fallback_flags;
    return BSX_OK;
}

int bsx_recon_graph_launches(const bsx_recon* h, int64_t* n) {
    BSX_REQUIRE(h && n, BSX_ERR_ARG, "bsx_recon_graph_launches: null argument");
    *n = h->graph_launches;
    return BSX_OK;
}

int bsx_recon_last_timing(const bsx_recon* h, double* insert_ms, int64_t* launches,
                          double* stage_ms) {
    BSX_REQUIRE(h, BSX_ERR_ARG, "null handle");
    const double* t = h->ktime;
    if (insert_ms) *insert_ms = t[KT_SCAN] + t[KT_FILL] + t[KT_TILE] + t[KT_DIRECT];
    if (launches) *launches = h->last_launches;
    if (stage_ms) *stage_ms = t[KT_BG] + t[KT_ROWS];
    return BSX_OK;
}

int bsx_recon_kernel_times(const bsx_recon* h, double* ms, int n) {
    BSX_REQUIRE(h && ms && n >= 0, BSX_ERR_ARG, "null argument");
    for (int q = 0; q < n && q < KT_END; ++q) ms[q] = h->ktime[q];
    if (n > KT_END) ms[KT_END] = h->last_entries;
    return BSX_OK;
}

// Brings the binned accumulator into the volume records (stream-ordered after
// the inserts) where entries were binned since the last fold; a recorded fold
// always, since its graph may be replayed after any insert.
static int fold(bsx_recon* h, hipStream_t s) {
    const bool rec = recording(s);
    if (!h->binned || !(rec || h->xdirty)) return BSX_OK;
    const long long n3 = (long long)h->K.N * h->K.N * h->K.N;
    const long long nrec = (long long)h->K.NT * h->K.NT * h->K.NT * 4096;
    hipLaunchKernelGGL(k_fold, dim3(2048), dim3(256), 0, s, h->acc, h->xacc, n3, h->K.N, h->K.NT,
                       nrec, h->p.nhalves, h->K.stride);
    BSX_HIP(hipGetLastError());
    if (!rec) h->xdirty = false;
    return BSX_OK;
}

int bsx_recon_accumulators(bsx_recon* h, int half, float* planes_dev, void* stream) {
    BSX_REQUIRE(h && planes_dev, BSX_ERR_ARG, "null argument");
    BSX_REQUIRE(half >= 0 && half < h->p.nhalves, BSX_ERR_ARG, "half %d out of range", half);
    const int rf = fold(h, (hipStream_t)stream);
    if (rf) return rf;
    const long long n3 = (long long)h->K.N * h->K.N * h->K.N;
    const long long nrec = (long long)h->K.NT * h->K.NT * h->K.NT * 4096;
    hipLaunchKernelGGL(k_planes, dim3(1024), dim3(256), 0, (hipStream_t)stream,
                       h->acc + (size_t)half * nrec * h->K.stride, n3, h->K.N, h->K.NT,
                       h->K.stride, h->K.fom, planes_dev);
    BSX_HIP(hipGetLastError());
    return BSX_OK;
}

int bsx_recon_set_accumulators(bsx_recon* h, int half, const float* planes_dev, int64_t count,
                               void* stream) {
    BSX_REQUIRE(h && planes_dev, BSX_ERR_ARG, "null argument");
    BSX_REQUIRE(half >= 0 && half < h->p.nhalves, BSX_ERR_ARG, "half %d out of range", half);
    BSX_REQUIRE(count >= 0, BSX_ERR_ARG, "negative particle count");
    hipStream_t s = (hipStream_t)stream;
    BSX_HIP(hipSetDevice(h->dev));
    const int rf = fold(h, s);   // the pair accumulator is empty afterwards
    if (rf) return rf;
    const long long n3 = (long long)h->K.N * h->K.N * h->K.N;
    const long long nrec = (long long)h->K.NT * h->K.NT * h->K.NT * 4096;
    hipLaunchKernelGGL(k_set_planes, dim3(1024), dim3(256), 0, s,
                       h->acc + (size_t)half * nrec * h->K.stride, n3, h->K.N, h->K.NT,
                       h->K.stride, planes_dev);
    BSX_HIP(hipGetLastError());
    h->inserted[half] = count;
    return BSX_OK;
}

int bsx_recon_stats(bsx_recon* h, int imap, int nmaps, double resolution, double* rows,
                    int32_t cap, int32_t* nrows, double* estimates, void* stream) {
    BSX_REQUIRE(h && nrows, BSX_ERR_ARG, "bsx_recon_stats: null argument");
    BSX_REQUIRE(h->K.fom, BSX_ERR_STATE, "bsx_recon_stats needs BSX_FLAG_FOM");
    BSX_REQUIRE(nmaps >= 1 && nmaps <= 3 && imap >= 0 && imap < nmaps, BSX_ERR_ARG,
                "imap %d / nmaps %d invalid", imap, nmaps);
    BSX_REQUIRE(std::isfinite(resolution), BSX_ERR_ARG, "bsx_recon_stats: resolution not finite");
    int hmask = 3;
    if (nmaps == 2) hmask = 1 << (imap % 2);
    if (nmaps == 3 && imap % 3) hmask = 1 << (imap % 3 - 1);
    if (h->p.nhalves == 1) {
        BSX_REQUIRE(hmask == 3, BSX_ERR_STATE, "half maps need nhalves = 2");
        hmask = 1;
    }
    const int N = h->K.N, nz = h->K.nz;   // nz = 1: a 2D map
    const double rs = N * h->p.sampling;   // real size = rad_scale (sampling ratio 1)
    // fspace_maximum_radius (Bimage_fspace.cpp:26-38) of the resolution as
    // given (the table's rows) and as check_resolution clamps it (the radial
    // power spectrum); Bimage::radial keeps at most N/2 shells
    auto maxrad = [&](double res) -> long { return res > 0.1 ? (long)(rs / res) : (long)(N / 2.0); };
    const long nr_stats = maxrad(resolution);
    const long nr1 = std::max<long>(
        1, maxrad(check_resolution(resolution, N, h->p.sampling, nz > 1 ? 3 : 2)));
    long nr2 = nr_stats < 1 ? N / 2 : std::min<long>(nr_stats, N / 2);
    nr2 = std::min(nr2, nr1);
    const size_t shm = sizeof(double) * 6 * nr1;
    BSX_REQUIRE(shm <= 64 * 1024, BSX_ERR_ARG, "bsx_recon_stats: %ld shells exceed the LDS table",
                nr1);
    hipStream_t s = (hipStream_t)stream;
    BSX_HIP(hipSetDevice(h->dev));
    const int rf = fold(h, s);
    if (rf) return rf;
    const int nblk = 1024;
    const int m = (int)(6 * nr1);
    double* part = nullptr;
    BSX_HIP(device_malloc(&part, sizeof(double) * ((size_t)nblk * m + m)));
    double* dsum = part + (size_t)nblk * m;
    const long long n3 = (long long)N * N * nz;
    const long long nrec = (long long)h->K.NT * h->K.NT * h->K.NT * 4096;
    hipLaunchKernelGGL(k_recon_stats, dim3(nblk), dim3(256), shm, s, h->acc, n3, N, nz, h->K.NT, nrec,
                       h->K.stride, hmask, h->p.nhalves, rs, 1.0 / rs, (int)nr1, (int)nr2, part);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_stats_sum, dim3((m + 255) / 256), dim3(256), 0, s, part, nblk, m, dsum);
        e = hipGetLastError();
    }
    std::vector<double> S((size_t)m);
    if (e == hipSuccess)
        e = hipMemcpyAsync(S.data(), dsum, sizeof(double) * m, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    (void)hipFree(part);
    BSX_HIP(e);
    // radial averages: sum / count where the count is nonzero, else 0
    auto avg = [&](int q, int c, long i) {
        const double n = S[(size_t)c * nr1 + i];
        return n != 0 ? S[(size_t)q * nr1 + i] / n : 0.0;
    };
    // the table (fspace_reconstruction_stats :547-593); rows beyond the
    // shorter radial arrays are not defined there and are left out
    const long nrow = std::max<long>(0, std::min(nr_stats, nr2) - 1);
    *nrows = (int32_t)nrow;
    double fscp = 1, snrp = 10, res_fsc = 0, res_snr = 0;
    const double fsc_cut = 0.3, snr_cut = 0.5;
    for (long i = 1; i <= nrow; ++i) {
        const double sfreq = i / rs, res = rs / i;
        const double prad = avg(1, 0, i), pfom = avg(3, 2, i);
        const double w = avg(4, 2, i);
        double fsc = 0, snr = 0, signal = 0, noise = 0;
        if (w > 1e-3) {
            const double w2 = avg(5, 2, i);
            noise = (pfom - prad) / w2;
            signal = (w * prad - pfom) / w2;
            if (noise > 0) snr = signal / noise;
            fsc = snr / (snr + 1);
            if (fsc < 0) fsc = 0;
        }
        if (fscp >= fsc_cut && fsc < fsc_cut) res_fsc = 1 / (sfreq - (fsc_cut - fsc) / ((fscp - fsc) * rs));
        if (snrp >= snr_cut && snr < snr_cut) res_snr = 1 / (sfreq - (snr_cut - snr) / ((snrp - snr) * rs));
        fscp = fsc;
        snrp = snr;
        if (rows && i <= cap) {
            double* r = rows + 9 * (i - 1);
            r[0] = (double)i;
            r[1] = sfreq;
            r[2] = res;
            r[3] = w;
            r[4] = prad;
            r[5] = signal;
            r[6] = noise;
            r[7] = snr;
            r[8] = fsc;
        }
    }
    if (estimates) {
        estimates[0] = res_snr;
        estimates[1] = res_fsc;
    }
    return BSX_OK;
}

// Weighing of the summed halves in hmask into vol (and the FOM map), after
// folding the binned accumulator where `fold` is set; the coverage count and the
// weight and Friedel sums are added to fin (5 doubles), which the caller has
// cleared; with `flags` the fallback flags move from there to fin's sixth place.
static int launch_weigh(bsx_recon* h, int hmask, bool fold, float2* vol, float* fom_dev, double* fin,
                        int* flags, hipStream_t s) {
    const int N = h->K.N, nz = h->K.nz;
    const long long nrec = (long long)h->K.NT * h->K.NT * h->K.NT * 4096;
    const long long pairs = (long long)(N / 2 + 1) * N * nz;
    const dim3 grid((unsigned)std::min(512LL, (pairs + 1023) / 1024));
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(1024), 0, s, h->acc, h->xacc, N, nz, h->K.NT, nrec, hmask,
                           h->p.nhalves, vol, fom_dev, fin, flags);
    };
    if (h->K.fom) fold ? go(k_weigh_pairs<true, true>) : go(k_weigh_pairs<true, false>);
    else fold ? go(k_weigh_pairs<false, true>) : go(k_weigh_pairs<false, false>);
    BSX_HIP(hipGetLastError());
    return BSX_OK;
}

// Inverse transform of the weighed (centre-shifted) transform in work, which
// it overwrites; the real part, scaled by 1/sqrt(voxels), goes to map_dev.
static int launch_inverse(bsx_recon* h, float2* work, float* map_dev, hipStream_t s) {
    const int N = h->K.N, nz = h->K.nz;
    const float sc = (float)(1.0 / sqrt((double)N * N * nz));
    int r = fft_axis_ex(work, nullptr, N, N, nz, 1, 0, +1, 1.0f, s);
    if (nz == 1) {
        if (r == BSX_OK) r = fft_axis_ex(work, map_dev, N, N, 1, 1, 1, +1, sc, s);
    } else {
        if (r == BSX_OK) r = fft_axis_ex(work, nullptr, N, N, N, 1, 1, +1, 1.0f, s);
        if (r == BSX_OK) r = fft_axis_ex(work, map_dev, N, N, N, 1, 2, +1, sc, s);
    }
    return r;
}

// The stats of a finish from the sums of launch_weigh.
static void fill_stats(const bsx_recon* h, int hmask, const double* fin, bsx_stats* stats) {
    stats->coverage = (int64_t)fin[0];
    stats->weight_sum = fin[1];
    double sw = fin[2], rr = fin[3], ri = fin[4];
    double fr = 0;
    if (sw > 0) {
        rr = sqrt(rr / sw);
        ri = sqrt(ri / sw);
        fr = sqrt(rr * rr + ri * ri);
    }
    stats->friedel = fr;
    int64_t np = 0;
    for (int q = 0; q < h->p.nhalves; ++q)
        if ((hmask >> q) & 1) np += h->inserted[q];
    stats->particles = np;
}

int bsx_recon_finish(bsx_recon* h, int imap, int nmaps, float* map_dev, float* fom_dev,
                     float* ft_dev, bsx_stats* stats, void* stream) {
    BSX_REQUIRE(h, BSX_ERR_ARG, "null handle");
    BSX_REQUIRE(nmaps >= 1 && nmaps <= 3 && imap >= 0 && imap < nmaps, BSX_ERR_ARG,
                "imap %d / nmaps %d invalid", imap, nmaps);
    BSX_REQUIRE(!fom_dev || h->K.fom, BSX_ERR_STATE, "FOM map requested without BSX_FLAG_FOM");
    int hmask = 3;
    if (nmaps == 2) hmask = 1 << (imap % 2);
    if (nmaps == 3 && imap % 3) hmask = 1 << (imap % 3 - 1);
    if (h->p.nhalves == 1) {
        BSX_REQUIRE(hmask == 3, BSX_ERR_STATE, "half maps need nhalves = 2");
        hmask = 1;
    }
    hipStream_t s = (hipStream_t)stream;
    BSX_HIP(hipSetDevice(h->dev));
    const int N = h->K.N, nz = h->K.nz;
    const long long n3 = (long long)N * N * nz;   // a 2D map: one plane
    float2* vol = (float2*)ft_dev;
    Scratch tmp, wtmp, fin, pin(true);
    if (!vol) {
        BSX_HIP(tmp.get(sizeof(float2) * n3));
        vol = tmp.as<float2>();
    }
    // the finish sums and, after them, the atomic-fallback flags of the inserts
    // since the last read (graph replays included; cleared for the next inserts)
    BSX_HIP(fin.get(6 * sizeof(double)));
    BSX_HIP(pin.get(6 * sizeof(double)));
    BSX_HIP(hipMemsetAsync(fin.as<double>(), 0, 6 * sizeof(double), s));
    {
        const int rw = launch_weigh(h, hmask, h->binned && h->xdirty, vol, fom_dev, fin.as<double>(),
                                    h->binned ? h->pool + 1 : nullptr, s);
        if (rw) return rw;
        h->xdirty = false;
    }
    BSX_HIP(hipMemcpyAsync(pin.as<double>(), fin.as<double>(), 6 * sizeof(double), hipMemcpyDeviceToHost, s));
    int r = BSX_OK;
    if (map_dev) {
        // inverse transform: work on a copy when the caller wants the transform back
        float2* work = vol;
        if (ft_dev) {
            BSX_HIP(wtmp.get(sizeof(float2) * n3));
            work = wtmp.as<float2>();
            BSX_HIP(hipMemcpyAsync(work, vol, sizeof(float2) * n3, hipMemcpyDeviceToDevice, s));
        }
        r = launch_inverse(h, work, map_dev, s);
    }
    BSX_HIP(hipStreamSynchronize(s));
    int flags = 0;
    memcpy(&flags, pin.as<double>() + 5, sizeof(flags));
    h->fallback_flags |= flags;
    if (r == BSX_OK && stats) fill_stats(h, hmask, pin.as<double>(), stats);
    tmp.release();
    wtmp.release();
    fin.release();
    pin.release();
    return r;
}


// ---- group runs: several reconstructions (e.g. one per particle box) as one graph ----

static void set32(void* p, long long n, unsigned v, hipStream_t s) {
    const long long blocks = std::max(1LL, std::min(2048LL, (n / 4 + 255) / 256));
    hipLaunchKernelGGL(k_set32, dim3((unsigned)blocks), dim3(256), 0, s, (unsigned*)p, n, v,
                       ((uintptr_t)p & 15) == 0 ? 1 : 0);
}

// One member's part of a group run, kernels only: accumulator and bin-state
// clears, staging of the n records uploaded by insert_prepare, the batch
// loop, then the fold, weighing and inverse transform into map_dev.
static int group_member_launch(bsx_recon* h, const float* imgs, int64_t n, float* map_dev,
                               hipStream_t s) {
    set32(h->acc, (long long)h->acc_elems, 0u, s);
    if (h->binned) {
        set32(h->xacc, (long long)h->acc_elems, 0u, s);
        set32(h->fill, h->nbins, 0u, s);
        set32(h->chunks, (long long)h->nbins * h->maxc, 0xFFFFFFFFu, s);
        set32(h->pool, 2, 0u, s);
        set32(h->entries, 2, 0u, s);
    }
    set32(h->gfin, 10, 0u, s);
    hipLaunchKernelGGL(k_background, dim3((unsigned)n), dim3(256), 0, s, imgs, h->recs, h->p.box,
                       h->bkg, nullptr, (h->p.flags & BSX_FLAG_RESCALE) ? h->resc : nullptr);
    BSX_HIP(hipGetLastError());
    const int64_t nbatches = (n + h->batch - 1) / h->batch;
    for (int64_t b = 0; b < nbatches; ++b) {
        const int64_t p0 = b * h->batch;
        const int rr = run_batch(h, imgs, p0, (int)std::min<int64_t>(h->batch, n - p0), s);
        if (rr) return rr;
    }
    const int r = launch_weigh(h, h->p.nhalves > 1 ? 3 : 1, h->binned, h->gvol, nullptr, h->gfin, nullptr, s);
    if (r) return r;
    return launch_inverse(h, h->gvol, map_dev, s);
}

struct bsx_recon_group {
    std::vector<bsx_recon*> hs;
    int dev = 0;
    hipGraphExec_t gexec = nullptr;
    hipStream_t cap_stream = nullptr;
    std::vector<uintptr_t> key;    // everything a captured launch depends on
    int seen = 0;                  // identical runs seen (capture on the second)
    int64_t graph_launches = 0;
};

int bsx_recon_group_create(bsx_recon* const* recons, int count, bsx_recon_group** out) {
    BSX_REQUIRE(out && recons && count >= 1 && count <= 64, BSX_ERR_ARG,
                "bsx_recon_group_create: bad arguments");
    *out = nullptr;
    for (int i = 0; i < count; ++i) {
        BSX_REQUIRE(recons[i], BSX_ERR_ARG, "bsx_recon_group_create: null handle %d", i);
        BSX_REQUIRE(recons[i]->dev == recons[0]->dev, BSX_ERR_ARG,
                    "bsx_recon_group_create: handles on different devices");
        for (int j = 0; j < i; ++j)
            BSX_REQUIRE(recons[j] != recons[i], BSX_ERR_ARG,
                        "bsx_recon_group_create: handle %d repeated", i);
    }
    bsx_recon_group* g = new bsx_recon_group();
    g->hs.assign(recons, recons + count);
    g->dev = recons[0]->dev;
    *out = g;
    return BSX_OK;
}

int bsx_recon_group_destroy(bsx_recon_group* g) {
    if (!g) return BSX_OK;
    (void)hipSetDevice(g->dev);
    if (g->gexec) (void)hipGraphExecDestroy(g->gexec);
    if (g->cap_stream) (void)hipStreamDestroy(g->cap_stream);
    delete g;
    return BSX_OK;
}

int bsx_recon_group_graph_launches(const bsx_recon_group* g, int64_t* n) {
    BSX_REQUIRE(g && n, BSX_ERR_ARG, "bsx_recon_group_graph_launches: null argument");
    *n = g->graph_launches;
    return BSX_OK;
}

int bsx_recon_group_run(bsx_recon_group* g, const float* const* imgs_dev,
                        const bsx_particle* const* parts, const int64_t* counts,
                        float* const* maps_dev, bsx_stats* stats, void* stream) {
    BSX_REQUIRE(g && imgs_dev && parts && counts && maps_dev, BSX_ERR_ARG,
                "bsx_recon_group_run: null argument");
    hipStream_t s = (hipStream_t)stream;
    BSX_HIP(hipSetDevice(g->dev));
    const int m = (int)g->hs.size();
    for (int i = 0; i < m; ++i) {
        const bsx_recon* h = g->hs[i];
        BSX_REQUIRE(counts[i] > 0 && imgs_dev[i] && parts[i] && maps_dev[i], BSX_ERR_ARG,
                    "bsx_recon_group_run: member %d: bad arguments", i);
        BSX_REQUIRE(!(h->p.flags & BSX_FLAG_CHECK_NAN), BSX_ERR_STATE,
                    "bsx_recon_group_run: member %d: BSX_FLAG_CHECK_NAN needs a host check "
                    "between staging and insertion, which a single graph cannot hold", i);
    }
    // finish buffers (allocated outside any capture)
    for (bsx_recon* h : g->hs) {
        const size_t n3 = (size_t)h->K.N * h->K.N * h->K.nz;
        if (!h->gvol) BSX_HIP(device_malloc(&h->gvol, sizeof(float2) * n3));
        if (!h->gfin) BSX_HIP(device_malloc(&h->gfin, 64));
    }
    // a run that stops half-way leaves its members to be cleared
    for (bsx_recon* h : g->hs) h->xdirty = h->bins_dirty = h->binned;
    // host side of every member's insert: records uploaded on s
    std::vector<int64_t> nrec(m), add(2 * m);
    for (int i = 0; i < m; ++i) {
        bsx_recon* h = g->hs[i];
        h->timing = false;
        const int r = insert_prepare(h, parts[i], counts[i], s, &nrec[i], &add[2 * i]);
        if (r) return r;
    }
    std::vector<uintptr_t> key;
    key.reserve(12 * m);
    for (int i = 0; i < m; ++i) {
        const bsx_recon* h = g->hs[i];
        const uintptr_t k[] = {(uintptr_t)h, (uintptr_t)imgs_dev[i], (uintptr_t)nrec[i],
                               (uintptr_t)h->batch, (uintptr_t)h->K.merge, (uintptr_t)h->piece,
                               (uintptr_t)maps_dev[i], (uintptr_t)h->recs, (uintptr_t)h->bkg,
                               (uintptr_t)h->resc, (uintptr_t)h->gvol, (uintptr_t)h->gfin};
        key.insert(key.end(), k, k + 12);
    }
    auto launch_all = [&](hipStream_t st) -> int {
        for (int i = 0; i < m; ++i) {
            const int r = group_member_launch(g->hs[i], imgs_dev[i], nrec[i], maps_dev[i], st);
            if (r) return r;
        }
        return BSX_OK;
    };
    const bool same = key == g->key;
    if (same && g->gexec) {
        BSX_HIP(hipGraphLaunch(g->gexec, s));
        g->graph_launches++;
    } else if (same && g->seen >= 1) {
        // second identical run: the lazily created resources (twiddle tables)
        // exist, so the whole run is captured once and replayed from now on
        hipGraph_t gr = nullptr;
        if (!g->cap_stream)
            BSX_HIP(hipStreamCreateWithFlags(&g->cap_stream, hipStreamNonBlocking));
        // the capture stream starts after the record uploads queued on s
        hipEvent_t up = nullptr;
        BSX_HIP(hipEventCreateWithFlags(&up, hipEventDisableTiming));
        BSX_HIP(hipEventRecord(up, s));
        BSX_HIP(hipStreamWaitEvent(g->cap_stream, up, 0));
        (void)hipEventDestroy(up);
        BSX_HIP(hipStreamBeginCapture(g->cap_stream, hipStreamCaptureModeThreadLocal));
        const int r = launch_all(g->cap_stream);
        const hipError_t ce = hipStreamEndCapture(g->cap_stream, &gr);
        if (r) {
            if (gr) (void)hipGraphDestroy(gr);
            return r;
        }
        BSX_HIP(ce);
        const hipError_t ie = hipGraphInstantiate(&g->gexec, gr, nullptr, nullptr, 0);
        (void)hipGraphDestroy(gr);
        if (ie != hipSuccess) g->gexec = nullptr;
        BSX_HIP(ie);
        BSX_HIP(hipGraphLaunch(g->gexec, s));
        g->graph_launches++;
    } else {
        if (g->gexec) (void)hipGraphExecDestroy(g->gexec);
        g->gexec = nullptr;
        g->key = key;
        g->seen = 1;
        const int r = launch_all(s);
        if (r) {
            g->key.clear();
            return r;
        }
    }
    if (same) g->seen++;
    // finish sums and capacity-fallback flags of every member
    std::vector<double> fin(5 * m);
    std::vector<int> flags(m, 0);
    for (int i = 0; i < m; ++i) {
        bsx_recon* h = g->hs[i];
        BSX_HIP(hipMemcpyAsync(&fin[5 * i], h->gfin, 5 * sizeof(double),
                               hipMemcpyDeviceToHost, s));
        if (h->binned)
            BSX_HIP(hipMemcpyAsync(&flags[i], h->pool + 1, sizeof(int), hipMemcpyDeviceToHost, s));
    }
    BSX_HIP(hipStreamSynchronize(s));
    for (int i = 0; i < m; ++i) {
        bsx_recon* h = g->hs[i];
        h->inserted[0] = add[2 * i];
        h->inserted[1] = add[2 * i + 1];
        h->fallback_flags |= flags[i];
        h->last_launches = (nrec[i] + h->batch - 1) / h->batch;
        h->xdirty = h->bins_dirty = false;   // cleared, inserted and folded above
        if (stats) fill_stats(h, h->p.nhalves > 1 ? 3 : 1, &fin[5 * i], &stats[i]);
    }
    return BSX_OK;
}

}  // extern "C"
