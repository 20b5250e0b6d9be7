// bsx_cnn.hip — the orientation-proposal network: a 5-layer CNN trained and
// run by hand-written HIP kernels (no library GEMMs).
//
// Architecture (input S x S, one channel; S a multiple of 8):
//   conv3x3 stride 1 (1 -> c1) + ReLU    S   x S
//   conv3x3 stride 2 (c1 -> c2) + ReLU   S/2 x S/2
//   conv3x3 stride 2 (c2 -> c3) + ReLU   S/4 x S/4
//   conv3x3 stride 2 (c3 -> c4) + ReLU   S/8 x S/8
//   fully connected (c4 (S/8)^2 -> nclasses), softmax cross-entropy
// Parameters are one flat FP32 array (W1 b1 W2 b2 W3 b3 W4 b4 Wfc bfc; conv
// weights [cout][cin][3][3], Wfc [class][feature]). Training: Adam on the
// FP32 master weights. Inference: BF16 copies of the weights with FP32
// accumulation and a fused per-row top-k of the softmax.
#include <cmath>
#include <cstring>
#include <algorithm>
#include <vector>

#include "bsx_common.h"

using namespace bsx;

namespace {

__device__ inline float bf16_to_f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

__host__ __device__ inline uint16_t f_to_bf16(float f) {
    uint32_t u = __builtin_bit_cast(uint32_t, f);
    if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)((u >> 16) | ((u & 0xffff) ? 0x40 : 0));
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

unsigned nblk(long n, int t = 256) { return (unsigned)std::min<long>((n + t - 1) / t, 1l << 30); }

template <typename T> __device__ inline float ldw(const T* p, long i);
template <> __device__ inline float ldw<float>(const float* p, long i) { return p[i]; }
template <> __device__ inline float ldw<uint16_t>(const uint16_t* p, long i) { return bf16_to_f(p[i]); }

// ---------------------------------------------------------------- conv fwd
// y[b][co][yo][xo] = relu(bias[co] + sum W[co][ci][ky][kx] x[b][ci][yo*s-1+ky][xo*s-1+kx]);
// one thread per (b, 4 output channels, yo, xo).
template <typename TW>
__global__ __launch_bounds__(256) void k_conv_fwd(const float* __restrict__ x, const TW* __restrict__ W,
                                                  const TW* __restrict__ bias, float* __restrict__ y,
                                                  int B, int Cin, int H, int Wd, int Cout, int Ho,
                                                  int Wo, int stride) {
    const long total = (long)B * (Cout / 4) * Ho * Wo;
    const long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= total) return;
    const int xo = (int)(g % Wo);
    const int yo = (int)((g / Wo) % Ho);
    const int c4 = (int)((g / ((long)Wo * Ho)) % (Cout / 4));
    const int b = (int)(g / ((long)Wo * Ho * (Cout / 4)));
    const int co = 4 * c4;
    float acc[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[q] = ldw(bias, co + q);
    const float* xb = x + (long)b * Cin * H * Wd;
    for (int ci = 0; ci < Cin; ++ci) {
        const float* xc = xb + (long)ci * H * Wd;
#pragma unroll
        for (int ky = 0; ky < 3; ++ky) {
            const int yi = yo * stride - 1 + ky;
            if (yi < 0 || yi >= H) continue;
#pragma unroll
            for (int kx = 0; kx < 3; ++kx) {
                const int xi = xo * stride - 1 + kx;
                if (xi < 0 || xi >= Wd) continue;
                const float v = xc[yi * Wd + xi];
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    acc[q] = fmaf(ldw(W, (((long)(co + q) * Cin + ci) * 3 + ky) * 3 + kx), v, acc[q]);
            }
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q)
        y[(((long)b * Cout + co + q) * Ho + yo) * Wo + xo] = fmaxf(acc[q], 0.f);
}

// g <- g * (y > 0): the ReLU backward, in place.
__global__ void k_relu_bwd(float* __restrict__ g, const float* __restrict__ y, long n) {
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        if (!(y[i] > 0.f)) g[i] = 0.f;
}

// dx[b][ci][yi][xi] = sum_{co,ky,kx} W[co][ci][ky][kx] g[b][co][yo][xo],
// yo = (yi + 1 - ky) / s when divisible and in range.
__global__ __launch_bounds__(256) void k_conv_bwd_data(const float* __restrict__ g,
                                                       const float* __restrict__ W,
                                                       float* __restrict__ dx, int B, int Cin, int H,
                                                       int Wd, int Cout, int Ho, int Wo, int stride) {
    const long total = (long)B * Cin * H * Wd;
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= total) return;
    const int xi = (int)(t % Wd);
    const int yi = (int)((t / Wd) % H);
    const int ci = (int)((t / ((long)Wd * H)) % Cin);
    const int b = (int)(t / ((long)Wd * H * Cin));
    float acc = 0.f;
    for (int co = 0; co < Cout; ++co) {
        const float* gc = g + ((long)b * Cout + co) * Ho * Wo;
        const float* wc = W + ((long)co * Cin + ci) * 9;
#pragma unroll
        for (int ky = 0; ky < 3; ++ky) {
            const int ny = yi + 1 - ky;
            if (ny < 0 || ny % stride) continue;
            const int yo = ny / stride;
            if (yo >= Ho) continue;
#pragma unroll
            for (int kx = 0; kx < 3; ++kx) {
                const int nx = xi + 1 - kx;
                if (nx < 0 || nx % stride) continue;
                const int xo = nx / stride;
                if (xo >= Wo) continue;
                acc = fmaf(wc[ky * 3 + kx], gc[yo * Wo + xo], acc);
            }
        }
    }
    dx[t] = acc;
}

// dW[co][ci][9] = sum_{b,yo,xo} g[b][co][yo][xo] x[b][ci][yo*s-1+ky][xo*s-1+kx];
// one workgroup per (co, ci); blockIdx.y == Cin gives db[co] = sum g.
__global__ __launch_bounds__(256) void k_conv_bwd_weight(const float* __restrict__ g,
                                                         const float* __restrict__ x,
                                                         float* __restrict__ dW, float* __restrict__ db,
                                                         int B, int Cin, int H, int Wd, int Cout,
                                                         int Ho, int Wo, int stride) {
    __shared__ float red[10][256];
    const int co = blockIdx.x, ci = blockIdx.y;
    float acc[9];
#pragma unroll
    for (int q = 0; q < 9; ++q) acc[q] = 0.f;
    float sb = 0.f;
    const long per = (long)Ho * Wo;
    for (long e = threadIdx.x; e < (long)B * per; e += blockDim.x) {
        const int b = (int)(e / per);
        const int r = (int)(e % per);
        const int yo = r / Wo, xo = r % Wo;
        const float gv = g[((long)b * Cout + co) * per + r];
        if (ci == Cin) {
            sb += gv;
            continue;
        }
        const float* xc = x + ((long)b * Cin + ci) * H * Wd;
#pragma unroll
        for (int ky = 0; ky < 3; ++ky) {
            const int yi = yo * stride - 1 + ky;
            if (yi < 0 || yi >= H) continue;
#pragma unroll
            for (int kx = 0; kx < 3; ++kx) {
                const int xi = xo * stride - 1 + kx;
                if (xi < 0 || xi >= Wd) continue;
                acc[ky * 3 + kx] = fmaf(gv, xc[yi * Wd + xi], acc[ky * 3 + kx]);
            }
        }
    }
#pragma unroll
    for (int q = 0; q < 9; ++q) red[q][threadIdx.x] = acc[q];
    red[9][threadIdx.x] = sb;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s)
#pragma unroll
            for (int q = 0; q < 10; ++q) red[q][threadIdx.x] += red[q][threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        if (ci == Cin) db[co] = red[9][0];
        else
            for (int q = 0; q < 9; ++q) dW[((long)co * Cin + ci) * 9 + q] = red[q][0];
    }
}

// ------------------------------------------------------------------ GEMM
// C[m][n] = sum_k A[m*am + k*ak] * B[k*bk + n*bn] (+ bias[n]) with BF16 B and bias
// (inference of networks that the matrix-core kernels do not take); 64x64 tiles,
// K step 16 through LDS, 4x4 outputs per thread, edges guarded.
__global__ __launch_bounds__(256) void k_sgemm(int M, int N, int K, const float* __restrict__ A,
                                               long am, long ak, const uint16_t* __restrict__ Bm,
                                               long bk, long bn, const uint16_t* __restrict__ bias,
                                               float* __restrict__ Cm, long ldc) {
    __shared__ float As[16][64 + 4];
    __shared__ float Bs[16][64 + 4];
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
    float acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;
    for (int k0 = 0; k0 < K; k0 += 16) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int e = threadIdx.x + 256 * q;          // 0..1023
            // A tile: 64 rows x 16 k; consecutive threads walk k when ak == 1
            const int ar = ak == 1 ? e / 16 : e % 64, ac = ak == 1 ? e % 16 : e / 64;
            const int gm = m0 + ar, gk = k0 + ac;
            As[ac][ar] = (gm < M && gk < K) ? A[gm * am + gk * ak] : 0.f;
            const int br = bn == 1 ? e / 64 : e % 16, bc = bn == 1 ? e % 64 : e / 16;
            const int gk2 = k0 + br, gn = n0 + bc;
            Bs[br][bc] = (gk2 < K && gn < N) ? ldw(Bm, gk2 * bk + gn * bn) : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < 16; ++kk) {
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = As[kk][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = Bs[kk][tx * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int gm = m0 + ty * 4 + i;
        if (gm >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int gn = n0 + tx * 4 + j;
            if (gn >= N) continue;
            Cm[(long)gm * ldc + gn] = acc[i][j] + (bias ? ldw(bias, gn) : 0.f);
        }
    }
}

// ------------------------------------------- FP32 training on matrix cores
// The stride-2 layers (2-4), the fully connected layer and the pair scores
// are contractions, run on v_mfma_f32_32x32x2_f32 (A: row lane & 31,
// k lane >> 5; B: column lane & 31, k lane >> 5; FP32 products and sums, twice
// the rate of scalar FP32 FMAs). An instruction takes 64 cycles for two
// 4-byte LDS reads per lane, so neither LDS nor the gathers bound the
// kernels; tiles are small so that the last layers still fill the chip.
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;
constexpr int TK = 16;   // k per LDS stage

// Row of an accumulator register: D[8 (r / 4) + 4 (lane / 32) + r % 4][lane % 32].
__device__ __forceinline__ int acc_row(int r, int lane) {
    return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
}

// Conv weights [co][ci][tap] of layers 2-4 as [tap][ci][co] (forward) and
// [tap][co][ci] (data gradient), so that the kernels below read them with
// consecutive lanes; one launch for the three layers.
struct PermLayers {
    long woff[3], ofs[3];   // weights in the parameters, copies in the output
    int cin[3], cout[3];
};
__global__ void k_perm_train(const float* __restrict__ P, PermLayers L, float* __restrict__ wf,
                             float* __restrict__ wb) {
    const int l = blockIdx.y;
    const int ci = L.cin[l], co = L.cout[l];
    const long n = (long)ci * co * 9;
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        const float v = P[L.woff[l] + i];
        const int tap = (int)(i % 9), c = (int)((i / 9) % ci), o = (int)(i / (9l * ci));
        wf[L.ofs[l] + ((long)tap * ci + c) * co + o] = v;
        wb[L.ofs[l] + ((long)tap * co + o) * ci + c] = v;
    }
}

// Implicit-GEMM convolution of a stride-2 layer, TC channels x TP positions
// per workgroup, one 32 x 32 block per wave; k = (16 channels, tap).
// BWD 0: y[b][n][yo][xo] = relu(bias[n] + sum W x), in = x (K channels, H x W),
//   positions the Ho x Wo outputs.
// BWD 1: dx[b][n][yi][xi] = (act > 0) sum W g (the ReLU backward of the layer
//   below included), in = g (K channels, Ho x Wo). An input row 2 y receives
//   tap 1 of output row y; row 2 y + 1 taps 0 and 2 of rows y + 1 and y: the
//   four parities of (yi, xi) (blockIdx.z) are dense contractions over 1, 2, 2
//   and 4 taps at Ho x Wo positions each.
// Bound by the MFMA rate: at 512 x 32^2 inputs, 32-64-128-128 channels, 66 us
// a layer forward and 63-97 us backward, 4.8 GFLOP each, 73 of 157 TFLOP/s
// (direct FP32 kernels, one thread per output: 433 and 2,329 us a layer).
template <int TC, int TP, bool BWD>
__global__ __launch_bounds__(256) void k_conv32(const float* __restrict__ in, const float* __restrict__ Wt,
                                                const float* __restrict__ bias,
                                                const float* __restrict__ act,
                                                float* __restrict__ out, int B, int K, int N, int H,
                                                int W, int Ho, int Wo) {
    static_assert(TC * TP == 4096, "four 32 x 32 blocks");
    constexpr int RP = TP * TK / 256, RC = TC * TK / 256;   // loads per thread and stage
    __shared__ float sp[2][TK][TP], sc[2][TK][TC];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wc = wave % (TC / 32), wp = wave / (TC / 32);
    const int P = B * Ho * Wo, p0 = (int)blockIdx.x * TP;   // < 2^31: batch and input size are bounded
    const int n0 = blockIdx.y * TC;
    // the four-tap parity first: its workgroups run longest
    const int par = BWD ? 3 - (int)blockIdx.z : 0;
    const int py = par >> 1, px = par & 1;
    const int ntx = BWD ? 1 + px : 3, ntap = BWD ? (1 + py) * ntx : 9;
    const int ih = BWD ? Ho : H, iw = BWD ? Wo : W;
    // this thread's position and channels of a stage
    const int mp = tid % TP, kp = tid / TP * RP, mc = tid % TC, kc = tid / TC * RC;
    const bool pok = p0 + mp < P;
    const int pq = pok ? p0 + mp : 0;
    const int x = pq % Wo, y = (pq / Wo) % Ho;
    const long plane = (long)ih * iw;
    const float* src = in + ((long)(pq / (Wo * Ho)) * K + kp) * plane;
    const bool cok = n0 + mc < N;
    const float* wsrc = Wt + (long)kc * N + n0 + mc;
    float rp[RP], rc[RC];
    int cb = 0, tap = 0;
    auto load = [&]() {
        int ky = tap / ntx, kx = tap - ky * ntx, iy, ix;
        if (BWD) {
            iy = y + (py && ky == 0);
            ix = x + (px && kx == 0);
            ky = py ? 2 * ky : 1;
            kx = px ? 2 * kx : 1;
        } else {
            iy = 2 * y - 1 + ky;
            ix = 2 * x - 1 + kx;
        }
        const bool ok = pok && iy >= 0 && iy < ih && ix >= 0 && ix < iw;
        const float* s = src + cb * TK * plane + (ok ? (long)iy * iw + ix : 0);
        const float* w = wsrc + ((long)(ky * 3 + kx) * K + cb * TK) * N;
#pragma unroll
        for (int j = 0; j < RP; ++j) rp[j] = ok ? s[j * plane] : 0.f;
#pragma unroll
        for (int j = 0; j < RC; ++j) rc[j] = cok ? w[(long)j * N] : 0.f;
        if (++tap == ntap) { tap = 0; ++cb; }
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int j = 0; j < RP; ++j) sp[buf][kp + j][mp] = rp[j];
#pragma unroll
        for (int j = 0; j < RC; ++j) sc[buf][kc + j][mc] = rc[j];
    };
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    const int nst = K / TK * ntap;
    load();
    store(0);
    __syncthreads();
    for (int st = 0; st < nst; ++st) {
        if (st + 1 < nst) load();
        const int buf = st & 1;
#pragma unroll
        for (int k = 0; k < TK; k += 2)
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(sc[buf][k + (lane >> 5)][wc * 32 + (lane & 31)],
                                                       sp[buf][k + (lane >> 5)][wp * 32 + (lane & 31)],
                                                       acc, 0, 0, 0);
        if (st + 1 < nst) store(buf ^ 1);
        __syncthreads();
    }
    const int po = p0 + wp * 32 + (lane & 31);
    if (po >= P) return;
    const int xo = po % Wo, yo = (po / Wo) % Ho;
    const long b = po / (Wo * Ho);
    const long oplane = BWD ? (long)H * W : (long)Ho * Wo;
    const long at = b * N * oplane + (BWD ? (long)(2 * yo + py) * W + 2 * xo + px : (long)yo * Wo + xo);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int n = n0 + wc * 32 + acc_row(r, lane);
        if (n >= N) continue;
        const long o = at + n * oplane;
        if (BWD) out[o] = act[o] > 0.f ? acc[r] : 0.f;
        else out[o] = fmaxf(acc[r] + bias[n], 0.f);
    }
}

// Weight gradient of a stride-2 layer: partial sums over a share of the
// B Ho Wo positions (blockIdx.z) of 64 output x 32 input channels for all 9
// taps, part[z] = [tap][co][ci] and the bias gradient [co]. Each stage holds
// 16 positions: g (64 channels) and the 9 shifted x (32 channels); waves are
// 2 channel blocks x 2 halves of the positions, 9 accumulators each, so one
// read of g serves 9 instructions. k_part_sum adds the shares in order.
// 69 us a layer at the
// sizes above (one workgroup per (co, ci), which read all of g and x each: 1,916 us).
__global__ __launch_bounds__(256, 2) void k_conv32_dw(const float* __restrict__ g,
                                                   const float* __restrict__ xin,
                                                   float* __restrict__ part, int B, int Cin, int H,
                                                   int W, int Cout, int Ho, int Wo) {
    constexpr int NP = 16, LG = 65, LX = 33;
    __shared__ float lds[NP * LG + 9 * NP * LX];
    static_assert(sizeof(lds) >= 4 * 2 * 64 * 16, "one tap of the halves' exchange");
    float* sg = lds;             // [pos][co]
    float* sx = lds + NP * LG;   // [tap][pos][ci]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wc = wave & 1, wh = wave >> 1;
    const int co0 = blockIdx.x * 64, ci0 = blockIdx.y * 32;
    const int P = B * Ho * Wo;
    const int nst = (P + NP - 1) / NP;
    const int per = (nst + (int)gridDim.z - 1) / (int)gridDim.z;
    const int s0 = (int)blockIdx.z * per, s1 = min(nst, s0 + per);
    const int mp = tid & 15, q = tid >> 4;   // position; g channels q + 16 j, x channels q, q + 16
    const long oplane = (long)Ho * Wo, iplane = (long)H * W;
    float rg[4], rx[2][9], gsum[4] = {0.f, 0.f, 0.f, 0.f};
    auto load = [&](int st) {
        const int p = st * NP + mp;
        const bool pok = p < P;
        const int pq = pok ? p : 0;
        const int x = pq % Wo, y = (pq / Wo) % Ho;
        const long b = pq / (Ho * Wo);
        const float* gs = g + (b * Cout + co0 + q) * oplane + (long)y * Wo + x;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            rg[j] = (pok && co0 + q + 16 * j < Cout) ? gs[16l * j * oplane] : 0.f;
        const float* xs = xin + (b * Cin + ci0 + q) * iplane;
#pragma unroll
        for (int t = 0; t < 9; ++t) {
            const int iy = 2 * y - 1 + t / 3, ix = 2 * x - 1 + t % 3;
            const bool ok = pok && iy >= 0 && iy < H && ix >= 0 && ix < W;
            const long o = ok ? (long)iy * W + ix : 0;
#pragma unroll
            for (int j = 0; j < 2; ++j)
                rx[j][t] = (ok && ci0 + q + 16 * j < Cin) ? xs[16l * j * iplane + o] : 0.f;
        }
    };
    f32x16 acc[9];
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;
    if (s0 < s1) load(s0);
    for (int st = s0; st < s1; ++st) {
        __syncthreads();   // the stage before has been read
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            sg[mp * LG + q + 16 * j] = rg[j];
            gsum[j] += rg[j];
        }
#pragma unroll
        for (int t = 0; t < 9; ++t)
#pragma unroll
            for (int j = 0; j < 2; ++j) sx[(t * NP + mp) * LX + q + 16 * j] = rx[j][t];
        __syncthreads();
        if (st + 1 < s1) load(st + 1);
#pragma unroll
        for (int k = 0; k < NP / 2; k += 2) {
            const int p = wh * (NP / 2) + k + (lane >> 5);
            const float a = sg[p * LG + wc * 32 + (lane & 31)];
#pragma unroll
            for (int t = 0; t < 9; ++t)
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, sx[(t * NP + p) * LX + (lane & 31)],
                                                              acc[t], 0, 0, 0);
        }
    }
    float* out = part + (long)blockIdx.z * ((long)Cout * Cin * 9 + Cout);
    // the second half of the positions joins the first, one tap at a time
#pragma unroll
    for (int t = 0; t < 9; ++t) {
        __syncthreads();
        if (wh == 1)
#pragma unroll
            for (int r = 0; r < 16; ++r) lds[(wc * 16 + r) * 64 + lane] = acc[t][r];
        __syncthreads();
        if (wh == 0)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int co = co0 + wc * 32 + acc_row(r, lane), ci = ci0 + (lane & 31);
                if (co < Cout && ci < Cin)
                    out[((long)t * Cout + co) * Cin + ci] = acc[t][r] + lds[(wc * 16 + r) * 64 + lane];
            }
    }
    if (blockIdx.y == 0) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float v = gsum[j];
            for (int o = 8; o > 0; o >>= 1) v += __shfl_xor(v, o, 16);
            if (mp == 0 && co0 + q + 16 * j < Cout)
                out[(long)Cout * Cin * 9 + co0 + q + 16 * j] = v;
        }
    }
}

// Four consecutive floats at float alignment (inputs may start anywhere).
struct Float4u {
    float v[4];
};

// First layer (one input channel, stride 1), forward: a thread holds the 3 x 6
// window of 4 consecutive outputs and runs over 8 output channels (uniform
// weights: scalar loads); bound by writing y.
__global__ __launch_bounds__(256) void k_conv1_32(const float* __restrict__ x, const float* __restrict__ Wt,
                                                  const float* __restrict__ bias, float* __restrict__ y,
                                                  int B, int S, int Cout) {
    const int quads = S * S / 4;
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    if (t >= (long)B * quads) return;
    const long b = t / quads;
    const int q = (int)(t - b * quads), yo = q / (S / 4), xo = (q - yo * (S / 4)) * 4;
    float v[3][6];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        const int yi = yo - 1 + r;
        const float* row = x + (b * S + yi) * S + xo;
        const bool ok = yi >= 0 && yi < S;
        Float4u x4 = {{0.f, 0.f, 0.f, 0.f}};
        if (ok) x4 = *(const Float4u*)row;
        v[r][0] = ok && xo > 0 ? row[-1] : 0.f;
#pragma unroll
        for (int c = 0; c < 4; ++c) v[r][c + 1] = x4.v[c];
        v[r][5] = ok && xo + 4 < S ? row[4] : 0.f;
    }
    const int c0 = blockIdx.y * 8, c1 = min(Cout, c0 + 8);
    for (int co = c0; co < c1; ++co) {
        float a[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) a[e] = bias[co];
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            const float w = Wt[co * 9 + k];
#pragma unroll
            for (int e = 0; e < 4; ++e) a[e] = fmaf(w, v[k / 3][k % 3 + e], a[e]);
        }
        *(float4*)(y + ((b * Cout + co) * S + yo) * (long)S + xo) =
            make_float4(fmaxf(a[0], 0.f), fmaxf(a[1], 0.f), fmaxf(a[2], 0.f), fmaxf(a[3], 0.f));
    }
}

// First layer, weight and bias gradients: partial sums of `per` inputs per
// workgroup (blockIdx.x), 32 output channels x 8 lanes that share a channel's
// positions, 4 consecutive ones at a time; part[z] = [co][9] and [co]. Bound
// by reading g.
__global__ __launch_bounds__(256) void k_conv1_32_dw(const float* __restrict__ g,
                                                     const float* __restrict__ x,
                                                     float* __restrict__ part, int B, int S, int Cout,
                                                     int per) {
    const int co = blockIdx.y * 32 + (threadIdx.x >> 3), pg = threadIdx.x & 7;
    const bool cok = co < Cout;
    const int quads = S * S / 4;
    float acc[10];
#pragma unroll
    for (int k = 0; k < 10; ++k) acc[k] = 0.f;
    for (long b = (long)blockIdx.x * per; b < min((long)B, ((long)blockIdx.x + 1) * per); ++b) {
        const float* gs = g + (b * Cout + (cok ? co : 0)) * (long)S * S;
        for (int q = pg; q < quads; q += 8) {
            const int yo = q / (S / 4), xo = (q - yo * (S / 4)) * 4;
            const float4 g4 = *(const float4*)(gs + yo * S + xo);   // rows are multiples of 8 floats
            const float gv[4] = {g4.x, g4.y, g4.z, g4.w};
#pragma unroll
            for (int r = 0; r < 3; ++r) {
                const int yi = yo - 1 + r;
                if (yi < 0 || yi >= S) continue;
                const float* row = x + (b * S + yi) * S + xo;
                const Float4u x4 = *(const Float4u*)row;
                const float v[6] = {xo > 0 ? row[-1] : 0.f, x4.v[0], x4.v[1], x4.v[2], x4.v[3],
                                    xo + 4 < S ? row[4] : 0.f};
#pragma unroll
                for (int c = 0; c < 3; ++c)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[3 * r + c] = fmaf(gv[e], v[c + e], acc[3 * r + c]);
            }
            acc[9] += (gv[0] + gv[1]) + (gv[2] + gv[3]);
        }
    }
    float* out = part + (long)blockIdx.x * Cout * 10;
#pragma unroll
    for (int k = 0; k < 10; ++k) {
        float v = acc[k];
        for (int o = 4; o > 0; o >>= 1) v += __shfl_xor(v, o, 8);
        if (pg == 0 && cok) out[k < 9 ? (long)co * 9 + k : (long)Cout * 9 + co] = v;
    }
}

// out[i] = sum over nz shares of part[z][i], n values each, 16 groups of
// shares per value (4 groups: 12 us a sum of 38 MB, 16: 8 us). taps > 1: the first nw values are [tap][co][ci] and go to
// [co][ci][tap]; bias (or null) is added by column i % ncol.
__global__ __launch_bounds__(1024) void k_part_sum(const float* __restrict__ part, int nz, long n, long nw,
                                                  int taps, const float* __restrict__ bias, int ncol,
                                                  float* __restrict__ out) {
    __shared__ float red[16][64];
    const int c = threadIdx.x & 63, grp = threadIdx.x >> 6;
    const long i = (long)blockIdx.x * 64 + c;
    float s = 0.f;
    if (i < n) {
#pragma unroll 4
        for (int z = grp; z < nz; z += 16) s += part[z * n + i];
    }
    red[grp][c] = s;
    __syncthreads();
    if (grp != 0 || i >= n) return;
    float v = 0.f;
#pragma unroll
    for (int q = 0; q < 16; ++q) v += red[q][c];
    if (bias) v += bias[i % ncol];
    const long per = taps > 1 ? nw / taps : 1;
    out[taps > 1 && i < nw ? (i % per) * taps + i / per : i] = v;
}

// C[m][n] = sum_k A[m am + k ak] B[k bk + n bn] (+ bias[n]) in FP32 on matrix
// cores, 64 x 64 per workgroup, blockIdx.z a share of K. One share: the result
// goes to C; several: share z to C + z M N for k_part_sum (bias null). The fully
// connected layer of 512 x 2048 -> 128 has 16 tiles only; its K is split so
// that some 512 workgroups run.
__global__ __launch_bounds__(256) void k_gemm32(int M, int N, int K, const float* __restrict__ A, long am,
                                                long ak, const float* __restrict__ Bm, long bk, long bn,
                                                const float* __restrict__ bias, float* __restrict__ Cm,
                                                int kper) {
    constexpr int LR = 65;
    __shared__ float sa[2][TK][LR], sb[2][TK][LR];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
    const int k0 = blockIdx.z * kper, k1 = min(K, k0 + kper);
    // consecutive threads walk the dimension that is contiguous in memory
    const bool ka = ak == 1, kb = bk == 1;
    const int ar = ka ? tid >> 4 : tid & 63, ac = ka ? tid & 15 : tid >> 6;
    const int br = kb ? tid >> 4 : tid & 63, bc = kb ? tid & 15 : tid >> 6;
    float ra[4], rb[4];
    auto load = [&](int kk) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int m = m0 + ar + (ka ? 16 * j : 0), k = kk + ac + (ka ? 0 : 4 * j);
            ra[j] = (m < M && k < k1) ? A[m * am + k * ak] : 0.f;
            const int n = n0 + br + (kb ? 16 * j : 0), q = kk + bc + (kb ? 0 : 4 * j);
            rb[j] = (n < N && q < k1) ? Bm[q * bk + n * bn] : 0.f;
        }
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            sa[buf][ac + (ka ? 0 : 4 * j)][ar + (ka ? 16 * j : 0)] = ra[j];
            sb[buf][bc + (kb ? 0 : 4 * j)][br + (kb ? 16 * j : 0)] = rb[j];
        }
    };
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    load(k0);
    store(0);
    __syncthreads();
    for (int kk = k0, buf = 0; kk < k1; kk += TK, buf ^= 1) {
        if (kk + TK < k1) load(kk + TK);
#pragma unroll
        for (int k = 0; k < TK; k += 2)
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(sa[buf][k + (lane >> 5)][wm * 32 + (lane & 31)],
                                                       sb[buf][k + (lane >> 5)][wn * 32 + (lane & 31)],
                                                       acc, 0, 0, 0);
        if (kk + TK < k1) store(buf ^ 1);
        __syncthreads();
    }
    const int n = n0 + wn * 32 + (lane & 31);
    if (n >= N) return;
    const float bv = bias ? bias[n] : 0.f;
    float* C = Cm + (long)blockIdx.z * M * N;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int m = m0 + wm * 32 + acc_row(r, lane);
        if (m < M) C[(long)m * N + n] = acc[r] + bv;
    }
}

// C[m][n] = scale * sum_k A[m][k] B[n][k] (rows of d values, FP32 sums in the order
// of k), 128 x 128 per workgroup, 64 x 64 per wave as 2 x 2 blocks: each LDS value
// feeds two instructions. Particle embeddings against class references; the scale
// (1 / tau) was a pass of its own over the scores (143 us for 16,384 x 4,368), and
// the product on the VALU took 338 us, now 253 us (72 TFLOP/s).
__global__ __launch_bounds__(256) void k_scores32(int M, int N, int K, const float* __restrict__ A,
                                                  const float* __restrict__ Bm, float scale,
                                                  float* __restrict__ C) {
    constexpr int LR = 129;
    __shared__ float sa[2][TK][LR], sb[2][TK][LR];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int m0 = blockIdx.y * 128, n0 = blockIdx.x * 128;
    const int lr = tid >> 4, lk = tid & 15;   // rows lr + 16 j, k lk
    float ra[8], rb[8];
    auto load = [&](int k0) {
        const int k = k0 + lk;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int m = m0 + lr + 16 * j, n = n0 + lr + 16 * j;
            ra[j] = (m < M && k < K) ? A[(long)m * K + k] : 0.f;
            rb[j] = (n < N && k < K) ? Bm[(long)n * K + k] : 0.f;
        }
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            sa[buf][lk][lr + 16 * j] = ra[j];
            sb[buf][lk][lr + 16 * j] = rb[j];
        }
    };
    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    load(0);
    store(0);
    __syncthreads();
    for (int k0 = 0, buf = 0; k0 < K; k0 += TK, buf ^= 1) {
        if (k0 + TK < K) load(k0 + TK);
#pragma unroll
        for (int k = 0; k < TK; k += 2) {
            const int kk = k + (lane >> 5);
            float a[2], b[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                a[i] = sa[buf][kk][wm * 64 + i * 32 + (lane & 31)];
                b[i] = sb[buf][kk][wn * 64 + i * 32 + (lane & 31)];
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        if (k0 + TK < K) store(buf ^ 1);
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int n = n0 + wn * 64 + j * 32 + (lane & 31);
            if (n >= N) continue;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = m0 + wm * 64 + i * 32 + acc_row(r, lane);
                if (m < M) C[(long)m * N + n] = acc[i][j][r] * scale;
            }
        }
}

// db[n] = sum_m g[m][n]: 64 columns per workgroup, the rows over its 16 waves
__global__ __launch_bounds__(1024) void k_colsum(const float* __restrict__ g, int M, int N,
                                                 float* __restrict__ db) {
    __shared__ float red[16][64];
    const int c = threadIdx.x & 63, grp = threadIdx.x >> 6;
    const int n = blockIdx.x * 64 + c;
    float s = 0.f;
    if (n < N) {
#pragma unroll 4
        for (int m = grp; m < M; m += 16) s += g[(long)m * N + n];
    }
    red[grp][c] = s;
    __syncthreads();
    if (grp != 0 || n >= N) return;
    float v = 0.f;
#pragma unroll
    for (int q = 0; q < 16; ++q) v += red[q][c];
    db[n] = v;
}

// ------------------------------------------------------ softmax / top-k
__device__ __forceinline__ float wave_add(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// One workgroup per row: loss[b] = logsumexp - logit[label]; dl = (p - onehot) / B.
__global__ __launch_bounds__(256) void k_softmax_ce(const float* __restrict__ logits,
                                                    const int* __restrict__ labels, int B, int C,
                                                    float* __restrict__ dl, float* __restrict__ loss) {
    __shared__ float red[256];
    const int b = blockIdx.x;
    const float* l = logits + (long)b * C;
    float mx = -INFINITY;
    for (int c = threadIdx.x; c < C; c += blockDim.x) mx = fmaxf(mx, l[c]);
    red[threadIdx.x] = mx;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] = fmaxf(red[threadIdx.x], red[threadIdx.x + s]);
        __syncthreads();
    }
    mx = red[0];
    __syncthreads();
    float se = 0.f;
    for (int c = threadIdx.x; c < C; c += blockDim.x) se += expf(l[c] - mx);
    red[threadIdx.x] = se;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    se = red[0];
    const int t = labels[b];
    const float inv = 1.f / (float)B;
    for (int c = threadIdx.x; c < C; c += blockDim.x)
        dl[(long)b * C + c] = (expf(l[c] - mx) / se - (c == t ? 1.f : 0.f)) * inv;
    if (threadIdx.x == 0 && loss) loss[b] = logf(se) + mx - l[t];
}

// The k largest logits of a row (k <= 32) as classes and softmax probabilities,
// best first (ties: lower class; NaN and -inf are never taken, missing places
// -1 and 0). W wavefronts per row, two passes over it: the lanes' maxima, the
// k-th largest of which bounds the k-th value from below, then the exponential
// sum and the values that reach the bound, listed in LDS. Before a list could
// overflow (values equal to the bound, or large ones on fewer than k lanes) it is
// cut to its k best, whose last one is the new bound: the classes come in
// ascending order, so that a later equal value never belongs to them. Bound by
// reading the row: 16,384 x 4,368 179 us (388 with 16 block-wide arg-max rounds over
// per-thread lists). Rows of equal values, the whole call with its scores: 1 x 2^20
// 0.6 ms, 16,384 x 4,368 0.4 ms; with a pass for each of 16 places once a list
// was full they took 46.8 and 1.5 ms.
constexpr int ROWCAP = 256;   // listed values of a wavefront

__device__ __forceinline__ unsigned long long logit_key(float v, int c) {
    const unsigned u = __float_as_uint(v + 0.f);   // -0 counts as 0
    const unsigned o = (u & 0x80000000u) ? ~u : u | 0x80000000u;
    return ((unsigned long long)o << 32) | (unsigned)~c;
}
__device__ __forceinline__ unsigned long long wave_max64(unsigned long long m) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long x = __shfl_xor(m, o, 64);
        m = x > m ? x : m;
    }
    return m;
}
// LDS written by lanes of this wavefront before is read by others after.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// The k largest of the keys x (Q a lane, all different, 0: none), largest first,
// to out[0..k); returns the k-th, 0 if there are fewer.
template <int Q>
__device__ __forceinline__ unsigned long long wave_best(unsigned long long (&x)[Q], int k, int lane,
                                                        unsigned long long* out) {
    unsigned long long m = 0;
    for (int r = 0; r < k; ++r) {
        m = x[0];
#pragma unroll
        for (int q = 1; q < Q; ++q) m = x[q] > m ? x[q] : m;
        m = wave_max64(m);
        if (lane == 0) out[r] = m;
#pragma unroll
        for (int q = 0; q < Q; ++q) x[q] = x[q] == m ? 0 : x[q];
    }
    return m;
}

template <int W>
__global__ __launch_bounds__(W > 4 ? 64 * W : 256) void k_row_topk(const float* __restrict__ logits, long n,
                                                                   int C, int k, int* __restrict__ cls,
                                                                   float* __restrict__ prob) {
    constexpr int ROWS = W >= 4 ? 1 : 4 / W;   // rows per workgroup
    __shared__ unsigned long long list[ROWS * W][ROWCAP];
    __shared__ float red[3][W];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, part = wave % W;
    const long b = (long)blockIdx.x * ROWS + wave / W;
    if (b >= n) return;   // whole wavefronts; with W > 1 a workgroup has one row
    const float* l = logits + b * C;
    unsigned long long* mine = list[wave];
    float lm = -INFINITY;
#pragma unroll 4
    for (int c = part * 64 + lane; c < C; c += 64 * W) lm = fmaxf(lm, l[c]);
    float mx = lm;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    // the k-th largest lane maximum (each round drops one lane)
    float bound = -INFINITY, left = lm;
    for (int r = 0; r < k; ++r) {
        float m = left;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
        bound = m;
        const unsigned long long has = __ballot(left == m);
        if (lane == __builtin_ctzll(has | (1ull << 63))) left = -INFINITY;
    }
    if (W > 1) {   // every wavefront's bound is one of the row
        if (lane == 0) {
            red[0][part] = mx;
            red[1][part] = bound;
        }
        __syncthreads();
#pragma unroll
        for (int w = 0; w < W; ++w) {
            mx = fmaxf(mx, red[0][w]);
            bound = fmaxf(bound, red[1][w]);
        }
    }
    float se = 0.f;
    int cnt = 0;
    unsigned long long above = 0;   // keys up to this one are out of the running
    auto cut = [&]() {
        unsigned long long x[ROWCAP / 64];
        wave_lds_sync();
#pragma unroll
        for (int q = 0; q < ROWCAP / 64; ++q) x[q] = lane + 64 * q < cnt ? mine[lane + 64 * q] : 0;
        wave_lds_sync();
        above = wave_best(x, k, lane, mine);
        wave_lds_sync();
        cnt = min(cnt, k);
    };
    for (int c0 = part * 64; c0 < C; c0 += 64 * W) {
        const int c = c0 + lane;
        const float v = c < C ? l[c] : -INFINITY;
        if (c < C) se += expf(v - mx);
        bool in = v >= bound && v > -INFINITY;
        if (__ballot(in)) {
            const unsigned long long key = logit_key(v, c);
            in = in && key > above;
            const unsigned long long has = __ballot(in);
            if (in) mine[cnt + __popcll(has & ((1ull << lane) - 1ull))] = key;
            cnt += __popcll(has);
            if (cnt > ROWCAP - 64) cut();
        }
    }
    se = wave_add(se);
    cut();
    if (W > 1) {
        if (lane == 0) red[2][part] = se;
        __syncthreads();
        if (wave) return;
        se = 0.f;
#pragma unroll
        for (int w = 0; w < W; ++w) se += red[2][w];
        constexpr int Q = W > 1 ? W / 2 : 1;   // 64 Q >= W * 32
        unsigned long long x[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int i = lane + 64 * q;
            x[q] = i < W * k ? list[i / k][i % k] : 0;
        }
        wave_lds_sync();
        (void)wave_best(x, k, lane, mine);
        wave_lds_sync();
    }
    if (lane < k) {
        const unsigned long long m = mine[lane];
        const unsigned o = (unsigned)(m >> 32);
        const float v = __uint_as_float((o & 0x80000000u) ? o & 0x7fffffffu : ~o);
        cls[b * k + lane] = m ? (int)~(unsigned)m : -1;
        prob[b * k + lane] = m ? expf(v - mx) / se : 0.f;
    }
}

// --------------------------------------------- contrastive (embedding) head
// Unit rows u = z / |z| of an n x d matrix (|z| floored at 1e-12); one
// wavefront per row, so that rows are read and written with consecutive
// lanes (one thread per row: 58 us for 4,096 x 128).
__global__ __launch_bounds__(256) void k_unit_rows(const float* __restrict__ z, long n, int d,
                                                   float* __restrict__ u, float* __restrict__ nrm) {
    const long i = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (i >= n) return;
    const float* r = z + i * d;
    float ss = 0.f;
    for (int c = lane; c < d; c += 64) ss = fmaf(r[c], r[c], ss);
    const float nz = fmaxf(sqrtf(wave_add(ss)), 1e-12f), inv = 1.f / nz;
    for (int c = lane; c < d; c += 64) u[i * d + c] = r[c] * inv;
    if (nrm && lane == 0) nrm[i] = nz;
}

// Softmax of the pair scores S (B x B, cosines) over temperature tau, by row
// (dim 0: p_ij over j) or by column (dim 1: q_ij over i), one workgroup per
// row / column; loss[i] = -log of the matched pair's probability.
__global__ __launch_bounds__(256) void k_pair_softmax(const float* __restrict__ S, int B,
                                                      float inv_tau, int dim, float* __restrict__ P,
                                                      float* __restrict__ loss) {
    __shared__ float red[256];
    const int i = blockIdx.x;
    const long st = dim == 0 ? 1 : B, base = dim == 0 ? (long)i * B : i;
    float mx = -INFINITY;
    for (int j = threadIdx.x; j < B; j += blockDim.x) mx = fmaxf(mx, S[base + j * st] * inv_tau);
    red[threadIdx.x] = mx;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] = fmaxf(red[threadIdx.x], red[threadIdx.x + w]);
        __syncthreads();
    }
    mx = red[0];
    __syncthreads();
    float se = 0.f;
    for (int j = threadIdx.x; j < B; j += blockDim.x) se += expf(S[base + j * st] * inv_tau - mx);
    red[threadIdx.x] = se;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    se = red[0];
    for (int j = threadIdx.x; j < B; j += blockDim.x)
        P[base + j * st] = expf(S[base + j * st] * inv_tau - mx) / se;
    if (threadIdx.x == 0) loss[i] = logf(se) + mx - S[base + (long)i * st] * inv_tau;
}

// dL/dS of the symmetric loss mean_i (row_i + col_i) / 2 over the B pairs:
// (p + q - 2 I) / (2 B tau); loss_out[i] = (row_i + col_i) / 2.
__global__ void k_pair_grad(const float* __restrict__ P, const float* __restrict__ Q, int B,
                            float inv_tau, const float* __restrict__ lrow,
                            const float* __restrict__ lcol, float* __restrict__ dS,
                            float* __restrict__ loss_out) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long)B * B) return;
    const int i = (int)(t / B), j = (int)(t % B);
    dS[t] = (P[t] + Q[t] - (i == j ? 2.f : 0.f)) * inv_tau / (2.f * B);
    if (j == 0 && loss_out) loss_out[i] = 0.5f * (lrow[i] + lcol[i]);
}

// Backward of u = z / |z|: dz = (du - (du . u) u) / |z|, one wavefront per row.
__global__ __launch_bounds__(256) void k_unit_rows_bwd(const float* __restrict__ du,
                                                       const float* __restrict__ u,
                                                       const float* __restrict__ nrm, long n, int d,
                                                       float* __restrict__ dz) {
    const long i = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (i >= n) return;
    float dot = 0.f;
    for (int c = lane; c < d; c += 64) dot = fmaf(du[i * d + c], u[i * d + c], dot);
    dot = wave_add(dot);
    const float inv = 1.f / nrm[i];
    for (int c = lane; c < d; c += 64) dz[i * d + c] = (du[i * d + c] - dot * u[i * d + c]) * inv;
}

__global__ void k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, long n, float lr, float b1, float b2, float eps,
                       float c1, float c2, float wd) {
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        const float gi = g[i] + wd * p[i];
        const float mi = b1 * m[i] + (1 - b1) * gi;
        const float vi = b2 * v[i] + (1 - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    }
}

__global__ void k_to_bf16(const float* __restrict__ p, uint16_t* __restrict__ q, long n) {
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        q[i] = f_to_bf16(p[i]);
}

// ------------------------------------------------------ MFMA inference
// Activations are NHWC BF16. Layer 1 (one input channel) runs on the VALU;
// layers 2-4 and the fully connected layer are implicit GEMMs on
// v_mfma_f32_32x32x16_bf16: rows = output positions (b, yo, xo), columns =
// output channels, k = (tap, input channel) with the channel fastest, so
// that 8 consecutive k are one 16-byte load from the NHWC input.
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;

// y[b][yo][xo][co] = bf16(relu(bias + sum_{ky,kx} W[co][0][ky][kx] x[b][yo-1+ky][xo-1+kx]))
// thread = (4 consecutive positions, 8 channels): a weight read from LDS (taps
// outermost, two 16-byte reads per tap) serves the four positions; a wavefront's
// 16-byte stores of 8 BF16 channels join in the NHWC output, whose writing bounds
// it (one position per thread, 80 LDS reads for its 72 products: 613 us for
// 16,384 x 32^2 x 32, now 391 us).
__global__ __launch_bounds__(256) void k_conv1_nhwc(const float* __restrict__ x,
                                                    const uint16_t* __restrict__ W,
                                                    const uint16_t* __restrict__ bias, int B, int S,
                                                    int C1, uint16_t* __restrict__ y) {
    extern __shared__ float w[];   // 9 x C1 weights [tap][channel], then C1 biases
    for (int i = threadIdx.x; i < C1 * 9; i += blockDim.x) w[i % 9 * C1 + i / 9] = bf16_to_f(W[i]);
    for (int i = threadIdx.x; i < C1; i += blockDim.x) w[C1 * 9 + i] = bf16_to_f(bias[i]);
    __syncthreads();
    const int ng = C1 / 8, quads = S * S / 4;
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long)B * quads * ng) return;
    const int g = (int)(t % ng);
    const long pq = t / ng;
    const long b = pq / quads;
    const int q = (int)(pq - b * quads), yo = q / (S / 4), xo = (q - yo * (S / 4)) * 4;
    float v[3][6];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        const int yi = yo - 1 + r;
        const float* row = x + (b * S + yi) * S + xo;
        const bool ok = yi >= 0 && yi < S;
        Float4u x4 = {{0.f, 0.f, 0.f, 0.f}};
        if (ok) x4 = *(const Float4u*)row;
        v[r][0] = ok && xo > 0 ? row[-1] : 0.f;
#pragma unroll
        for (int c = 0; c < 4; ++c) v[r][c + 1] = x4.v[c];
        v[r][5] = ok && xo + 4 < S ? row[4] : 0.f;
    }
    float a[4][8];
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int c = 0; c < 8; ++c) a[e][c] = w[C1 * 9 + g * 8 + c];
#pragma unroll
    for (int k = 0; k < 9; ++k) {
        const float4* wk = (const float4*)(w + k * C1 + g * 8);
        const float4 w0 = wk[0], w1 = wk[1];
        const float ww[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int c = 0; c < 8; ++c) a[e][c] = fmaf(ww[c], v[k / 3][k % 3 + e], a[e][c]);
    }
    uint16_t* o = y + (pq * 4) * C1 + g * 8;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        uint32_t p[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            p[j] = (uint32_t)f_to_bf16(fmaxf(a[e][2 * j], 0.f)) |
                   ((uint32_t)f_to_bf16(fmaxf(a[e][2 * j + 1], 0.f)) << 16);
        *(uint4*)(o + (long)e * C1) = make_uint4(p[0], p[1], p[2], p[3]);
    }
}

// Implicit-GEMM convolution (KS = 3: pad 1, stride 2; KS = 1: a plain GEMM over
// H = W = 1) of NHWC BF16 input with BF16 weights [Cout][KS*KS][Cin] and
// BF16 biases. OUTF32: FP32 output rows of stride ldo without ReLU (logits);
// else BF16 NHWC output with ReLU. Cin must be a multiple of 32.
// A workgroup's 4 waves (WM x WN) compute BM x BN blocks of 32 x 32 each; the
// loads of the next 32-deep K step are in flight during a step. With 2 x 2 blocks
// a wave reads 4 KB of LDS for 4 instructions (with 1 x 2, as before, 3 KB for 2:
// more than the LDS delivers at the MFMA rate). The valid taps of a row are a
// bit mask made once, a tap is a uniform offset. The BF16 output goes through LDS
// and leaves in 16-byte stores. 16,384 x 32^2 inputs, 32-64-128-128 channels: the
// three layers 1,471 us before, 1,284 us now.
template <int BM, int BN, int WM, int WN, int KS, bool OUTF32>
__global__ __launch_bounds__(256) void k_conv_mfma(const uint16_t* __restrict__ x, int B, int H,
                                                   int Wd, int Cin, int Ho, int Wo,
                                                   const uint16_t* __restrict__ Wt,
                                                   const uint16_t* __restrict__ bias, int Cout,
                                                   long ldo, void* __restrict__ out) {
    static_assert(WM * WN == 4, "four waves");
    constexpr int IM = 32 * BM * WM, IN = 32 * BN * WN, IK = 32, IROW = IK * 2 + 16;
    constexpr int NA = IM / 64, NB = IN / 64;   // 16-byte chunks per thread and step
    constexpr int OR = IN * 2 + 16;             // bytes per output row in LDS
    constexpr int LDS = 2 * (IM + IN) * IROW > IM * OR ? 2 * (IM + IN) * IROW : IM * OR;
    __shared__ __attribute__((aligned(16))) char lds[LDS];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WN, wn = wave % WN;
    const long M = (long)B * Ho * Wo, m0 = (long)blockIdx.x * IM;
    const int n0 = blockIdx.y * IN;
    const int K = KS * KS * Cin, nk = K / IK;
    // rows (tid >> 2) + 64 j, 8 channels from 8 (tid & 3)
    const int lr = tid >> 2, lp = tid & 3;
    const uint16_t* ap[NA];
    unsigned av[NA];
#pragma unroll
    for (int j = 0; j < NA; ++j) {
        const long m = m0 + lr + 64 * j;
        const long mm = m < M ? m : 0;
        const int xo = (int)(mm % Wo), yo = (int)((mm / Wo) % Ho);
        const long b = mm / ((long)Wo * Ho);
        const int y0 = KS == 3 ? 2 * yo - 1 : yo, x0 = KS == 3 ? 2 * xo - 1 : xo;
        ap[j] = x + ((b * H + y0) * Wd + x0) * (long)Cin + lp * 8;
        av[j] = 0;
#pragma unroll
        for (int t = 0; t < KS * KS; ++t) {
            const int yi = y0 + t / KS, xi = x0 + t % KS;
            if (m < M && yi >= 0 && yi < H && xi >= 0 && xi < Wd) av[j] |= 1u << t;
        }
    }
    const uint16_t* bp[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const int co = n0 + lr + 64 * j;
        bp[j] = co < Cout ? Wt + (long)co * K + lp * 8 : nullptr;
    }
    uint4 ra[NA], rb[NB];
    int tap = 0, ci = 0;   // of the next step to load
    auto load = [&](int kt) {
        const long o = ((long)(tap / KS) * Wd + tap % KS) * Cin + ci;
#pragma unroll
        for (int j = 0; j < NA; ++j) {
            ra[j] = make_uint4(0, 0, 0, 0);
            if ((av[j] >> tap) & 1) ra[j] = *(const uint4*)(ap[j] + o);
        }
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            rb[j] = make_uint4(0, 0, 0, 0);
            if (bp[j]) rb[j] = *(const uint4*)(bp[j] + (long)kt * IK);
        }
        ci += IK;
        if (ci == Cin) { ci = 0; ++tap; }
    };
    auto store = [&](int buf) {
        char* d = lds + buf * (IM + IN) * IROW + lr * IROW + lp * 16;
#pragma unroll
        for (int j = 0; j < NA; ++j) *(uint4*)(d + 64 * j * IROW) = ra[j];
#pragma unroll
        for (int j = 0; j < NB; ++j) *(uint4*)(d + (IM + 64 * j) * IROW) = rb[j];
    };
    f32x16 acc[BM][BN];
#pragma unroll
    for (int i = 0; i < BM; ++i)
#pragma unroll
        for (int j = 0; j < BN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    load(0);
    store(0);
    __syncthreads();
    for (int kt = 0; kt < nk; ++kt) {
        if (kt + 1 < nk) load(kt + 1);
        const char* buf = lds + (kt & 1) * (IM + IN) * IROW;
#pragma unroll
        for (int sub = 0; sub < IK / 16; ++sub) {
            const int off = sub * 32 + (lane >> 5) * 16;
            bf16x8 fa[BM], fb[BN];
#pragma unroll
            for (int i = 0; i < BM; ++i)
                fa[i] = *(const bf16x8*)(buf + ((wm * BM + i) * 32 + (lane & 31)) * IROW + off);
#pragma unroll
            for (int j = 0; j < BN; ++j)
                fb[j] = *(const bf16x8*)(buf + (IM + (wn * BN + j) * 32 + (lane & 31)) * IROW + off);
#pragma unroll
            for (int i = 0; i < BM; ++i)
#pragma unroll
                for (int j = 0; j < BN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
        }
        if (kt + 1 < nk) store((kt + 1) & 1);
        __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < BN; ++j) {
        const int cl = (wn * BN + j) * 32 + (lane & 31), co = n0 + cl;
        const float bv = co < Cout ? bf16_to_f(bias[co]) : 0.f;
#pragma unroll
        for (int i = 0; i < BM; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = (wm * BM + i) * 32 + acc_row(r, lane);
                const float v = acc[i][j][r] + bv;
                if (OUTF32) {
                    if (m0 + row < M && co < Cout) ((float*)out)[(m0 + row) * ldo + co] = v;
                } else {
                    *(uint16_t*)(lds + row * OR + cl * 2) = f_to_bf16(fmaxf(v, 0.f));
                }
            }
    }
    if (OUTF32) return;
    __syncthreads();
    if (Cout & 7) {   // last layer only: rows are not 16-byte aligned
        const int w = min(IN, Cout - n0);
        for (int c = tid; c < IM * w; c += 256) {
            const int row = c / w, q = c - row * w;
            if (m0 + row < M)
                ((uint16_t*)out)[(m0 + row) * Cout + n0 + q] = *(const uint16_t*)(lds + row * OR + q * 2);
        }
        return;
    }
    const int per = min(IN, Cout - n0) / 8;   // 16-byte chunks per row
    for (int c = tid; c < IM * per; c += 256) {
        const int row = c / per, q = c - row * per;
        if (m0 + row < M)
            *(uint4*)((uint16_t*)out + (m0 + row) * Cout + n0 + q * 8) = *(const uint4*)(lds + row * OR + q * 16);
    }
}

// BF16 inference weights: conv [co][ci][ky][kx] -> [co][ky*3+kx][ci]; FC
// [class][c*hw + pos] -> [class][pos*C + c] (NHWC flattening).
__global__ void k_perm_conv(const float* __restrict__ W, int Cout, int Cin, uint16_t* __restrict__ o) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long)Cout * Cin * 9) return;
    const int tap = (int)(t % 9);
    const int ci = (int)((t / 9) % Cin);
    const long co = t / (9l * Cin);
    o[(co * 9 + tap) * Cin + ci] = f_to_bf16(W[t]);
}

__global__ void k_perm_fc(const float* __restrict__ W, int ncls, int C, int hw, uint16_t* __restrict__ o) {
    const long F = (long)C * hw;
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long)ncls * F) return;
    const long cls = t / F;
    const int f = (int)(t % F);
    const int c = f / hw, pos = f % hw;
    o[cls * F + (long)pos * C + c] = f_to_bf16(W[t]);
}

}  // namespace

// ================================================================ host
struct bsx_cnn {
    int S = 0, ch[5] = {1, 0, 0, 0, 0}, nclass = 0, maxb = 0;
    int hw[5];                 // spatial edge per activation level
    long woff[5], boff[5];     // offsets of W/b of layers 1..4 and the FC (index 4)
    long nparam = 0, feat = 0;
    float* d_p = nullptr;      // parameters
    float* d_g = nullptr;      // gradients
    float* d_m = nullptr;
    float* d_v = nullptr;
    uint16_t* d_pb = nullptr;  // BF16 copy for inference
    bool pb_valid = false;
    float* d_act[5] = {};      // activations 1..4 (index 1..4), logits at [0]
    float* d_gact[5] = {};
    float* d_loss = nullptr;
    // training: conv weights of layers 2-4 reordered for k_conv32 (forward,
    // data gradient), and the shares of split sums, sized for every batch up to
    // max_batch, so that no step allocates
    float* d_wt[2] = {};
    long wt_ofs[5] = {};
    float* d_part = nullptr;
    long step = 0;
    // MFMA inference: permuted BF16 weights of layers 2-4 and the FC; NHWC
    // BF16 activations of layers 1-4 and FP32 logits, sized for chunks larger
    // than the training batch (a 512-particle chunk leaves most of the chip
    // idle in layers 3-4 and the FC)
    uint16_t* d_wi[5] = {};
    int icap = 0;
    uint16_t* d_ib[5] = {};
    float* d_ilog = nullptr;
    // contrastive training scratch (pairs of up to maxb / 2): unit rows,
    // norms, pair scores and their softmaxes, gradients
    float* d_nce = nullptr;
    long nce_cap = 0;
    float* d_match = nullptr;    // embedding top-k: scores of a particle chunk
    long match_cap = 0;
};

namespace {

void free_cnn(bsx_cnn* h) {
    void* ptrs[] = {h->d_p, h->d_g, h->d_m, h->d_v, h->d_pb, h->d_loss};
    for (void* q : ptrs)
        if (q) (void)hipFree(q);
    for (int i = 0; i < 5; ++i) {
        if (h->d_act[i]) (void)hipFree(h->d_act[i]);
        if (h->d_gact[i]) (void)hipFree(h->d_gact[i]);
        if (h->d_wi[i]) (void)hipFree(h->d_wi[i]);
        if (h->d_ib[i]) (void)hipFree(h->d_ib[i]);
    }
    for (float* q : h->d_wt)
        if (q) (void)hipFree(q);
    if (h->d_part) (void)hipFree(h->d_part);
    if (h->d_ilog) (void)hipFree(h->d_ilog);
    if (h->d_nce) (void)hipFree(h->d_nce);
    if (h->d_match) (void)hipFree(h->d_match);
}

long act_size(const bsx_cnn* h, int l, int B) {
    if (l == 0) return (long)B * h->nclass;
    return (long)B * h->ch[l] * h->hw[l] * h->hw[l];
}

// splitmix64 + Box-Muller: reproducible He-normal initialisation
struct Rng {
    uint64_t s;
    uint64_t next() {
        uint64_t z = (s += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        return z ^ (z >> 31);
    }
    double uniform() { return ((next() >> 11) + 0.5) * (1.0 / 9007199254740992.0); }
    double normal() { return sqrt(-2 * log(uniform())) * cos(2 * M_PI * uniform()); }
};

// The k best of each of n rows of C logits. One wavefront reads a row in about
// 4 us a thousand logits, which few long rows wait for; several share it where
// the rows leave CUs idle and their reading outweighs the 5 us (4 wavefronts) and
// 20 us (16) that a row's join takes, or 2 x and 8 x the rows a CU holds (scores of
// 16 values and the top 16, 1 / 4 / 16 wavefronts a row): 16 x 65,536 295 / 98 / 60 us,
// 16 x 16,384 88 / 44 / 45, 16 x 1,200 26 / 27 / 40; 256 x 4,368 42 / 33 / 44,
// 512 x 4,368 44 / 39 / 70, 1,024 x 4,368 48 / 54 / 118; 512 x 65,536 471 / 170 / 125,
// 1,024 x 65,536 530 / 229 / 223; 2,048 x 16,384 161 / 123 / 243, 4,096 x 16,384
// 222 / 220 / 468.
int row_topk(const float* logits, long n, int C, int k, int* cls, float* prob, hipStream_t s) {
    auto go = [&](auto kernel, int rows, int threads) {
        hipLaunchKernelGGL(kernel, dim3(nblk(n, rows)), dim3(threads), 0, s, logits, n, C, k, cls, prob);
    };
    if (C >= 32768 && n <= 512) go(k_row_topk<16>, 1, 1024);
    else if ((C >= 4096 && n <= 256) || (C >= 16384 && n <= 2048)) go(k_row_topk<4>, 1, 256);
    else go(k_row_topk<1>, 4, 256);
    BSX_HIP(hipGetLastError());
    return BSX_OK;
}

// Shares that a sum over `steps` stages is split into so that some 512
// workgroups (two per CU) run, with at least 4 stages a share.
int shares(long tiles, long steps) {
    return (int)std::max<long>(1, std::min<long>((512 + tiles - 1) / tiles, steps / 4));
}

// The matrix-core kernels of a stride-2 layer take input channels in whole
// 16-channel stages (the data gradient: output channels too); other channel
// counts keep the direct kernels.
bool conv32_ok(const bsx_cnn* h, int l) { return l >= 2 && h->ch[l - 1] % TK == 0 && h->ch[l] % TK == 0; }

// Shares of a k_gemm32 product, and the K range of each.
int gemm32_shares(int M, int N, int K, int* kper) {
    const int z = shares(((N + 63) / 64) * (long)((M + 63) / 64), (K + TK - 1) / TK);
    *kper = ((K + z - 1) / z + TK - 1) / TK * TK;
    return (K + *kper - 1) / *kper;
}

// Tiles and shares of a layer's weight gradient.
dim3 dw_grid(const bsx_cnn* h, int l, int B) {
    const int Cin = h->ch[l - 1], Cout = h->ch[l], Ho = h->hw[l];
    if (l == 1) return dim3(1, (Cout + 31) / 32, std::min(B, 512));
    const dim3 t((Cout + 63) / 64, (Cin + 31) / 32);
    return dim3(t.x, t.y, shares((long)t.x * t.y, ((long)B * Ho * Ho + 15) / 16));
}

// Values of the largest split sum of a forward or training step of up to
// h->maxb inputs or h->maxb / 2 pairs. A smaller batch may need more than a larger
// one (fewer tiles, more shares), so every batch is looked at.
long part_values(const bsx_cnn* h) {
    const int C = h->nclass, F = (int)h->feat;
    long n = 0;
    auto product = [&](int M, int N, int K) {
        int kper;
        const int nz = gemm32_shares(M, N, K, &kper);
        if (nz > 1) n = std::max(n, (long)M * N * nz);
    };
    for (int B = 1; B <= h->maxb; ++B) {
        for (int l = 1; l <= 4; ++l)
            if (l == 1 || conv32_ok(h, l))
                n = std::max(n, ((long)h->ch[l] * h->ch[l - 1] * 9 + h->ch[l]) * dw_grid(h, l, B).z);
        product(B, C, F);
        product(C, F, B);
        product(B, F, C);
        if (B % 2 == 0) {
            product(B / 2, B / 2, C);
            product(B / 2, C, B / 2);
        }
    }
    return n;
}

// C = A B (+ bias) on k_gemm32, K split over shares where C has few tiles.
int gemm32(bsx_cnn* h, int M, int N, int K, const float* A, long am, long ak, const float* B, long bk,
           long bn, const float* bias, float* C, hipStream_t s) {
    const dim3 g((N + 63) / 64, (M + 63) / 64);
    int kper;
    const int nz = gemm32_shares(M, N, K, &kper);
    if (nz == 1) {
        hipLaunchKernelGGL(k_gemm32, g, dim3(256), 0, s, M, N, K, A, am, ak, B, bk, bn, bias, C, K);
        BSX_HIP(hipGetLastError());
        return BSX_OK;
    }
    const long n = (long)M * N;
    hipLaunchKernelGGL(k_gemm32, dim3(g.x, g.y, nz), dim3(256), 0, s, M, N, K, A, am, ak, B, bk, bn,
                       (const float*)nullptr, h->d_part, kper);
    BSX_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_part_sum, dim3(nblk(n, 64)), dim3(1024), 0, s, h->d_part, nz, n, 0l, 1, bias, N, C);
    BSX_HIP(hipGetLastError());
    return BSX_OK;
}

// Fully connected layer of the forward pass; BF16 weights keep k_sgemm.
int forward_fc(bsx_cnn* h, int B, const float* W, const float* bias, hipStream_t s) {
    return gemm32(h, B, h->nclass, (int)h->feat, h->d_act[4], h->feat, 1, W, 1, h->feat, bias, h->d_act[0], s);
}
int forward_fc(bsx_cnn* h, int B, const uint16_t* W, const uint16_t* bias, hipStream_t s) {
    const int F = (int)h->feat, C = h->nclass;
    hipLaunchKernelGGL(k_sgemm, dim3((C + 63) / 64, (B + 63) / 64), dim3(256), 0, s, B, C, F,
                       h->d_act[4], (long)F, 1l, W, 1l, (long)F, bias, h->d_act[0], (long)C);
    BSX_HIP(hipGetLastError());
    return BSX_OK;
}

// Activations of the layers and the outputs d_act[0] for B inputs, with the
// FP32 parameters (training) or their BF16 copies.
template <typename TW>
int forward(bsx_cnn* h, const float* x, int B, const TW* P, hipStream_t s) {
    constexpr bool F32 = sizeof(TW) == 4;
    const float* in = x;
    if (F32 && (conv32_ok(h, 2) || conv32_ok(h, 3) || conv32_ok(h, 4))) {
        PermLayers L;
        for (int l = 2; l <= 4; ++l) {
            L.woff[l - 2] = h->woff[l - 1];
            L.ofs[l - 2] = h->wt_ofs[l];
            L.cin[l - 2] = h->ch[l - 1];
            L.cout[l - 2] = h->ch[l];
        }
        hipLaunchKernelGGL(k_perm_train, dim3(256, 3), dim3(256), 0, s, (const float*)P, L, h->d_wt[0],
                           h->d_wt[1]);
        BSX_HIP(hipGetLastError());
    }
    for (int l = 1; l <= 4; ++l) {
        const int Cin = h->ch[l - 1], Cout = h->ch[l], H = h->hw[l - 1], Ho = h->hw[l];
        const int stride = l == 1 ? 1 : 2;
        if (F32 && l == 1) {
            hipLaunchKernelGGL(k_conv1_32, dim3(nblk((long)B * H * H / 4), (Cout + 7) / 8), dim3(256), 0, s,
                               in, (const float*)P + h->woff[0], (const float*)P + h->boff[0],
                               h->d_act[1], B, H, Cout);
        } else if (F32 && conv32_ok(h, l)) {
            const float* w = h->d_wt[0] + h->wt_ofs[l];
            const float* bias = (const float*)P + h->boff[l - 1];
            const long pos = (long)B * Ho * Ho;
            if (Cout <= 32)
                hipLaunchKernelGGL((k_conv32<32, 128, false>), dim3(nblk(pos, 128)), dim3(256), 0, s, in, w,
                                   bias, (const float*)nullptr, h->d_act[l], B, Cin, Cout, H, H, Ho, Ho);
            else
                hipLaunchKernelGGL((k_conv32<64, 64, false>), dim3(nblk(pos, 64), (Cout + 63) / 64),
                                   dim3(256), 0, s, in, w, bias, (const float*)nullptr, h->d_act[l], B,
                                   Cin, Cout, H, H, Ho, Ho);
        } else {
            const long tot = (long)B * (Cout / 4) * Ho * Ho;
            hipLaunchKernelGGL((k_conv_fwd<TW>), dim3(nblk(tot)), dim3(256), 0, s, in, P + h->woff[l - 1],
                               P + h->boff[l - 1], h->d_act[l], B, Cin, H, H, Cout, Ho, Ho, stride);
        }
        BSX_HIP(hipGetLastError());
        in = h->d_act[l];
    }
    return forward_fc(h, B, P + h->woff[4], P + h->boff[4], s);
}

// Backpropagation from dL/dlogits in d_gact[0] (B rows) to the parameter
// gradients in d_g.
int backward_body(bsx_cnn* h, const float* x, int B, hipStream_t s) {
    const int F = (int)h->feat, C = h->nclass;
    float* P = h->d_p;
    float* G = h->d_g;
    // FC: dW = dl^T x, db = colsum(dl), dx = dl W
    int rc = gemm32(h, C, F, B, h->d_gact[0], 1, C, h->d_act[4], F, 1, nullptr, G + h->woff[4], s);
    if (rc) return rc;
    hipLaunchKernelGGL(k_colsum, dim3((C + 63) / 64), dim3(1024), 0, s, h->d_gact[0], B, C, G + h->boff[4]);
    BSX_HIP(hipGetLastError());
    rc = gemm32(h, B, F, C, h->d_gact[0], C, 1, P + h->woff[4], F, 1, nullptr, h->d_gact[4], s);
    if (rc) return rc;
    bool masked = false;   // d_gact[l] already holds the gradient before the ReLU
    for (int l = 4; l >= 1; --l) {
        const int Cin = h->ch[l - 1], Cout = h->ch[l], H = h->hw[l - 1], Ho = h->hw[l];
        const int stride = l == 1 ? 1 : 2;
        if (!masked) {
            const long na = act_size(h, l, B);
            hipLaunchKernelGGL(k_relu_bwd, dim3(nblk(na)), dim3(256), 0, s, h->d_gact[l], h->d_act[l], na);
            BSX_HIP(hipGetLastError());
        }
        masked = false;
        const float* in = l == 1 ? x : h->d_act[l - 1];
        const bool c32 = conv32_ok(h, l);
        const long nw = (long)Cout * Cin * 9, n = nw + Cout;
        if (l == 1 || c32) {
            // weights and biases are neighbours in the parameter vector
            const dim3 tiles = dw_grid(h, l, B);
            const int nz = (int)tiles.z;
            if (l == 1)
                hipLaunchKernelGGL(k_conv1_32_dw, dim3(nz, tiles.y), dim3(256), 0, s, h->d_gact[1], in,
                                   h->d_part, B, H, Cout, (B + nz - 1) / nz);
            else
                hipLaunchKernelGGL(k_conv32_dw, tiles, dim3(256), 0, s, h->d_gact[l], in,
                                   h->d_part, B, Cin, H, H, Cout, Ho, Ho);
            BSX_HIP(hipGetLastError());
            hipLaunchKernelGGL(k_part_sum, dim3(nblk(n, 64)), dim3(1024), 0, s, h->d_part, nz, n, nw,
                               l == 1 ? 1 : 9, (const float*)nullptr, 1, G + h->woff[l - 1]);
        } else {
            hipLaunchKernelGGL(k_conv_bwd_weight, dim3(Cout, Cin + 1), dim3(256), 0, s, h->d_gact[l], in,
                               G + h->woff[l - 1], G + h->boff[l - 1], B, Cin, H, H, Cout, Ho, Ho, stride);
        }
        BSX_HIP(hipGetLastError());
        if (l > 1 && c32) {
            const float* w = h->d_wt[1] + h->wt_ofs[l];
            const long pos = (long)B * Ho * Ho;
            if (Cin <= 32)
                hipLaunchKernelGGL((k_conv32<32, 128, true>), dim3(nblk(pos, 128), 1, 4), dim3(256), 0, s,
                                   h->d_gact[l], w, (const float*)nullptr, h->d_act[l - 1],
                                   h->d_gact[l - 1], B, Cout, Cin, H, H, Ho, Ho);
            else
                hipLaunchKernelGGL((k_conv32<64, 64, true>), dim3(nblk(pos, 64), (Cin + 63) / 64, 4),
                                   dim3(256), 0, s, h->d_gact[l], w, (const float*)nullptr,
                                   h->d_act[l - 1], h->d_gact[l - 1], B, Cout, Cin, H, H, Ho, Ho);
            BSX_HIP(hipGetLastError());
            masked = true;
        } else if (l > 1) {
            const long nx = (long)B * Cin * H * H;
            hipLaunchKernelGGL(k_conv_bwd_data, dim3(nblk(nx)), dim3(256), 0, s, h->d_gact[l],
                               P + h->woff[l - 1], h->d_gact[l - 1], B, Cin, H, H, Cout, Ho, Ho, stride);
            BSX_HIP(hipGetLastError());
        }
    }
    return BSX_OK;
}


int backward(bsx_cnn* h, const float* x, const int* labels, int B, hipStream_t s) {
    hipLaunchKernelGGL(k_softmax_ce, dim3(B), dim3(256), 0, s, h->d_act[0], labels, B, h->nclass,
                       h->d_gact[0], h->d_loss);
    BSX_HIP(hipGetLastError());
    return backward_body(h, x, B, s);
}

// Network outputs of n inputs in chunks (BF16 MFMA layers when the channel
// counts allow, else the FP32-accumulating BF16 path): calls
// use(logits, first, count) for each chunk, on stream s.
template <class Use>
int infer_chunks(bsx_cnn* h, const float* x_dev, int64_t n, hipStream_t s, const char* who, Use use) {
    // the MFMA layers need input channel counts (c1..c3 and the FC input) in multiples of 32
    const bool mfma = h->ch[1] % 32 == 0 && h->ch[2] % 32 == 0 && h->ch[3] % 32 == 0 &&
                      h->feat % 32 == 0;
    if (!h->pb_valid) {
        hipLaunchKernelGGL(k_to_bf16, dim3(nblk(h->nparam)), dim3(256), 0, s, h->d_p, h->d_pb, h->nparam);
        BSX_HIP(hipGetLastError());
        if (mfma) {
            for (int l = 1; l < 4; ++l) {
                const long nw = (long)h->ch[l + 1] * h->ch[l] * 9;
                hipLaunchKernelGGL(k_perm_conv, dim3(nblk(nw)), dim3(256), 0, s, h->d_p + h->woff[l],
                                   h->ch[l + 1], h->ch[l], h->d_wi[l]);
                BSX_HIP(hipGetLastError());
            }
            const long nf = h->feat * h->nclass;
            hipLaunchKernelGGL(k_perm_fc, dim3(nblk(nf)), dim3(256), 0, s, h->d_p + h->woff[4],
                               h->nclass, h->ch[4], h->hw[4] * h->hw[4], h->d_wi[4]);
            BSX_HIP(hipGetLastError());
        }
        h->pb_valid = true;
    }
    const long in = (long)h->S * h->S;
    // MFMA path: chunks of up to 4096 particles in the inference buffers
    int chunk = h->maxb;
    if (mfma) {
        chunk = (int)std::min<int64_t>(std::max<int64_t>(n, 1), 4096);
        chunk = std::max(chunk, std::min(h->maxb, 4096));
        if (chunk > h->icap) {
            for (int l = 1; l < 5; ++l) {
                if (h->d_ib[l]) (void)hipFree(h->d_ib[l]);
                h->d_ib[l] = nullptr;
            }
            if (h->d_ilog) (void)hipFree(h->d_ilog);
            h->d_ilog = nullptr;
            h->icap = 0;
            for (int l = 1; l < 5; ++l)
                if (device_malloc(&h->d_ib[l], sizeof(uint16_t) * act_size(h, l, chunk)) != hipSuccess) {
                    set_error("%s: inference activations (%d particles)", who, chunk);
                    return BSX_ERR_NOMEM;
                }
            if (device_malloc(&h->d_ilog, sizeof(float) * (size_t)chunk * h->nclass) != hipSuccess) {
                set_error("%s: logits (%d particles)", who, chunk);
                return BSX_ERR_NOMEM;
            }
            h->icap = chunk;
        }
        chunk = h->icap;
    }
    for (int64_t b0 = 0; b0 < n; b0 += chunk) {
        const int nb = (int)std::min<int64_t>(chunk, n - b0);
        if (!mfma) {
            int rc = forward<uint16_t>(h, x_dev + b0 * in, nb, h->d_pb, s);
            if (rc) return rc;
        } else {
            const uint16_t* P = h->d_pb;
            const long pos1 = (long)nb * (in / 4) * (h->ch[1] / 8);
            hipLaunchKernelGGL(k_conv1_nhwc, dim3(nblk(pos1)), dim3(256),
                               sizeof(float) * 10 * h->ch[1], s, x_dev + b0 * in, P + h->woff[0],
                               P + h->boff[0], nb, h->S, h->ch[1], h->d_ib[1]);
            BSX_HIP(hipGetLastError());
            for (int l = 2; l <= 4; ++l) {
                // up to 64 output channels 256 x 64 tiles, else 128 x 128; 64 x 64
                // where those would leave CUs without a tile
                const long M = (long)nb * h->hw[l] * h->hw[l];
                const int N = h->ch[l], im = N <= 64 ? 256 : 128, in_ = N <= 64 ? 64 : 128;
                const bool few = ((M + im - 1) / im) * ((N + in_ - 1) / in_) < 256;
                auto go = [&](auto kernel, int tm, int tn) {
                    hipLaunchKernelGGL(kernel, dim3((unsigned)((M + tm - 1) / tm), (unsigned)((N + tn - 1) / tn)),
                                       dim3(256), 0, s, h->d_ib[l - 1], nb, h->hw[l - 1], h->hw[l - 1],
                                       h->ch[l - 1], h->hw[l], h->hw[l], h->d_wi[l - 1], P + h->boff[l - 1],
                                       N, (long)N, (void*)h->d_ib[l]);
                };
                if (few) go(k_conv_mfma<1, 1, 2, 2, 3, false>, 64, 64);
                else if (N <= 64) go(k_conv_mfma<2, 2, 4, 1, 3, false>, 256, 64);
                else go(k_conv_mfma<2, 2, 2, 2, 3, false>, 128, 128);
                BSX_HIP(hipGetLastError());
            }
            const bool few = ((nb + 127l) / 128) * ((h->nclass + 127l) / 128) < 256;
            auto fc = [&](auto kernel, int t) {
                hipLaunchKernelGGL(kernel, dim3((unsigned)((nb + t - 1) / t), (unsigned)((h->nclass + t - 1) / t)),
                                   dim3(256), 0, s, h->d_ib[4], nb, 1, 1, (int)h->feat, 1, 1, h->d_wi[4],
                                   P + h->boff[4], h->nclass, (long)h->nclass, (void*)h->d_ilog);
            };
            if (few) fc(k_conv_mfma<1, 1, 2, 2, 1, true>, 64);
            else fc(k_conv_mfma<2, 2, 2, 2, 1, true>, 128);
            BSX_HIP(hipGetLastError());
        }
        const int rc = use(mfma ? h->d_ilog : h->d_act[0], b0, nb);
        if (rc) return rc;
    }
    return BSX_OK;
}

}  // namespace

extern "C" {

int bsx_cnn_create(bsx_cnn** out, int32_t in_size, const int32_t* channels, int32_t nclasses,
                   int32_t max_batch, uint64_t seed) {
    BSX_REQUIRE(out && channels, BSX_ERR_ARG, "bsx_cnn_create: null argument");
    *out = nullptr;
    BSX_REQUIRE(in_size >= 8 && in_size <= 256 && in_size % 8 == 0, BSX_ERR_ARG,
                "bsx_cnn_create: input size %d must be a multiple of 8 in 8..256", in_size);
    for (int i = 0; i < 4; ++i)
        BSX_REQUIRE(channels[i] >= 4 && channels[i] <= 1024 && channels[i] % 4 == 0, BSX_ERR_ARG,
                    "bsx_cnn_create: channel count %d must be a multiple of 4 in 4..1024", channels[i]);
    BSX_REQUIRE(channels[0] <= 1024 && channels[0] % 2 == 0, BSX_ERR_ARG,
                "bsx_cnn_create: first-layer channel count must be even");
    BSX_REQUIRE(nclasses >= 2 && nclasses <= (1 << 20), BSX_ERR_ARG,
                "bsx_cnn_create: %d classes out of range", nclasses);
    BSX_REQUIRE(max_batch >= 1 && max_batch <= 65536, BSX_ERR_ARG,
                "bsx_cnn_create: max_batch %d out of range", max_batch);
    bsx_cnn* h = new bsx_cnn();
    h->S = in_size;
    for (int i = 0; i < 4; ++i) h->ch[i + 1] = channels[i];
    h->nclass = nclasses;
    h->maxb = max_batch;
    h->hw[0] = h->hw[1] = in_size;
    h->hw[2] = in_size / 2;
    h->hw[3] = in_size / 4;
    h->hw[4] = in_size / 8;
    h->feat = (long)h->ch[4] * h->hw[4] * h->hw[4];
    long o = 0;
    for (int l = 0; l < 4; ++l) {
        h->woff[l] = o;
        o += (long)h->ch[l + 1] * h->ch[l] * 9;
        h->boff[l] = o;
        o += h->ch[l + 1];
    }
    h->woff[4] = o;
    o += h->feat * nclasses;
    h->boff[4] = o;
    o += nclasses;
    h->nparam = o;
    // He-normal initialisation, zero biases
    std::vector<float> p((size_t)o, 0.f);
    Rng r{seed ? seed : 0x5eedull};
    for (int l = 0; l < 5; ++l) {
        const long fan_in = l < 4 ? (long)h->ch[l] * 9 : h->feat;
        const long nw = l < 4 ? (long)h->ch[l + 1] * h->ch[l] * 9 : h->feat * nclasses;
        const double sd = sqrt(2.0 / fan_in) * (l == 4 ? 0.5 : 1.0);
        for (long i = 0; i < nw; ++i) p[h->woff[l] + i] = (float)(sd * r.normal());
    }
    auto fail = [&](hipError_t e, const char* what) {
        set_error("bsx_cnn_create: %s: %s", what, hipGetErrorString(e));
        free_cnn(h);
        delete h;
        return BSX_ERR_NOMEM;
    };
    hipError_t e;
    if ((e = device_malloc(&h->d_p, sizeof(float) * o)) != hipSuccess) return fail(e, "parameters");
    if ((e = device_malloc(&h->d_g, sizeof(float) * o)) != hipSuccess) return fail(e, "gradients");
    if ((e = device_malloc(&h->d_m, sizeof(float) * o)) != hipSuccess) return fail(e, "moments");
    if ((e = device_malloc(&h->d_v, sizeof(float) * o)) != hipSuccess) return fail(e, "moments");
    if ((e = device_malloc(&h->d_pb, sizeof(uint16_t) * o)) != hipSuccess) return fail(e, "bf16 copy");
    if ((e = device_malloc(&h->d_loss, sizeof(float) * max_batch)) != hipSuccess) return fail(e, "loss");
    for (int l = 0; l < 5; ++l) {
        const long n = act_size(h, l, max_batch);
        if ((e = device_malloc(&h->d_act[l], sizeof(float) * n)) != hipSuccess) return fail(e, "activations");
        if ((e = device_malloc(&h->d_gact[l], sizeof(float) * n)) != hipSuccess) return fail(e, "activations");
    }
    for (int l = 2; l <= 4; ++l) h->wt_ofs[l] = l == 2 ? 0 : h->wt_ofs[l - 1] + (long)h->ch[l - 1] * h->ch[l - 2] * 9;
    for (float*& q : h->d_wt)
        if ((e = device_malloc(&q, sizeof(float) * (h->wt_ofs[4] + (long)h->ch[4] * h->ch[3] * 9))) != hipSuccess)
            return fail(e, "training weights");
    if ((e = device_malloc(&h->d_part, sizeof(float) * std::max(1l, part_values(h)))) != hipSuccess)
        return fail(e, "training sums");
    for (int l = 1; l < 4; ++l)
        if ((e = device_malloc(&h->d_wi[l], sizeof(uint16_t) * h->ch[l + 1] * h->ch[l] * 9)) != hipSuccess)
            return fail(e, "inference weights");
    if ((e = device_malloc(&h->d_wi[4], sizeof(uint16_t) * h->feat * nclasses)) != hipSuccess)
        return fail(e, "inference weights");
    if ((e = hipMemcpy(h->d_p, p.data(), sizeof(float) * o, hipMemcpyHostToDevice)) != hipSuccess ||
        (e = hipMemset(h->d_m, 0, sizeof(float) * o)) != hipSuccess ||
        (e = hipMemset(h->d_v, 0, sizeof(float) * o)) != hipSuccess ||
        (e = hipMemset(h->d_g, 0, sizeof(float) * o)) != hipSuccess)
        return fail(e, "initialisation");
    *out = h;
    return BSX_OK;
}

int bsx_cnn_destroy(bsx_cnn* h) {
    if (!h) return BSX_OK;
    free_cnn(h);
    delete h;
    return BSX_OK;
}

int bsx_cnn_nparams(const bsx_cnn* h, int64_t* n, int64_t* feature_size) {
    BSX_REQUIRE(h, BSX_ERR_ARG, "bsx_cnn_nparams: null handle");
    if (n) *n = h->nparam;
    if (feature_size) *feature_size = h->feat;
    return BSX_OK;
}

int bsx_cnn_params(bsx_cnn* h, float* get_dev, const float* set_dev, void* stream) {
    BSX_REQUIRE(h, BSX_ERR_ARG, "bsx_cnn_params: null handle");
    hipStream_t s = (hipStream_t)stream;
    if (get_dev)
        BSX_HIP(hipMemcpyAsync(get_dev, h->d_p, sizeof(float) * h->nparam, hipMemcpyDeviceToDevice, s));
    if (set_dev) {
        BSX_HIP(hipMemcpyAsync(h->d_p, set_dev, sizeof(float) * h->nparam, hipMemcpyDeviceToDevice, s));
        h->pb_valid = false;
    }
    return BSX_OK;
}

int bsx_cnn_forward(bsx_cnn* h, const float* x_dev, int32_t batch, float* logits_dev, void* stream) {
    BSX_REQUIRE(h && x_dev, BSX_ERR_ARG, "bsx_cnn_forward: null argument");
    BSX_REQUIRE(batch >= 1 && batch <= h->maxb, BSX_ERR_ARG, "bsx_cnn_forward: batch %d out of 1..%d",
                batch, h->maxb);
    hipStream_t s = (hipStream_t)stream;
    int rc = forward<float>(h, x_dev, batch, h->d_p, s);
    if (rc) return rc;
    if (logits_dev)
        BSX_HIP(hipMemcpyAsync(logits_dev, h->d_act[0], sizeof(float) * batch * h->nclass,
                               hipMemcpyDeviceToDevice, s));
    return BSX_OK;
}

int bsx_cnn_gradients(bsx_cnn* h, const float* x_dev, const int32_t* labels_dev, int32_t batch,
                      float* grad_dev, float* loss_dev, void* stream) {
    BSX_REQUIRE(h && x_dev && labels_dev, BSX_ERR_ARG, "bsx_cnn_gradients: null argument");
    BSX_REQUIRE(batch >= 1 && batch <= h->maxb, BSX_ERR_ARG,
                "bsx_cnn_gradients: batch %d out of 1..%d", batch, h->maxb);
    hipStream_t s = (hipStream_t)stream;
    int rc = forward<float>(h, x_dev, batch, h->d_p, s);
    if (!rc) rc = backward(h, x_dev, labels_dev, batch, s);
    if (rc) return rc;
    if (grad_dev)
        BSX_HIP(hipMemcpyAsync(grad_dev, h->d_g, sizeof(float) * h->nparam, hipMemcpyDeviceToDevice, s));
    if (loss_dev)
        BSX_HIP(hipMemcpyAsync(loss_dev, h->d_loss, sizeof(float) * batch, hipMemcpyDeviceToDevice, s));
    return BSX_OK;
}

int bsx_cnn_train_step(bsx_cnn* h, const float* x_dev, const int32_t* labels_dev, int32_t batch,
                       float lr, float weight_decay, float* loss_dev, void* stream) {
    BSX_REQUIRE(lr > 0 && std::isfinite(lr) && weight_decay >= 0, BSX_ERR_ARG,
                "bsx_cnn_train_step: bad learning rate / weight decay");
    int rc = bsx_cnn_gradients(h, x_dev, labels_dev, batch, nullptr, loss_dev, stream);
    if (rc) return rc;
    hipStream_t s = (hipStream_t)stream;
    h->step++;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - powf(b1, (float)h->step), c2 = 1.f - powf(b2, (float)h->step);
    hipLaunchKernelGGL(k_adam, dim3(nblk(h->nparam)), dim3(256), 0, s, h->d_p, h->d_g, h->d_m, h->d_v,
                       h->nparam, lr, b1, b2, 1e-8f, c1, c2, weight_decay);
    BSX_HIP(hipGetLastError());
    h->pb_valid = false;
    return BSX_OK;
}

int bsx_cnn_infer_topk(bsx_cnn* h, const float* x_dev, int64_t n, int32_t k, int32_t* cls_dev,
                       float* prob_dev, void* stream) {
    BSX_REQUIRE(h && (n == 0 || (x_dev && cls_dev && prob_dev)), BSX_ERR_ARG,
                "bsx_cnn_infer_topk: null argument");
    BSX_REQUIRE(k >= 1 && k <= 32 && k <= h->nclass, BSX_ERR_ARG, "bsx_cnn_infer_topk: k %d out of range", k);
    hipStream_t s = (hipStream_t)stream;
    return infer_chunks(h, x_dev, n, s, "bsx_cnn_infer_topk", [&](const float* lg, int64_t b0, int nb) {
        return row_topk(lg, nb, h->nclass, k, cls_dev + b0 * k, prob_dev + b0 * k, s);
    });
}

int bsx_cnn_embed(bsx_cnn* h, const float* x_dev, int64_t n, float* emb_dev, void* stream) {
    BSX_REQUIRE(h && (n == 0 || (x_dev && emb_dev)), BSX_ERR_ARG, "bsx_cnn_embed: null argument");
    hipStream_t s = (hipStream_t)stream;
    const int d = h->nclass;
    return infer_chunks(h, x_dev, n, s, "bsx_cnn_embed", [&](const float* lg, int64_t b0, int nb) {
        hipLaunchKernelGGL(k_unit_rows, dim3(nblk(nb, 4)), dim3(256), 0, s, lg, (long)nb, d,
                           emb_dev + b0 * d, (float*)nullptr);
        BSX_HIP(hipGetLastError());
        return BSX_OK;
    });
}

int bsx_cnn_match_topk(bsx_cnn* h, const float* p_dev, int64_t n, const float* r_dev, int32_t m,
                       int32_t k, float tau, int32_t* cls_dev, float* prob_dev, void* stream) {
    BSX_REQUIRE(h && (n == 0 || (p_dev && r_dev && cls_dev && prob_dev)), BSX_ERR_ARG,
                "bsx_cnn_match_topk: null argument");
    BSX_REQUIRE(m >= 1 && k >= 1 && k <= 32 && k <= m, BSX_ERR_ARG,
                "bsx_cnn_match_topk: k %d / references %d out of range", k, m);
    BSX_REQUIRE(tau > 0 && std::isfinite(tau), BSX_ERR_ARG, "bsx_cnn_match_topk: bad temperature");
    if (n == 0) return BSX_OK;
    hipStream_t s = (hipStream_t)stream;
    const int d = h->nclass;
    const int64_t chunk = std::max<int64_t>(1, std::min<int64_t>(n, (256ll << 20) / (4ll * m)));
    if (chunk * m > h->match_cap) {
        if (h->d_match) (void)hipFree(h->d_match);
        h->d_match = nullptr;
        h->match_cap = 0;
        BSX_HIP(device_malloc(&h->d_match, sizeof(float) * chunk * m));
        h->match_cap = chunk * m;
    }
    for (int64_t b0 = 0; b0 < n; b0 += chunk) {
        const int nb = (int)std::min<int64_t>(chunk, n - b0);
        // scores = P R^T / tau: the rows' softmax over the references
        hipLaunchKernelGGL(k_scores32, dim3((m + 127) / 128, (nb + 127) / 128), dim3(256), 0, s, nb, m, d,
                           p_dev + b0 * d, r_dev, 1.f / tau, h->d_match);
        BSX_HIP(hipGetLastError());
        const int rc = row_topk(h->d_match, nb, m, k, cls_dev + b0 * k, prob_dev + b0 * k, s);
        if (rc) return rc;
    }
    return BSX_OK;
}

int bsx_cnn_pair_gradients(bsx_cnn* h, const float* x_dev, int32_t batch, float tau,
                           float* grad_dev, float* loss_dev, void* stream) {
    BSX_REQUIRE(h && x_dev, BSX_ERR_ARG, "bsx_cnn_pair_gradients: null argument");
    BSX_REQUIRE(batch >= 2 && 2 * batch <= h->maxb, BSX_ERR_ARG,
                "bsx_cnn_pair_gradients: batch %d out of 2..%d (pairs of the network's batch)",
                batch, h->maxb / 2);
    BSX_REQUIRE(tau > 0 && std::isfinite(tau), BSX_ERR_ARG,
                "bsx_cnn_pair_gradients: bad temperature");
    hipStream_t s = (hipStream_t)stream;
    const int B = batch, B2 = 2 * batch, d = h->nclass;
    // scratch: U (2B d), dU (2B d), norms (2B), S, P, Q, dS (B^2 each), losses (2B)
    const long need = 2l * B2 * d + 2l * B2 + 4l * B * B;
    if (need > h->nce_cap) {
        if (h->d_nce) (void)hipFree(h->d_nce);
        h->d_nce = nullptr;
        h->nce_cap = 0;
        BSX_HIP(device_malloc(&h->d_nce, sizeof(float) * need));
        h->nce_cap = need;
    }
    float* U = h->d_nce;
    float* dU = U + (long)B2 * d;
    float* nrm = dU + (long)B2 * d;
    float* lrl = nrm + B2;                // row losses (B), column losses (B)
    float* S = lrl + B2;
    float* P = S + (long)B * B;
    float* Q = P + (long)B * B;
    float* dS = Q + (long)B * B;
    int rc = forward<float>(h, x_dev, B2, h->d_p, s);
    if (rc) return rc;
    hipLaunchKernelGGL(k_unit_rows, dim3(nblk(B2, 4)), dim3(256), 0, s, h->d_act[0], (long)B2, d, U, nrm);
    BSX_HIP(hipGetLastError());
    const float* Up = U;
    const float* Ur = U + (long)B * d;
    // S = Up Ur^T (cosines)
    if ((rc = gemm32(h, B, B, d, Up, d, 1, Ur, 1, d, nullptr, S, s))) return rc;
    const float it = 1.f / tau;
    hipLaunchKernelGGL(k_pair_softmax, dim3(B), dim3(256), 0, s, S, B, it, 0, P, lrl);
    hipLaunchKernelGGL(k_pair_softmax, dim3(B), dim3(256), 0, s, S, B, it, 1, Q, lrl + B);
    hipLaunchKernelGGL(k_pair_grad, dim3(nblk((long)B * B)), dim3(256), 0, s, P, Q, B, it, lrl,
                       lrl + B, dS, h->d_loss);
    BSX_HIP(hipGetLastError());
    // dUp = dS Ur, dUr = dS^T Up
    if ((rc = gemm32(h, B, d, B, dS, B, 1, Ur, d, 1, nullptr, dU, s))) return rc;
    if ((rc = gemm32(h, B, d, B, dS, 1, B, Up, d, 1, nullptr, dU + (long)B * d, s))) return rc;
    hipLaunchKernelGGL(k_unit_rows_bwd, dim3(nblk(B2, 4)), dim3(256), 0, s, dU, U, nrm, (long)B2, d,
                       h->d_gact[0]);
    BSX_HIP(hipGetLastError());
    rc = backward_body(h, x_dev, B2, s);
    if (rc) return rc;
    if (grad_dev)
        BSX_HIP(hipMemcpyAsync(grad_dev, h->d_g, sizeof(float) * h->nparam, hipMemcpyDeviceToDevice, s));
    if (loss_dev)
        BSX_HIP(hipMemcpyAsync(loss_dev, h->d_loss, sizeof(float) * B, hipMemcpyDeviceToDevice, s));
    return BSX_OK;
}

int bsx_cnn_train_pairs(bsx_cnn* h, const float* x_dev, int32_t batch, float tau, float lr,
                        float weight_decay, float* loss_dev, void* stream) {
    BSX_REQUIRE(lr > 0 && std::isfinite(lr) && weight_decay >= 0, BSX_ERR_ARG,
                "bsx_cnn_train_pairs: bad learning rate / weight decay");
    int rc = bsx_cnn_pair_gradients(h, x_dev, batch, tau, nullptr, loss_dev, stream);
    if (rc) return rc;
    hipStream_t s = (hipStream_t)stream;
    h->step++;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - powf(b1, (float)h->step), c2 = 1.f - powf(b2, (float)h->step);
    hipLaunchKernelGGL(k_adam, dim3(nblk(h->nparam)), dim3(256), 0, s, h->d_p, h->d_g, h->d_m, h->d_v,
                       h->nparam, lr, b1, b2, 1e-8f, c1, c2, weight_decay);
    BSX_HIP(hipGetLastError());
    h->pb_valid = false;
    return BSX_OK;
}

}  // extern "C"
