// bsx_insert.hip — row transforms (K2) and insertion (K3) of the particle
// transforms for the transform size BSX_INSERT_FT (one translation unit each).
#include "bsx_insert.h"

// ------------------------------------------------------------------- K2
// One workgroup: 2*LINES rows of one particle (rows y0 + 2j, y0 + 2j + 1 form
// complex line j). Output: inter[p][x][y], x in [0, FT/2], y in [0, box).
template <int FT, int LINES>
__global__ __launch_bounds__(256) void k_rows(const float* __restrict__ imgs,
                                              const PartDev* __restrict__ recs,
                                              const float* __restrict__ bkg, int box,
                                              int tiles_per_part, float2* __restrict__ inter,
                                              const float2* __restrict__ twg,
                                              const double2* __restrict__ resc) {
    constexpr int T = FftThreads<FT>::value;
    constexpr int G = 256 / T;
    constexpr int NT = G * T;
    constexpr int HX = FT / 2 + 1;
    __shared__ __attribute__((aligned(16))) float2 lds[LINES * FT + FT];
    float2* tw = lds + LINES * FT;
    const int tid = threadIdx.x;
    const int p = blockIdx.x / tiles_per_part;
    const int y0 = (blockIdx.x % tiles_per_part) * 2 * LINES;
    const float* img = imgs + (size_t)recs[p].src * box * box;
    const float b = bkg[p];
    for (int i = tid; i < FT; i += NT) tw[i] = twg[i];
    // load: line j = rows (y0+2j, y0+2j+1), x < box from the image (rescaled
    // when resc is given) minus the background, zero elsewhere (the padded
    // region equals the background).
    if (resc) {
        const double2 rs = resc[p];
        for (int idx = tid; idx < LINES * FT; idx += NT) {
            const int j = idx / FT, x = idx - j * FT;
            const int ya = y0 + 2 * j, yb = ya + 1;
            float a = 0.f, c = 0.f;
            if (x < box) {
                if (ya < box) a = rescaled(img[(size_t)ya * box + x], rs) - b;
                if (yb < box) c = rescaled(img[(size_t)yb * box + x], rs) - b;
            }
            lds[j * FT + x] = make_float2(a, c);
        }
    } else if ((box & 3) == 0) {
        // rows y0 + 2j and y0 + 2j + 1 as float4 loads, written as four
        // (a, c) pairs; x in [box, FT) zero
        const int q4 = box >> 2;
        for (int idx = tid; idx < LINES * q4; idx += NT) {
            const int j = idx / q4, x4 = idx - j * q4;
            const int ya = y0 + 2 * j, yb = ya + 1;
            float4 a = make_float4(0.f, 0.f, 0.f, 0.f), c = a;
            if (ya < box) {
                a = *(const float4*)(img + (size_t)ya * box + 4 * x4);
                a.x -= b; a.y -= b; a.z -= b; a.w -= b;
            }
            if (yb < box) {
                c = *(const float4*)(img + (size_t)yb * box + 4 * x4);
                c.x -= b; c.y -= b; c.z -= b; c.w -= b;
            }
            float4* d = (float4*)(lds + j * FT + 4 * x4);
            d[0] = make_float4(a.x, c.x, a.y, c.y);
            d[1] = make_float4(a.z, c.z, a.w, c.w);
        }
        const int zq = (FT - box) >> 1;   // float4 (two pairs) per line beyond the image
        for (int idx = tid; idx < LINES * zq; idx += NT) {
            const int j = idx / zq, x2 = idx - j * zq;
            *(float4*)(lds + j * FT + box + 2 * x2) = make_float4(0.f, 0.f, 0.f, 0.f);
        }
    } else {
        for (int idx = tid; idx < LINES * FT; idx += NT) {
            const int j = idx / FT, x = idx - j * FT;
            const int ya = y0 + 2 * j, yb = ya + 1;
            float a = 0.f, c = 0.f;
            if (x < box) {
                if (ya < box) a = img[(size_t)ya * box + x] - b;
                if (yb < box) c = img[(size_t)yb * box + x] - b;
            }
            lds[j * FT + x] = make_float2(a, c);
        }
    }
    __syncthreads();
    const int g = tid / T, t = tid - g * T;
#pragma unroll 1
    for (int r0 = 0; r0 < LINES; r0 += G) FftLine<FT, -1, T>::run(lds + (r0 + g) * FT, tw, t);
    // store: for each x in [0, FT/2], the 2*LINES consecutive rows
    constexpr int ROWS = 2 * LINES;
    float2* out = inter + (size_t)p * HX * box;
    if ((box & 1) == 0) {
        // rows y0 + 2j (A) and y0 + 2j + 1 (B) of column x as one 16-byte store
        for (int idx = tid; idx < HX * LINES; idx += NT) {
            const int x = idx / LINES, j = idx - x * LINES;
            const int y = y0 + 2 * j;
            if (y >= box) continue;
            const float2 z = lds[j * FT + x];
            const float2 zm = lds[j * FT + ((FT - x) & (FT - 1))];
            *(float4*)(out + (size_t)x * box + y) =
                make_float4(0.5f * (z.x + zm.x), 0.5f * (z.y - zm.y),
                            0.5f * (z.y + zm.y), -0.5f * (z.x - zm.x));
        }
        return;
    }
    for (int idx = tid; idx < HX * ROWS; idx += NT) {
        const int x = idx / ROWS, r = idx - x * ROWS;
        const int y = y0 + r;
        if (y >= box) continue;
        const int j = r >> 1;
        const float2 z = lds[j * FT + x];
        const float2 zm = lds[j * FT + ((FT - x) & (FT - 1))];
        float2 v;
        if ((r & 1) == 0) v = make_float2(0.5f * (z.x + zm.x), 0.5f * (z.y - zm.y));   // A(x)
        else v = make_float2(0.5f * (z.y + zm.y), -0.5f * (z.x - zm.x));              // B(x)
        out[(size_t)x * box + y] = v;
    }
}

// 32-bit forms for the insertion hot path (coordinates stay within a few
// box sizes; record indices below 2^31 per half).
__device__ __forceinline__ unsigned rec_index32(int x, int y, int z, int NT) {
    return (unsigned)(((((z >> 4) * NT + (y >> 4)) * NT + (x >> 4)) << 12) | ((z & 15) << 8) |
                      ((y & 15) << 4) | (x & 15));
}
__device__ __forceinline__ int wrap32(int c, int n) {
    if (c >= 0 && c < n) return c;
    if (c < 0 && c >= -n) return c + n;
    if (c >= n && c < 2 * n) return c - n;
    c %= n;
    return c < 0 ? c + n : c;
}

enum { MODE_DIRECT = 0, MODE_FILL = 2 };

// One emission: a contribution to the record `key`; `kk` is the sample row
// (runs are merged only along unbroken k steps); `incl` marks samples the
// reference inserts (decided from geometry alone, so the count and fill
// passes agree exactly).
struct Emit {
    int key, kk, incl;
    int bin;         // MODE_FILL: 1 = binned entry, 0 = added to the volume directly
    float re, im, w, p, w2;
};

// Fill-pass staging in LDS: a workgroup appends its merged entries to a dense LDS list (one
// 16-B record each; a wavefront takes its slots with one LDS atomic) and
// counts them per bin in a small LDS hash table; at each flush one integer
// atomic per (workgroup, bin) reserves the bin range (at most two chunks)
// and the entries are written out.
#define BSX_STAGE_CAP 512      // entries per flush: 2 rounds x 1 binned emission x 256 threads
#define BSX_STAGE_HASH 128     // bins per flush (more fall back to direct reservations)
static_assert(BSX_STAGE_CAP <= BSX_CHUNK, "a flushed bin range must span at most two chunks");
static_assert(BSX_STAGE_CAP <= 1024 && BSX_STAGE_HASH <= 256, "list ranks take 10 bits, slots 8");

struct Stage {
    float4* ent;     // entries: (sum w re, sum w im, sum w, r) with r =
                     // (hash slot << 22) | (rank in the bin << 12) | record in tile,
                     // r = -1: slot taken by an entry reserved on its own
    int* nent;       // entries in the list
    int* hkey;       // bin per hash slot, -1 = free
    int* hcnt;       // entries per hash slot
    int4* hinfo;     // at a flush, per hash slot: reserved base, chunks of the
                     // range start and end, bin
    float2* ent2;    // FOM: (sum w|F|^2, sum w^2) of each entry, else null
};

struct BinCtx {
    int* fill;       // per-bin reservation counters (bin sizes after the fill)
    int* chunks;     // [nbins][maxc] pool chunk of each bin chunk, -1 = not yet, -2 = none
    int* pool;       // [0] next free pool chunk, [1] fallback flags (1 table, 2 pool, 4 wait)
    float4* bins;    // the pool: (re, im, w, record-in-tile) entries
    float* acc;      // volume records (3 floats), target of the atomic fallback
    int npool;       // chunks in the pool
    int maxc;        // chunks per bin
    Stage st;        // fill-pass staging
    float2* bins2;   // FOM: (sum w|F|^2, sum w^2) of each pool entry, else null
    int stride;      // floats per volume record (3, or 5 with the FOM sums)
};

// Takes a pool chunk (-2 when the pool is exhausted) and installs it as chunk
// ci of bin b unless one is there already; returns the installed value.
__device__ __forceinline__ int chunk_take(const BinCtx& bc, int b, int ci) {
    int nc = atomicAdd(bc.pool, 1);
    if (nc >= bc.npool) nc = -2;
    const int prev = atomicCAS(bc.chunks + (size_t)b * bc.maxc + ci, -1, nc);
    return prev == -1 ? nc : prev;
}

// Called by the reservation holding position ci * BSX_CHUNK of bin b.
__device__ __forceinline__ void chunk_alloc(const BinCtx& bc, int b, int ci) {
    if (ci < bc.maxc) (void)chunk_take(bc, b, ci);
}

// Pool chunk of chunk ci of bin b once its allocator has installed it. A wait
// past its bound installs a chunk itself (the allocator's chunk then goes
// unused), so every writer of a bin chunk agrees on it. -1 selects the atomic
// fallback (beyond the table or pool exhausted; then all writers of the chunk
// fall back and the tile pass skips it).
__device__ __forceinline__ int chunk_wait(const BinCtx& bc, int b, int ci) {
    if (ci >= bc.maxc) {
        atomicOr(bc.pool + 1, 1);
        return -1;
    }
    const int* slot = bc.chunks + (size_t)b * bc.maxc + ci;
    int c = -1;
    for (int i = 0; i < BSX_SPIN_LIMIT && c == -1; ++i) {
        c = __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (c == -1) __builtin_amdgcn_s_sleep(2);
    }
    if (c == -1) {
        atomicOr(bc.pool + 1, 4);
        c = chunk_take(bc, b, ci);
    }
    if (c == -2) {
        atomicOr(bc.pool + 1, 2);
        return -1;
    }
    return c;
}

__device__ __forceinline__ void put_entry(const BinCtx& bc, int c, int pos, float re, float im,
                                          float w, int key, float p = 0.f, float w2 = 0.f) {
    if (c >= 0) {
        const size_t e = (size_t)c * BSX_CHUNK + (pos & (BSX_CHUNK - 1));
        bc.bins[e] = make_float4(re, im, w, __int_as_float(key & 4095));
        if (bc.bins2) bc.bins2[e] = make_float2(p, w2);
    } else {
        float* rec = bc.acc + (size_t)(unsigned)key * bc.stride;
        unsafeAtomicAdd(rec + 0, re);
        unsafeAtomicAdd(rec + 1, im);
        unsafeAtomicAdd(rec + 2, w);
        if (bc.bins2) {
            unsafeAtomicAdd(rec + 3, p);
            unsafeAtomicAdd(rec + 4, w2);
        }
    }
}

// Resolves the (at most two) chunks of a reserved range [base, base + cnt):
// allocations first, then waits, so that no allocator is held up behind a
// wait of its own wavefront.
__device__ __forceinline__ void range_chunks(const BinCtx& bc, int b, int base, int cnt,
                                             bool any, int& c0, int& c1) {
    const int i0 = base / BSX_CHUNK, i1 = (base + cnt - 1) / BSX_CHUNK;
    if (any) {
        if ((base & (BSX_CHUNK - 1)) == 0) chunk_alloc(bc, b, i0);
        if (i1 != i0) chunk_alloc(bc, b, i1);
    }
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    if (any) {
        c0 = chunk_wait(bc, b, i0);
        c1 = i1 != i0 ? chunk_wait(bc, b, i1) : c0;
    }
}

// One entry into slot i of the workgroup's list (per-lane LDS atomics for
// the bin table: measured faster here than grouping the lanes of a
// wavefront by bin first).
__device__ __forceinline__ void stage_entry(const BinCtx& bc, int i, int key, float re, float im,
                                           float w, float p = 0.f, float w2 = 0.f) {
    const int bin = (int)((unsigned)key >> 12);
    int slot = -1;
    int hs = (int)(((unsigned)bin * 2654435761u) >> 25) & (BSX_STAGE_HASH - 1);
    for (int t = 0; t < BSX_STAGE_HASH; ++t) {
        const int prev = atomicCAS(&bc.st.hkey[hs], -1, bin);
        if (prev == -1 || prev == bin) { slot = hs; break; }
        hs = (hs + 1) & (BSX_STAGE_HASH - 1);
    }
    const bool alone = slot < 0;   // table full: reserve this entry on its own
    int pos = 0, c0 = -1, c1 = -1;
    if (alone) pos = atomicAdd(bc.fill + bin, 1);
    range_chunks(bc, bin, pos, 1, alone, c0, c1);
    if (alone) {
        put_entry(bc, c0, pos, re, im, w, key, p, w2);
        bc.st.ent[i] = make_float4(0.f, 0.f, 0.f, __int_as_float(-1));
        return;
    }
    const int rank = atomicAdd(&bc.st.hcnt[slot], 1);
    bc.st.ent[i] = make_float4(re, im, w, __int_as_float((slot << 22) | (rank << 12) | (key & 4095)));
    if (bc.st.ent2) bc.st.ent2[i] = make_float2(p, w2);
}

// The lanes with `out` set append their entries: dense slots from one LDS
// atomic per wavefront (all lanes call this together).
__device__ __forceinline__ void stage_append(const BinCtx& bc, bool out, int key, float re,
                                            float im, float w, float p = 0.f, float w2 = 0.f) {
    const unsigned long long m = __ballot(out);
    if (m == 0) return;
    const int lane = __lane_id();
    const int leader = __builtin_ctzll(m);
    int base = 0;
    if (lane == leader) base = atomicAdd(bc.st.nent, __popcll(m));
    base = __shfl(base, leader, 64);
    if (out) stage_entry(bc, base + __popcll(m & ((1ull << lane) - 1ull)), key, re, im, w, p, w2);
}

// Workgroup-uniform: reserve every staged bin range, write the staged
// entries, clear the list (r = -1: empty slot) and the table.
__device__ __forceinline__ void stage_flush(const BinCtx& bc) {
    __syncthreads();
    const int tid = threadIdx.x;
    int b = -1, cnt = 0, base = 0, c0 = -1, c1 = -1;
    if (tid < BSX_STAGE_HASH) {
        b = bc.st.hkey[tid];
        if (b >= 0) {
            cnt = bc.st.hcnt[tid];
            base = atomicAdd(bc.fill + b, cnt);
        }
    }
    range_chunks(bc, b, base, cnt, b >= 0, c0, c1);
    if (b >= 0) bc.st.hinfo[tid] = make_int4(base, c0, c1, b);
    __syncthreads();
    const int n = *bc.st.nent;
    for (int i = tid; i < n; i += blockDim.x) {
        const float4 e = bc.st.ent[i];
        const int pr = __float_as_int(e.w);
        if (pr < 0) continue;
        const int4 hi = bc.st.hinfo[pr >> 22];
        const int pos = hi.x + ((pr >> 12) & 1023);
        const int c = pos / BSX_CHUNK == hi.x / BSX_CHUNK ? hi.y : hi.z;
        // full record key (bin from the hash slot) for the atomic fallback
        const int key = (int)(((unsigned)hi.w << 12) | (unsigned)(pr & 4095));
        const float2 e2 = bc.st.ent2 ? bc.st.ent2[i] : make_float2(0.f, 0.f);
        put_entry(bc, c, pos, e.x, e.y, e.z, key, e2.x, e2.y);
    }
    __syncthreads();
    if (tid < BSX_STAGE_HASH) {
        bc.st.hkey[tid] = -1;
        bc.st.hcnt[tid] = 0;
    }
    if (tid == 0) *bc.st.nent = 0;
    __syncthreads();
}

// Row shifts of a wavefront (DPP, rows of 16 lanes): dpp_down<D> gives lane
// i the value of lane i + D of its row, dpp_up1 that of lane i - 1; lanes
// whose source lies outside the row read 0 (the merge conditions exclude
// them).
template <int D>
__device__ __forceinline__ int dpp_down(int v) {
    static_assert(D >= 1 && D <= 15, "row shift");
    return __builtin_amdgcn_update_dpp(0, v, 0x100 + D, 0xF, 0xF, true);
}
template <int D>
__device__ __forceinline__ float dpp_downf(float v) {
    return __int_as_float(dpp_down<D>(__float_as_int(v)));
}
__device__ __forceinline__ int dpp_up1(int v) {
    return __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, true);
}

// One step of the segmented suffix sum below: lane l takes lane l + D's sums
// when both hold the same key and bin flag and their sample rows differ by D.
// pk packs (row << 2) | (bin << 1) | incl.
template <int D, int MG, bool FOM>
__device__ __forceinline__ void merge_step(Emit& e, int& pk, int lg) {
    if (D >= MG) return;
    const int nk = dpp_down<D>(e.key);
    const int np = dpp_down<D>(pk);
    const float r0 = dpp_downf<D>(e.re);
    const float r1 = dpp_downf<D>(e.im);
    const float r2 = dpp_downf<D>(e.w);
    float r3 = 0.f, r4 = 0.f;
    if (FOM) {
        r3 = dpp_downf<D>(e.p);
        r4 = dpp_downf<D>(e.w2);
    }
    if (lg + D < MG && nk == e.key && ((np ^ pk) & 2) == 0 && abs((np >> 2) - e.kk) == D) {
        pk |= np & 1;
        e.re += r0;
        e.im += r1;
        e.w += r2;
        if (FOM) { e.p += r3; e.w2 += r4; }
    }
}

// Merges runs of equal keys inside aligned groups of MG <= 16 lanes (segmented
// Hillis-Steele suffix sums over DPP row shifts); lanes l and l+d merge only if their keys are
// equal and their sample rows differ by exactly d, so the samples between lie
// on one straight segment and equal keys are contiguous (a periodic revisit
// would need a segment longer than N-1 voxels, excluded on the host). The
// first lane of each run then adds to the volume with atomics (MODE_DIRECT, and
// samples without a pair entry) or appends to the workgroup's list.
template <int MG, bool FOM, int MODE, int FAST = 0>
__device__ __forceinline__ void emit(float* __restrict__ acc, int stride, int merge, Emit e,
                                     const BinCtx& bc) {
    bool head = true;
    if (MG > 1 && merge) {
        const int lg = __lane_id() & (MG - 1);
        // sample row, bin flag and inclusion in one word for the shifts
        int pk = (e.kk * 4) | (e.bin << 1) | e.incl;
        merge_step<1, MG, FOM>(e, pk, lg);
        merge_step<2, MG, FOM>(e, pk, lg);
        if (merge == 1) {   // runs may exceed 4 samples (merge 2: the host showed they do not)
            merge_step<4, MG, FOM>(e, pk, lg);
            merge_step<8, MG, FOM>(e, pk, lg);
        }
        e.incl = pk & 1;
        const int prev_key = dpp_up1(e.key);
        const int prev_pk = dpp_up1(pk);
        head = !(lg != 0 && prev_key == e.key && ((prev_pk ^ pk) & 2) == 0 &&
                 abs(e.kk - (prev_pk >> 2)) == 1);
    }
    const bool out0 = head && e.incl;
    if (MODE == MODE_DIRECT || !e.bin) {
        if (!out0) return;
        float* rec = acc + (size_t)(unsigned)e.key * stride;
        unsafeAtomicAdd(rec + 0, e.re);
        unsafeAtomicAdd(rec + 1, e.im);
        unsafeAtomicAdd(rec + 2, e.w);
        if (FOM) {
            unsafeAtomicAdd(rec + 3, e.p);
            unsafeAtomicAdd(rec + 4, e.w2);
        }
        return;
    }
    stage_append(bc, out0, e.key, e.re, e.im, e.w, e.p, e.w2);   // lanes still here hold binned entries
}

template <bool FOM>
__device__ __forceinline__ Emit make_emit(unsigned key, int kk, bool incl, float fr, float fi,
                                          double w, int bin) {
    Emit e;
    e.key = (int)key;
    e.kk = kk;
    e.incl = incl ? 1 : 0;
    e.bin = bin;
    if (!incl) w = 0;
    e.re = (float)(fr * w);
    e.im = (float)(fi * w);
    e.w = (float)w;
    e.p = FOM ? (float)(w * ((double)fr * fr + (double)fi * fi)) : 0.f;
    e.w2 = FOM ? (float)(w * w) : 0.f;
    return e;
}

// sin and cos of a double-precision angle: exact reduction to [-pi, pi] in
// FP64, then FP32 evaluation (absolute error ~1e-7, below the FP32 rounding
// the reference applies when it stores the shifted / CTF-multiplied values).
__device__ __forceinline__ void sincos_red(double a, float* s, float* c) {
    const double r = a - 6.283185307179586 * rint(a * 0.15915494309189535);
    sincosf((float)r, s, c);
}
__device__ __forceinline__ float sin_red(double a) {
    const double r = a - 6.283185307179586 * rint(a * 0.15915494309189535);
    return sinf((float)r);
}

// Band, taper, phase shift and CTF of one sample (fspace_pack_2D :147-157,
// phase_shift_to_origin, img_ctf_calculate): returns whether the sample is in
// the resolution band, its weight and (unless counting) its value.
// ph: the phase factor exp(i (h phx + k phy)) when the caller tracks it
// (nullptr: evaluated here).
template <int MODE>
__device__ __forceinline__ bool sample_value(const ReconConst& K, const PartDev& P, bool active,
                                             long h, long k, float2 F, double* s0, double* s1,
                                             double* s2, double* w, float* fr, float* fi,
                                             const float2* ph = nullptr) {
    *s0 = (double)h * P.invscale;
    *s1 = (double)k * P.invscale;
    *s2 = *s0 * *s0 + *s1 * *s1;
    const bool inband = active && *s2 >= K.mins2 && *s2 <= K.maxs2;
    *w = 0;
    *fr = 0.f;
    *fi = 0.f;
    if (!inband) return false;
    double ww = P.wp;
    // taper of the outermost shell: most wavefronts hold no such sample and
    // skip it; FP32 square root (the weight is stored in FP32)
    const double d = (K.maxs2 - *s2) * K.mscz;
    if (__ballot(d < 1) != 0) {
        if (d < 1) ww *= (double)__builtin_amdgcn_sqrtf((float)d);
    }
    *w = ww;
    float sn, cs;
    if (ph) {
        cs = ph->x;
        sn = ph->y;
    } else {
        sincos_red((double)h * P.phx + (double)k * P.phy, &sn, &cs);
    }
    float vr = F.x * cs - F.y * sn, vi = F.x * sn + F.y * cs;
    if (K.ctf_mode) {
        const double fx = (double)h * P.fscale, fy = (double)k * P.fscale;
        const double cs2 = fx * fx + fy * fy;
        float c = 0.f;
        if (cs2 <= K.shi2) {
            // chi = c0 + c2m2 s^2 sin 2a + c20 s^2 + c22 s^2 cos 2a + c40 s^4 with
            // s^2 cos 2a = fx^2 - fy^2 and s^2 sin 2a = 2 fx fy (no division)
            double dphi = P.c0;
            dphi += P.c2m2 * (2 * fx * fy);
            dphi += P.c20 * cs2;
            dphi += P.c22 * (fx * fx - fy * fy);
            dphi += P.c40 * cs2 * cs2;
            if (K.ctf_mode == 1) {
                // phase flip needs the sign only: sin chi < 0 iff the reduced
                // angle lies in (-pi, 0)
                const double r = dphi - 6.283185307179586 * rint(dphi * 0.15915494309189535);
                c = (r < 0) ? -1.f : 1.f;
            } else {
                c = sin_red(dphi);
                if (K.ctf_mode == 3) c = (float)((K.wiener + 1) * c / ((double)c * c + K.wiener));
            }
        }
        vr *= c;
        vi *= c;
    }
    *fr = vr;
    *fi = vi;
    return true;
}

// Interpolation of one sample at voxel coordinates m (fspace_2D_interpolate,
// Bimage_reconstruct.cpp:25-88): nearest / weighted nearest / trilinear.
template <int MG, bool FOM, int MODE, int FAST = 0>
__device__ __forceinline__ void interp_emit(float* __restrict__ acc, const ReconConst& K,
                                            const double m[3], bool inband, double w, float fr,
                                            float fi, int kk, int merge, unsigned keybase,
                                            const BinCtx& bc, int bin = 1, bool flush = false) {
    if (FAST == 1 || FAST == 2 || (!FAST && K.interp < 2)) {
        const double fx = floor(m[0] + 0.5), fy = floor(m[1] + 0.5), fz = floor(m[2] + 0.5);
        double ww = w;
        if (FAST == 2 || (!FAST && K.interp == 1)) {   // weighted nearest neighbour
            const double dx = m[0] - fx, dy = m[1] - fy, dz = m[2] - fz;
            ww *= 1 - sqrt(dx * dx + dy * dy + dz * dz);
        }
        const int cx = wrap32((int)fx, K.N), cy = wrap32((int)fy, K.N), cz = wrap32((int)fz, K.nz);
        emit<MG, FOM, MODE, FAST>(acc, K.stride, merge,
                            make_emit<FOM>(keybase + rec_index32(cx, cy, cz, K.NT), kk,
                                           inband && ww > 0, fr, fi, ww, bin),
                            bc);
    } else {
        const double fx = floor(m[0]), fy = floor(m[1]), fz = floor(m[2]);
        const double dx = m[0] - fx, dy = m[1] - fy, dz = m[2] - fz;
        const int cx = (int)fx, cy = (int)fy, cz = (int)fz;
#pragma unroll
        for (int corner = 0; corner < 8; ++corner) {
            const int xx = corner & 1, yy = (corner >> 1) & 1, zz = corner >> 2;
            const int jx = wrap32(cx + xx, K.N), jy = wrap32(cy + yy, K.N), jz = wrap32(cz + zz, K.nz);
            const double ww = (xx ? dx : 1 - dx) * (yy ? dy : 1 - dy) * (zz ? dz : 1 - dz) * w;
            emit<MG, FOM, MODE, FAST>(acc, K.stride, merge,
                                make_emit<FOM>(keybase + rec_index32(jx, jy, jz, K.NT), kk,
                                               inband, fr, fi, ww, bin),
                                bc);
            // staged pair entries: at most one per thread and corner, so the list
            // is flushed once it could not take another corner's
            // (workgroup-uniform: only the sample's own emission, which every
            // thread makes, asks)
            if (MODE == MODE_FILL && flush) {
                __syncthreads();
                const bool full = *bc.st.nent > BSX_STAGE_CAP - (int)blockDim.x;
                __syncthreads();   // every wave has read the count
                if (full) stage_flush(bc);
            }
        }
    }
}

__device__ __forceinline__ void coords(const ReconConst& K, const PartDev& P, double s0, double s1,
                                       double sz, double m[3]) {
    m[0] = (s0 * P.R[0] + s1 * P.R[1] + sz * P.R[2]) * K.mscale;
    m[1] = (s0 * P.R[3] + s1 * P.R[4] + sz * P.R[5]) * K.mscale;
    m[2] = (s0 * P.R[6] + s1 * P.R[7] + sz * P.R[8]) * K.mscz;
}

// One sample (h, k) with raw value F and the Friedel mate of its array
// position, (-h, km) with value conj(F): fspace_pack_2D's loop body for both.
// Away from the Nyquist row and without the Ewald offset the mate's
// frequency is exactly -(h, k), so its coordinates are -m and its value the
// conjugate: computed once, emitted twice. Every lane of a wavefront runs the
// same emits (excluded samples carry incl = 0), so shuffles and ballots stay
// uniform.
//
// In the fill pass (the Ewald offsets have their own branch) a sample whose mate
// lands on exactly the opposite voxels (-v for v:
// nearest neighbour all but exact .5 ties, trilinear always) is emitted
// once, as pair entries at v that the fold later also adds, conjugated, at
// -v. Samples without such a mate (the x = 0 and x = FT/2
// columns, the Nyquist row, ties) add to the volume directly, and the mate
// of a tie is emitted on its own, as before.
template <int MG, bool FOM, int MODE, int FAST = 0>
__device__ __forceinline__ void insert_pair(float* __restrict__ acc, const ReconConst& K,
                                            const PartDev& P, bool active, bool mirror, long h,
                                            long k, long km, float2 F, int merge,
                                            unsigned keybase, const BinCtx& bc, float2 ph) {
    double s0, s1, s2, w;
    float fr, fi;
    const bool inband =
        sample_value<MODE>(K, P, active, h, k, F, &s0, &s1, &s2, &w, &fr, &fi, &ph);
    double m[3];
    const double mz0 = FAST ? 0.0 : P.ew * s2;
    if (FAST) {
        // no Ewald offset: the z term of coords is a signed zero, which
        // changes neither a non-zero sum nor the voxel that a zero rounds to
        m[0] = (s0 * P.R[0] + s1 * P.R[1]) * K.mscale;
        m[1] = (s0 * P.R[3] + s1 * P.R[4]) * K.mscale;
        m[2] = (s0 * P.R[6] + s1 * P.R[7]) * K.mscz;
    } else {
        coords(K, P, s0, s1, mz0, m);
    }
    if (!FAST && (MODE == MODE_FILL || K.ewald)) {   // the general fill serves Ewald insertion only
        // two emissions per frequency, at +mz0 (A) and -mz0 (B). Off the
        // Nyquist row the mate's emissions at +mz0 and -mz0 lie at exactly
        // -B and -A with the conjugate value, so with pair entries A stands
        // for the mate's -mz0 emission and B for its +mz0 one (where the
        // nearest voxels mirror too); the others are computed in full.
        constexpr bool pr = MODE == MODE_FILL;
        double mb[3];
        coords(K, P, s0, s1, -mz0, mb);
        bool sa = pr && km == -k, sb = sa;
        if (K.interp < 2) {
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                sa = sa && floor(-m[q] + 0.5) == -floor(m[q] + 0.5);
                sb = sb && floor(-mb[q] + 0.5) == -floor(mb[q] + 0.5);
            }
        }
        interp_emit<MG, FOM, MODE, FAST>(acc, K, m, inband, w, fr, fi, (int)k, merge, keybase, bc,
                                         mirror && sa ? 1 : 0, pr);
        interp_emit<MG, FOM, MODE, FAST>(acc, K, mb, inband, w, fr, fi, (int)k, merge, keybase, bc,
                                         mirror && sb ? 1 : 0, pr);
        // staged nearest-neighbour entries: at most two per thread here
        if (pr && K.interp < 2) stage_flush(bc);
        double t0, t1, t2, tw;
        float gr, gi;
        const bool ib = sample_value<MODE>(K, P, mirror, -h, km, make_float2(F.x, -F.y), &t0,
                                           &t1, &t2, &tw, &gr, &gi);
        const bool needc = ib && !sb, needd = ib && !sa;   // C = -B, D = -A when paired
        if (__ballot(needc || needd) == 0) return;   // wavefront-uniform
        const double mz = P.ew * t2;
        coords(K, P, t0, t1, mz, m);
        interp_emit<MG, FOM, MODE, FAST>(acc, K, m, needc, tw, gr, gi, (int)km, merge, keybase, bc,
                                         0);
        coords(K, P, t0, t1, -mz, m);
        interp_emit<MG, FOM, MODE, FAST>(acc, K, m, needd, tw, gr, gi, (int)km, merge, keybase, bc,
                                         0);
        return;
    }
    // the mate, per lane: -m and the conjugate away from the Nyquist row,
    // else computed in full; emitted below by all lanes together
    double mm[3];
    double tw = w;
    float gr = fr, gi = -fi;
    bool ib = inband && mirror;
    if (km == -k) {
        mm[0] = -m[0];
        mm[1] = -m[1];
        mm[2] = -m[2];
    } else if (FAST) {
        // the Nyquist row (k = km = -FT/2): the mate's phase angle is
        // -(h phx + k phy) - FT phy, so its factor follows from the sample's
        double t0, t1, t2;
        const float2 pm = make_float2(
            (float)((double)ph.x * P.nyq[0] + (double)ph.y * P.nyq[1]),
            (float)((double)ph.x * P.nyq[1] - (double)ph.y * P.nyq[0]));
        ib = sample_value<MODE>(K, P, mirror, -h, km, make_float2(F.x, -F.y), &t0, &t1, &t2,
                                &tw, &gr, &gi, &pm);
        mm[0] = (t0 * P.R[0] + t1 * P.R[1]) * K.mscale;
        mm[1] = (t0 * P.R[3] + t1 * P.R[4]) * K.mscale;
        mm[2] = (t0 * P.R[6] + t1 * P.R[7]) * K.mscz;
    } else {
        double t0, t1, t2;
        ib = sample_value<MODE>(K, P, mirror, -h, km, make_float2(F.x, -F.y), &t0, &t1, &t2,
                                &tw, &gr, &gi);
        coords(K, P, t0, t1, 0.0, mm);
    }
    if (FAST) {
        // trilinear: the mate's corners are the sample's negated, with the
        // same weights (floor(-m) = -floor(m) - 1 and 1 - dx; a coordinate
        // that is an integer only swaps a zero-weight corner)
        bool sym = km == -k;
        if (FAST < 3) {
#pragma unroll
            for (int q = 0; q < 3; ++q) sym = sym && floor(-m[q] + 0.5) == -floor(m[q] + 0.5);
        }
        const bool pair = mirror && sym;
        interp_emit<MG, FOM, MODE, FAST>(acc, K, m, inband, w, fr, fi, (int)k, merge, keybase, bc,
                                   pair ? 1 : 0, true);
        const bool mate = ib && !sym;
        if (__ballot(mate) == 0) return;   // wavefront-uniform
        interp_emit<MG, FOM, MODE, FAST>(acc, K, mm, mate, tw, gr, gi, (int)km, merge, keybase, bc, 0);
        return;
    }
    interp_emit<MG, FOM, MODE, FAST>(acc, K, m, inband, w, fr, fi, (int)k, merge, keybase, bc);
    interp_emit<MG, FOM, MODE, FAST>(acc, K, mm, ib, tw, gr, gi, (int)km, merge, keybase, bc);
}

// Column tasks: task = (particle, x) with x in [0, FT/2]; G tasks per WG.
// The specialisations (FAST 1: nearest, 2: weighted nearest, 3: trilinear, with
// pair entries and staging, no Ewald) are held to 5 waves per SIMD (at most 96
// VGPRs): their 31.7 KB of LDS allows 5 workgroups per CU, and one register
// more would round the allocation up to 104 and allow only 4 (the weighted one
// spills 12 B for it); with the FOM sums (35.8 KB) and for trilinear insertion to
// 4. Generic kernel (167 VGPRs) against the specialised ones, per batch: FOM sums
// of 128^2 particles 1,151 -> 889 us, trilinear insertion of 90^2 ones 836 -> 734.
template <int FT, bool FOM, int MODE, int FAST = 0>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(FAST ? (FOM || FAST == 3 ? 4 : 5) : 1)))
void k_cols(const float2* __restrict__ inter,
                                              const float* __restrict__ bkg,
                                              const PartDev* __restrict__ recs, int nb, int box,
                                              ReconConst K, float* __restrict__ acc,
                                              const float2* __restrict__ twg, BinCtx bc) {
    constexpr int T = FftThreads<FT>::value;
    constexpr int G = 256 / T;
    constexpr int NT = G * T;
    constexpr int HX = FT / 2 + 1;
    constexpr int MG = T < 16 ? T : 16;   // run-merge group: lanes of one column
    constexpr int LDSN = G * FT + FT;
    constexpr int SCAP = MODE == MODE_FILL ? BSX_STAGE_CAP : 1;
    constexpr int SHASH = MODE == MODE_FILL ? BSX_STAGE_HASH : 1;
    __shared__ float2 lds[LDSN];
    __shared__ float4 st_ent[SCAP];
    __shared__ float2 st_ent2[FOM ? SCAP : 1];
    __shared__ int4 st_hinfo[SHASH];
    __shared__ int st_hkey[SHASH], st_hcnt[SHASH], st_nent;
    const int tid = threadIdx.x;
    const int g = tid / T, t = tid - g * T;
    const long task = (long)blockIdx.x * G + g;
    const int p = (int)(task / HX);
    const int x = (int)(task - (long)p * HX);
    const bool valid = p < nb;
    float2* line = lds + g * FT;
    {
        float2* tw = lds + G * FT;
        for (int i = tid; i < FT; i += NT) tw[i] = twg[i];
        const float2* col = inter + ((size_t)p * HX + x) * box;
        for (int i = t; i < FT; i += T) line[i] = (valid && i < box) ? col[i] : make_float2(0.f, 0.f);
        __syncthreads();
        FftLine<FT, -1, T>::run(line, tw, t);
    }
    // staging (pair entries: at most one binned emission per thread and
    // round, so 2 rounds fit the list; the 512-entry list keeps the LDS of a
    // workgroup under 32 KB, 5 workgroups per CU)
    static_assert(NT == 256 && 2 * NT <= BSX_STAGE_CAP, "two rounds fit the list");
    bc.st = Stage{st_ent, &st_nent, st_hkey, st_hcnt, st_hinfo, FOM ? st_ent2 : nullptr};
    if (MODE == MODE_FILL) {
        if (tid < BSX_STAGE_HASH) {
            st_hkey[tid] = -1;
            st_hcnt[tid] = 0;
        }
        if (tid == 0) st_nent = 0;
        __syncthreads();
    }
    // At FT 512 a wavefront is one column (T == 64), so its particle is
    // uniform: the record is then read with scalar loads, kept in SGPRs.
    const int prec = valid ? p : 0;
    const PartDev& P = recs[T == 64 ? __builtin_amdgcn_readfirstlane(prec) : prec];
    const unsigned keybase = (unsigned)P.half * (unsigned)(K.NT * K.NT * K.NT) * 4096u;
    const float inv = 1.0f / FT;
    const float b = valid ? bkg[p] : 0.f;
    const long h = (x <= (FT - 1) / 2) ? x : x - FT;
    const bool mirror = valid && x >= 1 && x <= FT / 2 - 1;
    const int merge = K.merge;
    // phase factor of this thread's sample, advanced by exact FP64 rotations
    // (k grows by T per round and wraps by -FT after round 3, as y passes FT/2)
    double er, ei;
    {
        float sn, cs;
        sincos_red((double)h * P.phx + (double)t * P.phy, &sn, &cs);
        er = cs;
        ei = sn;
    }
#pragma unroll 1
    for (int r = 0; r < 8; ++r) {
        const int y = t + r * T;
        float2 F = line[y];
        F.x *= inv;
        F.y *= inv;
        if (x == 0 && y == 0) F.x += b * FT;
        const long k = (y <= (FT - 1) / 2) ? y : y - FT;
        // Friedel mate of the column: array position (FT-x, FT-y), value conj
        const int ym = (FT - y) & (FT - 1);
        const long km = (ym <= (FT - 1) / 2) ? ym : ym - FT;
        insert_pair<MG, FOM, MODE, FAST>(acc, K, P, valid, mirror, h, k, km, F, merge, keybase, bc,
                                   make_float2((float)er, (float)ei));
        {
            const double c = r == 3 ? P.rot[2] : P.rot[0], sd = r == 3 ? P.rot[3] : P.rot[1];
            const double nr = er * c - ei * sd;
            ei = er * sd + ei * c;
            er = nr;
        }
        if (MODE == MODE_FILL && (FAST == 3 ? r == 7 : (r & 1) == 1)) stage_flush(bc);
    }
}

template <int FT>
int insert_batch(bsx_recon* h, const float* imgs, int64_t p0, int nb, hipStream_t s,
                 int (*mark)(bsx_recon*, hipStream_t, int)) {
    constexpr int T = FftThreads<FT>::value;
    constexpr int G = 256 / T;
    // one line per column group: 8 rows per workgroup at FT = 512 (20 KB of
    // LDS, 8 workgroups per CU; 16 rows measured 12 % slower)
    constexpr int LINES = G;
    constexpr int NT = G * T;
    const int box = h->p.box;
    const float2* tw = twiddles(FT, s);
    BSX_REQUIRE(tw, BSX_ERR_DEVICE, "twiddles(%d) failed", FT);
    const int tiles = (box + 2 * LINES - 1) / (2 * LINES);
    hipLaunchKernelGGL((k_rows<FT, LINES>), dim3(nb * tiles), dim3(NT), 0, s, imgs,
                       h->recs + p0, h->bkg + p0, box, tiles, h->inter, tw,
                       h->resc ? h->resc + p0 : nullptr);
    BSX_HIP(hipGetLastError());
    int r = mark(h, s, KT_ROWS);
    if (r) return r;
    const long ntask = (long)nb * (FT / 2 + 1);
    const dim3 grid((unsigned)((ntask + G - 1) / G));
    const PartDev* rec = h->recs + p0;
    const float* bk = h->bkg + p0;
    const BinCtx bc{h->fill,  h->chunks, h->pool, h->bins,  h->xacc,
                    h->npool, h->maxc,   Stage{}, h->bins2, h->K.stride};
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(NT), 0, s, h->inter, bk, rec, nb, box, h->K, h->acc, tw, bc);
    };
    if (!h->binned) {
        h->K.fom ? go(k_cols<FT, true, MODE_DIRECT>) : go(k_cols<FT, false, MODE_DIRECT>);
    } else if (h->K.ewald) {
        h->K.fom ? go(k_cols<FT, true, MODE_FILL>) : go(k_cols<FT, false, MODE_FILL>);
    } else {
        // specialised on the interpolation
        switch (h->K.interp) {
            case 0: h->K.fom ? go(k_cols<FT, true, MODE_FILL, 1>) : go(k_cols<FT, false, MODE_FILL, 1>); break;
            case 1: h->K.fom ? go(k_cols<FT, true, MODE_FILL, 2>) : go(k_cols<FT, false, MODE_FILL, 2>); break;
            default: h->K.fom ? go(k_cols<FT, true, MODE_FILL, 3>) : go(k_cols<FT, false, MODE_FILL, 3>);
        }
    }
    BSX_HIP(hipGetLastError());
    return mark(h, s, h->binned ? KT_FILL : KT_DIRECT);
}

template int insert_batch<BSX_INSERT_FT>(bsx_recon*, const float*, int64_t, int, hipStream_t,
                                         int (*)(bsx_recon*, hipStream_t, int));
