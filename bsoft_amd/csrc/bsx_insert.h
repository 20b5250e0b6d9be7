// bsx_insert.h — particle records, the accumulator layout, the binned insertion's
// data structures and the reconstruction handle, shared by bsx_recon.hip (host
// side, tile pass, finish) and bsx_insert.hip (row transforms and the fill, one
// translation unit per transform size, since their instances take minutes to
// compile).
#pragma once

#include <vector>

#include "bsx_fft_dev.h"
#include "bsx_common.h"

using namespace bsx;

// Device record of one particle, all derived quantities computed on the host
// in double precision.
struct alignas(16) PartDev {
    double R[9];        // View::matrix (row-major d[i][j])
    double invscale;    // (1/mag) / (ft * pixel_size)      fspace_pack_2D invscale
    double phx, phy;    // 2 pi ori / ft                      phase_shift_to_origin
    double rot[4];      // cos, sin of T phy and (T - ft) phy, T = ft / 8: the phase
                        // steps between the rounds of a column thread
    double c0, c20, c22, c2m2, c40;   // aberration weights   ctf.h:321-335
    double fscale;      // 1 / (ft * pixel_size)              img_ctf_calculate freq_scale
    double ew;          // Ewald offset lambda/2, 0 if off
    double nyq[2];      // cos, sin of -ft phy: the phase factor of a Nyquist-row
                        // mate is conj(sample's) times this
    double hox, hoy;    // background-ellipse origin (image header)
    long long src;      // index of the image in the caller's stack
    float wp;           // particle weight incl. pad ratio
    int half;           // accumulator set
};

struct ReconConst {
    int N, ft, box, stride, interp, ctf_mode, fom, nhalves;   // ctf_mode 0 none 1 flip 2 apply 3 wiener
    int merge, ewald, NT;                                     // NT: 16^3 tiles per edge
    double mins2, maxs2, mscale, shi2, wiener;
    // z extent: a 2D map (breconstruct -TwoD) has one plane (nz = 1) and z
    // real size 1 (particle_reconstruct sets the z sampling to 1,
    // mg_reconstruct.cpp:117), which scales m_z and the resolution taper
    double mscz;
    int nz;
};

// Rescaled pixel value: the FP64 product and sum of Bimage::rescale
// (Bimage_rescale.cpp:27-45) stored back as FP32.
__device__ __forceinline__ float rescaled(float v, double2 r) {
    return (float)((double)v * r.x + r.y);
}

// ------------------------------------------------------------------- K3
// Accumulator layout: records of `stride` floats (sum w re, sum w im, sum w
// [, sum w|F|^2, sum w^2]) in 16^3-voxel tiles; a tile is 4096 contiguous
// records (48 KB lean). Key = half * NREC + record index, NREC = NT^3 * 4096,
// so key >> 12 is the (half, tile) bin and key & 4095 the record in the tile.
__host__ __device__ __forceinline__ long rec_index(long x, long y, long z, long NT) {
    return ((((z >> 4) * NT + (y >> 4)) * NT + (x >> 4)) << 12) | ((z & 15) << 8) |
           ((y & 15) << 4) | (x & 15);
}

// Bins live in chunks of BSX_CHUNK entries taken from a pool while the fill
// pass reserves them: a bin's reservation counter gives each entry a position,
// position / BSX_CHUNK indexes the bin's chunk table, and the reservation that
// holds a chunk's first position allocates it (one pool atomic, then a
// compare-and-swap into the table) while the other writers of that chunk wait
// for the table entry. No counting pass is needed: after the fill the counters are the bin
// sizes, k_piece_scan turns them into work pieces, and k_bin_reset clears the
// counters and the used table entries for the next batch. An entry whose
// chunk cannot be had (table or pool exhausted) is added to the volume with
// float atomics instead, so capacity only costs speed.
#define BSX_CHUNK 4096
#define BSX_SPIN_LIMIT 4096    // polls of a chunk-table entry before the atomic fallback

// Bins are processed in pieces of at most `piece` entries (a whole number of
// chunks, 8192 to 32768; 16384 by default, chosen by bsx_recon_autotune) so
// that the few hot bins around the origin (every plane passes through the
// low-frequency core) are spread over many workgroups.
#define BSX_PIECE_DEFAULT 16384
#define BSX_PIECE_MIN 8192
#define BSX_PIECE_MAX 32768

// ================================================================== host side
struct bsx_recon {
    bsx_recon_params p;
    ReconConst K;
    double hi_res;
    int dev;
    bool binned = true;            // tile-binned insertion (else direct atomics)
    float* acc = nullptr;
    float* xacc = nullptr;         // binned accumulator, folded into acc
    bool xdirty = false;           // xacc may hold entries that have not been folded
    bool bins_dirty = false;       // an insert stopped between its fill and its bin reset
    size_t acc_elems = 0;
    float2* inter = nullptr;
    float* bkg = nullptr;
    double2* resc = nullptr;       // per record (scale, shift) of -rescale (flags bit 1)
    PartDev* recs = nullptr;
    int* nonfinite = nullptr;
    int64_t recs_cap = 0;
    int* fill = nullptr;           // per (half, tile) bin: entries reserved
    int* chunks = nullptr;         // per bin: pool chunk of each bin chunk
    int* pool = nullptr;           // next free chunk, fallback flags
    int npool = 0;
    int maxc = 0;
    int* poff = nullptr;           // piece offsets per bin
    int* pbin = nullptr;           // bin of each piece
    unsigned long long* entries = nullptr;   // bin entries of the current insert
    float4* bins = nullptr;
    float2* bins2 = nullptr;       // FOM sums of the pool entries (FOM only)
    size_t bins_cap = 0;
    int nbins = 0;
    int batch = 0;
    int batch_cap = 0;               // batch the buffers were sized for
    int piece = BSX_PIECE_DEFAULT;   // tile-pass piece length (entries)
    int64_t inserted[2] = {0, 0};
    int fallback_flags = 0;        // atomic-fallback flags seen (1 table, 2 pool, 4 wait bound)
    double ktime[7] = {0, 0, 0, 0, 0, 0, 0};   // background rows fallback scan fill tile direct
    double last_entries = 0;
    int64_t last_launches = 0;
    std::vector<hipEvent_t> evs;
    std::vector<int> evlab;
    size_t nev = 0;
    size_t bytes = 0;
    PartDev* hrecs = nullptr;      // pinned staging of the records
    int64_t hrecs_cap = 0;
    hipEvent_t copied = nullptr;   // staging buffer reusable once this completes
    bool timing = false;
    // BSX_FLAG_GRAPH: the batch loop of an insert, captured on the second
    // call with the same (images, record count, batch, run merge, piece) and
    // replayed while that set is inserted again; up to 8 such sets (e.g. the
    // chunks of a pipelined insert) are kept, the least recently used evicted
    struct GraphEntry {
        const float* imgs;
        int64_t n;
        int batch, merge, piece;   // kernel constants baked into the graph
        int seen;                  // calls seen (capture on the second)
        hipGraphExec_t exec;
        uint64_t used;
    };
    std::vector<GraphEntry> graphs;
    uint64_t graph_clock = 0;
    int64_t graph_launches = 0;
    hipStream_t cap_stream = nullptr;   // capture happens here (the caller's stream may be
                                        // the legacy default stream, which cannot capture)
    std::vector<int> sym_order;         // point-group operator orders (empty: C1)
    std::vector<double> sym_axis;       // their unit axes, 3 per operator
    // group runs (bsx_recon_group_run): weighed transform and the finish
    // sums (5 doubles), kept so that the finish needs no allocation inside a
    // captured graph
    float2* gvol = nullptr;
    double* gfin = nullptr;
};

// KT_FALLBACK holds the atomic-fallback flags of the insert, not a time
enum { KT_BG = 0, KT_ROWS, KT_FALLBACK, KT_SCAN, KT_FILL, KT_TILE, KT_DIRECT, KT_END };

// Row transforms and insertion (binned fill or direct atomics) of the nb
// particles from record p0 on, for transform size FT; `mark` records the timing
// marks.
template <int FT>
int insert_batch(bsx_recon* h, const float* imgs, int64_t p0, int nb, hipStream_t s,
                 int (*mark)(bsx_recon*, hipStream_t, int));
