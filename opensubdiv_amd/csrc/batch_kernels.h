// Batched evaluation: many meshes, each with many frames of control points,
// in one graph launch of two kernels.
//
//   phase A  k_batch_stencils  every stencil segment (one table in compact
//                              slices applied to F frames): refinement
//                              tables and the patch-point tables that fill
//                              each mesh's vertex buffer [control | points];
//   phase B  k_batch_patches   every patch segment (one mesh's PatchCoords
//                              evaluated on its F frames), reading the
//                              vertex buffers phase A completed.
//
// Frames are extra right-hand-side columns: a wave loads a table slice's
// entries once for all frames (once per chunk of frames where the slice is
// wider than 16 entries or lists no control vertices), and a PatchCoord's basis
// is evaluated once for all frames.  Element (v, f, k) of a multi-frame buffer
// lives at base + v * vStride + f * fStride + k, so both frame-major and
// vertex-major (frames interleaved) layouts work.
//
// Work is cut into items of up to `itemSlices` 64-row slices (phase A) or
// kBlock coords (phase B).  Static scheduling maps one item to one block;
// persistent scheduling launches a fixed grid whose blocks claim items from
// a device counter (one vector atomic per item, by lane 0 of wave 0) until
// the list is exhausted -- every block exits when the counter passes the
// item count.
//
// Every sum accumulates w * x in the same order as the single-mesh kernels
// (k_stencils_compact / k_patches), so batched results equal one-mesh-per-launch
// results bit for bit.
#pragma once
#include <type_traits>

#include "../../include/osdhip.h"
#include "common.h"
#include "patch_basis_device.h"
#include "stencil_compact.h"

namespace osdhip {

struct BatchStencilSeg {
    const unsigned *rec;          // compact slices (stencil_compact.h), one weight array
    const SliceDesc *slices;
    const int *perm;              // slice row -> table row; NULL: the same
    const int *ctrl;
    const float *src;
    long long srcV, srcF;
    float *dst;
    long long dstV, dstF;
    int nrows, nslices, frames, pad;
};

struct BatchPatchSeg {
    const osdhip_patch_coord *coords;
    const osdhip_patch_array *arrays;
    const int *indices;
    const osdhip_patch_param *params;
    const float *src;
    long long srcV, srcF;
    float *out[3];                // P, dPdu, dPdv (NULL = skip)
    long long outV, outF;
    int ncoords, frames;
    // point staging of regular-interior coords, per wave of 64 coords
    // (NULL: gathers only): nuniq[w] distinct points listed at
    // pts[ptsOff[w] ...] (nuniq < 0: more than kPatchSlots), and per coord
    // the list positions of its 16 points, one byte each
    const int *nuniq;
    const long long *ptsOff;
    const int *pts;
    const unsigned *slots;        // 4 words per coord
    const int *ngen;              // per wave: coords that are not regular-interior
};

// Device views of the segments with global-qualified pointers (the
// descriptors are read from memory, so the compiler would otherwise treat
// their pointers as generic and emit flat accesses).
#define G_ OSDHIP_GLOBAL
#define C_ OSDHIP_CONST
struct GStencilSeg {
    const G_ unsigned *rec;
    const C_ SliceDesc *slices;
    const G_ int *perm;
    const G_ int *ctrl;
    const G_ float *src;
    long long srcV, srcF;
    G_ float *dst;
    long long dstV, dstF;
    int nrows, nslices, frames;
};

struct GPatchSeg {
    const G_ osdhip_patch_coord *coords;
    const G_ osdhip_patch_array *arrays;
    const G_ int *indices;
    const G_ osdhip_patch_param *params;
    const G_ float *src;
    long long srcV, srcF;
    G_ float *out[3];
    long long outV, outF;
    int ncoords, frames;
    const G_ int *nuniq;
    const G_ long long *ptsOff;
    const G_ int *pts;
    const G_ unsigned *slots;
    const G_ int *ngen;
};

__device__ __forceinline__ GStencilSeg gseg(const C_ BatchStencilSeg &s)
{
    GStencilSeg g;
    g.rec = gptr(s.rec);
    g.slices = cptr(s.slices);
    g.perm = gptr(s.perm);
    g.ctrl = gptr(s.ctrl);
    g.src = gptr(s.src);
    g.srcV = s.srcV;
    g.srcF = s.srcF;
    g.dst = gptr_w(s.dst);
    g.dstV = s.dstV;
    g.dstF = s.dstF;
    g.nrows = s.nrows;
    g.nslices = s.nslices;
    g.frames = s.frames;
    return g;
}

__device__ __forceinline__ GPatchSeg gseg(const C_ BatchPatchSeg &s)
{
    GPatchSeg g;
    g.coords = gptr(s.coords);
    g.arrays = gptr(s.arrays);
    g.indices = gptr(s.indices);
    g.params = gptr(s.params);
    g.src = gptr(s.src);
    g.srcV = s.srcV;
    g.srcF = s.srcF;
    for (int k = 0; k < 3; ++k) g.out[k] = s.out[k] ? gptr_w(s.out[k]) : nullptr;
    g.outV = s.outV;
    g.outF = s.outF;
    g.ncoords = s.ncoords;
    g.frames = s.frames;
    g.nuniq = gptr(s.nuniq);
    g.ptsOff = gptr(s.ptsOff);
    g.pts = gptr(s.pts);
    g.slots = gptr(s.slots);
    g.ngen = gptr(s.ngen);
    return g;
}

// Field-wise loads of the Osd structs through global pointers.
__device__ __forceinline__ osdhip_patch_coord ld(const G_ osdhip_patch_coord *p)
{
    osdhip_patch_coord c;
    c.arrayIndex = p->arrayIndex;
    c.patchIndex = p->patchIndex;
    c.vertIndex = p->vertIndex;
    c.s = p->s;
    c.t = p->t;
    return c;
}
__device__ __forceinline__ osdhip_patch_array ld(const G_ osdhip_patch_array *p)
{
    osdhip_patch_array a;
    a.regDesc = p->regDesc;
    a.desc = p->desc;
    a.numPatches = p->numPatches;
    a.indexBase = p->indexBase;
    a.stride = p->stride;
    a.primitiveIdBase = p->primitiveIdBase;
    return a;
}
__device__ __forceinline__ osdhip_patch_param ld(const G_ osdhip_patch_param *p)
{
    osdhip_patch_param q;
    q.field0 = p->field0;
    q.field1 = p->field1;
    q.sharpness = p->sharpness;
    return q;
}

struct BatchItem {
    int seg, first, count;        // phase A: slices [first, first+count); B: coords
    int f0;                       // phase B: first frame
};

__device__ __forceinline__ BatchItem ld(const C_ BatchItem *p)
{
    BatchItem it;
    it.seg = p->seg;
    it.first = p->first;
    it.count = p->count;
    it.f0 = p->f0;
    return it;
}

struct BatchArgs {
    const BatchStencilSeg *sseg;
    const BatchPatchSeg *pseg;
    const BatchItem *items;
    int nitems;
    int persistent;
    int itemFrames;               // phase B: an item's frames are [f0, f0 + itemFrames)
    unsigned *counter;            // persistent: one claim counter per XCD queue
};

__global__ void k_batch_reset(unsigned *counters, int n)
{
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i < n) counters[i] = 0u;
}

// Next item of this block; neighbouring slices, which share control points, go
// to one XCD (the hardware places block b on XCD b % 8) and share its L2.
// Static: block b takes item xcd_logical_block() once, runs of eight items per
// XCD in turn.  Persistent: the items are split into kNumXcd contiguous ranges,
// one per XCD; block b claims items from its XCD's range through that range's
// counter and, when the range is exhausted, from the other ranges in turn; it
// returns -1 once every range is exhausted.  Must be reached by every thread of
// the block (it contains __syncthreads).  The result is wave-uniform.  claim:
// two ints of LDS that nothing else uses while the kernel runs.
__device__ __forceinline__ int batch_next_item(const BatchArgs &a, int iter, int *claim)
{
    if (!a.persistent) {
        if (iter) return -1;
        const int lb = xcd_logical_block();
        return lb < a.nitems ? lb : -1;
    }
    int &slot = claim[0], &queue = claim[1];
    __syncthreads();                          // previous item's readers are done
    if (threadIdx.x == 0) {
        if (iter == 0) queue = (int)(blockIdx.x % kNumXcd);
        const int per = (a.nitems + kNumXcd - 1) / kNumXcd;
        int it = -1;
        for (int k = 0; k < kNumXcd && it < 0; ++k) {
            const int q = (queue + k) % kNumXcd;
            const int lo = q * per, n = min(a.nitems, lo + per) - lo;
            if (n <= 0) continue;
            const int c = (int)atomicAdd(a.counter + q, 1u);
            if (c < n) {
                it = lo + c;
                queue = q;
            }
        }
        slot = it;
    }
    __syncthreads();
    // block-uniform: the item's descriptors are then read with scalar loads
    return __builtin_amdgcn_readfirstlane(slot);
}

// Phase A: one wave per compact slice, all frames of its segment.
//
// A listed slice's control vertices are staged in LDS for FC frames at a
// time.  Each lane copies one 16-byte quad of one (vertex, frame): the lanes
// of a load instruction cover whole vertices side by side (with the frames
// of a vertex adjacent, 8 lines of 128 B per instruction where one vertex
// per lane touched 64), which is what the vector cache is paid by.  The
// quads of the next chunk are in flight, in registers, while the current
// one is summed.
//
// In LDS a slot's FC * LC values lie side by side, padded (for FC > 1) to an
// odd number of quads, so a lane reads an entry's values with 16-byte reads and slots
// spread over all banks (109 of 128 B per clock and CU for 45 random slots
// at FC * LC = 28, 228 B when four lanes share a slot, as neighbouring rows
// in Far's order do; value-major 4-byte reads gave 57).
constexpr int kBatchWidth = 16;                       // widest slice held in registers

template <int LC, int FC>
struct BatchChunk {
    static constexpr int Q = FC * LC;
    static constexpr int NQ = (Q + 3) / 4;            // quads per slot
    // floats per slot; one frame packs its quads, so that the longest list
    // fits; one and two floats take no more (221 K rows, 12 frames of 2 floats:
    // 33.8 -> 32.9 us)
    static constexpr int STR = Q <= 2 ? Q : FC == 1 ? 4 * NQ : 4 * (NQ | 1);
};

// Quads a lane copies per chunk (list length x quads per vertex / 64, at
// most): lists of up to 64 vertices at FC = 4 and 5 to 8 floats, longer ones
// at fewer frames.
constexpr int kStageQuads = 8;

// Longest list staged at FC frames: the quads a lane copies, and the LDS of
// a wave (BatchArea).
template <int LC, int FC, int FLOATS>
constexpr int batch_list()
{
    const int byQuads = kStageQuads * kWave / (FC * ((LC + 3) / 4));
    const int byLds = FLOATS / BatchChunk<LC, FC>::STR - 1;
    const int n = byQuads < byLds ? byQuads : byLds;
    return n < kSliceList ? n : kSliceList;
}

// LDS floats per wave: the longest list at one frame, 63 vertices and the
// zero slot at FC, or the store transpose (64 rows of an odd number of
// floats).
template <int LC, int FC>
struct BatchArea {
    static constexpr int LIST = (kSliceList + 1) * BatchChunk<LC, 1>::STR;
    static constexpr int CHUNK = kWave * BatchChunk<LC, FC>::STR;
    static constexpr int RUNS = kWave * ((FC * LC) | 1);
    static constexpr int MOST = LIST > CHUNK ? (LIST > RUNS ? LIST : RUNS)
                                             : (CHUNK > RUNS ? CHUNK : RUNS);
    static constexpr int FLOATS = (MOST + 3) / 4 * 4;
};

// The lane index through an empty asm: what a path forms from it is formed
// there, instead of being held in registers across the whole kernel.
__device__ __forceinline__ int lane_here()
{
    int lane = (int)threadIdx.x & (kWave - 1);
    asm volatile("" : "+v"(lane));
    return lane;
}

// Stores a chunk's results for vertex-major outputs (dstF == LC): each lane
// parks its row's FC * LC values in LDS, then every store instruction
// writes RPI rows, SEG consecutive lanes per row covering the row's
// contiguous run of FC * LC floats.
template <int LC, int FC>
__device__ __forceinline__ void store_runs(const GStencilSeg &sg, float *area, const int *rowsL,
                                           const float (&acc)[FC][LC], int f0)
{
    constexpr int Q = FC * LC, TP = Q | 1;            // odd row stride: no bank conflicts
    constexpr int SEG = Q <= 8 ? 8 : Q <= 16 ? 16 : Q <= 32 ? 32 : 64;   // lanes per row
    constexpr int RPI = kWave / SEG;                  // rows per store instruction
    const int lane = lane_here();
    wave_lds_sync();                                   // compute reads of the area are done
#pragma unroll
    for (int c = 0; c < FC; ++c)
#pragma unroll
        for (int k = 0; k < LC; ++k) area[lane * TP + c * LC + k] = acc[c][k];
    wave_lds_sync();
    const int q = lane % SEG, hi = lane / SEG;
    const int nq = min(FC, sg.frames - f0) * LC;       // valid values per row
    G_ float *base = sg.dst + (size_t)f0 * LC + q;
#pragma unroll 4
    for (int it = 0; it < kWave / RPI; ++it) {
        const int r = it * RPI + hi;
        const int rr = rowsL[r];
        if (q < nq && rr >= 0) base[(size_t)rr * sg.dstV] = area[r * TP + q];
    }
}

// Reads a slot's first Q values, 16 bytes at a time where there are more than two
// (x: whole quads).
template <int Q, int N>
__device__ __forceinline__ void read_values(const float *p, float (&x)[N])
{
    if constexpr (Q <= 2) {
#pragma unroll
        for (int k = 0; k < Q; ++k) x[k] = p[k];
    } else {
#pragma unroll
        for (int q = 0; q < (Q + 3) / 4; ++q) {
            const v4f v = *(const v4f *)(p + 4 * q);
#pragma unroll
            for (int k = 0; k < 4; ++k) x[4 * q + k] = v[k];
        }
    }
}

// acc[c][k] += the first NF * LC values at p times w.
template <int LC, int FC, int NF>
__device__ __forceinline__ void add_entry(const float *p, float w, float (&acc)[FC][LC])
{
    float x[(NF * LC + 3) / 4 * 4];
    read_values<NF * LC>(p, x);
#pragma unroll
    for (int c = 0; c < NF; ++c)
#pragma unroll
        for (int k = 0; k < LC; ++k) acc[c][k] = acc[c][k] + x[c * LC + k] * w;
}

// One listed slice for every frame, FC per chunk (U <= batch_list at FC).
// RES: the slice's entries (W <= kBatchWidth) stay in registers.  A wider
// slice reads them from the caches for every chunk, four at a time, and
// stages a chunk when it gets to it: this keeps its registers below the RES
// path's, whose waves per SIMD it shares (eight or sixteen entries read ahead:
// 14 to 25 VGPRs more).  1.3 M rows of 14 entries on average, slices up to 18
// wide (valence-6 vertices), 16 frames of 7 floats: 606 us at FC = 4, 940 one
// frame at a time.
template <int LC, int FC, bool RES>
__device__ __forceinline__ void batch_listed_slice(const GStencilSeg &sg, float *area, int *rowsL,
                                                   const G_ unsigned *rp, const G_ float *wp, int W,
                                                   int U, const G_ int *list, int row, bool active)
{
    using A = BatchChunk<LC, FC>;
    constexpr int GR = RES ? kBatchWidth / 4 : 1;      // entry groups held
    constexpr int H = (LC + 3) / 4;                    // quads per (vertex, frame)
    constexpr int N = LC < 4 ? LC : 4;                 // floats per copied quad
    constexpr int QV = FC * H;                         // quads per vertex: 1, 2, 4 or 8
    constexpr int VI = kWave / QV;                     // vertices per copy instruction
    constexpr int LISTS = (kStageQuads + QV - 1) / QV; // list registers (64 vertices each)
    const int lane = lane_here();
    const int G = (W + 3) / 4;
    EntryGroup<1> e[GR];
    auto load = [&](int g0) {
#pragma unroll
        for (int c = 0; c < GR; ++c)
            if (g0 + c < G) {                          // wave-uniform
                e[c].slots = load_entry<RES>(rp + (size_t)(g0 + c) * kWave + lane);
                load_weights<1, RES>(wp, W, g0 + c, lane, e[c].w);
            }
    };
    int vtx[LISTS];
#pragma unroll
    for (int h = 0; h < LISTS; ++h) {
        vtx[h] = 0;
        if (h * kWave < U) vtx[h] = list[min(h * kWave + lane, U - 1)];
    }
    if (RES) load(0);
    // this lane's quad of its vertices: frame c of the chunk, floats
    // [k0, k0 + N) (the last quad of 5 to 7 floats overlaps the one before)
    const int q = lane % QV, c = q / H, k0 = min(4 * (q % H), LC - N);
    float x[kStageQuads][N];
    auto stage = [&](int f0) {
        // frames past the end repeat the last one (never stored)
        const G_ float *p = sg.src + (size_t)min(f0 + c, sg.frames - 1) * sg.srcF + k0;
#pragma unroll
        for (int r = 0; r < kStageQuads; ++r)
            if (r * VI < U) {                          // wave-uniform
                int v = vtx[r / QV];                   // one quad per vertex: the lane's own
                if (QV > 1) v = __shfl(v, (r * VI + lane / QV) % kWave, kWave);
                const G_ float *pv = p + (size_t)(unsigned)v * sg.srcV;
#pragma unroll
                for (int k = 0; k < N; ++k) x[r][k] = pv[k];
            }
    };
    // vertex-major outputs with a row's frames adjacent: results leave
    // through LDS so that consecutive lanes store one row's run
    const bool runs = sg.dstF == LC && sg.frames > 1;
    if (runs) rowsL[lane] = active ? row : -1;
    if (RES) stage(0);
    for (int f0 = 0; f0 < sg.frames; f0 += FC) {
        if (!RES) stage(f0);
        wave_lds_sync();                               // previous chunk's reads are done
#pragma unroll
        for (int r = 0; r < kStageQuads; ++r) {
            const int u = r * VI + lane / QV;
            if (r * VI < U && u < U) {
                float *d = area + u * A::STR + c * LC + k0;
#pragma unroll
                for (int k = 0; k < N; ++k) d[k] = x[r][k];
            }
        }
        if (lane < A::STR) area[U * A::STR + lane] = 0.0f;   // the zero slot
        wave_lds_sync();
        // the next chunk's loads are in flight while this one is summed
        if (RES && f0 + FC < sg.frames) stage(f0 + FC);
        float acc[FC][LC];
#pragma unroll
        for (int f = 0; f < FC; ++f)
#pragma unroll
            for (int k = 0; k < LC; ++k) acc[f][k] = 0.0f;
        auto entries = [&](auto frames) {
            constexpr int NF = decltype(frames)::value, NQ = (NF * LC + 3) / 4;
            // entries whose LDS reads are in flight together: 16 floats of
            // them, where a batch is small enough to wait for them (221 K
            // rows, 12 frames of 2 floats: 36.2 us one by one, 33.8 in fours);
            // hoisting all reads would cut occupancy
            constexpr int FLIGHT = NQ == 1 ? 4 : NQ == 2 ? 2 : 1;
            for (int g0 = 0; g0 < (RES ? 1 : G); g0 += GR) {
                if (!RES) {
                    asm volatile("" ::: "memory");     // no loads moved up here
                    load(g0);
                }
#pragma unroll
                for (int g = 0; g < GR; ++g) {
                    if (g0 + g < G) {                  // wave-uniform
                        // through an empty asm each chunk: the LDS addresses
                        // are formed per chunk instead of held across the
                        // frame loop
                        unsigned slots = e[g].slots;
                        asm volatile("" : "+v"(slots));
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            add_entry<LC, FC, NF>(area + ((slots >> (8 * u)) & 0xffu) * A::STR,
                                                  e[g].w[0][u], acc);
                            if ((u + 1) % FLIGHT == 0) __builtin_amdgcn_sched_barrier(0);
                        }
                    }
                }
            }
        };
        // a last chunk of at most half its frames reads and adds only those
        if (FC > 1 && sg.frames - f0 <= FC / 2)        // wave-uniform
            entries(std::integral_constant<int, (FC + 1) / 2>{});
        else
            entries(std::integral_constant<int, FC>{});
        if (runs) {
            store_runs<LC, FC>(sg, area, rowsL, acc, f0);
        } else if (active) {
#pragma unroll
            for (int f = 0; f < FC; ++f) {
                if (f0 + f >= sg.frames) break;
                G_ float *d = sg.dst + (size_t)row * sg.dstV + (size_t)(f0 + f) * sg.dstF;
#pragma unroll
                for (int k = 0; k < LC; ++k) d[k] = acc[f][k];
            }
        }
    }
}

// An unlisted slice (more distinct control vertices than a list holds) for
// every frame, FC per chunk: control points gathered from memory, 8 / FC
// entries in flight.  Bound by the gathers; the entries are read once per
// chunk and stay in the caches.  200 K rows of 16 random vertices, 16 frames of
// 7 floats: 351 us at FC = 4; one frame at a time with its entries streamed
// 813.
template <int LC, int FC>
__device__ __forceinline__ void batch_gather_slice(const GStencilSeg &sg, const G_ unsigned *idx,
                                                   const G_ float *wp, int W, int row, bool active)
{
    constexpr int N = 8 / FC, GC = (N + 3) / 4;        // entries in flight, of GC groups
    const int lane = lane_here();
    for (int f0 = 0; f0 < sg.frames; f0 += FC) {
        float acc[FC][LC];
#pragma unroll
        for (int c = 0; c < FC; ++c)
#pragma unroll
            for (int k = 0; k < LC; ++k) acc[c][k] = 0.0f;
        const G_ float *src = sg.src + (size_t)f0 * sg.srcF;
        for (int g = 0; 4 * g < W; g += GC) {
            unsigned ii[4 * GC];
            float w[GC][1][4];
#pragma unroll
            for (int u = 0; u < 4 * GC; ++u)
                ii[u] = idx[(size_t)min(4 * g + u, W - 1) * kWave + lane];
#pragma unroll
            for (int c = 0; c < GC; ++c)               // past the width: the last group, skipped below
                load_weights<1, false>(wp, W, min(g + c, (W - 1) / 4), lane, w[c]);
#pragma unroll
            for (int u0 = 0; u0 < 4 * GC; u0 += N) {
                if (u0 && 4 * g + u0 >= W) break;      // wave-uniform
                float v[N][FC][LC];
#pragma unroll
                for (int u = 0; u < N; ++u) {
                    const unsigned x = 4 * g + u0 + u < W ? ii[u0 + u] : kSliceNoIndex;
                    const G_ float *p = src + (size_t)(x == kSliceNoIndex ? 0u : x) * sg.srcV;
#pragma unroll
                    for (int c = 0; c < FC; ++c) {
                        const G_ float *q = p + (size_t)(f0 + c < sg.frames ? c : 0) * sg.srcF;
#pragma unroll
                        for (int k = 0; k < LC; ++k) v[u][c][k] = q[k];
                    }
                }
#pragma unroll
                for (int u = 0; u < N; ++u) {
                    const bool take = 4 * g + u0 + u < W && ii[u0 + u] != kSliceNoIndex;
#pragma unroll
                    for (int c = 0; c < FC; ++c)
#pragma unroll
                        for (int k = 0; k < LC; ++k) {
                            const float wj = w[(u0 + u) / 4][0][(u0 + u) % 4];
                            const float t = acc[c][k] + v[u][c][k] * wj;
                            acc[c][k] = take ? t : acc[c][k];
                        }
                }
            }
        }
        if (active) {
#pragma unroll
            for (int c = 0; c < FC; ++c) {
                if (f0 + c >= sg.frames) break;
                G_ float *d = sg.dst + (size_t)row * sg.dstV + (size_t)(f0 + c) * sg.dstF;
#pragma unroll
                for (int k = 0; k < LC; ++k) d[k] = acc[c][k];
            }
        }
    }
}

template <int LC, int FC>
__global__ __launch_bounds__(kBlock) void k_batch_stencils(BatchArgs a)
{
    constexpr int FLOATS = BatchArea<LC, FC>::FLOATS;
    __shared__ __attribute__((aligned(16))) float lds[kWavesPerBlock][FLOATS];
    __shared__ int rowsLds[kWavesPerBlock][kWave];
    __shared__ int claim[2];
    const int wv = wave_in_block();
    for (int iter = 0;; ++iter) {
        const int itx = batch_next_item(a, iter, claim);
        if (itx < 0) break;
        const BatchItem item = ld(cptr(a.items) + itx);
        const GStencilSeg sg = gseg(cptr(a.sseg)[item.seg]);
        for (int sl = wv; sl < item.count; sl += kWavesPerBlock) {
            const int s = item.first + sl, lane = lane_here();
            const C_ SliceDesc &ds = sg.slices[s];     // scalar loads
            const int W = ds.width, U = ds.nuniq;
            int row = s * kWave + lane;
            if (sg.perm) row = sg.perm[(long long)s * kWave + lane];
            const bool active = row < sg.nrows;
            const G_ unsigned *rp = sg.rec + ds.off;
            const G_ float *wp = (const G_ float *)(rp + slice_index_dwords(W, U));
            if (U < 0) {
                if (FC > 1 && sg.frames > 1)
                    batch_gather_slice<LC, FC>(sg, rp, wp, W, row, active);
                else
                    batch_gather_slice<LC, 1>(sg, rp, wp, W, row, active);
                continue;
            }
            const G_ int *list = sg.ctrl + ds.ctrlOff;
            float *area = lds[wv];
            int *rowsL = rowsLds[wv];
            // a list too long for FC frames at once takes fewer per chunk, and
            // so does a segment of fewer frames
            static_assert(batch_list<LC, 1, FLOATS>() == kSliceList, "every list fits at one frame");
            auto listed = [&](auto frames) {
                constexpr int F = decltype(frames)::value;
                if (W <= kBatchWidth)
                    batch_listed_slice<LC, F, true>(sg, area, rowsL, rp, wp, W, U, list, row,
                                                    active);
                else
                    batch_listed_slice<LC, F, false>(sg, area, rowsL, rp, wp, W, U, list, row,
                                                     active);
            };
            if (FC == 4 && sg.frames > 2 && U <= batch_list<LC, FC, FLOATS>())
                listed(std::integral_constant<int, FC>{});
            else if (FC >= 2 && sg.frames > 1 && U <= batch_list<LC, FC < 2 ? 1 : 2, FLOATS>())
                listed(std::integral_constant<int, FC < 2 ? 1 : 2>{});
            else
                listed(std::integral_constant<int, 1>{});
        }
    }
}

// Most points listed per wave of 64 coords (slot bytes: up to 256); the
// staged regular-patch kernel comes in 128- and 256-slot variants.
constexpr int kPatchSlots = 256;

// One wave per 64 coords of a patch segment (coords [64 w, 64 w + 64)):
// count pass (FILL false) -- distinct points of the wave's regular-interior
// coords (nuniq = -1 when more than kPatchSlots), list length and the
// number of other coords (ngen); fill pass -- the ascending point list and
// each regular-interior coord's 16 slot bytes.
// Distinct points are extracted in ascending order by repeated wave minima.
template <bool FILL>
__global__ __launch_bounds__(kBlock) void k_patch_slots(BatchPatchSeg sg, int *nuniq,
                                                        long long *listLen, const long long *ptsOff,
                                                        int *pts, unsigned *slots, int *ngen)
{
    const int lane = (int)threadIdx.x & (kWave - 1);
    const int w = (int)blockIdx.x * kWavesPerBlock + wave_in_block();
    const int nw = (sg.ncoords + kWave - 1) / kWave;
    if (w >= nw) return;                                  // whole wave
    if (FILL && nuniq[w] < 0) return;
    const int i = w * kWave + lane;
    bool reg = false;
    int idx[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) idx[j] = 0;
    if (i < sg.ncoords) {
        const osdhip_patch_coord c = sg.coords[i];
        const osdhip_patch_array arr = sg.arrays[c.arrayIndex];
        const unsigned f1 = sg.params[c.patchIndex].field1;
        const int type = ((f1 >> 5) & 1u) ? arr.regDesc : arr.desc;
        reg = type == OSDHIP_PATCH_REGULAR && ((f1 >> 7) & 0x1fu) == 0;
        if (reg) {
            const int *cvs = sg.indices + arr.indexBase + arr.stride * (c.patchIndex - arr.primitiveIdBase);
#pragma unroll
            for (int j = 0; j < 16; ++j) idx[j] = cvs[j];
        }
    }
    unsigned sw[4] = { 0u, 0u, 0u, 0u };
    long long last = -1;
    int U = 0;
    bool over = false;
    for (;;) {
        unsigned m = 0xffffffffu;
        if (reg) {
#pragma unroll
            for (int j = 0; j < 16; ++j)
                if ((long long)(unsigned)idx[j] > last) m = min(m, (unsigned)idx[j]);
        }
        m = wave_min_u(m);
        if (m == 0xffffffffu) break;
        if (U == kPatchSlots) {
            over = true;
            break;
        }
        if (FILL) {
            if (lane == 0) pts[ptsOff[w] + U] = (int)m;
#pragma unroll
            for (int j = 0; j < 16; ++j)
                if (reg && (unsigned)idx[j] == m) sw[j / 4] |= (unsigned)U << (8 * (j % 4));
        }
        last = m;
        ++U;
    }
    if (!FILL) {
        const bool gen = i < sg.ncoords && !reg;
        const int ng = __popcll(__ballot(gen));
        if (lane == 0) {
            nuniq[w] = over ? -1 : U;
            listLen[w] = over ? 0 : U;
            ngen[w] = ng;
        }
        return;
    }
    if (reg) {
#pragma unroll
        for (int r = 0; r < 4; ++r) slots[(size_t)i * 4 + r] = sw[r];
    }
}

// acc[o][q][k] += x * w_o[j] for frames q of a chunk, reference order.
template <int LC, int FC>
__device__ __forceinline__ void batch_patch_point(const G_ float *p, long long fstride, int nq,
                                                  float wp, float wu, float wv,
                                                  float (&acc)[3][FC][LC])
{
#pragma unroll
    for (int q = 0; q < FC; ++q) {
        if (q < nq) {                                   // uniform per segment
#pragma unroll
            for (int k = 0; k < LC; ++k) {
                const float x = p[q * fstride + k];
                acc[0][q][k] += x * wp;
                acc[1][q][k] += x * wu;
                acc[2][q][k] += x * wv;
            }
        }
    }
}

// Phase B in kernels of their own register budgets:
//   k_batch_patches_staged,
//   k_batch_patches_gather   regular B-spline patches without boundary (nearly
//                            all coords): the 16 weights are formed in-line
//                            from the separable curves -- the same single
//                            products basis_bspline stores;
//   k_batch_patches          every other coord (Gregory, boundary, bilinear),
//                            skipping the regular-interior ones.
__device__ __forceinline__ float pick4(const float (&v)[4], int r)
{
    return r == 0 ? v[0] : r == 1 ? v[1] : r == 2 ? v[2] : v[3];
}

// A regular-interior coord (REGULAR type, no boundary) and its parameters.
struct RegularCoord {
    bool ok;
    float s, t, k1;
    const G_ int *cvs;
};

__device__ __forceinline__ RegularCoord regular_coord(const GPatchSeg &sg, int i)
{
    RegularCoord rc;
    const osdhip_patch_coord c = ld(sg.coords + i);
    const osdhip_patch_array arr = ld(sg.arrays + c.arrayIndex);
    const osdhip_patch_param pp = ld(sg.params + c.patchIndex);
    const unsigned f1 = pp.field1;
    const int type = ((f1 >> 5) & 1u) ? arr.regDesc : arr.desc;
    const int boundary = (int)((f1 >> 7) & 0x1fu);
    rc.ok = type == OSDHIP_PATCH_REGULAR && boundary == 0;
    const int depth = (int)(f1 & 0xfu);
    const int nonquad = (int)((f1 >> 4) & 1u);
    const int pv = (int)((f1 >> 12) & 0x3ffu);
    const int pu = (int)((f1 >> 22) & 0x3ffu);
    const float frac_inv = (float)(1 << (depth - nonquad));
    rc.s = c.s * frac_inv - (float)pu;
    rc.t = c.t * frac_inv - (float)pv;
    rc.k1 = (float)(1 << depth);
    rc.cvs = sg.indices + arr.indexBase + arr.stride * (c.patchIndex - arr.primitiveIdBase);
    return rc;
}

template <int LC, int FC>
__device__ __forceinline__ void store_patch_chunk(const GPatchSeg &sg, int i, int f0, int nq,
                                                  float k1, const float (&acc)[3][FC][LC])
{
#pragma unroll
    for (int q = 0; q < FC; ++q) {
        if (q >= nq) break;
#pragma unroll
        for (int o = 0; o < 3; ++o) {
            G_ float *d = sg.out[o];
            if (!d) continue;
            const float f = o == 0 ? 1.0f : k1;
            d += (size_t)i * sg.outV + (size_t)(f0 + q) * sg.outF;
#pragma unroll
            for (int k = 0; k < LC; ++k) d[k] = acc[o][q][k] * f;
        }
    }
}

// Regular coords of waves that are not staged (k_batch_patches_gather: every
// wave with ALL, else those whose list is longer than kPatchSlots) gather
// their points from memory; k_batch_patches_staged takes the waves whose
// coords reference at most SLOTS distinct points (listed by k_patch_slots).
// Same products and order in both.  An item takes itemFrames frames of its
// coords: small batches split a coord's frames over several items, because
// one wave's frames follow one another at a load latency each.
template <int LC, int FC, bool ALL>
__global__ __launch_bounds__(kBlock) void k_batch_patches_gather(BatchArgs a)
{
    __shared__ int claim[2];
    const int wv = wave_in_block();
    for (int iter = 0;; ++iter) {
        const int itx = batch_next_item(a, iter, claim);
        if (itx < 0) break;
        const BatchItem item = ld(cptr(a.items) + itx);
        const GPatchSeg sg = gseg(cptr(a.pseg)[item.seg]);
        const int i = item.first + (int)threadIdx.x;
        if (i >= item.first + item.count) continue;
        // the wave's entry in the staging lists (items start at multiples of
        // kBlock coords; a wave past the segment's end has none)
        if (!ALL && sg.nuniq && sg.nuniq[(item.first >> 6) + wv] >= 0) continue;
        const RegularCoord rc = regular_coord(sg, i);
        if (!rc.ok) continue;
        Curve cs, ct;
        bspline_curve(rc.s, cs);
        bspline_curve(rc.t, ct);
        const int fEnd = item.f0 + min(a.itemFrames, sg.frames - item.f0);
        for (int f0 = item.f0; f0 < fEnd; f0 += FC) {
            const int nq = min(FC, fEnd - f0);
            float acc[3][FC][LC];
#pragma unroll
            for (int o = 0; o < 3; ++o)
#pragma unroll
                for (int q = 0; q < FC; ++q)
#pragma unroll
                    for (int k = 0; k < LC; ++k) acc[o][q][k] = 0.0f;
            const G_ float *base = sg.src + (size_t)f0 * sg.srcF;
#pragma unroll 1
            for (int r = 0; r < 4; ++r) {                 // point j = 4 r + q
                const float tb = pick4(ct.b, r), td = pick4(ct.d, r);
                int idx[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) idx[q] = rc.cvs[4 * r + q];
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    batch_patch_point<LC, FC>(base + (size_t)(unsigned)idx[q] * sg.srcV, sg.srcF,
                                              nq, cs.b[q] * tb, cs.d[q] * tb, cs.b[q] * td, acc);
            }
            store_patch_chunk<LC, FC>(sg, i, f0, nq, rc.k1, acc);
        }
    }
}

// Staged waves: the wave copies its listed points' FC frames into LDS, each
// lane one 16-byte quad of one (point, frame) as k_batch_stencils does, and
// every lane reads its coord's 16 points through its slot bytes with 16-byte
// reads (slot-major, as BatchChunk pads them).  12 meshes of 679 K coords, 1
// to 16 frames of 7 floats, with the frames of a coord split over items:
// lists up to 128 172 -> 146 us, longer lists 119 -> 70 us against one point
// per lane and value-major 4-byte reads (2.0 TB/s of output).
template <int LC, int FC, int SLOTS>
__global__ __launch_bounds__(kBlock) void k_batch_patches_staged(BatchArgs a)
{
    using A = BatchChunk<LC, FC>;
    constexpr int STR = A::STR;
    constexpr int H = (LC + 3) / 4;                       // quads per (point, frame)
    constexpr int N = LC < 4 ? LC : 4;                    // floats per copied quad
    constexpr int QP = FC * H;                            // quads per point: 1, 2, 4 or 8
    constexpr int PI = kWave / QP;                        // points per copy instruction
    __shared__ __attribute__((aligned(16))) float lds[kWavesPerBlock][SLOTS * STR];
    // the claimed item's ints, in floats that no slot uses where there are some:
    // at 7 floats of 2 frames, 8 bytes of their own leave room for three blocks
    // per CU instead of four (1 M coords, 1 frame 54.1 -> 48.9 us, 14 frames 387
    // -> 378 us)
    int *claim;
    if constexpr (STR - 4 * A::NQ >= 2) {
        claim = (int *)(lds[0] + 4 * A::NQ);
    } else {
        __shared__ int own[2];
        claim = own;
    }
    const int wv = wave_in_block();
    for (int iter = 0;; ++iter) {
        const int itx = batch_next_item(a, iter, claim);
        if (itx < 0) break;
        const BatchItem item = ld(cptr(a.items) + itx);
        const GPatchSeg sg = gseg(cptr(a.pseg)[item.seg]);
        const int i = item.first + (int)threadIdx.x;
        const bool inRange = i < item.first + item.count;
        // the wave's entry in the staging lists (items start at multiples of
        // kBlock coords); a wave past the segment's end has none
        const int U = wv * kWave < item.count ? sg.nuniq[(item.first >> 6) + wv] : -1;
        // 128 slots take U <= 128, 256 slots 128 < U <= 256
        if (U < 0 || U > SLOTS || (SLOTS > 128 && U <= 128)) continue;

        // every lane takes part in the copies
        float *area = lds[wv];
        const int lane = lane_here();
        const G_ int *lst = sg.pts + sg.ptsOff[(item.first >> 6) + wv];
        RegularCoord rc;
        rc.ok = false;
        if (inRange) rc = regular_coord(sg, i);
        unsigned sw[4] = { 0u, 0u, 0u, 0u };
        if (rc.ok) {
#pragma unroll
            for (int r = 0; r < 4; ++r) sw[r] = sg.slots[(size_t)i * 4 + r];
        }
        Curve cs, ct;
        bspline_curve(rc.ok ? rc.s : 0.0f, cs);
        bspline_curve(rc.ok ? rc.t : 0.0f, ct);
        // this lane's quad of its points: frame c of the chunk, floats
        // [k0, k0 + N) (the last quad of 5 to 7 floats overlaps the one before)
        const int q = lane % QP, c = q / H, k0 = min(4 * (q % H), LC - N);
        const int fEnd = item.f0 + min(a.itemFrames, sg.frames - item.f0);
        for (int f0 = item.f0; f0 < fEnd; f0 += FC) {
            const int nq = min(FC, fEnd - f0);
            wave_lds_sync();                              // previous chunk's reads are done
            const G_ float *p = sg.src + (size_t)(f0 + min(c, nq - 1)) * sg.srcF + k0;
            for (int u0 = 0; u0 < U; u0 += 4 * PI) {      // four copies in flight
                float x[4][N];
                int pt[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) pt[r] = lst[min(u0 + r * PI + lane / QP, U - 1)];
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int k = 0; k < N; ++k) x[r][k] = p[(size_t)(unsigned)pt[r] * sg.srcV + k];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int u = u0 + r * PI + lane / QP;
                    if (u < U) {
                        float *d = area + u * STR + c * LC + k0;
#pragma unroll
                        for (int k = 0; k < N; ++k) d[k] = x[r][k];
                    }
                }
            }
            wave_lds_sync();
            if (!rc.ok) continue;
            float acc[3][FC][LC];
#pragma unroll
            for (int o = 0; o < 3; ++o)
#pragma unroll
                for (int f = 0; f < FC; ++f)
#pragma unroll
                    for (int k = 0; k < LC; ++k) acc[o][f][k] = 0.0f;
            // the curves' values pass through an empty asm each chunk, so the
            // 48 weight products are formed per chunk instead of being held
            // in registers across the frame loop (they are the same products)
            float cb[4], cd[4], tbv[4], tdv[4];
            unsigned swv[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                cb[r] = cs.b[r];
                cd[r] = cs.d[r];
                tbv[r] = ct.b[r];
                tdv[r] = ct.d[r];
                swv[r] = sw[r];
                asm volatile("" : "+v"(cb[r]), "+v"(cd[r]), "+v"(tbv[r]), "+v"(tdv[r]), "+v"(swv[r]));
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {                 // point j = 4 r + qq, in order
                const float tb = tbv[r], td = tdv[r];
#pragma unroll
                for (int qq = 0; qq < 4; ++qq) {
                    const float wp = cb[qq] * tb, wu = cd[qq] * tb, wvv = cb[qq] * td;
                    const float *ps = area + ((swv[r] >> (8 * qq)) & 0xffu) * STR;
                    // every frame of the chunk without branches, so the point's
                    // LDS reads issue together (frames past the end are not stored)
                    float x[4 * A::NQ];
                    read_values<FC * LC>(ps, x);
#pragma unroll
                    for (int f = 0; f < FC; ++f)
#pragma unroll
                        for (int k = 0; k < LC; ++k) {
                            acc[0][f][k] += x[f * LC + k] * wp;
                            acc[1][f][k] += x[f * LC + k] * wu;
                            acc[2][f][k] += x[f * LC + k] * wvv;
                        }
                    // one point's reads in flight: the point's sums are taken
                    // as asm inputs before a memory clobber, so its products
                    // are formed before the next point's LDS reads issue
                    // (otherwise every point's values are held at once)
#pragma unroll
                    for (int o = 0; o < 3; ++o)
#pragma unroll
                        for (int f = 0; f < FC; ++f)
#pragma unroll
                            for (int k = 0; k < LC; ++k) asm volatile("" ::"v"(acc[o][f][k]));
                    asm volatile("" ::: "memory");
                }
            }
            store_patch_chunk<LC, FC>(sg, i, f0, nq, rc.k1, acc);
        }
    }
}

template <int LC, int FC>
__global__ __launch_bounds__(kBlock) void k_batch_patches(BatchArgs a)
{
    __shared__ int claim[2];
    const int wv = wave_in_block();
    for (int iter = 0;; ++iter) {
        const int itx = batch_next_item(a, iter, claim);
        if (itx < 0) break;
        const BatchItem item = ld(cptr(a.items) + itx);
        const GPatchSeg sg = gseg(cptr(a.pseg)[item.seg]);
        const int i = item.first + (int)threadIdx.x;
        if (i >= item.first + item.count) continue;
        // waves without such coords (counted when the batch was built)
        if (sg.ngen && sg.ngen[(item.first >> 6) + wv] == 0) continue;

        const osdhip_patch_coord c = ld(sg.coords + i);
        const osdhip_patch_array arr = ld(sg.arrays + c.arrayIndex);
        const osdhip_patch_param pp = ld(sg.params + c.patchIndex);
        const unsigned f1 = pp.field1;
        const int type = ((f1 >> 5) & 1u) ? arr.regDesc : arr.desc;
        const int boundary = (int)((f1 >> 7) & 0x1fu);
        if (type == OSDHIP_PATCH_REGULAR && boundary == 0) continue;   // the regular kernel's
        float s = c.s, t = c.t, sign;
        const float k1 = patch_normalize(type, f1, s, t, sign);
        const int n = patch_points(type);
        const G_ int *cvs = sg.indices + arr.indexBase + arr.stride * (c.patchIndex - arr.primitiveIdBase);
        Basis<true, false> B;
        if (n == 16) basis_bspline<true, false>(s, t, boundary, B);
        else if (n == 20) basis_gregory<true, false>(s, t, B);
        else if (n == 4) basis_linear<true, false>(s, t, B);
        else if (n == 12) basis_box_tri<true, false>(s, t, boundary, B);
        else if (n == 18) basis_gregory_tri<true, false>(s, t, B);
        else if (n == 3) basis_linear_tri<true, false>(s, t, B);
        // a negative (invalid) point index reads point 0, as in k_patches
        int cv[20];
#pragma unroll
        for (int j = 0; j < 20; ++j) cv[j] = j < n ? max(cvs[j], 0) : 0;

        const int fEnd = item.f0 + min(a.itemFrames, sg.frames - item.f0);
        for (int f0 = item.f0; f0 < fEnd; f0 += FC) {
            const int nq = min(FC, fEnd - f0);
            float acc[3][FC][LC];
#pragma unroll
            for (int o = 0; o < 3; ++o)
#pragma unroll
                for (int q = 0; q < FC; ++q)
#pragma unroll
                    for (int k = 0; k < LC; ++k) acc[o][q][k] = 0.0f;
            const G_ float *base = sg.src + (size_t)f0 * sg.srcF;
            // the point count follows from the type: 16 / 20 points without
            // per-point predicates, the others (at most 18) predicated, all
            // in the reference's point order
            if (n == 16 || n == 20) {
#pragma unroll
                for (int j = 0; j < 16; ++j)
                    batch_patch_point<LC, FC>(base + (size_t)(unsigned)cv[j] * sg.srcV, sg.srcF,
                                              nq, B.p[j], B.ds[j], B.dt[j], acc);
                if (n == 20) {
#pragma unroll
                    for (int j = 16; j < 20; ++j)
                        batch_patch_point<LC, FC>(base + (size_t)(unsigned)cv[j] * sg.srcV,
                                                  sg.srcF, nq, B.p[j], B.ds[j], B.dt[j], acc);
                }
            } else {
#pragma unroll
                for (int j = 0; j < 18; ++j)
                    if (j < n)
                        batch_patch_point<LC, FC>(base + (size_t)(unsigned)cv[j] * sg.srcV,
                                                  sg.srcF, nq, B.p[j], B.ds[j], B.dt[j], acc);
            }
#pragma unroll
            for (int q = 0; q < FC; ++q) {
                if (q >= nq) break;
#pragma unroll
                for (int o = 0; o < 3; ++o) {
                    G_ float *d = sg.out[o];
                    if (!d) continue;
                    const float f = o == 0 ? 1.0f : k1;
                    d += (size_t)i * sg.outV + (size_t)(f0 + q) * sg.outF;
#pragma unroll
                    for (int k = 0; k < LC; ++k) d[k] = acc[o][q][k] * f;
                }
            }
        }
    }
}

// Frame uploads of an epoch (osdhip_batch_upload): the kernel reads the pinned
// frames over the host link itself.  A block of threads copies kUploadBlock
// bytes, all its loads in flight before the first store.  Bound by the link;
// what it saves is a copy command, with its own start and completion, per
// frame (an epoch of 10 requests: 162 -> 115 us a call, most of it spent
// queueing).
constexpr int kUploadBlocks = 32;               // host blocks per launch
constexpr int kUploadLoads = 2;                 // 16-byte loads per thread
constexpr long long kUploadBlock = 16LL * kUploadLoads * kBlock;
struct UploadArgs {
    int n;
    int end[kUploadBlocks];                     // first grid block past each host block
    int *dst[kUploadBlocks];
    const int *src[kUploadBlocks];
    long long words[kUploadBlocks];
};
typedef int v4i_word __attribute__((ext_vector_type(4), aligned(4)));
__global__ __launch_bounds__(kBlock) void k_batch_upload(UploadArgs a)
{
    const int b = (int)blockIdx.x;
    int s = 0;
    while (s < a.n - 1 && b >= a.end[s]) ++s;
    const long long first = (long long)(b - (s ? a.end[s - 1] : 0)) * (kUploadBlock / 4);
    const int *src = a.src[s] + first;
    int *dst = a.dst[s] + first;
    const long long left = a.words[s] - first;  // >= 1
    const int t = 4 * (int)threadIdx.x;
    if (left >= kUploadBlock / 4) {
        v4i_word v[kUploadLoads];
#pragma unroll
        for (int k = 0; k < kUploadLoads; ++k)
            v[k] = *(const v4i_word *)(src + t + 4 * kBlock * k);
#pragma unroll
        for (int k = 0; k < kUploadLoads; ++k) *(v4i_word *)(dst + t + 4 * kBlock * k) = v[k];
        return;
    }
    const int m = (int)left;
    const int whole = m & ~3;
    for (int j = t; j < whole; j += 4 * kBlock)
        *(v4i_word *)(dst + j) = *(const v4i_word *)(src + j);
    const int j = whole + (int)threadIdx.x;
    if (j < m) dst[j] = src[j];
}

}  // namespace osdhip
