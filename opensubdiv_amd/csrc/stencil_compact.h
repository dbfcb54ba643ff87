// EvalStencils on compact slices (HipStencilTable layouts 0 and 2).
//
// Rows are cut into 64-row slices, one per wavefront, in Far's order or in
// a locality order (perm).  A slice lists its distinct control vertices in
// ascending order; a wavefront copies those vertices' primvars into LDS and
// every entry then names its control point by one byte, its position in the
// list, instead of a 4-byte index: a one-weight entry costs 5 bytes of HBM
// where an {index, weight} record costs 8, and a control point is fetched
// once per slice instead of once per entry.
//
// Stored per slice, as dwords from SliceDesc::off:
//   slot bytes   ceil(W / 4) x 64 dwords: dword g of lane l holds the list
//                positions of entries 4 g .. 4 g + 3 of row l (past the
//                row's size: U, the zero slot);
//   weights      one array:  column groups of four, lane l's four weights
//                side by side (the last group holds W % 4 per lane);
//                3 or 6 arrays: column by column, lane l's 3 or 6 weights
//                side by side.
// W is the slice's widest row; weights past a row's size are 0.  The zero
// slot holds zeros, and adding 0 * 0 = +0 leaves every partial sum as it is
// (a sum that starts at +0 is never -0 under round-to-nearest), so no
// predicate is needed and the sums are CpuEvalStencils' bit for bit.
//
// A slice with more distinct control vertices than its table lists
// (U = -1) keeps 4-byte control indices, W x 64 dwords, in place of the slot
// bytes (padding: kSliceNoIndex, skipped) and gathers from memory.
#pragma once
#include "common.h"

namespace osdhip {

// Most control vertices a slice lists: its list positions and the zero slot
// are bytes.
constexpr int kSliceList = 255;
// Slices of a locality order list at most 63: a wave then stages its list
// with one vertex per lane.
constexpr int kLocalityList = kWave - 1;
constexpr unsigned kSliceNoIndex = 0xffffffffu;

struct SliceDesc {
    long long off;          // first dword of the slice's stored entries
    long long ctrlOff;      // first entry of its control list
    int width;              // widest row
    int nuniq;              // listed control vertices; -1: not listed
    int pad[2];
};

struct CompactArgs {
    const float *src;       // includes srcDesc.offset and the element window start
    int srcStride;
    float *dst[6];          // NULL = output not requested
    int dstStride[6];
    const int *perm;        // slice row -> Far row; NULL: Far's order
    const SliceDesc *slices;
    const int *ctrl;
    const unsigned *rec;
    int rowBegin, rowEnd;   // Far rows [rowBegin, rowEnd); output row = row - rowBegin
    int sliceBegin, nslices;
    int nblocks;
    int slots;              // LDS slots per wave
};

// Entries 4 g .. 4 g + 3 of one lane: slot bytes (or, unlisted, nothing) and
// weights.
template <int NWT>
struct EntryGroup {
    unsigned slots;
    float w[NWT][4];
};

// Reads *p; STREAM: data the call reads once.
template <bool STREAM, class P>
__device__ __forceinline__ auto load_entry(P p)
{
    if constexpr (STREAM) return __builtin_nontemporal_load(p);
    else return *p;
}

// Loads group g of a slice's weights: wp = the slice's weights (wave-uniform);
// 4 g < W.  Columns past W get weight 0.
template <int NWT, bool STREAM = true, class P>
__device__ __forceinline__ void load_weights(P wp, int W, int g, int lane, float (&w)[NWT][4])
{
    const int left = W - 4 * g;                        // wave-uniform
    if constexpr (NWT == 1) {
        P p = wp + (size_t)g * (4 * kWave);
        if (left >= 4) {
            const v4f q = load_entry<STREAM>((const OSDHIP_GLOBAL v4f *)(p + 4 * lane));
#pragma unroll
            for (int u = 0; u < 4; ++u) w[0][u] = q[u];
        } else {
            p += left * lane;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                w[0][u] = 0.0f;
                if (u < left) w[0][u] = p[u];
            }
        }
    } else {
        P p = wp + (size_t)(4 * g) * (NWT * kWave) + NWT * lane;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            // past the width: the last column again, with weight 0
            P q = p + (size_t)min(u, left - 1) * (NWT * kWave);
#pragma unroll
            for (int k = 0; k < NWT; ++k) w[k][u] = load_entry<STREAM>(q + k);
        }
#pragma unroll
        for (int u = 1; u < 4; ++u)
#pragma unroll
            for (int k = 0; k < NWT; ++k) w[k][u] = u < left ? w[k][u] : 0.0f;
    }
}

// Floats per LDS slot of LC values: whole 16-byte reads.
template <int LC>
struct SlotShape {
    static constexpr int STR = LC <= 2 ? LC : LC <= 4 ? 4 : 8;
};

// One slot's LC values from LDS, 16 bytes at a time.
template <int LC>
__device__ __forceinline__ void read_slot(const float *p, float (&x)[LC])
{
    if constexpr (LC <= 2) {
#pragma unroll
        for (int k = 0; k < LC; ++k) x[k] = p[k];
    } else {
#pragma unroll
        for (int q = 0; q < (LC + 3) / 4; ++q) {
            const v4f v = *(const v4f *)(p + 4 * q);
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (4 * q + k < LC) x[4 * q + k] = v[k];
        }
    }
}

// Stores one slot's LC values (floats past LC: not read).
template <int LC>
__device__ __forceinline__ void write_slot(float *p, const float (&x)[LC])
{
    if constexpr (LC <= 2) {
#pragma unroll
        for (int k = 0; k < LC; ++k) p[k] = x[k];
    } else {
#pragma unroll
        for (int q = 0; q < (LC + 3) / 4; ++q) {
            v4f v;
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = 4 * q + k < LC ? x[4 * q + k < LC ? 4 * q + k : 0] : 0.0f;
            *(v4f *)(p + 4 * q) = v;
        }
    }
}

// Sums of an unlisted slice's row: control points gathered from memory, the
// gathers of GC entry groups in flight; idx / wp: the slice's indices and
// weights.
template <int NWT, int LC, int GC, class IP, class P, class S>
__device__ __forceinline__ void gather_slice(S src, size_t sstride, IP idx, P wp, int W, int lane,
                                             float (&acc)[NWT][LC])
{
    constexpr int N = 4 * GC;
    for (int g = 0; 4 * g < W; g += GC) {
        unsigned ii[N];
        float w[GC][NWT][4], v[N][LC];
#pragma unroll
        for (int u = 0; u < N; ++u)
            ii[u] = __builtin_nontemporal_load(idx + (size_t)min(4 * g + u, W - 1) * kWave + lane);
#pragma unroll
        for (int c = 0; c < GC; ++c)                  // past the width: the last group, skipped below
            load_weights<NWT>(wp, W, min(g + c, (W - 1) / 4), lane, w[c]);
#pragma unroll
        for (int u = 0; u < N; ++u) {
            ii[u] = 4 * g + u < W ? ii[u] : kSliceNoIndex;
            S p = src + (size_t)(ii[u] == kSliceNoIndex ? 0u : ii[u]) * sstride;
#pragma unroll
            for (int k = 0; k < LC; ++k) v[u][k] = p[k];
        }
#pragma unroll
        for (int u = 0; u < N; ++u) {
            const bool take = ii[u] != kSliceNoIndex;
#pragma unroll
            for (int a = 0; a < NWT; ++a)
#pragma unroll
                for (int k = 0; k < LC; ++k) {
                    const float t = acc[a][k] + v[u][k] * w[u / 4][a][u % 4];
                    acc[a][k] = take ? t : acc[a][k];
                }
        }
    }
}

// Dwords of a slice's index part: slot bytes or control indices.
__device__ __forceinline__ size_t slice_index_dwords(int W, int U)
{
    return (size_t)(U >= 0 ? (W + 3) / 4 : W) * kWave;
}

// LISTS: some slice of the table lists its control vertices.  The other
// variant, for one-weight tables of 5 to 8 floats without any list, keeps the
// gathers of two entry groups in flight, whose registers would cost listed
// slices their waves (2.1 M rows of 7 floats: 58.9 -> 62.4 us; 500 K rows of
// 16 random vertices, 7 floats: 56.8 us with two groups, 63.5 with one).
template <int NWT, int LC, bool LISTS>
__global__ __launch_bounds__(kBlock) void k_stencils_compact(CompactArgs a)
{
    constexpr int GATHER = LC <= 4 || !LISTS ? 2 : 1;   // entry groups gathered at a time
    constexpr int STR = SlotShape<LC>::STR;
    constexpr int GC = NWT == 6 ? 2 : 4;            // entry groups in flight
    // a.slots * STR floats per wave: the table's longest list and the zero slot
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int lane = (int)threadIdx.x & (kWave - 1);
    const int wv = wave_in_block();
    const int lb = xcd_logical_block();
    if (lb >= a.nblocks) return;
    const int sl = lb * kWavesPerBlock + wv;
    if (sl >= a.nslices) return;                     // whole wave idle
    const int s = a.sliceBegin + sl;
    const OSDHIP_CONST SliceDesc &ds = cptr(a.slices)[s];
    const int W = ds.width, U = LISTS ? ds.nuniq : -1;
    int row = s * kWave + lane;
    if (a.perm) row = gptr(a.perm)[row];             // wave-uniform branch
    const bool active = row >= a.rowBegin && row < a.rowEnd;
    const OSDHIP_GLOBAL unsigned *rp = gptr(a.rec) + ds.off;
    const OSDHIP_GLOBAL float *wp =
        (const OSDHIP_GLOBAL float *)(rp + slice_index_dwords(W, U));
    const OSDHIP_GLOBAL float *src = gptr(a.src);
    const size_t sstride = (size_t)a.srcStride;

    float acc[NWT][LC];
#pragma unroll
    for (int w = 0; w < NWT; ++w)
#pragma unroll
        for (int k = 0; k < LC; ++k) acc[w][k] = 0.0f;

    if (LISTS && U >= 0) {
        float *area = lds + wv * a.slots * STR;
        const OSDHIP_GLOBAL int *list = gptr(a.ctrl) + ds.ctrlOff;
        const int G = (W + 3) / 4;
        EntryGroup<NWT> e[GC];
        auto load = [&](int g0) {
#pragma unroll
            for (int c = 0; c < GC; ++c)
                if (g0 + c < G) {                    // wave-uniform
                    e[c].slots = __builtin_nontemporal_load(rp + (size_t)(g0 + c) * kWave + lane);
                    load_weights<NWT>(wp, W, g0 + c, lane, e[c].w);
                }
        };
        load(0);                                     // in flight while the list is staged
        // the list (up to four rounds of 64), all its loads before any is used
        constexpr int R = (kSliceList + kWave) / kWave;
        int v[R];
        float x[R][LC];
#pragma unroll
        for (int h = 0; h < R; ++h)
            if (h * kWave < U) v[h] = list[min(h * kWave + lane, U - 1)];   // wave-uniform
#pragma unroll
        for (int h = 0; h < R; ++h)
            if (h * kWave < U) {
                const OSDHIP_GLOBAL float *p = src + (size_t)(unsigned)v[h] * sstride;
#pragma unroll
                for (int k = 0; k < LC; ++k) x[h][k] = p[k];
            }
#pragma unroll
        for (int h = 0; h < R; ++h)
            if (h * kWave + lane < U) write_slot<LC>(area + (h * kWave + lane) * STR, x[h]);
        if (lane < STR) area[U * STR + lane] = 0.0f;     // the zero slot
        wave_lds_sync();
        for (int g0 = 0; g0 < G; g0 += GC) {
            if (g0) load(g0);
#pragma unroll
            for (int c = 0; c < GC; ++c)
                if (g0 + c < G) {
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        float x[LC];
                        read_slot<LC>(area + ((e[c].slots >> (8 * u)) & 0xffu) * STR, x);
#pragma unroll
                        for (int w = 0; w < NWT; ++w)
#pragma unroll
                            for (int k = 0; k < LC; ++k)
                                acc[w][k] = acc[w][k] + x[k] * e[c].w[w][u];
                    }
                }
        }
    } else {
        gather_slice<NWT, LC, GATHER>(src, sstride, rp, wp, W, lane, acc);
    }
    if (active) {
        const size_t r = (size_t)(row - a.rowBegin);
#pragma unroll
        for (int w = 0; w < NWT; ++w) {
            float *d = a.dst[w];
            if (!d) continue;
            d += r * (size_t)a.dstStride[w];
#pragma unroll
            for (int k = 0; k < LC; ++k) d[k] = acc[w][k];
        }
    }
}

}  // namespace osdhip
