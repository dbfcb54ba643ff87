// Device-side construction of HipStencilTable's slice layouts from the
// uploaded CSR arrays (used by osdhip_stencil_table_create only).
#pragma once
#include "common.h"
#include "stencil_compact.h"
#include "stencil_sliced.h"

namespace osdhip {

// Per slice: widest stencil, and 64 * width entries (the scan input).
__global__ __launch_bounds__(kBlock) void k_slice_widths(const int *sizes, int n, int S,
                                                         int *width, long long *entries,
                                                         int paired = 0)
{
    const int s = (int)(blockIdx.x * kBlock + threadIdx.x);
    if (s >= S) return;
    int w = 0;
    const int r1 = min(n, (s + 1) * kWave);
    for (int r = s * kWave; r < r1; ++r) w = max(w, sizes[r]);
    width[s] = w;
    // paired records: a slice holds whole column pairs
    entries[s] = (long long)(paired ? w + (w & 1) : w) * kWave;
}

// Slice-row sizes padded to whole slices (rows past the end: 0).
__global__ __launch_bounds__(kBlock) void k_pad_sizes(const int *sizes, int n, int rows,
                                                      int *padded)
{
    const int r = (int)(blockIdx.x * kBlock + threadIdx.x);
    if (r >= rows) return;
    padded[r] = r < n ? sizes[r] : 0;
}

// Paired records (one weight array): entries 2p and 2p + 1 of a row sit
// side by side, {index, w, index, w}, so a lane reads both with one 16-byte
// load; column pair p of a slice holds its 64 rows' pairs contiguously,
// record (j, lane) at dword 2 * sliceOff + 256 * (j / 2) + 4 * lane +
// 2 * (j % 2).  An odd width is padded to a whole pair.
__global__ __launch_bounds__(kBlock) void k_fill_records_paired(
    const int *sizes, const int *offsets, const int *indices, const float *w0, int n, int rows,
    const long long *sliceOff, const int *sliceWidth, unsigned *rec)
{
    const int r = (int)(blockIdx.x * kBlock + threadIdx.x);
    if (r >= rows) return;
    const int s = r / kWave, lane = r % kWave;
    const int W = sliceWidth[s], W2 = W + (W & 1);
    const int sz = r < n ? sizes[r] : 0;
    const long long off = r < n ? (long long)offsets[r] : 0;
    for (int j = 0; j < W2; ++j) {
        unsigned q0 = 0u, q1 = 0u;
        if (j < sz) {
            q0 = (unsigned)indices[off + j];
            q1 = __float_as_uint(w0[off + j]);
        }
        unsigned *d = rec + (size_t)(2 * sliceOff[s] + 256LL * (j >> 1) + 4 * lane + 2 * (j & 1));
        d[0] = q0;
        d[1] = q1;
    }
}

// Split-stream layout (layout 1: index and each weight array in its own
// column-major slice stream).
__global__ __launch_bounds__(kBlock) void k_fill_split(
    const int *sizes, const int *offsets, const int *indices, const float *w0, const float *w1,
    const float *w2, const float *w3, const float *w4, const float *w5, int nw, int n, int rows,
    const long long *sliceOff, const int *sliceWidth, int *sidx, float *s0, float *s1, float *s2,
    float *s3, float *s4, float *s5)
{
    const int r = (int)(blockIdx.x * kBlock + threadIdx.x);
    if (r >= rows) return;
    const int s = r / kWave, lane = r % kWave;
    const int W = sliceWidth[s];
    const int sz = r < n ? sizes[r] : 0;
    const long long off = r < n ? (long long)offsets[r] : 0;
    const float *ws[6] = { w0, w1, w2, w3, w4, w5 };
    float *ds[6] = { s0, s1, s2, s3, s4, s5 };
    for (int j = 0; j < W; ++j) {
        const size_t e = (size_t)(sliceOff[s] + (long long)j * kWave + lane);
        sidx[e] = j < sz ? indices[off + j] : 0;
        for (int k = 0; k < nw; ++k) ds[k][e] = j < sz ? ws[k][off + j] : 0.0f;
    }
}

// ---------------------------------------------------------------------------
// Compact slices (layouts 0 and 2; stencil_compact.h).
//
// Layout 0 keeps Far's row order.  Layout 2's locality order sorts rows by
// their dominant control vertex (the entry of largest |weight|, the first
// one on ties; a stable sort keeps Far order among equal keys), so the 64
// rows of a slice surround a few control vertices and share most of their
// support: 26-38 distinct control vertices per slice on creased
// cube-spheres at levels 2-4, against 30 (level 4) to 100 (level 2) on
// average in Far order -- which keeps a slice's 64 outputs consecutive.

// Sort key per slice row: the dominant control vertex (empty rows and rows
// past n: 0xffffffff; the sort is stable, so padding stays last); value:
// the row.
__global__ __launch_bounds__(kBlock) void k_row_dominant(const int *sizes, const int *offsets,
                                                         const int *indices, const float *w0, int n,
                                                         int rows, unsigned *keys, int *vals)
{
    const int r = (int)(blockIdx.x * kBlock + threadIdx.x);
    if (r >= rows) return;
    unsigned key = 0xffffffffu;
    if (r < n && sizes[r] > 0) {
        const long long off = offsets[r];
        key = (unsigned)indices[off];
        float best = fabsf(w0[off]);
        for (int j = 1; j < sizes[r]; ++j) {
            const float a = fabsf(w0[off + j]);
            if (a > best) {
                best = a;
                key = (unsigned)indices[off + j];
            }
        }
    }
    keys[r] = key;
    vals[r] = r;
}

// Rows of the dominant-vertex order regrouped by size within windows of K
// consecutive rows (one block per window): a slice costs its widest row in
// every lane, and rows of one neighbourhood differ in size (9, 12, 16
// entries at a regular vertex, edge and face), so sorting each window's rows
// by size -- stable, by counting -- makes a slice's rows alike while its
// rows still come from a few neighbouring control vertices.  Rows past n
// (slice padding) stay after every real row.
template <int K>
__global__ __launch_bounds__(kBlock) void k_window_size_sort(const int *in, const int *sizes,
                                                             int n, long long rows, int *out)
{
    __shared__ unsigned char key[K];
    __shared__ int start[65];
    const long long w0 = (long long)blockIdx.x * K;
    const int m = (int)(rows - w0 < K ? rows - w0 : K);
    for (int b = (int)threadIdx.x; b < 65; b += kBlock) start[b] = 0;
    for (int i = (int)threadIdx.x; i < m; i += kBlock) {
        const int r = in[w0 + i];
        key[i] = (unsigned char)(r >= 0 && r < n ? min(sizes[r], 63) : 64);
    }
    __syncthreads();
    if (threadIdx.x == 0) {                    // counts, then their exclusive sums
        for (int i = 0; i < m; ++i) ++start[key[i]];
        int s = 0;
        for (int b = 0; b < 65; ++b) {
            const int c = start[b];
            start[b] = s;
            s += c;
        }
    }
    __syncthreads();
    for (int i = (int)threadIdx.x; i < m; i += kBlock) {
        const int k = key[i];
        int before = 0;
        for (int j = 0; j < i; ++j) before += key[j] == k;
        out[w0 + start[k] + before] = in[w0 + i];
    }
}

// Open-addressed set of a slice's control indices in LDS.  A slice stops
// inserting once more than `cap` <= kSliceList are distinct, so at most
// kSliceList + 64 of the kSetSize places are ever taken and every probe
// ends at a free place or its own key.
constexpr int kSetSize = 512;
static_assert(kSliceList + kWave < kSetSize, "probes end");
__device__ __forceinline__ int set_home(unsigned x) { return (int)((x * 2654435761u) >> 23); }

// True when x was not in the set yet.
__device__ __forceinline__ bool set_insert(unsigned *h, unsigned x)
{
    for (int p = set_home(x);; p = (p + 1) & (kSetSize - 1)) {
        const unsigned old = atomicCAS(h + p, kSliceNoIndex, x);
        if (old == kSliceNoIndex) return true;
        if (old == x) return false;
    }
}

__device__ __forceinline__ int set_find(const unsigned *h, unsigned x)
{
    int p = set_home(x);
    while (h[p] != x) p = (p + 1) & (kSetSize - 1);
    return p;
}

// What the slices before one hold (an exclusive scan) and what one holds.
struct SliceCount {
    long long entries;      // 64 * width
    long long dwords;       // stored entries
    long long list;         // listed control vertices
    int listed;             // 1: the slice lists its control vertices
    int longest;            // longest list (a maximum, not a sum)
};
struct SliceCountAdd {
    __host__ __device__ SliceCount operator()(const SliceCount &a, const SliceCount &b) const
    {
        return { a.entries + b.entries, a.dwords + b.dwords, a.list + b.list, a.listed + b.listed,
                 a.longest > b.longest ? a.longest : b.longest };
    }
};

// One wave per slice of the ordered rows perm[] (NULL: Far's order).  Count
// pass (FILL false): slice width, distinct control vertices (nuniq = -1 when
// more than `cap`) and what it holds.  Fill pass: the descriptor, the ascending control
// list, the slot bytes (or control indices) and the weights, as
// stencil_compact.h lays them out.
template <int NWT, bool FILL>
__global__ __launch_bounds__(kBlock) void k_compact_slices(
    const int *perm, const int *sizes, const int *offsets, const int *indices, const float *w0,
    const float *w1, const float *w2, const float *w3, const float *w4, const float *w5, int n, int S,
    int cap, int *width, int *nuniq, SliceCount *counts, const SliceCount *before,
    SliceDesc *slices, int *ctrl, unsigned *rec)
{
    __shared__ unsigned set[kWavesPerBlock][kSetSize];
    __shared__ unsigned char rank[FILL ? kWavesPerBlock : 1][kSetSize];
    __shared__ unsigned vals[FILL ? kWavesPerBlock : 1][kSliceList];
    __shared__ unsigned short place[FILL ? kWavesPerBlock : 1][kSliceList];
    const int lane = (int)threadIdx.x & (kWave - 1);
    const int wv = wave_in_block();
    const int s = (int)blockIdx.x * kWavesPerBlock + wv;
    if (s >= S) return;                                // whole wave
    unsigned *h = set[wv];
    const long long i = (long long)s * kWave + lane;
    const int r = perm ? perm[i] : (int)min(i, (long long)n);
    const bool valid = r >= 0 && r < n;
    const int sz = valid ? sizes[r] : 0;
    const long long off = valid ? (long long)offsets[r] : 0;
    const int W = FILL ? width[s] : wave_max_i(sz);
    int U = FILL ? nuniq[s] : 0;
    if (!FILL || U >= 0) {
        for (int k = lane; k < kSetSize; k += kWave) h[k] = kSliceNoIndex;
        wave_lds_sync();
        int found = 0;
        bool over = false;
        for (int j = 0; j < W && !over; ++j) {         // wave-uniform
            bool fresh = false, bad = false;
            if (j < sz) {
                const unsigned x = (unsigned)indices[off + j];
                bad = x == kSliceNoIndex;              // the free mark: such a slice is not listed
                if (!bad) fresh = set_insert(h, x);
            }
            found += __popcll(__ballot(fresh));
            over = found > cap || __ballot(bad) != 0;
        }
        if (!FILL) U = over ? -1 : found;
    }
    if (!FILL) {
        if (lane == 0) {
            width[s] = W;
            nuniq[s] = U;
            counts[s] = { (long long)W * kWave,
                          (long long)slice_index_dwords(W, U) + (long long)W * NWT * kWave,
                          max(U, 0), U >= 0, max(U, 0) };
        }
        return;
    }
    const long long recOff = before[s].dwords, ctrlOff = before[s].list;
    if (lane == 0) {
        SliceDesc d;
        d.off = recOff;
        d.ctrlOff = ctrlOff;
        d.width = W;
        d.nuniq = U;
        d.pad[0] = d.pad[1] = 0;
        slices[s] = d;
    }
    if (U >= 0) {
        // the set's members side by side, then each one's rank among them
        wave_lds_sync();
        int count = 0;
        for (int k = 0; k < kSetSize; k += kWave) {
            const unsigned x = h[k + lane];
            const unsigned long long m = __ballot(x != kSliceNoIndex);
            if (x != kSliceNoIndex) {
                const int at = count + __popcll(m & ((1ull << lane) - 1));
                vals[wv][at] = x;
                place[wv][at] = (unsigned short)(k + lane);
            }
            count += __popcll(m);
        }
        wave_lds_sync();
        for (int k = lane; k < U; k += kWave) {
            const unsigned x = vals[wv][k];
            int below = 0;
            for (int q = 0; q < U; ++q) below += vals[wv][q] < x;
            rank[wv][place[wv][k]] = (unsigned char)below;
            ctrl[ctrlOff + below] = (int)x;
        }
        wave_lds_sync();
    }
    unsigned *rp = rec + recOff;
    float *wp = (float *)(rp + slice_index_dwords(W, U));
    const float *ws[6] = { w0, w1, w2, w3, w4, w5 };
    for (int g = 0; 4 * g < W; ++g) {
        unsigned bytes = 0u;
        const int left = min(4, W - 4 * g);            // wave-uniform
        for (int u = 0; u < 4; ++u) {
            const int j = 4 * g + u;
            const bool in = j < sz;
            const unsigned x = in ? (unsigned)indices[off + j] : kSliceNoIndex;
            if (U >= 0) bytes |= (in ? (unsigned)rank[wv][set_find(h, x)] : (unsigned)U) << (8 * u);
            if (u >= left) continue;
            if (U < 0) rp[(size_t)j * kWave + lane] = x;
            float *d = NWT == 1 ? wp + (size_t)g * (4 * kWave) + left * lane + u
                                : wp + (size_t)j * (NWT * kWave) + NWT * lane;
#pragma unroll
            for (int k = 0; k < NWT; ++k) d[k] = in ? ws[k][off + j] : 0.0f;
        }
        if (U >= 0) rp[(size_t)g * kWave + lane] = bytes;
    }
}

}  // namespace osdhip
