// Patch-ordered evaluation of PatchCoords, in two levels.  The coords are
// binned by patch (bin = (patchIndex >> 8) mod 4096: 256 consecutive patches
// per bin, which share control points); the evaluating blocks then order
// their part of the binned coords by patch in LDS (k_patches_sorted), so that
// neighbouring lanes evaluate the same patch: their index rows and control
// points are the same lines, and their patch type is the same.  Each coord's
// result depends on that coord only and goes to its own row, so any visit
// order gives the same bits.
//
// One pass over the coords counts bins per tile of coords in LDS (no global
// atomics), a second turns the tiles' counts of each bin into first
// positions within the bin, and a third places each coord's number (LDS
// atomics per tile; every block forms the bins' own first positions from
// their totals itself).  Workspace (device memory, PatchSortLayout): every
// launch writes what it reads, with kernels only (no memset), so the sequence
// may be captured into a graph and a workspace reused by calls that do not
// overlap.  1.5 M random coords on 280 K patches, P and tangents of 4 floats:
// binning 24.3 us (5 launches of 256 threads, 1,024-patch bins and a scan
// spread over three of them: 39.3 us), the whole call, nothing cached, 155 us
// against 189 with those bins alone.
#pragma once
#include <hip/hip_runtime.h>

#include "../../include/osdhip.h"
#include "common.h"
#include "patch_kernels.h"
#include "patch_sort_layout.h"

namespace osdhip {

constexpr int kSortBlock = 1024;          // threads of the binning kernels
constexpr int kBinsPerThread = kPatchBins / kSortBlock;
static_assert(kPatchBins % kSortBlock == 0, "bins are cleared and scanned kSortBlock at a time");

__device__ __forceinline__ int patch_bin(int patchIndex)
{
    return patchIndex < 0 ? 0 : (patchIndex >> kPatchBinShift) & (kPatchBins - 1);
}

// Block b: bin counts of coords [b * tile, min(n, (b + 1) * tile)) into
// hist[b * kPatchBins + bin].
__global__ __launch_bounds__(kSortBlock) void k_patch_bin_hist(const osdhip_patch_coord *coords,
                                                               int n, int tile, unsigned *hist)
{
    __shared__ unsigned h[kPatchBins];
    for (int k = (int)threadIdx.x; k < kPatchBins; k += kSortBlock) h[k] = 0u;
    __syncthreads();
    const long long i0 = (long long)blockIdx.x * tile;
    const long long i1 = i0 + tile < n ? i0 + tile : n;
    for (long long i = i0 + threadIdx.x; i < i1; i += kSortBlock)
        atomicAdd(&h[patch_bin(coords[i].patchIndex)], 1u);
    __syncthreads();
    for (int k = (int)threadIdx.x; k < kPatchBins; k += kSortBlock)
        hist[(size_t)blockIdx.x * kPatchBins + k] = h[k];
}

// Block b: bins [64 b, 64 b + 64), 64 lanes of one bin each times 16 groups of
// tiles: the tiles' counts become first positions within the bin, their sum
// its total.
constexpr int kScanBins = 64, kScanGroups = kSortBlock / kScanBins;
constexpr int kScanTiles = kMaxBinBlocks / kScanGroups;    // tiles per thread at most
__global__ __launch_bounds__(kSortBlock) void k_patch_bin_scan(unsigned *hist, int blocks,
                                                               unsigned *totals)
{
    __shared__ unsigned part[kScanGroups][kScanBins];
    const int lane = (int)threadIdx.x % kScanBins, g = (int)threadIdx.x / kScanBins;
    unsigned *col = hist + (size_t)blockIdx.x * kScanBins + lane;
    unsigned v[kScanTiles];
    unsigned mine = 0;
#pragma unroll
    for (int k = 0; k < kScanTiles; ++k) {
        const int b = g * kScanTiles + k;
        v[k] = b < blocks ? col[(size_t)b * kPatchBins] : 0u;
    }
#pragma unroll
    for (int k = 0; k < kScanTiles; ++k) mine += v[k];
    part[g][lane] = mine;
    __syncthreads();
    unsigned at = 0;
    for (int k = 0; k < g; ++k) at += part[k][lane];
#pragma unroll
    for (int k = 0; k < kScanTiles; ++k) {
        const int b = g * kScanTiles + k;
        if (b < blocks) col[(size_t)b * kPatchBins] = at;
        at += v[k];
    }
    if (g == kScanGroups - 1) totals[blockIdx.x * kScanBins + lane] = at;
}

// Block b places coords [b * tile, ...) of each bin from the bin's first
// position for this tile (the order within a tile's share of a bin is
// whatever the LDS atomics give; it does not change any result).
__global__ __launch_bounds__(kSortBlock) void k_patch_bin_scatter(const osdhip_patch_coord *coords,
                                                                  int n, int tile,
                                                                  const unsigned *hist,
                                                                  const unsigned *totals, int *order)
{
    __shared__ unsigned cur[kPatchBins];
    __shared__ unsigned waveSums[kSortBlock / kWave];
    const int t = (int)threadIdx.x, lane = t & (kWave - 1), w = t / kWave;
    // exclusive scan of the bins' totals, kBinsPerThread neighbours per thread
    unsigned x[kBinsPerThread], mine = 0;
#pragma unroll
    for (int k = 0; k < kBinsPerThread; ++k) {
        x[k] = totals[t * kBinsPerThread + k];
        mine += x[k];
    }
    unsigned incl = mine;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const unsigned y = (unsigned)__shfl_up((int)incl, d, kWave);
        if (lane >= d) incl += y;
    }
    if (lane == kWave - 1) waveSums[w] = incl;
    __syncthreads();
    unsigned at = incl - mine;
    for (int k = 0; k < w; ++k) at += waveSums[k];
#pragma unroll
    for (int k = 0; k < kBinsPerThread; ++k) {
        const int bin = t * kBinsPerThread + k;
        cur[bin] = at + hist[(size_t)blockIdx.x * kPatchBins + bin];
        at += x[k];
    }
    __syncthreads();
    const long long i0 = (long long)blockIdx.x * tile;
    const long long i1 = i0 + tile < n ? i0 + tile : n;
    for (long long i = i0 + t; i < i1; i += kSortBlock) {
        const unsigned pos = atomicAdd(&cur[patch_bin(coords[i].patchIndex)], 1u);
        order[pos] = (int)i;
    }
}

// Queues the binning of n coords on st in the workspace at ws (laid out by
// PatchSortLayout(n)); returns the order array.
inline int *queue_patch_sort(const osdhip_patch_coord *coords, int n, char *ws, hipStream_t st)
{
    const PatchSortLayout L(n);
    unsigned *hist = (unsigned *)(ws + L.hist), *totals = (unsigned *)(ws + L.totals);
    int *order = (int *)(ws + L.order);
    hipLaunchKernelGGL(k_patch_bin_hist, dim3(L.blocks), dim3(kSortBlock), 0, st, coords, n, L.tile,
                       hist);
    hipLaunchKernelGGL(k_patch_bin_scan, dim3(kPatchBins / kScanBins), dim3(kSortBlock), 0, st, hist,
                       L.blocks, totals);
    hipLaunchKernelGGL(k_patch_bin_scatter, dim3(L.blocks), dim3(kSortBlock), 0, st, coords, n,
                       L.tile, hist, totals, order);
    return order;
}

// EvalPatches of binned coords: a block takes kBlock of them, orders them by
// patch (a counting sort on the patch's last ten bits, which tells apart the
// patches of four neighbouring bins) and evaluates one coord per lane.  The
// coords' fields wait in LDS: they were gathered once, by number.  Bound by
// memory latency and by the results' stores, which go to scattered rows (with
// the stores left out the same call takes 79.5 us instead of 157): ordering
// more coords per block shares more lines between lanes but leaves fewer waves
// in flight.  The call on 1.5 M coords: 162.7 us without the ordering, 155
// with 256 coords, 157 with 512, 161 with 768, 170 with 1,024.
constexpr int kSortKeys = 1024;
template <bool D1, bool D2, int LC>
__global__ __launch_bounds__(kBlock) void k_patches_sorted(PatchArgs a, const int *order)
{
    constexpr int KT = kSortKeys / kBlock;
    __shared__ v4i rec[kBlock];                 // arrayIndex, patchIndex, s, t
    __shared__ int num[kBlock];
    __shared__ unsigned cnt[kSortKeys];
    __shared__ unsigned waveSums[kWavesPerBlock];
    const int t = (int)threadIdx.x, lane = t & (kWave - 1), w = t / kWave;
    const long long first = (long long)xcd_logical_block() * kBlock;
    if (first >= a.n) return;                   // whole block
    const int m = (int)(a.n - first < kBlock ? a.n - first : kBlock);
    const int id = t < m ? order[first + t] : -1;
#pragma unroll
    for (int k = 0; k < KT; ++k) cnt[t + k * kBlock] = 0u;
    v4i r = v4i{ 0, 0, 0, 0 };
    if (id >= 0) {
        const osdhip_patch_coord *c = a.coords + id;
        r = v4i{ c->arrayIndex, c->patchIndex, __float_as_int(c->s), __float_as_int(c->t) };
    }
    const int key = r.y & (kSortKeys - 1);
    __syncthreads();
    const unsigned rank = id >= 0 ? atomicAdd(&cnt[key], 1u) : 0u;
    __syncthreads();
    unsigned x[KT], mine = 0;                   // exclusive scan of the counts, in place
#pragma unroll
    for (int k = 0; k < KT; ++k) {
        x[k] = cnt[t * KT + k];
        mine += x[k];
    }
    unsigned incl = mine;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const unsigned y = (unsigned)__shfl_up((int)incl, d, kWave);
        if (lane >= d) incl += y;
    }
    if (lane == kWave - 1) waveSums[w] = incl;
    __syncthreads();
    unsigned at = incl - mine;
    for (int k = 0; k < w; ++k) at += waveSums[k];
#pragma unroll
    for (int k = 0; k < KT; ++k) {
        cnt[t * KT + k] = at;
        at += x[k];
    }
    __syncthreads();
    if (id >= 0) {
        const unsigned pos = cnt[key] + rank;
        rec[pos] = r;
        num[pos] = id;
    }
    __syncthreads();
    if (t >= m) return;
    const v4i q = rec[t];
    osdhip_patch_coord c;
    c.arrayIndex = q.x;
    c.patchIndex = q.y;
    c.vertIndex = 0;                            // not read
    c.s = __int_as_float(q.z);
    c.t = __int_as_float(q.w);
    eval_patch_coord<D1, D2, LC>(a, c, num[t]);
}

}  // namespace osdhip
