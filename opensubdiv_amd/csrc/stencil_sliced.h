// EvalStencils on 64-row slices with 4-byte control indices: split streams
// (HipStencilTable layout 1) and paired records (layout 3).
//
// HipStencilTable::Create re-lays the Far CSR table out for wave64: the
// entries of the 64 stencils of slice s are stored column-major, entry j of
// row r at sliceOffset[s] + 64*j + (r % 64), padded to the slice's widest
// stencil.  Lane r of a wavefront then reads entry j of its own stencil
// with one fully coalesced 256-byte load per stream, without LDS (so the
// kernel runs at full occupancy), and accumulates entries in table order
// (bit-identical to CpuEvalStencils).  Padding entries are loaded but never
// accumulated (per-lane predicate j < size).  The control-point gathers of
// kSliceGroup consecutive entries are issued before any is consumed.
#pragma once
#include "common.h"

namespace osdhip {

struct SlicedArgs {
    const float *src;       // includes srcDesc.offset and the element window start
    int srcStride;
    float *dst[6];
    int dstStride[6];
    const int *rowSize;     // per stencil
    const long long *sliceOff;
    const int *sliceWidth;
    const int *idx;
    const float *w[6];
    int rowBegin, rowEnd;   // stencils [rowBegin, rowEnd); output row = row - rowBegin
    int sliceBegin, nslices;
    int nblocks;
};

constexpr int kSliceGroup = 4;

template <int NW, int LC>
__global__ __launch_bounds__(kBlock) void k_stencils_sliced(SlicedArgs a)
{
    const int lane = (int)threadIdx.x & (kWave - 1);
    const int lb = xcd_logical_block();
    if (lb >= a.nblocks) return;
    const int sl = lb * kWavesPerBlock + wave_in_block();
    if (sl >= a.nslices) return;                     // whole wave idle
    const int s = a.sliceBegin + sl;
    const int row = s * kWave + lane;
    const bool active = row >= a.rowBegin && row < a.rowEnd;
    const int sz = active ? a.rowSize[row] : 0;
    const int W = a.sliceWidth[s];
    const long long eo = a.sliceOff[s] + lane;

    float acc[NW][LC];
#pragma unroll
    for (int w = 0; w < NW; ++w)
#pragma unroll
        for (int k = 0; k < LC; ++k) acc[w][k] = 0.0f;

    const float *__restrict__ src = a.src;
    const size_t sstride = (size_t)a.srcStride;
    for (int j = 0; j < W; j += kSliceGroup) {
        int ii[kSliceGroup];
        float ww[NW][kSliceGroup];
#pragma unroll
        for (int u = 0; u < kSliceGroup; ++u) {
            // columns past the width re-read the last one (never accumulated:
            // j + u >= W >= size), so the loads are unconditional
            const long long e = eo + (long long)min(j + u, W - 1) * kWave;
            ii[u] = __builtin_nontemporal_load(a.idx + e);
#pragma unroll
            for (int w = 0; w < NW; ++w) ww[w][u] = __builtin_nontemporal_load(a.w[w] + e);
        }
        float v[kSliceGroup][LC];
#pragma unroll
        for (int u = 0; u < kSliceGroup; ++u) {
            if (j + u < sz) {
                const float *p = src + (size_t)(unsigned)ii[u] * sstride;
#pragma unroll
                for (int k = 0; k < LC; ++k) v[u][k] = p[k];
            }
        }
#pragma unroll
        for (int u = 0; u < kSliceGroup; ++u) {
            if (j + u < sz) {
#pragma unroll
                for (int w = 0; w < NW; ++w)
#pragma unroll
                    for (int k = 0; k < LC; ++k) acc[w][k] += v[u][k] * ww[w][u];
            }
        }
    }
    if (active) {
        const size_t r = (size_t)(row - a.rowBegin);
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            float *d = a.dst[w];
            if (!d) continue;
            d += r * (size_t)a.dstStride[w];
#pragma unroll
            for (int k = 0; k < LC; ++k) d[k] = acc[w][k];
        }
    }
}

// Paired records (layout 3, one weight array).
struct RecArgs {
    const float *src;       // includes srcDesc.offset and the element window start
    int srcStride;
    float *dst[6];          // NULL = output not requested
    int dstStride[6];
    const int *rowSize;     // per slice row (padded to a multiple of 64)
    const long long *sliceOff;
    const int *sliceWidth;
    const unsigned *rec;
    int rowBegin, rowEnd;   // stencils [rowBegin, rowEnd); output row = row - rowBegin
    int sliceBegin, nslices;
    int nblocks;
};

// One weight array, paired records (layout 3): a lane loads the records of
// entries 2p and 2p + 1 of its row with one 16-byte load, so a wave streams
// 1 KiB of {index, weight} records per load instruction.  Padding records
// (past a row's size) hold index 0 and weight 0, so every gather address is
// valid; only the accumulation is predicated.  G entries (G / 2 pair loads) are loaded, then all their
// control-point gathers are issued; past the width the last pair is
// re-read and not accumulated.  Same products and order as CpuEvalStencils.
template <int LC, int G>
__global__ __launch_bounds__(kBlock) void k_stencils_rec_paired(RecArgs a)
{
    static_assert(G % 2 == 0, "pairs");
    const int lane = (int)threadIdx.x & (kWave - 1);
    const int lb = xcd_logical_block();
    if (lb >= a.nblocks) return;
    const int sl = lb * kWavesPerBlock + wave_in_block();
    if (sl >= a.nslices) return;                     // whole wave idle
    const int s = a.sliceBegin + sl;
    const int row = s * kWave + lane;
    const bool active = row >= a.rowBegin && row < a.rowEnd;
    const int sz = active ? a.rowSize[row] : 0;
    const int W = a.sliceWidth[s];
    const int P = (W + 1) >> 1;                      // column pairs
    const unsigned *rp = a.rec + (size_t)(2 * a.sliceOff[s] + 4 * lane);

    float acc[LC];
#pragma unroll
    for (int k = 0; k < LC; ++k) acc[k] = 0.0f;
    const float *__restrict__ src = a.src;
    const size_t sstride = (size_t)a.srcStride;
    for (int p0 = 0; p0 < P; p0 += G / 2) {
        int ii[G];
        float ww[G];
#pragma unroll
        for (int u = 0; u < G / 2; ++u) {
            const v4i q = __builtin_nontemporal_load(
                (const v4i *)(rp + (size_t)min(p0 + u, P - 1) * (kWave * 4)));
            ii[2 * u] = q.x;
            ww[2 * u] = __int_as_float(q.y);
            ii[2 * u + 1] = q.z;
            ww[2 * u + 1] = __int_as_float(q.w);
        }
        float v[G][LC];
#pragma unroll
        for (int u = 0; u < G; ++u) {
            const float *pp = src + (size_t)(unsigned)ii[u] * sstride;
#pragma unroll
            for (int k = 0; k < LC; ++k) v[u][k] = pp[k];
        }
#pragma unroll
        for (int u = 0; u < G; ++u) {
            const bool take = 2 * p0 + u < sz;
#pragma unroll
            for (int k = 0; k < LC; ++k) {
                const float t = acc[k] + v[u][k] * ww[u];
                acc[k] = take ? t : acc[k];
            }
        }
    }
    if (active) {
        float *d = a.dst[0];
        if (d) {
            d += (size_t)(row - a.rowBegin) * (size_t)a.dstStride[0];
#pragma unroll
            for (int k = 0; k < LC; ++k) d[k] = acc[k];
        }
    }
}

}  // namespace osdhip
