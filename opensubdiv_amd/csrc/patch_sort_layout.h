// Workspace layout of the patch-order binning (patch_sort.h): the tiles' bin
// histograms hist[blocks x kPatchBins] (turned in place into each tile's first
// position within the bin), the bins' totals, and order[n]; 256-byte aligned.
#pragma once
#include <cstddef>

namespace osdhip {

constexpr int kPatchBins = 4096;          // bin = (patchIndex >> 8) mod 4096
constexpr int kPatchBinShift = 8;         // 256 consecutive patches per bin
constexpr int kMaxBinBlocks = 256;        // blocks (tiles of coords) at most
constexpr int kMinBinTile = 4096;         // coords per block at least

constexpr long long patch_tile(long long n)
{
    const long long t = (n + kMaxBinBlocks - 1) / kMaxBinBlocks;
    return t < kMinBinTile ? kMinBinTile : t;
}

struct PatchSortLayout {
    size_t hist = 0, totals = 0, order = 0, bytes = 0;
    int tile = 0, blocks = 0;
    constexpr explicit PatchSortLayout(long long n)
    {
        auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
        tile = (int)patch_tile(n);
        blocks = (int)((n + tile - 1) / tile);
        totals = up(hist + 4 * (size_t)kPatchBins * (size_t)(blocks > 0 ? blocks : 1));
        order = up(totals + 4 * (size_t)kPatchBins);
        bytes = up(order + 4 * (size_t)n);
    }
};

}  // namespace osdhip
