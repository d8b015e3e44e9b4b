// Batched views: one launch per stage over the work items of every view.
//
// Each view's arguments live in a device array of ViewDesc; a launch's blocks
// are numbered over the concatenation of all views' work items (tiles or
// pixel blocks), so a block finds its view with a short scan of the
// per-view first-item offsets (uniform per block, scalar loads) and then runs
// the same per-tile / per-block body as the single-view kernel.
#pragma once

#include "gi_device.h"

namespace sgi_batch {

struct ViewDesc {
    sgi_dev::GbufArgs g;
    sgi_dev::FrameArgs fr;
    sgi_dev::CsmArgs csm;
    int tilesX, tilesY;  // culling / gather tiles at the batch's tile size
    int tileStart;       // first batch tile of this view
    int dtileStart;      // first batch 16x16 tile (direct light)
    int dblockStart;     // first batch 64x4 block (denoiser)
    int dfilterStart;    // first batch block of the denoiser's filter (filterBlocks() a view)
    sgi_vpl* vplUpdated;
    int32_t* visible;
    sgi_atlas_entry* entries;
    uint8_t* visFlags;
    int32_t* tiles;
    float* direct;
    float* color;
    float* reservoir;
    const float* prevGi;
    const float* prevHistory;
    float* combined;
    float* giOut;
    float* reservoirOut;
    float* historyOut;
    float4* resA;
    float4* resB;
    float4* normals;
};

enum Offset { kTiles = 0, kDirectTiles = 1, kDenoiseBlocks = 2, kFilterBlocks = 3 };

// Pixels of a column that a thread of the a-trous filter takes, from the number of 64 x 4 pixel blocks of
// the launch (a batch: of all views).
// With few waves a thread's chain decides, with more its loads: the whole denoiser with 1 / 2 / 4 pixels
// takes 18 / 25 / 30 us at 320x180 (225 blocks), 33.3 / 33.5 / 35.9 at 560x315 (711), 40.2 / 35.2 / 37.2 at
// 640x360 (900), 54 / 47 / 52 at 800x450 (1469), 69 / 58 / 56 at 960x540 (2025).
constexpr int kRows2 = 750, kRows4 = 1800;
inline int filterRows(int blocks) { return blocks < kRows2 ? 1 : (blocks < kRows4 ? 2 : 4); }
// Blocks of its launch over a W x H view: two for each region of 64 x 8 rows pixels.
__host__ __device__ __forceinline__ int filterBlocks(int W, int H, int rows) {
    return ((W + 63) / 64) * ((H + 8 * rows - 1) / (8 * rows)) * 2;
}

// The view whose work items contain batch item `item` (views are in item order).
template <int OFF>
__device__ __forceinline__ int findView(const ViewDesc* __restrict__ v, int n, int item) {
    int i = 0;
    for (int k = 1; k < n; ++k) {
        const int start = OFF == kTiles         ? v[k].tileStart
                          : OFF == kDirectTiles ? v[k].dtileStart
                          : OFF == kFilterBlocks ? v[k].dfilterStart
                                                 : v[k].dblockStart;
        if (start <= item) i = k;
    }
    return i;
}

}  // namespace sgi_batch
