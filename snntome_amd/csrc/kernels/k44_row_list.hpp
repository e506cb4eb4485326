// k44_row_list.hpp — private index rows of scattered positions on the VALU (see k44_row_list.hip).
#pragma once
#include "k44_mfma_tile.hpp"

namespace k44dev {

struct RowListArgs {
    const __half *X;        // canvas + the wave's lowest row offset
    const uint32_t *roff;   // [index rows][32 steps] element offset of every position from X
    const __half *W;        // [cout][32 steps], zero past the row
    const __half *bias;     // [cout] or nullptr
    const uint16_t *cmap;   // [cout] or nullptr
    __half *Y;              // canvas + y_off
    const __half *R;        // canvas + res_off or nullptr
    uint64_t out_stride;
    uint32_t cout, cluster;
    uint32_t B, steps;      // positions per row, ceil(B / 32)
    uint32_t ttiles;        // 64-token tiles
    int act;                // (rows, outputs and residuals on the 16-byte grid)
};

// kw: waves that share a neuron's positions (1 or 4).
hipError_t launch_row_list(const RowListArgs &a, uint32_t kw, hipStream_t stream);

}  // namespace k44dev
