// k44_mfma_rows.hpp — MFMA waves whose tiles gather arbitrary rows (see k44_mfma_rows.hip).
#pragma once
#include "k44_mfma_tile.hpp"
#include "k44_spatial.hpp"

namespace k44dev {

// Item of workgroup b of n: workgroups go round-robin over the 8 XCDs, each takes a contiguous run.
__device__ __forceinline__ uint32_t xcd_contiguous(uint32_t b, uint32_t n) {
    const uint32_t x = b & 7u, q = n >> 3, r = n & 7u;
    return x * q + min(x, r) + (b >> 3);
}

struct RowsArgs {
    const __half *X;       // canvas + the wave's lowest row offset
    const uint32_t *roff;  // [index rows][32 ksteps] element offset of every position from X
    const __half *Wf;      // A fragments [index row][k-step][blocks][lane][8], zero past the row
    const __half *bias;    // [cout] or nullptr
    const uint16_t *cmap;  // [cout] or nullptr
    __half *Y;             // canvas + y_off
    const __half *R;       // canvas + res_off or nullptr
    const uint32_t *tile_x, *tile_y;  // per 64-token tile offsets (2-D waves); nullptr: 64 t
    uint64_t out_stride;
    uint32_t B, ksteps;    // positions per row, ceil(B / 32)
    uint32_t blocks;       // 16-neuron blocks per index row
    uint32_t subs;         // sub-tiles of 16 NB neurons per index row
    uint32_t ttiles;       // 64-token tiles
    int act;
    uint32_t vec;          // output / residual rows: 8-, 4- or 1-element aligned stores
    uint32_t mask_w, mask_h, mask_wpad, mask_tpf;  // as in MfmaTileArgs
};

// A launch covers `n` independent waves of the same kernel shape (descriptors in device memory;
// workgroup column x belongs to the wave w with start[w] <= x < start[w + 1]), or, with n = 0, the
// one wave passed by value.
struct RowsLaunch {
    const RowsArgs *waves = nullptr;
    const uint32_t *start = nullptr;
    uint32_t n = 0;
    uint32_t by_cols = 0;  // token tiles when items are numbered column by column (launcher)
    RowsArgs one{};
    // 2-D waves (mis kernels only; not interleaved frames): the zero frame of the output planes,
    // cleared by a second layer of workgroups (blockIdx.z = 1), or nullptr.
    __half *halo = nullptr;
    uint32_t halo_planes = 0;
    Plane2D plane{};
};

// cols: workgroup columns (index rows x sub-tiles, all waves); ttiles: the most 64-token tiles of
// a wave.  nb: 16-neuron blocks per workgroup (1..4); kw: waves that share a tile's k-steps (1:
// four 64-token tiles per workgroup; 4 or 8: one).  mis: rows at any element offset.
hipError_t launch_mfma_rows(const RowsLaunch &l, uint32_t cols, uint32_t ttiles, uint32_t nb,
                            uint32_t kw, bool mis, hipStream_t stream);

}  // namespace k44dev
