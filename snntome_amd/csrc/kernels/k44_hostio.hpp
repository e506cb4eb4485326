// k44_hostio.hpp — kernels that move plan inputs and outputs between host memory and the canvas.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace k44dev {

// Where element (channel, y, x) of frame 0 sits in a tensor region (K44ResDesc::canvas_offset):
// channel * channel_stride + (y + y0) * row_stride + (x + x0) * x_step.  Token rows have
// row_stride 0: H rows of a channel share its one row of tokens (the last one given is kept).
struct FrameLayout {
    uint32_t H, W, row_stride, x_step, x0, y0;
    uint64_t channel_stride;
};

// region[0 .. channels * channel_stride): frame 0 from `in` ([channels][H][W] fp32, of which n_in
// elements exist; the rest reads as zero) rounded to fp16 as the plan compiler rounds, every
// other element (halos, padding, further frames) zero.
hipError_t launch_import_f32(uint16_t *region, const float *in, uint64_t n_in, uint32_t channels,
                             const FrameLayout &L, hipStream_t stream);

// dst[0 .. n) = elements [first, first + n) of frame 0 ([channels][H][W] order) as fp32.
// dst may be page-locked host memory.
hipError_t launch_export_f32(float *dst, const uint16_t *region, uint64_t first, uint64_t n,
                             const FrameLayout &L, hipStream_t stream);

// dst[0 .. n) = elements [first, first + n) of [rows][cols], row r at src + r * row_stride,
// packed.  dst may be page-locked host memory.
hipError_t launch_pack_rows(uint16_t *dst, const uint16_t *src, uint64_t first, uint64_t n,
                            uint64_t row_stride, uint64_t cols, hipStream_t stream);

}  // namespace k44dev
