// k44_hostio.hip — host fp32 <-> canvas fp16 (see k44_hostio.hpp).
//
// Bound by the host link: 4 bytes per element over PCIe (about 55 GB/s on MI355X), against
// about 5 us of device work per million elements.  The conversions replace a scalar host loop
// over every element (1-2 ns per element and direction, on top of the same transfers): a dense
// block over 200 tokens (205 k elements each way) 642 -> 266 us per call, an image block on a
// 32 x 160 x 160 input (819 k in, 410 k out) 1952 -> 472 us.
#include "k44_hostio.hpp"

#include "k44_pack_index.hpp"

#include <hip/hip_fp16.h>

#include <algorithm>

namespace k44dev {

typedef unsigned short us8 __attribute__((ext_vector_type(8)));

// The plan compiler's rounding (RNE; NaN keeps its upper payload bits and sets bit 0).
__device__ __forceinline__ unsigned short half_bits(float f) {
    const uint32_t u = __float_as_uint(f), mag = u & 0x7fffffffu;
    if (mag > 0x7f800000u)
        return (unsigned short)(((u >> 16) & 0x8000u) | 0x7c00u | ((mag & 0x7fffffu) >> 13) | 1u);
    return __half_as_ushort(__float2half_rn(f));
}

// Exact, NaN payloads kept (the conversion instruction would quiet a signalling NaN).
__device__ __forceinline__ float half_value(unsigned short h) {
    if ((h & 0x7c00u) == 0x7c00u)
        return __uint_as_float(((uint32_t)(h & 0x8000u) << 16) | 0x7f800000u |
                               ((uint32_t)(h & 0x3ffu) << 13));
    return __half2float(__ushort_as_half(h));
}

// Thread = 8 consecutive region elements of one channel.  VEC: region rows of channels are 8
// elements aligned (every layout of the compiler), one 16-byte store.
template <bool VEC>
__global__ __launch_bounds__(256) void k44_import_f32_kernel(uint16_t *region, const float *in,
                                                             uint64_t n_in, FrameLayout L) {
    const uint64_t e0 = ((uint64_t)blockIdx.x * 256u + threadIdx.x) * 8u;
    if (e0 >= L.channel_stride) return;
    const uint64_t src0 = (uint64_t)blockIdx.y * L.H * L.W;
    uint16_t *dst = region + (uint64_t)blockIdx.y * L.channel_stride + e0;
    us8 v;
    if (L.row_stride == 0u) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            unsigned short h = 0u;
            for (uint32_t y = L.H; e0 + i < L.W && y > 0u; --y) {
                const uint64_t s = src0 + (uint64_t)(y - 1u) * L.W + e0 + i;
                if (s >= n_in) continue;
                h = half_bits(in[s]);
                break;
            }
            v[i] = h;
        }
    }
    uint64_t row = L.row_stride ? e0 / L.row_stride : 0u;
    uint32_t col = (uint32_t)(e0 - row * L.row_stride);
#pragma unroll
    for (int i = 0; i < 8 && L.row_stride; ++i) {
        unsigned short h = 0u;
        const uint32_t xs = col / L.x_step;
        if (row >= L.y0 && row - L.y0 < L.H && xs >= L.x0 && xs - L.x0 < L.W &&
            col - xs * L.x_step == 0u) {
            const uint64_t s = src0 + (row - L.y0) * L.W + (xs - L.x0);
            if (s < n_in) h = half_bits(in[s]);
        }
        v[i] = h;
        if (++col == L.row_stride) {
            col = 0u;
            ++row;
        }
    }
    if constexpr (VEC) {
        *reinterpret_cast<us8 *>(dst) = v;
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (e0 + i < L.channel_stride) dst[i] = v[i];
    }
}

hipError_t launch_import_f32(uint16_t *region, const float *in, uint64_t n_in, uint32_t channels,
                             const FrameLayout &L, hipStream_t stream) {
    const uint64_t bx = (L.channel_stride + 2047u) / 2048u;
    if (bx > 0x7fffffffull) return hipErrorInvalidValue;
    const bool vec = L.channel_stride % 8u == 0u && reinterpret_cast<uintptr_t>(region) % 16u == 0u;
    for (uint32_t c = 0; c < channels; c += 65535u) {  // grid.y limit
        const uint32_t nc = std::min(65535u, channels - c);
        const uint64_t skip = (uint64_t)c * L.H * L.W;
        const dim3 grid((uint32_t)bx, nc, 1u);
        uint16_t *r = region + (uint64_t)c * L.channel_stride;
        const uint64_t n = n_in > skip ? n_in - skip : 0u;
        if (vec)
            hipLaunchKernelGGL(k44_import_f32_kernel<true>, grid, dim3(256), 0, stream, r, in + skip, n, L);
        else
            hipLaunchKernelGGL(k44_import_f32_kernel<false>, grid, dim3(256), 0, stream, r, in + skip, n, L);
    }
    return hipGetLastError();
}

// Thread = 4 consecutive output elements (one 16-byte store: full lines of host memory per wave).
__global__ __launch_bounds__(256) void k44_export_f32_kernel(float *dst, const uint16_t *region,
                                                             uint64_t first, uint64_t n,
                                                             FrameLayout L, uint32_t vec) {
    for (uint64_t q = (uint64_t)blockIdx.x * 256u + threadIdx.x; q * 4u < n;
         q += (uint64_t)gridDim.x * 256u) {
        const uint64_t i0 = first + q * 4u, line = i0 / L.W;
        uint32_t x = (uint32_t)(i0 - line * L.W);
        uint64_t ch = line / L.H;
        uint32_t y = (uint32_t)(line - ch * L.H);
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        float *vp = &v.x;
        const uint32_t cnt = n - q * 4u < 4u ? (uint32_t)(n - q * 4u) : 4u;
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i) {
            if (i < cnt)
                vp[i] = half_value(region[ch * L.channel_stride +
                                          (uint64_t)(y + L.y0) * L.row_stride +
                                          (uint64_t)(x + L.x0) * L.x_step]);
            if (++x == L.W) {
                x = 0u;
                if (++y == L.H) {
                    y = 0u;
                    ++ch;
                }
            }
        }
        if (vec && cnt == 4u) {
            *reinterpret_cast<float4 *>(dst + q * 4u) = v;
        } else {
#pragma unroll
            for (uint32_t i = 0; i < 4u; ++i)
                if (i < cnt) dst[q * 4u + i] = vp[i];
        }
    }
}

hipError_t launch_export_f32(float *dst, const uint16_t *region, uint64_t first, uint64_t n,
                             const FrameLayout &L, hipStream_t stream) {
    if (n == 0u) return hipSuccess;
    const uint64_t blocks = std::min<uint64_t>((n + 1023u) / 1024u, 4096u);
    hipLaunchKernelGGL(k44_export_f32_kernel, dim3((uint32_t)blocks), dim3(256), 0, stream, dst,
                       region, first, n, L,
                       reinterpret_cast<uintptr_t>(dst) % 16u == 0u ? 1u : 0u);
    return hipGetLastError();
}

// Thread = 8 consecutive packed elements.  VEC: rows and both ends on the 16-byte grid.
template <bool VEC, typename I>
__global__ __launch_bounds__(256) void k44_pack_rows_kernel(uint16_t *dst, const uint16_t *src,
                                                            I first, I n, uint64_t row_stride,
                                                            I cols) {
    for (I q = ((I)blockIdx.x * 256u + threadIdx.x) * 8u; q < n; q += (I)gridDim.x * 2048u) {
        RowCol<I> at = row_col<I>(first + q, cols);
        I &c = at.c;
        const uint16_t *p = src + (uint64_t)at.r * row_stride;
        if constexpr (VEC) {
            *reinterpret_cast<us8 *>(dst + q) = *reinterpret_cast<const us8 *>(p + c);
        } else {
            us8 v;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                v[i] = q + i < n ? p[c] : (unsigned short)0u;
                if (++c == cols) {
                    c = 0;
                    p += q + i + 1u < n ? row_stride : 0u;
                }
            }
            if (q + 8u <= n && reinterpret_cast<uintptr_t>(dst + q) % 16u == 0u) {
                *reinterpret_cast<us8 *>(dst + q) = v;
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (q + i < n) dst[q + i] = v[i];
            }
        }
    }
}

template <bool VEC>
static void pack_rows(uint16_t *dst, const uint16_t *src, uint64_t first, uint64_t n,
                      uint64_t row_stride, uint64_t cols, hipStream_t stream) {
    const dim3 grid((uint32_t)std::min<uint64_t>((n + 2047u) / 2048u, 2048u));
    with_pack_index(first, n, cols, [&](auto f, auto k, auto w) {
        hipLaunchKernelGGL((k44_pack_rows_kernel<VEC, decltype(f)>), grid, dim3(256), 0, stream, dst,
                           src, f, k, row_stride, w);
    });
}

hipError_t launch_pack_rows(uint16_t *dst, const uint16_t *src, uint64_t first, uint64_t n,
                            uint64_t row_stride, uint64_t cols, hipStream_t stream) {
    if (n == 0u) return hipSuccess;
    const bool vec = (first | n | row_stride | cols) % 8u == 0u &&
                     (reinterpret_cast<uintptr_t>(dst) | reinterpret_cast<uintptr_t>(src)) % 16u == 0u;
    if (vec)
        pack_rows<true>(dst, src, first, n, row_stride, cols, stream);
    else
        pack_rows<false>(dst, src, first, n, row_stride, cols, stream);
    return hipGetLastError();
}

}  // namespace k44dev
