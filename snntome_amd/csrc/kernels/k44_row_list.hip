// k44_row_list.hip — one neuron's scattered positions at a time, on the VALU.
//
// For waves whose neurons share index rows with fewer than 16 others (no matrix tile) and whose
// positions form short segments or none: the segment gathers fill batches of 16 rows per segment, of
// which a single position uses one.  Here a wave walks a table of row offsets 32 at a time: 8 lanes
// x 16 bytes per row, 4 loads in flight per lane and the offsets of the next step with them; the 8
// row groups meet by shuffles.  Bound by the gathered bytes from L2 (128 per position and 64-token
// tile, 10 to 11 TB/s).  The tiles of one token range run together: their rows stay in L2 while
// every neuron passes.  4,096 neurons x 256 positions over 64 tokens 137 -> 13.4 us, over 256
// tokens 251 -> 48, 256 x 250 over 10 tokens 76 -> 3.9.
#include "k44_row_list.hpp"

namespace k44dev {

template <int KW>
__global__ __launch_bounds__(256) void k44_row_list_kernel(RowListArgs a) {
    __shared__ float red[KW == 1 ? 1 : 4][KW == 1 ? 1 : 64];
    const int lane = (int)(threadIdx.x & 63u);
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t j = KW == 1 ? blockIdx.x * 4u + wave : blockIdx.x;
    if (j >= a.cout) return;  // (KW = 4: whole workgroups)
    const uint32_t k0 = KW == 1 ? 0u : wave, tok0 = blockIdx.y * 64u;
    const int gr = lane >> 3, gc = (lane & 7) * 8;  // rows 4 gr .. +3 of a step, tokens gc .. +7
    const u4_t *roff = reinterpret_cast<const u4_t *>(a.roff + (uint64_t)(j / a.cluster) * a.steps * 32u) + gr;
    const h4_t *wt = reinterpret_cast<const h4_t *>(a.W + (uint64_t)j * a.steps * 32u) + gr;
    const __half *xt = a.X + tok0 + (uint32_t)gc;
    float acc[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    if (k0 < a.steps) {
        u4_t ro = roff[(uint64_t)k0 * 8u];
        h4_t w = wt[(uint64_t)k0 * 8u];
        for (uint32_t ks = k0; ks < a.steps; ks += KW) {
            h8_t x[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = *reinterpret_cast<const h8_t *>(xt + ro[i]);
            const h4_t wc = w;
            const uint32_t kn = min(ks + KW, a.steps - 1u);
            ro = roff[(uint64_t)kn * 8u];
            w = wt[(uint64_t)kn * 8u];
            asm volatile("" ::: "memory");  // or the compiler sinks the next step's table loads
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                // past the row: nothing is added, whatever the repeated last position holds
                if (32u * ks + 4u * (uint32_t)gr + i >= a.B) x[i] = h8_t{};
#pragma unroll
                for (int e = 0; e < 8; ++e) acc[e] = fmaf((float)wc[i], (float)x[i][e], acc[e]);
            }
        }
    }
#pragma unroll
    for (int s = 8; s < 64; s *= 2)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += __shfl_xor(acc[e], s);
    if constexpr (KW == 4) {
        if (gr == 0)
#pragma unroll
            for (int e = 0; e < 8; ++e) red[wave][gc + e] = acc[e];
        __syncthreads();
        if (wave != 0u || gr != 0) return;
#pragma unroll
        for (int e = 0; e < 8; ++e)
            acc[e] = ((red[0][gc + e] + red[1][gc + e]) + red[2][gc + e]) + red[3][gc + e];
    }
    if (gr != 0) return;
    const uint64_t oj = a.cmap ? (uint64_t)a.cmap[j] : (uint64_t)j;
    if (a.cmap && oj == K44_CMAP_EMPTY) return;
    const float b = a.bias ? __half2float(a.bias[j]) : 0.0f;
    const uint64_t o = oj * a.out_stride + tok0 + (uint32_t)gc;
    __half r[8], out[8];
    if (a.R) *reinterpret_cast<u4_t *>(r) = *reinterpret_cast<const u4_t *>(a.R + o);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float v = acc[e] + b, rv = a.R ? __half2float(r[e]) : 0.0f;
        out[e] = __float2half_rn(a.cmap ? apply_act(v + rv, a.act) : apply_act(v, a.act) + rv);
    }
    *reinterpret_cast<u4_t *>(a.Y + o) = *reinterpret_cast<const u4_t *>(out);
}

hipError_t launch_row_list(const RowListArgs &a, uint32_t kw, hipStream_t stream) {
    if (a.cout == 0u || a.ttiles == 0u) return hipSuccess;
    if (a.ttiles > 65535u || a.steps == 0u) return hipErrorInvalidValue;
    if (kw == 4u)
        hipLaunchKernelGGL(k44_row_list_kernel<4>, dim3(a.cout, a.ttiles), dim3(256), 0, stream, a);
    else
        hipLaunchKernelGGL(k44_row_list_kernel<1>, dim3((a.cout + 3u) / 4u, a.ttiles), dim3(256), 0,
                           stream, a);
    return hipGetLastError();
}

}  // namespace k44dev
