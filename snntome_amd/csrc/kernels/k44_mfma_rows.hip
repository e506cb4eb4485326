// k44_mfma_rows.hip — dense contraction over arbitrary rows on v_mfma_f32_16x16x32_f16.
//
// For waves whose neurons come in clusters of a multiple of 16 that share an index row, whatever
// the row's positions are: scattered synapses, segments that do not fill 32-deep k-steps,
// convolutions over 8 or 16 channels, rows at any element offset.  The row's positions are a
// table of element offsets, so a k-step is any 32 rows; the last one is filled up with zero rows
// (zeros in LDS, not zero weights against data: an infinity elsewhere must not become a NaN).
//
// What bounds it: latency and gathered bytes from L2 (128 per row and 64-token tile), not
// MFMA.  A wave gathers its k-step's 32 rows (8 lanes x 16 bytes each) through registers into a
// private LDS tile, one step ahead of the MFMAs, and takes the B operand with
// ds_read_b64_tr_b16.  KW waves of a workgroup share one tile's k-steps (k = wave, wave + KW,
// ...) and add their accumulators in LDS, in a fixed order: the chain of dependent gathers is
// KW times shorter and no partial sums leave the workgroup.  KW = 1 gives each of 4 waves a
// 64-token tile of its own (same A fragments through L1) once there are enough tiles.
// The token tiles of one neuron tile share its weights, through one XCD's L2: in grid order when
// the columns are a multiple of 8, else with the items numbered column by column and each XCD
// taking a contiguous run of them.
#include <algorithm>

#include "k44_mfma_rows.hpp"

namespace k44dev {

namespace {
constexpr int PITCH = 72;                       // halves per LDS row: 64 tokens + 16-byte skew
constexpr int XS_BYTES = 32 * PITCH * 2;        // one wave's k-step
constexpr int RP = 68;                          // floats per neuron of the transposed sums
static_assert(XS_BYTES >= 16 * RP * 4, "a wave's k-step region holds 16 neurons' sums");

__device__ __forceinline__ bool rows_stored(const RowsArgs &a, uint32_t tile, uint32_t t) {
    if (!a.mask_w) return true;
    const uint32_t rel = 64u * (tile % a.mask_tpf) + t;
    const uint32_t row = rel / a.mask_wpad;
    return row < a.mask_h && rel - row * a.mask_wpad < a.mask_w;
}

// Epilogue of 8 consecutive tokens of neuron j: bias, activation, residual, fp16 (RNE) store.
template <int ACT>
__device__ __forceinline__ void rows_store8(const RowsArgs &a, float (&v)[8], uint32_t j,
                                            uint32_t tile, uint32_t t0, uint64_t ty) {
    typedef unsigned int u2_t __attribute__((ext_vector_type(2)));
    const uint64_t oj = a.cmap ? (uint64_t)a.cmap[j] : (uint64_t)j;
    if (a.cmap && oj == K44_CMAP_EMPTY) return;
    const float b = a.bias ? __half2float(a.bias[j]) : 0.0f;
    const uint64_t o = oj * a.out_stride + ty + t0;
    __half r[8], out[8];
    if (a.R) {
        if (a.vec == 8u) {
            *reinterpret_cast<u4_t *>(r) = *reinterpret_cast<const u4_t *>(a.R + o);
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                r[i] = rows_stored(a, tile, t0 + i) ? a.R[o + i] : __half(0.0f);
        }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float x = v[i] + b, rv = a.R ? __half2float(r[i]) : 0.0f;
        out[i] = __float2half_rn(a.cmap ? act_c<ACT>(x + rv) : act_c<ACT>(x) + rv);
    }
    if (a.vec == 8u) {
        *reinterpret_cast<u4_t *>(a.Y + o) = *reinterpret_cast<const u4_t *>(out);
    } else if (a.vec == 4u && !a.mask_w) {
        reinterpret_cast<u2_t *>(a.Y + o)[0] = reinterpret_cast<const u2_t *>(out)[0];
        reinterpret_cast<u2_t *>(a.Y + o)[1] = reinterpret_cast<const u2_t *>(out)[1];
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (rows_stored(a, tile, t0 + i)) a.Y[o + i] = out[i];
    }
}

// One wave's own tile, 16 neurons at a time through its LDS region.
template <int NB, int ACT>
__device__ __forceinline__ void rows_finish1(const RowsArgs &a, const f4_t (&acc)[NB][4], float *ws,
                                             int lane, uint32_t j0, uint32_t tile, uint64_t ty) {
    const int g = lane >> 4, c = lane & 15;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int tb = 0; tb < 4; ++tb) ws[(4 * g + i) * RP + 16 * tb + c] = acc[nb][tb][i];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int n = 8 * q + (lane >> 3), t0 = 8 * (lane & 7);
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = ws[n * RP + t0 + e];
            rows_store8<ACT>(a, v, j0 + 16u * nb + (uint32_t)n, tile, (uint32_t)t0, ty);
        }
    }
}

// The workgroup's four partial sums of every (neuron, 8-token chunk), in slot order.
template <int NB, int NW, int ACT>
__device__ __forceinline__ void rows_finish(const RowsArgs &a, const float *red, int tid,
                                            uint32_t j0, uint32_t tile, uint64_t ty) {
    for (int u = tid; u < NB * 128; u += 64 * NW) {
        const int n = u >> 3, t0 = 8 * (u & 7);
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = red[n * RP + t0 + e];
#pragma unroll
        for (int s = 1; s < 4; ++s)
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] += red[(s * NB * 16 + n) * RP + t0 + e];
        rows_store8<ACT>(a, v, j0 + (uint32_t)n, tile, (uint32_t)t0, ty);
    }
}
// Zero frame of the output planes (not interleaved): a wavefront per plane row, all of the rows
// above and below the image, the columns beside it otherwise.  As a second layer of the
// convolution's own workgroups instead of a kernel after it (3.75 us each, six in an image block:
// 89.5 us of device time, 75.2 so; 48 channels of 320 x 320 226 and 199): the tiles store image pixels only, so the two never meet.
__device__ __forceinline__ void clear_halo(__half *base, uint32_t planes, const Plane2D &p,
                                           uint32_t wave, uint32_t waves, uint32_t lane) {
    const uint32_t rows = ((uint32_t)p.single_stride + p.W_pad - 1u) / p.W_pad;
    for (uint32_t it = wave; it < planes * rows; it += waves) {
        const uint32_t pl = it / rows, row = it - pl * rows;
        const uint32_t c = pl / p.frames, f = pl - c * p.frames;
        const uint32_t e0 = row * p.W_pad, w = min(p.W_pad, (uint32_t)p.single_stride - e0);
        const bool inner = row >= 1u && row <= p.H;
        __half *r = base + (uint64_t)c * p.channel_stride + (uint64_t)f * p.single_stride + e0;
        for (uint32_t q = lane; q < w - (inner ? min(p.W, w - 4u) : 0u); q += 64u)
            r[inner && q >= 4u ? q + p.W : q] = __float2half_rn(0.0f);
    }
}
}  // namespace

template <int NB, int KW, bool MIS>
__global__ __launch_bounds__(64 * (KW == 1 ? 4 : KW)) void k44_mfma_rows_kernel(RowsLaunch l) {
    constexpr int NW = KW == 1 ? 4 : KW;
    constexpr int SLOTS = 4;                       // partial sums met in LDS at a time
    constexpr int RED = KW == 1 ? 0 : SLOTS * NB * 16 * RP * 4;
    constexpr int SMEM = NW * XS_BYTES > RED ? NW * XS_BYTES : RED;
    __shared__ __attribute__((aligned(16))) char smem[SMEM];
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if constexpr (MIS) {
        if (blockIdx.z) {
            clear_halo(l.halo, l.halo_planes, l.plane,
                       (blockIdx.y * gridDim.x + blockIdx.x) * NW + (uint32_t)wave,
                       gridDim.x * gridDim.y * NW, (uint32_t)lane);
            return;
        }
    }
    uint32_t col = blockIdx.x, ty0 = blockIdx.y;
    if (l.by_cols) {
        const uint32_t item = xcd_contiguous(blockIdx.x, gridDim.x);
        col = item / l.by_cols;
        ty0 = item - col * l.by_cols;
    }
    RowsArgs a = l.one;
    if (l.n) {
        const kconst_u32 *start = (const kconst_u32 *)l.start;
        uint32_t w = 0;
        while (w + 1u < l.n && col >= start[w + 1u]) ++w;
        col -= start[w];
        a = l.waves[w];
    }
    const uint32_t tile = KW == 1 ? ty0 * 4u + (uint32_t)wave : ty0;
    if (tile >= a.ttiles) return;  // whole workgroup, or a wave of one without barriers (KW = 1)
    const uint32_t row = col / a.subs, blk = (col - row * a.subs) * NB;
    const uint32_t k0 = KW == 1 ? 0u : (uint32_t)wave;
    _Float16(*xs)[PITCH] = reinterpret_cast<_Float16(*)[PITCH]>(smem + wave * XS_BYTES);

    const int gr = lane >> 3, gc = (lane & 7) * 8;  // gather: rows 4 gr .. +3, tokens gc .. +7
    const u4_t *roff = reinterpret_cast<const u4_t *>(a.roff + (uint64_t)row * a.ksteps * 32u) + gr;
    const h8_t *wf = reinterpret_cast<const h8_t *>(a.Wf) +
                     ((uint64_t)row * a.ksteps * a.blocks + blk) * 64u + lane;
    const uint32_t tx = (a.tile_x ? a.tile_x[tile] : 64u * tile) + (uint32_t)gc;
    const __half *xt = a.X + tx;
    // MIS: element offset of the lane's tokens past the 16-byte boundary below them
    const uint32_t xmis = MIS ? (uint32_t)((reinterpret_cast<uintptr_t>(xt) >> 1) & 7u) : 0u;

    f4_t acc[NB][4];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int tb = 0; tb < 4; ++tb) acc[nb][tb] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};

    u4_t xr[4], xh[MIS ? 4 : 1];
    uint32_t xm[MIS ? 4 : 1];
    h8_t ar[NB];
    auto load_x = [&](const u4_t &ro) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (MIS) {
                xm[i] = (ro[i] + xmis) & 7u;
                const u4_t *p = reinterpret_cast<const u4_t *>(xt + ro[i] - xm[i]);
                xr[i] = p[0];
                xh[i] = p[1];
            } else {
                xr[i] = *reinterpret_cast<const u4_t *>(xt + ro[i]);
            }
        }
    };
    auto load_a = [&](uint32_t ks) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) ar[nb] = wf[((uint64_t)ks * a.blocks + nb) * 64u];
    };
    const int tr_row = 8 * (lane >> 4) + ((lane & 15) >> 2), tr_col = 4 * (lane & 3);
    if (k0 < a.ksteps) {
        u4_t rn = roff[(uint64_t)k0 * 8u];
        load_a(k0);
        load_x(rn);
        rn = roff[(uint64_t)min(k0 + KW, a.ksteps - 1u) * 8u];
        for (uint32_t ks = k0; ks < a.ksteps; ks += KW) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                u4_t v = xr[i];
                if constexpr (MIS) v = shift_elems(xr[i], xh[i], xm[i]);
                if (32u * ks + 4u * (uint32_t)gr + i >= a.B) v = u4_t{0u, 0u, 0u, 0u};
                *reinterpret_cast<u4_t *>(&xs[4 * gr + i][gc]) = v;
            }
            h8_t af[NB];
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) af[nb] = ar[nb];
            // Next step in flight (past the end: the last step again, unused).  Two steps in
            // flight need 184 registers instead of 128 and were slower for it (4,096 x 512
            // scattered 7.0 us instead of 6.1, a dense block over 512 tokens 67 instead of 58).
            load_a(min(ks + KW, a.ksteps - 1u));
            load_x(rn);
            rn = roff[(uint64_t)min(ks + 2u * KW, a.ksteps - 1u) * 8u];
            // KW = 1: or the compiler sinks these loads to their use (a dense block over 4,096 tokens
            // 273 us, 258 so; with more waves per tile it costs up to 3 %)
            if constexpr (KW == 1) asm volatile("" ::: "memory");
#pragma unroll
            for (int tb = 0; tb < 4; ++tb) {
                const _Float16 *p = &xs[tr_row][tr_col + 16 * tb];
                const h4_t lo = lds_read_tr16(p);
                const h4_t hi = lds_read_tr16(p + 4 * PITCH);
                const h8_t b = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
                    acc[nb][tb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[nb], b, acc[nb][tb], 0, 0, 0);
            }
        }
    }

    const uint32_t j0 = (row * a.blocks + blk) * 16u;
    const uint64_t ty = a.tile_y ? (uint64_t)a.tile_y[tile] : 64ull * tile;
    const int g = lane >> 4, c = lane & 15;
    if constexpr (KW == 1) {
        float *ws = reinterpret_cast<float *>(smem + wave * XS_BYTES);
        K44_WITH_ACT(a.act, rows_finish1<NB, A_>(a, acc, ws, lane, j0, tile, ty))
        return;
    }
    __syncthreads();  // every wave is done with its k-step region
    if constexpr (KW == 8) {  // waves 4..7 add theirs to waves 0..3
        f4_t *ex = reinterpret_cast<f4_t *>(smem) + (wave & 3) * NB * 256 + lane;
        if (wave >= 4)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int tb = 0; tb < 4; ++tb) ex[(nb * 4 + tb) * 64] = acc[nb][tb];
        __syncthreads();
        if (wave < 4)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int tb = 0; tb < 4; ++tb) acc[nb][tb] += ex[(nb * 4 + tb) * 64];
        __syncthreads();
    }
    float *red = reinterpret_cast<float *>(smem);
    if (wave < SLOTS) {
        float *ws = red + wave * NB * 16 * RP;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int tb = 0; tb < 4; ++tb)
                    ws[(16 * nb + 4 * g + i) * RP + 16 * tb + c] = acc[nb][tb][i];
    }
    __syncthreads();
    K44_WITH_ACT(a.act, rows_finish<NB, NW, A_>(a, red, tid, j0, tile, ty))
}

template <int NB, int KW>
static hipError_t launch_rows_kw(RowsLaunch l, uint32_t cols, uint32_t ttiles, bool mis,
                                 hipStream_t stream) {
    const uint32_t tys = KW == 1 ? (ttiles + 3u) / 4u : ttiles;
    l.by_cols = cols % 8u != 0u && tys > 1u && cols > 8u ? tys : 0u;
    if (l.halo && !mis) return hipErrorInvalidValue;
    const uint32_t layers = l.halo ? 2u : 1u;
    const dim3 grid = l.by_cols ? dim3(cols * tys, 1u, layers) : dim3(cols, tys, layers);
    const dim3 block(64u * (KW == 1 ? 4u : KW), 1u, 1u);
    if (mis)
        hipLaunchKernelGGL((k44_mfma_rows_kernel<NB, KW, true>), grid, block, 0, stream, l);
    else
        hipLaunchKernelGGL((k44_mfma_rows_kernel<NB, KW, false>), grid, block, 0, stream, l);
    return hipGetLastError();
}

template <int NB>
static hipError_t launch_rows_nb(const RowsLaunch &l, uint32_t cols, uint32_t ttiles, uint32_t kw,
                                 bool mis, hipStream_t stream) {
    if (kw == 8u) return launch_rows_kw<NB, 8>(l, cols, ttiles, mis, stream);
    if (kw == 4u) return launch_rows_kw<NB, 4>(l, cols, ttiles, mis, stream);
    if (kw == 1u) return launch_rows_kw<NB, 1>(l, cols, ttiles, mis, stream);
    return hipErrorInvalidValue;
}

hipError_t launch_mfma_rows(const RowsLaunch &l, uint32_t cols, uint32_t ttiles, uint32_t nb,
                            uint32_t kw, bool mis, hipStream_t stream) {
    if (cols == 0u || ttiles == 0u) return hipSuccess;
    if ((uint64_t)cols * ttiles > 0x7fffffffull || (kw == 1u ? (ttiles + 3u) / 4u : ttiles) > 65535u)
        return hipErrorInvalidValue;
    switch (nb) {
    case 1u: return launch_rows_nb<1>(l, cols, ttiles, kw, mis, stream);
    case 2u: return launch_rows_nb<2>(l, cols, ttiles, kw, mis, stream);
    case 3u: return launch_rows_nb<3>(l, cols, ttiles, kw, mis, stream);
    case 4u: return launch_rows_nb<4>(l, cols, ttiles, kw, mis, stream);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace k44dev
