// k44_mfma_jobs.hip — neurons with dendritic segments of their own, on v_mfma_f32_16x16x32_f16.
//
// A neuron that shares its index row with no other has no dense contraction, and the VALU gathers
// read every segment once per neuron: 2.15 GB from L2 for 4,096 neurons x 16 segments x 128
// positions over 128 tokens, at 24 TB/s and with a fused multiply-add per product.  But segments
// of different neurons overlap: sorted by address, the 65,536 (neuron, segment) jobs of that wave
// over 36,864 positions start less than one position apart.  So 32 consecutive jobs make a tile
// over a window of 32-position k-steps that holds all their segments, with zero weights outside
// each job's own: the window's rows are read once for all of them (50 MB), and the products run on
// the matrix cores.  Every job's fp32 sums go to a row of their own, and a second kernel adds a
// neuron's K rows in segment order and runs the epilogue (34 MB written and read).
// That wave: 87 us as gathers, 25 as job tiles; 8,192 x 12 x 128 over 256 tokens of 130,000 rows
// 769 and 58; 4,096 x 8 x 64 over 64 tokens 19.1 and 12.1.  Tiles of 64 jobs, with half the
// windows but twice the zero products, were never faster (31, 61 and 12.5 us).
// Bound now by the gather's latency (a k-step's rows come one step ahead) and the sums' traffic.
//
// Zero weights must not meet infinities or NaNs of rows that a job does not read (0 * inf is
// NaN): a wave that gathers a non-finite value runs its tile again with those values taken out of the
// products (as zeros) and counted instead: per job and token, how many lie in the job's own segment,
// how many are infinities that meet a weight other than zero, and the sum of those products' signs, each
// one more matrix product of zeros and ones.  All infinite with one sign: that infinity is added,
// else NaN, as the products themselves would give (weights are finite: the host sends others to
// the gathers).  Window rows that no job of the tile reads are never loaded (their table entries
// repeat a row that is).  The wave of 4,096 x 16 x 128 with one infinity among its 36,864
// positions: 33 us, with 1,000 of them 38 (25 without; 88 as gathers, 201 and 325 job by job on the VALU).
#include "k44_mfma_jobs.hpp"

#include <algorithm>

#include "k44_mfma_rows.hpp"

namespace k44dev {

namespace {
constexpr int PITCH = 72;   // halves per LDS row: 64 tokens + 16-byte skew
constexpr int RP = 68;      // floats per job of the transposed sums
constexpr int NB = (int)K44_JOB_BLOCKS;
constexpr unsigned short ONE = 0x3c00;  // 1.0 in fp16

typedef unsigned short us8_t __attribute__((ext_vector_type(8)));

// Nonzero iff one of the two halves is infinite or NaN (exponent 31).
__device__ __forceinline__ uint32_t nonfinite2(uint32_t h) {
    return ((h & 0x7c007c00u) + 0x04000400u) & 0x80008000u;
}
}  // namespace

// Wave = one tile x 64 tokens; the token tiles of a job tile are neighbours, and each XCD takes a
// contiguous run of the address-sorted tiles, so a row is fetched into few L2s.
__global__ __launch_bounds__(256, 4) void k44_mfma_jobs_kernel(JobArgs a) {
    __shared__ __attribute__((aligned(16))) _Float16 smem[4][32][PITCH];
    const int lane = (int)(threadIdx.x & 63u);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t item = xcd_contiguous(blockIdx.x, gridDim.x) * 4u + (uint32_t)wave;
    const uint32_t tile = item / a.ttiles, tok0 = (item - tile * a.ttiles) * 64u;
    if (tile >= a.tiles) return;  // (no workgroup barrier in this kernel)
    _Float16(*xs)[PITCH] = smem[wave];
    const int gr = lane >> 3, gc = (lane & 7) * 8;  // gather: rows 4 gr .. +3, tokens gc .. +7
    const u4_t *roff = reinterpret_cast<const u4_t *>(a.roff + (uint64_t)tile * a.ksteps * 32u) + gr;
    const h8_t *wf = reinterpret_cast<const h8_t *>(a.Wf) + (uint64_t)tile * a.ksteps * NB * 64u + lane;
    const __half *xt = a.X + tok0 + (uint32_t)gc;

    f4_t acc[NB][4];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int tb = 0; tb < 4; ++tb) acc[nb][tb] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
    u4_t xr[4];
    h8_t ar[NB];
    uint32_t bad = 0u;
    auto load_x = [&](const u4_t &ro) {
#pragma unroll
        for (int i = 0; i < 4; ++i) xr[i] = *reinterpret_cast<const u4_t *>(xt + ro[i]);
    };
    auto load_a = [&](uint32_t ks) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) ar[nb] = wf[((uint64_t)ks * NB + nb) * 64u];
    };
    const int tr_row = 8 * (lane >> 4) + ((lane & 15) >> 2), tr_col = 4 * (lane & 3);
    const uint32_t last = a.ksteps - 1u;
    u4_t rn = roff[0];
    load_a(0u);
    load_x(rn);
    rn = roff[(uint64_t)min(1u, last) * 8u];
    for (uint32_t ks = 0; ks <= last; ++ks) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            *reinterpret_cast<u4_t *>(&xs[4 * gr + i][gc]) = xr[i];
#pragma unroll
            for (int q = 0; q < 4; ++q) bad |= nonfinite2(xr[i][q]);
        }
        h8_t af[NB];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) af[nb] = ar[nb];
        // next step in flight (past the end: the last step again, unused)
        load_a(min(ks + 1u, last));
        load_x(rn);
        rn = roff[(uint64_t)min(ks + 2u, last) * 8u];
        asm volatile("" ::: "memory");  // or the compiler sinks these loads to where they are used
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

    const uint32_t *jm = a.jmap + (uint64_t)tile * (16u * NB);
    if (__any(bad != 0u)) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int tb = 0; tb < 4; ++tb) acc[nb][tb] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
        uint32_t kn[NB];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) kn[nb] = a.koff[(uint64_t)tile * (16u * NB) + 16u * nb + (lane & 15)];
#pragma unroll 1
        for (uint32_t ks = 0; ks <= last; ++ks) {
            rn = roff[(uint64_t)ks * 8u];
            load_a(ks);
            load_x(rn);
#pragma unroll
            for (int i = 0; i < 4; ++i) *reinterpret_cast<u4_t *>(&xs[4 * gr + i][gc]) = xr[i];
            const uint32_t p0 = 32u * ks + 8u * (uint32_t)(lane >> 4);
#pragma unroll
            for (int tb = 0; tb < 4; ++tb) {
                const _Float16 *p = &xs[tr_row][tr_col + 16 * tb];
                const h4_t lo = lds_read_tr16(p);
                const h4_t hi = lds_read_tr16(p + 4 * PITCH);
                const us8_t x = __builtin_bit_cast(
                    us8_t, (h8_t)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                const us8_t out = (us8_t)((x & 0x7c00) == 0x7c00), inf = (us8_t)((x & 0x7fff) == 0x7c00);
                const h8_t fin = __builtin_bit_cast(h8_t, (us8_t)(x & ~out));
                const h8_t any = __builtin_bit_cast(h8_t, (us8_t)(out & ONE));
                const h8_t one = __builtin_bit_cast(h8_t, (us8_t)(inf & ONE));
                const h8_t sgn = __builtin_bit_cast(h8_t, (us8_t)(inf & (ONE | (x & 0x8000))));
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    f4_t &c = acc[nb][tb];
                    c = __builtin_amdgcn_mfma_f32_16x16x32_f16(ar[nb], fin, c, 0, 0, 0);
                    const us8_t w = __builtin_bit_cast(us8_t, ar[nb]), nz = (us8_t)((w & 0x7fff) != 0);
                    us8_t own;
#pragma unroll
                    for (int e = 0; e < 8; ++e) own[e] = p0 + e - kn[nb] < a.S ? ONE : 0;
                    const f4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
                    const f4_t met = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                        __builtin_bit_cast(h8_t, own), any, zero, 0, 0, 0);
                    const f4_t infs = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                        __builtin_bit_cast(h8_t, (us8_t)(nz & ONE)), one, zero, 0, 0, 0);
                    const f4_t signs = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                        __builtin_bit_cast(h8_t, (us8_t)(nz & (ONE | (w & 0x8000)))), sgn, zero, 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (met[i] != 0.0f)
                            c[i] += infs[i] == met[i] && fabsf(signs[i]) == met[i]
                                        ? copysignf(__builtin_inff(), signs[i])
                                        : __builtin_nanf("");
                }
            }
        }
    }
    float *ws = reinterpret_cast<float *>(smem[wave]);  // 16 jobs at a time
    static_assert(sizeof(smem[0]) >= 16 * RP * 4, "a wave's k-step region holds 16 jobs' sums");
    const int g = lane >> 4, c = lane & 15;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        uint32_t slot[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) slot[q] = jm[16 * nb + 8 * q + (lane >> 3)];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int tb = 0; tb < 4; ++tb) ws[(4 * g + i) * RP + 16 * tb + c] = acc[nb][tb][i];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int n = 8 * q + (lane >> 3), t0 = 8 * (lane & 7);
            const f4_t v0 = *reinterpret_cast<const f4_t *>(&ws[n * RP + t0]);
            const f4_t v1 = *reinterpret_cast<const f4_t *>(&ws[n * RP + t0 + 4]);
            if (slot[q] != 0xffffffffu) {
                f4_t *dst = reinterpret_cast<f4_t *>(a.part + (uint64_t)slot[q] * a.tokens + tok0 + t0);
                dst[0] = v0;
                dst[1] = v1;
            }
        }
    }
}

// Thread = 4 tokens of one neuron: K 16-byte loads, up to 8 in flight.
__global__ __launch_bounds__(256) void k44_jobs_reduce_kernel(JobReduceArgs a) {
    const uint32_t per = a.tokens / 4u;
    const uint64_t q = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    const uint32_t j = (uint32_t)(q / per), t = (uint32_t)(q - (uint64_t)j * per) * 4u;
    if (j >= a.cout) return;
    const f4_t *p = reinterpret_cast<const f4_t *>(a.part + (uint64_t)j * a.K * a.tokens + t);
    const uint64_t oj = a.cmap ? (uint64_t)a.cmap[j] : (uint64_t)j;
    if (a.cmap && oj == K44_CMAP_EMPTY) return;
    const float b = a.bias ? __half2float(a.bias[j]) : 0.0f;
    const uint64_t o = oj * a.out_stride + t;
    __half r[4], out[4];
    if (a.R) *reinterpret_cast<uint2 *>(r) = *reinterpret_cast<const uint2 *>(a.R + o);
    f4_t s = {0.0f, 0.0f, 0.0f, 0.0f};
    uint32_t k = 0;
    for (; k + 8u <= a.K; k += 8u) {
        f4_t v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = p[(uint64_t)(k + u) * per];
#pragma unroll
        for (int u = 0; u < 8; ++u) s += v[u];
    }
    for (; k < a.K; ++k) s += p[(uint64_t)k * per];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float x = s[i] + b, rv = a.R ? __half2float(r[i]) : 0.0f;
        out[i] = __float2half_rn(a.cmap ? apply_act(x + rv, a.act) : apply_act(x, a.act) + rv);
    }
    *reinterpret_cast<uint2 *>(a.Y + o) = *reinterpret_cast<const uint2 *>(out);
}

hipError_t launch_mfma_jobs(const JobArgs &a, hipStream_t stream) {
    const uint64_t items = (uint64_t)a.tiles * a.ttiles;
    if (items == 0u) return hipSuccess;
    if (a.ksteps == 0u || items > 0x3fffffffull) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k44_mfma_jobs_kernel, dim3((uint32_t)((items + 3u) / 4u)), dim3(256), 0, stream,
                       a);
    return hipGetLastError();
}

hipError_t launch_jobs_reduce(const JobReduceArgs &a, hipStream_t stream) {
    const uint64_t n = (uint64_t)a.cout * (a.tokens / 4u);
    if (n == 0u) return hipSuccess;
    if ((n + 255u) / 256u > 0x7fffffffull) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k44_jobs_reduce_kernel, dim3((uint32_t)((n + 255u) / 256u)), dim3(256), 0,
                       stream, a);
    return hipGetLastError();
}

}  // namespace k44dev
