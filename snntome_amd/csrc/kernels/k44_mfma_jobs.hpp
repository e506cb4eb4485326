// k44_mfma_jobs.hpp — private dendritic segments on MFMA (see k44_mfma_jobs.hip).
#pragma once
#include "k44_mfma_tile.hpp"

namespace k44dev {

constexpr uint32_t K44_JOB_BLOCKS = 2u;  // 16-job blocks per tile

struct JobArgs {
    const __half *X;        // canvas + the wave's lowest row offset
    const uint32_t *roff;   // [tiles][32 ksteps] element offset of every window row from X
    const __half *Wf;       // A fragments [tile][k-step][2][lane][8], zero outside a job's segment
    const uint32_t *jmap;   // [tiles][32] partial row of each job (neuron * K + segment), ~0 none
    const uint32_t *koff;   // [tiles][32] window row of each job's first position
    float *part;            // [neurons * K][tokens]
    uint32_t ksteps, tiles, ttiles, tokens, S;
};

struct JobReduceArgs {
    const float *part;
    const __half *bias;     // [cout] or nullptr
    const uint16_t *cmap;   // [cout] or nullptr
    __half *Y;
    const __half *R;        // or nullptr
    uint64_t out_stride;
    uint32_t cout, K, tokens;
    int act;                // (output and residual rows on the 8-byte grid)
};

// Fills part with every job's sums over its segment.
hipError_t launch_mfma_jobs(const JobArgs &a, hipStream_t stream);
// Adds each neuron's K sums in segment order and runs the epilogue.
hipError_t launch_jobs_reduce(const JobReduceArgs &a, hipStream_t stream);

}  // namespace k44dev
