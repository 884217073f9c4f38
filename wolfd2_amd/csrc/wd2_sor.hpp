// wd2_sor.hpp -- stopping test shared by the temporally blocked red-black
// SOR kernels (FP64 and mixed precision).
//
// The stopping test of sweep m is max|s| < sortol over the whole grid
// (pressure.f:534), which holds exactly when it holds on every tile: each tile
// publishes a bit mask of its sweeps whose owned-point maximum is below
// sortol, and the test of a launch is the AND of the masks.
#pragma once

#include "wd2_dev.hpp"

namespace wd2 {

// AND of the ntiles masks (every thread gets it): a reduction by lane moves
// within a wavefront, one LDS exchange across them.
__device__ inline unsigned tiled_mask(const unsigned *__restrict__ masks, int ntiles, unsigned *sh) {
    int m = ~0;
    for (int k = threadIdx.x; k < ntiles; k += blockDim.x) m &= (int)masks[k];
    m &= __builtin_amdgcn_update_dpp(~0, m, 0x111, 0xf, 0xf, false);   // row_shr:1, 2, 4, 8
    m &= __builtin_amdgcn_update_dpp(~0, m, 0x112, 0xf, 0xf, false);
    m &= __builtin_amdgcn_update_dpp(~0, m, 0x114, 0xf, 0xf, false);
    m &= __builtin_amdgcn_update_dpp(~0, m, 0x118, 0xf, 0xf, false);
    m &= __builtin_amdgcn_update_dpp(~0, m, 0x142, 0xa, 0xf, false);   // row_bcast:15
    m &= __builtin_amdgcn_update_dpp(~0, m, 0x143, 0xc, 0xf, false);   // row_bcast:31
    if ((threadIdx.x & 63) == 63) sh[threadIdx.x >> 6] = (unsigned)m;
    __syncthreads();
    unsigned r = ~0u;
    for (int w = 0; w < (int)(blockDim.x >> 6); w++) r &= sh[w];
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(r);
}

// 1-based sweep of a launch (nsweep <= 32 sweeps after sweep m0) after which
// the solve stops, or 0; *conv tells whether it stopped converged.
__device__ inline int tiled_stop(unsigned mask, int nsweep, int m0, int msorit, int *conv) {
    mask &= nsweep < 32 ? (1u << nsweep) - 1u : ~0u;
    if (m0 == 0) mask &= ~1u;                    // the first sweep of a solve never stops it
    const int first = mask ? __ffs(mask) : 33;   // first sweep below the tolerance
    const int last = max(msorit - m0, 1);        // the sweep that reaches msorit
    *conv = first <= last;
    const int k = min(first, last);
    return k <= nsweep ? k : 0;
}

}  // namespace wd2
