// Launches of the clipping kernels (clip_kernels.hip, compiled in parts) and
// the work-group numbering shared by the kernels.
#pragma once

#include <hip/hip_runtime.h>

#include "common.h"

namespace vgc {

// Work-groups go to the 8 XCDs of the chip in turn; renumber them so that
// each XCD takes one contiguous range of work-groups (cells in Morton order:
// neighbouring cells read the same seeds and tree nodes, from that XCD's L2).
// A bijection of [0, gridDim.x).
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_block() {
    const int nb = gridDim.x, b = blockIdx.x;
    const int q = nb / kXcds, r = nb % kXcds, x = b % kXcds;
    return x * q + (x < r ? x : r) + b / kXcds;
}

// FP64 signs or exact ones, neighbours gathered in the kernel or read from
// lists; S: 64-corner slots per lane; waves: wavefronts per work-group (S = 1)
void launch_clip_gather(int S, const ClipParams& P, int waves, hipStream_t stream);
void launch_clip_list(int S, const ClipParams& P, int waves, hipStream_t stream);
void launch_clip_exact_gather(int S, const ClipParams& P, int waves, hipStream_t stream);
void launch_clip_exact_list(int S, const ClipParams& P, int waves, hipStream_t stream);
// the first pass with FP64 corners of the *count cells in P.items (at most
// P.n_items), by wavefronts that take one after the other
void launch_clip_listed(const ClipParams& P, const unsigned* count, hipStream_t stream);
// the FP32 first pass (pair_cell.h)
void launch_pairs(const ClipParams& P, int waves, hipStream_t stream);

}  // namespace vgc
