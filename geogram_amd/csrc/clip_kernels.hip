// The clipping kernels, compiled once per VGC_CLIP_PART (0: gathered
// neighbours, 1: lists, 2 and 3: the same with exact signs, 4: the FP32 first
// pass, 5: the cells that leaves), so that the parts build in parallel.
#include <stdexcept>

#include "clip_launch.h"

namespace vgc {

static inline unsigned blocks_for(long long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

#if VGC_CLIP_PART < 4
// S = 1 with FP64 signs (every cell's first pass, and the second gather):
// registers capped at 128 for 4 waves per SIMD (some spill to scratch); with
// one-wave work-groups that measured 7 % faster than 168 registers and 3
// waves — the wait for dependent LDS and memory round trips is hidden by
// occupancy.  The exact re-clip (a few cells) keeps its registers.
template <int S, int WAVES, bool EXACT, bool GATHER, bool W, bool CORNER = W>
__global__ __launch_bounds__(64 * WAVES, (S == 1 && !EXACT) ? 4 : 1) void k_clip(ClipParams P) {
    __shared__ CellLds<S> lds[WAVES];
    const int wave = WAVES == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int item = xcd_block() * WAVES + wave;
    // From lists, the item in a vector register: with a scalar one the compiler
    // keeps all that follows from it in scalar registers, runs out of them and
    // spills (S = 4: 124 spilled and 308 vector registers, against 36 and 231).
    // Cells of the first 13 Newton steps of a clustered transport of 1M seeds:
    // 3.07 s scalar, 2.39 s so.  Gathering kernels spill either way, and run
    // 10 to 25 % faster scalar.
    if constexpr (!GATHER) asm volatile("" : "+v"(item));
    if (item >= P.n_items) return;  // whole wavefront
    process_cell<S, EXACT, GATHER, W, CORNER>(P, item, lds[wave]);
}

template <bool E, bool G, bool W>
static void clip_egw(int S, const ClipParams& P, int waves, hipStream_t stream) {
    const unsigned g4 = blocks_for(P.n_items, 4), g1 = blocks_for(P.n_items, 1);
    if (S == 1) {
        if constexpr (G && !W) {
            if (P.corner) {
                // second gather of Voronoi cells, with the corner test
                k_clip<1, 1, E, G, W, true><<<g1, 64, 0, stream>>>(P);
                return;
            }
        }
        if (waves == 1)
            k_clip<1, 1, E, G, W><<<g1, 64, 0, stream>>>(P);
        else
            k_clip<1, 4, E, G, W><<<g4, 256, 0, stream>>>(P);
    } else if (S == 2) {
        k_clip<2, 4, E, G, W><<<g4, 256, 0, stream>>>(P);
    } else if (S == 4) {
        k_clip<4, 1, E, G, W><<<g1, 64, 0, stream>>>(P);
    } else {
        // 512 corners: list mode only (the last tier)
        if constexpr (!G)
            k_clip<8, 1, E, false, W><<<g1, 64, 0, stream>>>(P);
        else
            throw std::runtime_error("clip: 512-corner cells run from lists only");
    }
}
template <bool E, bool G>
static void clip_eg(int S, const ClipParams& P, int waves, hipStream_t stream) {
    if (P.weighted)
        clip_egw<E, G, true>(S, P, waves, stream);
    else
        clip_egw<E, G, false>(S, P, waves, stream);
}

#if VGC_CLIP_PART == 0
void launch_clip_gather(int S, const ClipParams& P, int waves, hipStream_t stream) {
    clip_eg<false, true>(S, P, waves, stream);
}
#elif VGC_CLIP_PART == 1
void launch_clip_list(int S, const ClipParams& P, int waves, hipStream_t stream) {
    clip_eg<false, false>(S, P, waves, stream);
}
#elif VGC_CLIP_PART == 2
void launch_clip_exact_gather(int S, const ClipParams& P, int waves, hipStream_t stream) {
    clip_eg<true, true>(S, P, waves, stream);
}
#else
void launch_clip_exact_list(int S, const ClipParams& P, int waves, hipStream_t stream) {
    clip_eg<true, false>(S, P, waves, stream);
}
#endif
#elif VGC_CLIP_PART == 5
// The cells that the FP32 first pass left (0.3 % of the 2M mixture), their
// list and its length read on the device: up to 4096 wavefronts, the number
// the chip holds, share them.
template <bool W>
__global__ __launch_bounds__(64, 4) void k_clip_listed(ClipParams P, const unsigned* count) {
    __shared__ CellLds<1> lds;
    const int n = (int)*count;
    for (int item = blockIdx.x; item < n; item += gridDim.x)
        process_cell<1, false, true, W, W>(P, item, lds);
}
void launch_clip_listed(const ClipParams& P, const unsigned* count, hipStream_t stream) {
    const unsigned g = (unsigned)(P.n_items < 4096 ? P.n_items : 4096);
    if (P.weighted)
        k_clip_listed<true><<<g, 64, 0, stream>>>(P, count);
    else
        k_clip_listed<false><<<g, 64, 0, stream>>>(P, count);
}
#else
// The first pass with FP32 corner state: two cells per wavefront
// (pair_cell.h).
template <int WAVES, bool W, bool COUNT>
__global__ __launch_bounds__(64 * WAVES, 4) void k_pair(ClipParams P) {
    __shared__ PairLds lds[WAVES];
    const int wave = WAVES == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int first = P.group * (xcd_block() * WAVES + wave);
    if (first >= P.n_items) return;  // whole wavefront
    process_pairs<W, COUNT>(P, first, min(P.group, P.n_items - first), lds[wave]);
}

template <bool W, bool COUNT>
static void clip_pairs(const ClipParams& P, int waves, hipStream_t stream) {
    if (waves == 1)
        k_pair<1, W, COUNT><<<blocks_for(P.n_items, P.group), 64, 0, stream>>>(P);
    else
        k_pair<4, W, COUNT><<<blocks_for(P.n_items, 4 * P.group), 256, 0, stream>>>(P);
}

void launch_pairs(const ClipParams& P, int waves, hipStream_t stream) {
    if (P.weighted)
        P.counters ? clip_pairs<true, true>(P, waves, stream) : clip_pairs<true, false>(P, waves, stream);
    else
        P.counters ? clip_pairs<false, true>(P, waves, stream) : clip_pairs<false, false>(P, waves, stream);
}
#endif

}  // namespace vgc
