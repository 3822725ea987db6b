// Second half of a weight gradient in a fixed order: the partial sums that every workgroup left in a slot of its own are
// added to the result.
#pragma once
#include "common.hpp"

namespace aprnet {

// out[e] += sum of part[slot][e] over the slots, in an order that is fixed by the slot count alone: wave w of the block's W adds
// slots w, w + W, ... (eight loads in flight), the W sums of an element meet in LDS and are added in wave order.
// A wave reads 64 neighbouring elements of a slot, whole lines: with a wave per element, whose lanes read one element of 64
// slots, the 1x1x1 backward of 512 -> 512 channels took 9.80 ms on 103 k particles and 2.63 ms on 4 k, now 9.59 and 2.40 ms.
// Bound by the latency of the chain of loads when one thread walks all slots of an element (27 k elements fill a tenth of
// the chip): 128 us on average over the launches of a training step of the 16-32-64 network on 5.5 M particles, 48 us with
// 16 waves per 64 elements.
template <typename A, int W>
__device__ __forceinline__ void sum_slots_body(const A* __restrict__ part, int64_t ld, int slots, int64_t n, A* __restrict__ out) {
    __shared__ A sums[W][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t e = (int64_t)blockIdx.x * 64 + lane;
    const A* src = part + (e < n ? e : n - 1);
    A s[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) s[i] = 0;
    int k = w;
    for (; k + 7 * W < slots; k += 8 * W)
#pragma unroll
        for (int i = 0; i < 8; ++i) s[i] += src[(int64_t)(k + i * W) * ld];
    for (; k < slots; k += W) s[0] += src[(int64_t)k * ld];
    sums[w][lane] = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
    __syncthreads();
    if (w == 0 && e < n) {
        A t = 0;
#pragma unroll
        for (int i = 0; i < W; ++i) t += sums[i][lane];
        out[e] += t;
    }
}
template <typename A, int W>
__global__ void __launch_bounds__(64 * W) sum_slots_kernel(const A* __restrict__ part, int64_t ld, int slots, int64_t n, A* __restrict__ out) {
    sum_slots_body<A, W>(part, ld, slots, n, out);
}

// Several sums in one launch: slots first[k] .. first[k + 1] - 1 are added to out + out[k] * n.
struct SlotGroups { int n; int first[MAX_LEVELS + 2], out[MAX_LEVELS + 1]; };
// all: null, or a word that is 0 if only the first slot of every pair holds something.
template <typename A>
__global__ void __launch_bounds__(1024) sum_slot_groups_kernel(const A* __restrict__ part, int64_t ld, const SlotGroups g, int64_t n, A* __restrict__ out,
                                                               const int* __restrict__ all) {
    const int k = blockIdx.y, step = all && *all == 0 ? 2 : 1;
    sum_slots_body<A, 16>(part + (int64_t)g.first[k] * ld, step * ld, (g.first[k + 1] - g.first[k]) / step, n, out + (int64_t)g.out[k] * n);
}
template <typename A>
int launch_sum_slot_groups(const A* part, int64_t ld, const SlotGroups& g, int64_t n, A* out, hipStream_t st, const int* all = nullptr) {
    if (n <= 0 || g.n <= 0) return 0;
    hipLaunchKernelGGL(sum_slot_groups_kernel<A>, dim3((unsigned)((n + 63) / 64), (unsigned)g.n), dim3(1024), 0, st, part, ld, g, n, out, all);
    APRNET_LAUNCH_CHECK("sum_slot_groups_kernel");
    return 0;
}

// 16 waves, 4 where there are fewer slots than that (1x1x1 256 -> 512 on 4 k particles, 3 slots: 2.54 instead of 2.55 ms)
template <typename A>
int launch_sum_slots(const A* part, int64_t ld, int slots, int64_t n, A* out, hipStream_t st) {
    if (n <= 0 || slots <= 0) return 0;
    const dim3 grid((unsigned)((n + 63) / 64));
    if (slots < 16) hipLaunchKernelGGL((sum_slots_kernel<A, 4>), grid, dim3(64 * 4), 0, st, part, ld, slots, n, out);
    else hipLaunchKernelGGL((sum_slots_kernel<A, 16>), grid, dim3(64 * 16), 0, st, part, ld, slots, n, out);
    APRNET_LAUNCH_CHECK("sum_slots_kernel");
    return 0;
}

}  // namespace aprnet
