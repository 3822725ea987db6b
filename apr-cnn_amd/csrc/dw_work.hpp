// Weight gradient on the plan's window lists: which windows a workgroup takes, and where its sums go.
#pragma once
#include "conv_common.hpp"

namespace aprnet {

// Work of a launch on the plan's window lists: workgroups blk0[k] .. blk0[k + 1] - 1 (grid.x) take the windows of stencil
// index s_of[k].  One launch covers all stencil indices: with a launch and a sum of slots each, most of them left the chip
// idle (the coarse levels have a handful of windows), and the weight gradients of a training step of the 16-32-64-128 network on
// two APRs of 338 k particles took 76 + 102 launches; now 28 + 28, and the step 14.4 instead of 15.8 ms.
struct DwWork {
    int n_s;
    int s_of[MAX_LEVELS + 1], win0[MAX_LEVELS + 1], nwin[MAX_LEVELS + 1], blk0[MAX_LEVELS + 2];
    // The windows of an index are cut into n_run runs of len or (the first `rem`) len + 1 neighbours, which its workgroups take in turn.
    int n_run[MAX_LEVELS + 1], len[MAX_LEVELS + 1], rem[MAX_LEVELS + 1];
    int chain[MAX_LEVELS + 1];     // windows whose products are added up in registers before the sums go to the slots
    int first_coarse;              // windows from here on may stage tree nodes (below the finest level of the call)
};

// Partial sums of one workgroup and column half, rows of output channels from co0 on: its slot, or (no slots) the result itself.
struct DwSlot {
    __amdgpu_buffer_rsrc_t rs;
    float* p; bool own; int co_n, Cin, K;
    template <typename T>
    __device__ __forceinline__ DwSlot(const ConvArgs<T>& a, int bx, int co0, int kh, int rows, int K_, int s) : own(a.gw_part != nullptr), co_n(min(rows, a.Cout - co0)), Cin(a.Cin), K(K_) {
        p = (own ? a.gw_part + (int64_t)(2 * bx + kh) * a.gw_part_ld : a.gw + (int64_t)s * a.Cout * Cin * K) + (int64_t)co0 * Cin * K;
        rs = __builtin_amdgcn_make_buffer_rsrc(p, 0, co_n * Cin * K * 4, 0x00020000);
    }
    // first: nothing is in the slot yet.  Later sums come by atomic additions, which are not waited for; the lane that wrote an element is
    // the only one that adds to it, so they arrive in the order of the program.
    __device__ __forceinline__ void add(int row, int ci, int t, float v, bool first) const {
        const bool in = t < K && row < co_n;
        const int e = (row * Cin + ci) * K + t;
        if (own && first) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, v), rs, in ? e * 4 : (int)BUF_OOB, 0, 0);      // (past the end: not written)
        else if (in && v != 0.f) unsafeAtomicAdd(p + e, v);
    }
};

// conv_bwd_mfma.hip: the work of a launch, the same for every kernel that writes the slots
DwWork dw_work(int code, int Cout, int Cin, int S_exp, int Lc, const WinLists& wl);

}  // namespace aprnet
