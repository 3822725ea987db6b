// fp32 work spaces of the bfloat16 input gradient in groups of four channels, [C / 4][count][4], gfx950: the hand-down of the tree's
// gradient and the rounding to bfloat16 planes (helpers.hpp:255-350, there level by level from parent to child).
//
// A lane of the convolution holds four neighbouring channels of a position: grouped they are one 16-byte store (conv_mfma.hip), as planes
// four of 4 bytes into as many lines.  Here every node and particle pulls its parent's share, from a table of parents that the plan
// keeps, instead of a parent pushing to its children: what a particle pulls is added on the way to its rounded result, so the pass
// that added the lowest level's shares to the work space is gone.  Bound by memory (6 bytes per value, a quarter to an eighth of the
// parents' 16 bytes, 4 bytes of parent per particle and two groups): 64 channels of 15.4 M particles 1.67 ms, 4.2 TB/s, with the two levels
// of nodes before it 1.9 (planes: 1.7 handed down, 1.15 rounded).  With the stores of the convolution and clearing only where something
// is added (conv_bwd.hip, 1.04 -> 0.23 ms): 1x5x5 64 -> 64 forward and backward on 15.4 M particles 24.1 -> 21.9 ms, training step of the
// 16-32-64 network on 3.4 M 17.9 -> 16.5 ms.
#include "common.hpp"

#include <algorithm>

namespace aprnet {

// A parent: tree node | log2 of its children << 28 (their number is a power of two, helpers.hpp:133-153), or NO_PARENT.
constexpr uint32_t NO_PARENT = 0xffffffffu, PARENT_NODE = (1u << 28) - 1;
constexpr int GG_TB = 256;
__device__ __forceinline__ float parent_share(uint32_t p) { return 1.f / (float)(1 << ((p >> 28) & 3u)); }

__global__ void __launch_bounds__(GG_TB) no_parents_kernel(uint32_t* p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * GG_TB + threadIdx.x;
    if (i < n) p[i] = NO_PARENT;
}
__global__ void __launch_bounds__(GG_TB)
parents_kernel(const int32_t* __restrict__ children, int64_t n_tree, uint32_t* __restrict__ of_particle, uint32_t* __restrict__ of_node) {
    const int64_t t = (int64_t)blockIdx.x * GG_TB + threadIdx.x;
    if (t >= n_tree) return;
    int32_t v[8];
    int n = 0;
#pragma unroll
    for (int s = 0; s < 8; ++s) { v[s] = children[(int64_t)s * n_tree + t]; n += v[s] != NO_CHILD; }
    const uint32_t p = (uint32_t)t | ((uint32_t)(n >= 8 ? 3 : n >= 4 ? 2 : n >= 2 ? 1 : 0) << 28);
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        if (v[s] == NO_CHILD) continue;
        if (v[s] >= 0) of_particle[v[s]] = p; else of_node[~v[s]] = p;
    }
}

// The parents of all particles and tree nodes, 4 bytes each.  Built on first use (allocates; refused while `st` is capturing), then
// served from the plan.
int get_parents(aprnet_plan* p, hipStream_t st) {
    if (p->d_parents) return 0;
    if (p->parents_unavailable || p->n_tree >= (int64_t)PARENT_NODE) return fail(APRNET_ERR_UNSUPPORTED, "the table of parents is not available for this plan");
    if (stream_is_capturing(st)) return fail(APRNET_ERR_UNSUPPORTED, "the table of parents is built on the first backward call: run it once before capturing");
    const int64_t n = p->n_apr + p->n_tree;
    uint32_t* d = nullptr;
    if (hipMalloc((void**)&d, (size_t)std::max<int64_t>(n, 1) * sizeof(uint32_t)) != hipSuccess) {
        (void)hipGetLastError();
        p->parents_unavailable = true;
        return fail(APRNET_ERR_UNSUPPORTED, "no memory for the table of parents");
    }
    hipLaunchKernelGGL(no_parents_kernel, dim3((unsigned)((n + GG_TB - 1) / GG_TB)), dim3(GG_TB), 0, st, d, n);
    if (p->n_tree) hipLaunchKernelGGL(parents_kernel, dim3((unsigned)((p->n_tree + GG_TB - 1) / GG_TB)), dim3(GG_TB), 0, st, p->d_children, p->n_tree, d, d + p->n_apr);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(st);           // (calls on other streams read it from here on)
    if (e != hipSuccess) { (void)hipFree(d); return fail(APRNET_ERR_HIP, std::string("table of parents: ") + hipGetErrorString(e)); }
    p->d_parents = d;
    return 0;
}

// gt[q][t] += the share of t's parent, for the nodes of one level (listed, or t_begin ..); their parents' shares have arrived.
constexpr int PULL_Q = 4;           // groups per thread
__global__ void __launch_bounds__(GG_TB)
pull_level_kernel(const uint32_t* __restrict__ of_node, const int32_t* __restrict__ nodes, int64_t t_begin, int64_t count, float4* __restrict__ gt, int64_t ldt, int nq) {
    const int64_t i = (int64_t)blockIdx.x * GG_TB + threadIdx.x;
    if (i >= count) return;
    const int64_t t = nodes ? nodes[i] : t_begin + i;
    const uint32_t p = of_node[t];
    if (p == NO_PARENT) return;
    const float s = parent_share(p);
    const int64_t tp = p & PARENT_NODE;
    const int q0 = blockIdx.y * PULL_Q;
    float4 a[PULL_Q], b[PULL_Q];
#pragma unroll
    for (int k = 0; k < PULL_Q; ++k) {
        const int64_t row = (int64_t)min(q0 + k, nq - 1) * ldt;
        a[k] = gt[row + t]; b[k] = gt[row + tp];
    }
#pragma unroll
    for (int k = 0; k < PULL_Q; ++k)
        if (q0 + k < nq) gt[(int64_t)(q0 + k) * ldt + t] = make_float4(a[k].x + b[k].x * s, a[k].y + b[k].y * s, a[k].z + b[k].z * s, a[k].w + b[k].w * s);
}

// The coarse levels, a few thousand nodes together, in one launch: a workgroup per group of channels, nodes and parents read first, the levels
// meet in LDS.
constexpr int PULL_LEVELS = 12, PULL_NODES = 2048, PULL_TB = 1024;
struct PullLevels { int n; int64_t end[PULL_LEVELS], t0; };          // adjacent levels, coarsest first
__global__ void __launch_bounds__(PULL_TB)
pull_coarse_kernel(const uint32_t* __restrict__ of_node, const PullLevels lv, float4* __restrict__ gt, int64_t ldt) {
    __shared__ float4 g[PULL_NODES];
    constexpr int J = PULL_NODES / PULL_TB;
    const int64_t row = (int64_t)blockIdx.x * ldt, t1 = lv.end[lv.n - 1];
    uint32_t p[J];
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int64_t t = lv.t0 + j * PULL_TB + threadIdx.x;
        p[j] = t < t1 ? of_node[t] : NO_PARENT;
        if (t < t1) g[t - lv.t0] = gt[row + t];
    }
    __syncthreads();
    for (int i = 1; i < lv.n; ++i) {
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const int64_t t = lv.t0 + j * PULL_TB + threadIdx.x;
            if (t < lv.end[i - 1] || t >= lv.end[i] || p[j] == NO_PARENT) continue;
            const float s = parent_share(p[j]);
            const float4 b = g[(p[j] & PARENT_NODE) - lv.t0];            // (the level above, in this launch)
            float4 a = g[t - lv.t0];
            a = make_float4(a.x + b.x * s, a.y + b.y * s, a.z + b.z * s, a.w + b.w * s);
            g[t - lv.t0] = a;
            gt[row + t] = a;
        }
        __syncthreads();
    }
}

// dst[4 q + c][i] = bfloat16 of gx[q][i][c] + the share of i's parent.  Particles from n_part on are tree nodes i - tree_off.
constexpr int FIN_E = 4, FIN_Q = 2, FIN_N = GG_TB * FIN_E;
__global__ void __launch_bounds__(GG_TB)
finish_gradient_kernel(const float4* __restrict__ gx, int64_t ldx, const float4* __restrict__ gt, int64_t ldt, const uint32_t* __restrict__ of_particle,
                       const uint32_t* __restrict__ of_node, int64_t n_part, int64_t tree_off, int64_t n, int nq, bf16_t* __restrict__ dst, int64_t ldd) {
    typedef unsigned vech __attribute__((ext_vector_type(2), aligned(2)));
    __shared__ __attribute__((aligned(16))) unsigned short buf[FIN_Q][4][FIN_N];
    const int64_t b0 = (int64_t)blockIdx.x * FIN_N;
    const int q0 = blockIdx.y * FIN_Q;
    float4 v[FIN_Q][FIN_E], w[FIN_Q][FIN_E];
    uint32_t p[FIN_E];
#pragma unroll
    for (int e = 0; e < FIN_E; ++e) {
        const int64_t i = min(b0 + e * GG_TB + threadIdx.x, n - 1);
        p[e] = gt ? (i < n_part ? of_particle + i : of_node + (i - tree_off))[0] : NO_PARENT;       // (gt: uniform)
#pragma unroll
        for (int k = 0; k < FIN_Q; ++k) v[k][e] = gx[(int64_t)min(q0 + k, nq - 1) * ldx + i];
    }
    if (gt) {
#pragma unroll
        for (int e = 0; e < FIN_E; ++e)
#pragma unroll
            for (int k = 0; k < FIN_Q; ++k) w[k][e] = gt[(int64_t)min(q0 + k, nq - 1) * ldt + (p[e] == NO_PARENT ? 0 : p[e] & PARENT_NODE)];
#pragma unroll
        for (int e = 0; e < FIN_E; ++e) {
            const float s = p[e] == NO_PARENT ? 0.f : parent_share(p[e]);
            if (p[e] == NO_PARENT) continue;
#pragma unroll
            for (int k = 0; k < FIN_Q; ++k)
                v[k][e] = make_float4(v[k][e].x + w[k][e].x * s, v[k][e].y + w[k][e].y * s, v[k][e].z + w[k][e].z * s, v[k][e].w + w[k][e].w * s);
        }
    }
#pragma unroll
    for (int e = 0; e < FIN_E; ++e)
#pragma unroll
        for (int k = 0; k < FIN_Q; ++k) {
            const int at = e * GG_TB + threadIdx.x;
            buf[k][0][at] = float_to_bf16(v[k][e].x).bits; buf[k][1][at] = float_to_bf16(v[k][e].y).bits;
            buf[k][2][at] = float_to_bf16(v[k][e].z).bits; buf[k][3][at] = float_to_bf16(v[k][e].w).bits;
        }
    __syncthreads();
    const int at = threadIdx.x * FIN_E;
#pragma unroll
    for (int k = 0; k < FIN_Q; ++k) {
        if (q0 + k >= nq) break;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            bf16_t* row = dst + (int64_t)(4 * (q0 + k) + c) * ldd + b0 + at;
            if (b0 + at + FIN_E <= n) {
                const uint2 u = *reinterpret_cast<const uint2*>(&buf[k][c][at]);
                *reinterpret_cast<vech*>(row) = vech{u.x, u.y};
            } else {
#pragma unroll
                for (int e = 0; e < FIN_E; ++e)
                    if (b0 + at + e < n) row[e].bits = buf[k][c][at + e];
            }
        }
    }
}

// gx = bfloat16 of gx4 + what the tree hands down.  gx4 [C / 4][ldx][4], gt4 [C / 4][ldt][4], 16-byte aligned; the table of parents is there
// (get_parents).  `need`: see fill_tree_mean_bwd (tree_ops.hip).
int finish_grouped_gradient(const aprnet_plan* p, int d, const float* gx4, int64_t ldx, int C, float* gt4, int64_t ldt, bf16_t* gx, int64_t ldgx,
                            const NeedLists* need, hipStream_t st) {
    const int Lc = p->lc(d), nq = C / 4, l_top = std::min(Lc - 1, p->tree.level_max);
    const int64_t np = p->number_parts(d);
    const uint32_t* of_particle = p->d_parents;
    const uint32_t* of_node = p->d_parents + p->n_apr;
    float4* gt = (float4*)gt4;
    int l_first = p->tree.level_min;
    if (need) while (l_first <= l_top && need->cnt[l_first] == 0) ++l_first;
    const bool tree = p->tree_parts(d) > 0 && l_first <= l_top;
    if (tree) {
        PullLevels lv{};
        int l = l_first;
        for (; l <= l_top && lv.n < PULL_LEVELS; ++l) {
            const int64_t b = p->tree.level_begin(l), e = p->tree.level_end(l);
            if (lv.n == 0) lv.t0 = b;
            if (e - lv.t0 > PULL_NODES) break;
            lv.end[lv.n++] = e;
        }
        if (lv.n > 1) hipLaunchKernelGGL(pull_coarse_kernel, dim3((unsigned)nq), dim3(PULL_TB), 0, st, of_node, lv, gt, ldt);
        for (l = std::max(l, l_first + 1); l <= l_top; ++l) {
            const int64_t b = p->tree.level_begin(l), e = p->tree.level_end(l);
            const bool list = need && !need->whole[l];
            const int64_t n = list ? need->cnt[l] : e - b;
            if (n <= 0) continue;
            hipLaunchKernelGGL(pull_level_kernel, dim3((unsigned)((n + GG_TB - 1) / GG_TB), (unsigned)((nq + PULL_Q - 1) / PULL_Q)), dim3(GG_TB), 0, st, of_node,
                               list ? need->d_nodes + need->off[l] : nullptr, b, n, gt, ldt, nq);
        }
        APRNET_LAUNCH_CHECK("pull_level_kernel");
    }
    if (np > 0) {
        hipLaunchKernelGGL(finish_gradient_kernel, dim3((unsigned)((np + FIN_N - 1) / FIN_N), (unsigned)((nq + FIN_Q - 1) / FIN_Q)), dim3(GG_TB), 0, st, (const float4*)gx4,
                           ldx, tree ? gt : nullptr, ldt, of_particle, of_node, (int64_t)p->apr.level_end(Lc), p->tree_offset(Lc), np, nq, gx, ldgx);
        APRNET_LAUNCH_CHECK("finish_gradient_kernel");
    }
    return 0;
}

}  // namespace aprnet
