// Weight gradient of a stencil convolution of fp32 features on the bfloat16 matrix instructions, gfx950: both operands as three
// bfloat16 pieces (see conv_split.hip for the pieces, the six products and what they leave out).
//
//   dW[s][co][ci][t] = sum over the output positions (columns) of  gY[co][column] * patch[ci][cell(column) + off(t)]
//
// M = 16 output channels, N = 4 taps x 4 input channels, K = 32 columns of a window per v_mfma_f32_16x16x32_bf16.  Both operands want
// eight consecutive columns of one row per lane, while an LDS cell holds four channels of one position (8 bytes per piece):
// ds_read_b64_tr_b16 turns that round on the way out (conv_dw_g8.hip).  The sixteen lanes of a group name 8 bytes each, four
// columns x four "quads"; the quads of the output gradient are four groups of four channels, those of the patch four taps of the same
// four channels, so that 27 taps fill 28 quads (25 fill 28) and one chunk of four channels is staged at a time.
//
// A workgroup owns two chunks of input channels and 16 * NCO output channels; its eight waves are four pairs of tap groups x two halves
// of the columns (blocks of 32 in turn).  Large and small products have sums of their own, as in conv_split.hip, which stay in registers
// over the windows of a chain and go to the workgroup's slot (see dw_work.hpp).  The output gradient comes from the copy in groups of four
// channels that the input gradient's kernel reads, the features from their planes.
//
// Measured against the fp32 instructions (conv_bwd_mfma.hip), backward pass with the input gradient beside it, ms: 3x3x3, 9.8 M particles
// 32 -> 32 channels 14.0 (15.0), 16 -> 16 4.7 (5.6); 2.9 M sparse ones 24 -> 48 6.6 (8.8); 2.2 M dense ones 64 -> 64 9.8 (10.6); 320 k
// 32 -> 32 0.59 (0.73); 12 k 128 -> 128 0.58 (0.67); 1x5x5 64 -> 64 on 3.9 M 12.8 (17.4).  Error against 64 bits 0.3 to 0.6 of theirs.
// (On the windows of one row group that the plan's lists held then.  With those of the compressed axis, lists.hip, and the gradients in turn
// where each fills the chip, conv_bwd.hip: 12.6, 3.98, 5.7, 9.1, 0.51, 0.48 and 12.0; the kernel alone 6.4 of the first.)
// Bound by waiting, not by a unit: 32 -> 32 on 9.8 M, alone, matrix pipes busy 20 % of the launch, vector ALU and LDS 30 % each, a
// window takes lists, values, two rounds of staging and of products in turn, and two workgroups per CU overlap them in part.  What was
// tried: sixteen waves with both chunks staged at once and every load a window ahead 14.7 ms (one workgroup per CU, its phases in
// step); lists a window ahead 17.3 (spills; 16 -> 16, without any, 5.2 instead of 4.9); 128 columns of gradient at a time 15.1;
// three workgroups per CU for 16 outputs 6.7 (spills); stores of the sums straight from the registers 128 -> 128 on 12 k 0.73.
#include "dw_work.hpp"
#include "pieces.hpp"

namespace aprnet {

typedef float floatx4w __attribute__((ext_vector_type(4)));
typedef int intx4w __attribute__((ext_vector_type(4)));
typedef short shortx4w __attribute__((ext_vector_type(4)));

// Tap groups of four, and cells between two staged rows, searched so that the four taps of a group read different LDS banks
// (a half-wave reads eight columns of four taps, 8 bytes each: 256 bytes, every bank once if no two cells that differ fall together).
// -1: no tap, nothing of what it gives is kept.
template <int K> struct DwTaps;
template <> struct DwTaps<27> {
    static constexpr int ROW = 70;
    static constexpr signed char tap[32] = {25, 5, 24, 3, 16, 15, 1, 4, 20, 18, 19, 26, 2, 22, 21, 23, 9, 10, 17, 11, 0, 6, 8, 7, 14, 12, 13, -1, -1, -1, -1, -1};
};
template <> struct DwTaps<25> {
    static constexpr int ROW = 69;
    static constexpr signed char tap[32] = {24, 5, 9, 21, 6, 7, -1, 8, 10, -1, 23, 22, 11, 12, 14, 13, -1, 17, 4, 2, 15, 19, 18, 3, 1, 0, 16, 20, -1, -1, -1, -1};
};

constexpr int DW_CHUNKS = 2;               // chunks of four input channels that a workgroup owns, staged in turn
template <class G, int NCO> struct DwSplitShape {
    static constexpr int WT = 4, TPW = 2;                           // wave groups over taps, tap groups of a wave
    static constexpr int GC = NCO == 2 ? 192 : 256;                 // columns whose output gradient is staged at a time
    static constexpr int RS = DwTaps<G::K>::ROW, PS = G::NROW * RS; // cells of a piece's patch
    static constexpr int GS = GC + 4;                               // columns between two groups of channels (32 bytes more: other banks)
    static constexpr int IPT = (G::MAXITEM + G::NT - 1) / G::NT;
    static constexpr int GPT = NCO * 4 * GC / G::NT;                // 16-byte pieces of output gradient per thread
    static constexpr int CSTEP = G::NT / (4 * NCO);                 // columns between two of them
};

// four columns of one row for this lane from LDS (see above)
__device__ __forceinline__ shortx4w dw_tr(const char* p) {
    typedef __attribute__((address_space(3))) shortx4w lds_s4;
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)p);
}
__device__ __forceinline__ bf16x8s dw_join(shortx4w a, shortx4w b) {
    return __builtin_bit_cast(bf16x8s, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

// The windows of a workgroup, one after the other; past the last one: an empty window.
struct DwCursor {
    int run, w, w1;
    __device__ __forceinline__ void open(const DwWork& k, int si) {
        if (run >= k.n_run[si]) { w = w1 = -1; return; }
        w = k.win0[si] + run * k.len[si] + min(run, k.rem[si]);
        w1 = w + k.len[si] + (run < k.rem[si] ? 1 : 0);
    }
    __device__ __forceinline__ void next(const DwWork& k, int si) {
        if (w < 0 || ++w < w1) return;
        run += k.blk0[si + 1] - k.blk0[si];
        open(k, si);
    }
    __device__ __forceinline__ int4 header(const int4* __restrict__ win) const {
        int4 h = win[max(w, 0)];
        h.x = __builtin_amdgcn_readfirstlane(h.x); h.y = __builtin_amdgcn_readfirstlane(h.y);
        h.z = __builtin_amdgcn_readfirstlane(h.z); h.w = __builtin_amdgcn_readfirstlane(h.w);
        if (w < 0) h.y = h.w = 0;
        return h;
    }
};

// bytes of up to eight planes of `count` values, `ld` apart (0: none left)
__device__ __forceinline__ int plane_range(int planes, int64_t ld, int64_t count) {
    const int n = min(planes, DW_CHUNKS * SP_CIB);
    return n <= 0 || count <= 0 ? 0 : (int)(unsigned)(((n - 1) * ld + count) * 4);
}

template <class G, int NCO>
__global__ void __launch_bounds__(G::NT) __attribute__((amdgpu_waves_per_eu(4, 4)))
conv_dw_split_kernel(const ConvArgs<float> a, const DwWork wk, int* __restrict__ mark) {
    typedef DwSplitShape<G, NCO> S;
    static_assert(G::NT == 512 && G::RS == 64, "eight waves, cells of the plan's lists");
    static_assert(S::GPT * G::NT == NCO * 4 * S::GC && S::CSTEP * S::GPT == S::GC && S::CSTEP % 64 == 0, "every thread stages the same number of columns");
    struct Operands { uint2 patch[3][S::PS], gyl[3][NCO * 4 * S::GS]; };
    constexpr int SUMS = 16 * NCO * DW_CHUNKS * SP_CIB * G::K;           // of the workgroup: [output channel][input channel][tap]
    union Shared { Operands op; float sums[2][SUMS]; };
    __shared__ __attribute__((aligned(16))) Shared sh;
    __shared__ int cpl[S::GC];
    auto& patch = sh.op.patch;
    auto& gyl = sh.op.gyl;

    int si = 0;
    while (si + 1 < wk.n_s && (int)blockIdx.x >= wk.blk0[si + 1]) ++si;
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wt = wave & (S::WT - 1), kh = wave / S::WT;
    const int ci0 = blockIdx.y * (SP_CIB * DW_CHUNKS), co0 = blockIdx.z * 16 * NCO;

    int toff[S::TPW];                  // byte offset of this lane's tap of a tap group
#pragma unroll
    for (int i = 0; i < S::TPW; ++i) {
        const int t = max((int)DwTaps<G::K>::tap[4 * (wt * S::TPW + i) + (lane & 3)], 0);
        toff[i] = (((t / (G::KX * G::KY)) * G::RX + (t / G::KY) % G::KX) * S::RS + t % G::KY) * 8;
    }
    constexpr int TG = (G::K + 3) / 4;                                   // tap groups (the last wave pair has one)
    const int ntg = min(S::TPW, TG - wt * S::TPW);
    const int lrow = ((lane >> 4) << 3) + ((lane & 15) >> 2);            // this lane's column within 32 (first read)
    constexpr int PB = S::PS * 8, GB = NCO * 4 * S::GS * 8;              // bytes of a piece
    const char* pl = reinterpret_cast<const char*>(patch);
    const char* gl = reinterpret_cast<const char*>(gyl) + ((lane & 3) * S::GS + lrow) * 8;

    floatx4w acc[DW_CHUNKS][S::TPW][NCO], low[DW_CHUNKS][S::TPW][NCO];
#pragma unroll
    for (int q = 0; q < DW_CHUNKS; ++q)
#pragma unroll
    for (int i = 0; i < S::TPW; ++i)
#pragma unroll
        for (int h = 0; h < NCO; ++h) acc[q][i][h] = low[q][i][h] = floatx4w{0.f, 0.f, 0.f, 0.f};

    // The sums so far to the workgroup's slot (first: they start it), by way of LDS: a lane holds four output channels of one (input channel, tap),
    // and stores of those, 4 bytes at a time from sixteen lines each, were what small inputs of wide layers waited for.  The two halves
    // of the columns are added on the way.
    auto flush = [&](const bool first) {
        int l = lane;
        asm volatile("" : "+v"(l));         // addresses formed per call, not kept (and spilled) across the window loop
        __syncthreads();                    // the operands have been read
        float bad = 0.f;                    // stays 0 unless a sum is infinite or NaN
#pragma unroll
        for (int q = 0; q < DW_CHUNKS; ++q)
#pragma unroll
            for (int i = 0; i < S::TPW; ++i) {
                const int c = q * SP_CIB + (l & 3), t = DwTaps<G::K>::tap[4 * (wt * S::TPW + i) + ((l & 15) >> 2)];
                float* dst = sh.sums[kh] + (4 * (l >> 4) * (DW_CHUNKS * SP_CIB) + c) * G::K + t;
#pragma unroll
                for (int h = 0; h < NCO; ++h) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float v = (acc[q][i][h][r] + low[q][i][h][r]) * SPLIT_UNSCALE;
                        if (t < 0) continue;
                        if (ci0 + c < a.Cin) bad = fmaf(v, 0.f, bad);
                        dst[(h * 16 + r) * (DW_CHUNKS * SP_CIB) * G::K] = v;
                    }
                    acc[q][i][h] = low[q][i][h] = floatx4w{0.f, 0.f, 0.f, 0.f};
                }
            }
        if (bad != 0.f) *mark = 1;
        __syncthreads();
        constexpr int ROW = DW_CHUNKS * SP_CIB * G::K;
        const int nrow = min(16 * NCO, a.Cout - co0), ncol = min(DW_CHUNKS * SP_CIB, a.Cin - ci0) * G::K;
        float* slot = a.gw_part + (int64_t)(2 * blockIdx.x) * a.gw_part_ld + ((int64_t)co0 * a.Cin + ci0) * G::K;
        for (int e = threadIdx.x; e < SUMS; e += G::NT) {
            const int row = e / ROW, col = e - row * ROW;
            if (row >= nrow || col >= ncol) continue;
            const float v = sh.sums[0][e] + sh.sums[1][e];
            float* p = slot + (int64_t)row * a.Cin * G::K + col;
            // (later sums by atomic additions, which are not waited for: this thread alone adds to the element, in the order of the program)
            if (first) *p = v; else if (v != 0.f) unsafeAtomicAdd(p, v);
        }
    };

    auto contract = [&](auto qc, const int ng) {
        constexpr int q = decltype(qc)::value;
        for (int kb = kh; kb * 32 < ng; kb += 2) {
            const char* ca = pl + cpl[kb * 32 + lrow];
            const char* cb = pl + cpl[kb * 32 + lrow + 4];
            const char* g = gl + kb * 256;
            bf16x8s av[3][NCO];
#pragma unroll
            for (int p = 0; p < 3; ++p)
#pragma unroll
                for (int h = 0; h < NCO; ++h) av[p][h] = dw_join(dw_tr(g + p * GB + h * (4 * S::GS * 8)), dw_tr(g + p * GB + h * (4 * S::GS * 8) + 32));
#pragma unroll
            for (int i = 0; i < S::TPW; ++i) {
                if (i >= ntg) break;                                     // wave-uniform
                bf16x8s bv[3];
#pragma unroll
                for (int p = 0; p < 3; ++p) bv[p] = dw_join(dw_tr(ca + toff[i] + p * PB), dw_tr(cb + toff[i] + p * PB));
#define APRNET_PRODUCT(C, A, B) _Pragma("unroll") for (int h = 0; h < NCO; ++h) C[q][i][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[A][h], bv[B], C[q][i][h], 0, 0, 0);
                APRNET_PRODUCT(low, 2, 0) APRNET_PRODUCT(low, 0, 2) APRNET_PRODUCT(low, 1, 1)
                APRNET_PRODUCT(low, 1, 0) APRNET_PRODUCT(low, 0, 1) APRNET_PRODUCT(acc, 0, 0)
#undef APRNET_PRODUCT
            }
        }
    };

    // What a thread loads of a window: slots of its items and columns (lists), a window ahead of the values.
    struct Slots { int idx[S::IPT], pos[S::IPT], cidx[S::GPT], cpos[S::GPT]; };
    const int gp = wave & (4 * NCO - 1), gc0 = (wave / (4 * NCO)) * 64 + lane;      // output gradient: group of channels, first column (+ CSTEP per piece)
    const int ngrp = (a.Cout + SP_CIB - 1) / SP_CIB, grp = co0 / SP_CIB + gp;
    const __amdgpu_buffer_rsrc_t rg = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.xi + (int64_t)min(grp, ngrp - 1) * a.xi_ld * SP_CIB), 0,
                                                                        grp < ngrp ? (int)(a.x_count * 16) : 0, 0x00020000);
    auto load_cols = [&](unsigned c0, int ng, int (&cidx)[S::GPT], int (&cpos)[S::GPT]) {                 // unconditional: lanes past the columns read zero
        const __amdgpu_buffer_rsrc_t ri = __builtin_amdgcn_make_buffer_rsrc(const_cast<int*>(a.l_col_idx + c0), 0, ng * 4, 0x00020000);
        const __amdgpu_buffer_rsrc_t rp = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned short*>(a.l_col_pos + c0), 0, ng * 2, 0x00020000);
#pragma unroll
        for (int k = 0; k < S::GPT; ++k) {
            cidx[k] = __builtin_amdgcn_raw_buffer_load_b32(ri, (gc0 + k * S::CSTEP) * 4, 0, 0);
            cpos[k] = (int)__builtin_amdgcn_raw_buffer_load_b16(rp, (gc0 + k * S::CSTEP) * 2, 0, 0);
        }
    };
    auto load_slots = [&](const int4 hd, Slots& s) {
        const __amdgpu_buffer_rsrc_t ri = __builtin_amdgcn_make_buffer_rsrc(const_cast<int*>(a.l_item_idx + (unsigned)hd.x), 0, hd.y * 4, 0x00020000);
        const __amdgpu_buffer_rsrc_t rp = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned short*>(a.l_item_pos + (unsigned)hd.x), 0, hd.y * 2, 0x00020000);
#pragma unroll
        for (int k = 0; k < S::IPT; ++k) {
            s.idx[k] = __builtin_amdgcn_raw_buffer_load_b32(ri, (int)(threadIdx.x + k * G::NT) * 4, 0, 0);
            s.pos[k] = (int)__builtin_amdgcn_raw_buffer_load_b16(rp, (int)(threadIdx.x + k * G::NT) * 2, 0, 0);
        }
        load_cols((unsigned)hd.z, min(hd.w, S::GC), s.cidx, s.cpos);
    };
    struct Values { int x[S::IPT][SP_CIB]; intx4w g[S::GPT]; };
    auto load_gy = [&](const int (&cidx)[S::GPT], int ng, intx4w (&v)[S::GPT]) {
#pragma unroll
        for (int k = 0; k < S::GPT; ++k)
            v[k] = __builtin_amdgcn_raw_buffer_load_b128(rg, (int)(gc0 + k * S::CSTEP < ng ? (unsigned)cidx[k] * 16u : BUF_OOB), 0, 0);
    };
    // The eight planes of the workgroup as one range of memory, the plane in the scalar offset (one descriptor each for features and tree
    // instead of eight, which would not fit the scalar registers); fewer than 2^27 particles and tree nodes to a plane.
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.x + (int64_t)ci0 * a.ldx), 0, plane_range(a.Cin - ci0, a.ldx, a.x_count), 0x00020000);
    const __amdgpu_buffer_rsrc_t rt = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.tree_data + (int64_t)ci0 * a.ldt), 0, plane_range(a.Cin - ci0, a.ldt, a.t_count), 0x00020000);
    auto load_x = [&](const int q, const int nitem, const bool tree_items, const Slots& s, Values& v) {
        int plane[SP_CIB];          // (a channel past the last one reads the last one's plane; what it gives is not kept)
#pragma unroll
        for (int c = 0; c < SP_CIB; ++c) plane[c] = min(q * SP_CIB + c, a.Cin - 1 - ci0);
#pragma unroll
        for (int k = 0; k < S::IPT; ++k) {
            if (k * G::NT >= nitem) break;                                // wave-uniform
            const int off = (int)((unsigned)s.idx[k] * 4u);              // (no item: 0, a value that is not stored)
            if (tree_items) {                                            // (see load_values of conv_common.hpp)
                if (s.pos[k] & (int)ITEM_TREE) {
#pragma unroll
                    for (int c = 0; c < SP_CIB; ++c) v.x[k][c] = __builtin_amdgcn_raw_buffer_load_b32(rt, off, plane_offset(plane[c], a.ldt), 0);
                    asm volatile("" ::: "memory");
                } else {
#pragma unroll
                    for (int c = 0; c < SP_CIB; ++c) v.x[k][c] = __builtin_amdgcn_raw_buffer_load_b32(rx, off, plane_offset(plane[c], a.ldx), 0);
                }
            } else {
#pragma unroll
                for (int c = 0; c < SP_CIB; ++c) v.x[k][c] = __builtin_amdgcn_raw_buffer_load_b32(rx, off, plane_offset(plane[c], a.ldx), 0);
            }
        }
    };
    auto store_gy = [&](const intx4w (&g)[S::GPT], const int (&cpos)[S::GPT], int ng) {
#pragma unroll
        for (int k = 0; k < S::GPT; ++k) {
            const int col = gc0 + k * S::CSTEP;
            uint2 p[3];
            split_pair(__builtin_bit_cast(float, (int)g[k][0]), __builtin_bit_cast(float, (int)g[k][1]), p[0].x, p[1].x, p[2].x);
            split_pair(__builtin_bit_cast(float, (int)g[k][2]), __builtin_bit_cast(float, (int)g[k][3]), p[0].y, p[1].y, p[2].y);
#pragma unroll
            for (int i = 0; i < 3; ++i) gyl[i][gp * S::GS + col] = p[i];
            if (gp == 0) {
                const int cell = (cpos[k] & (int)COL_CELL) - G::TAP0;
                cpl[col] = col < ng ? ((cell >> 6) * S::RS + (cell & 63)) * 8 : 0;
            }
        }
    };
    auto store_x = [&](const Slots& s, const Values& v, int nitem) {
#pragma unroll
        for (int k = 0; k < S::IPT; ++k) {
            if ((int)threadIdx.x + k * G::NT >= nitem) break;
            const int c = ((s.pos[k] & (int)ITEM_CELL) >> 6) * S::RS + (s.pos[k] & 63);
            const bool pair = (s.pos[k] & (int)ITEM_PAIR) != 0;
            float f[SP_CIB];
#pragma unroll
            for (int e = 0; e < SP_CIB; ++e) f[e] = SPLIT_SCALE * RawLoad<float>::cast(v.x[k][e]);
            uint2 p[3];
            split_pair(f[0], f[1], p[0].x, p[1].x, p[2].x);
            split_pair(f[2], f[3], p[0].y, p[1].y, p[2].y);
#pragma unroll
            for (int i = 0; i < 3; ++i) patch[i][c] = p[i];
            if (pair) {
#pragma unroll
                for (int i = 0; i < 3; ++i) patch[i][c + 1] = p[i];
            }
        }
    };

    DwCursor cur;
    cur.run = (int)blockIdx.x - wk.blk0[si];
    cur.open(wk, si);
    const int chain = wk.chain[si];
    int left = chain;
    bool first = true;
    int4 hd = cur.header(a.win);
    bool tree_items = cur.w >= wk.first_coarse;
    for (;;) {
        const int nitem = hd.y, nc = hd.w;
        cur.next(wk, si);
        const int4 hn = cur.header(a.win);
        const bool tree_next = cur.w >= wk.first_coarse, last = cur.w < 0;
        int ng = min(nc, S::GC);
        Slots sl;
        Values v;
        load_slots(hd, sl);
        load_gy(sl.cidx, ng, v.g);
        load_x(0, nitem, tree_items, sl, v);
        __syncthreads();                                                 // the previous window's operands have been read
        for (int i = threadIdx.x; i < 3 * S::PS / 2; i += G::NT) reinterpret_cast<uint4*>(patch)[i] = make_uint4(0u, 0u, 0u, 0u);
        store_gy(v.g, sl.cpos, ng);
        for (int g0 = 0;;) {
            const bool more = g0 + S::GC < nc;
            __syncthreads();
            store_x(sl, v, nitem);
            __syncthreads();
            load_x(1, nitem, tree_items, sl, v);
            contract(std::integral_constant<int, 0>{}, ng);
            __syncthreads();
            store_x(sl, v, nitem);
            __syncthreads();
            if (more) load_x(0, nitem, tree_items, sl, v);
            contract(std::integral_constant<int, 1>{}, ng);
            if (!more) break;
            g0 += S::GC;
            ng = min(nc - g0, S::GC);
            load_cols((unsigned)hd.z + (unsigned)g0, ng, sl.cidx, sl.cpos);
            load_gy(sl.cidx, ng, v.g);
            __syncthreads();
            store_gy(v.g, sl.cpos, ng);
        }
        if (--left == 0 || last) { flush(first); left = chain; first = false; }
        if (last) break;
        hd = hn;
        tree_items = tree_next;
    }
}

using D333 = ConvGeom<3, 3, 3, 2, 4, 512>;
using D155 = ConvGeom<1, 5, 5, 1, 8, 512>;

template <class G>
static int launch_dw_split(const ConvArgs<float>& a, const DwWork& k, int* mark, hipStream_t st) {
    const int nco = a.Cout <= 16 ? 1 : 2, nci = SP_CIB * DW_CHUNKS;
    const dim3 grid((unsigned)k.blk0[k.n_s], (unsigned)((a.Cin + nci - 1) / nci), (unsigned)((a.Cout + 16 * nco - 1) / (16 * nco)));
    if (nco == 1) hipLaunchKernelGGL((conv_dw_split_kernel<G, 1>), grid, dim3(G::NT), 0, st, a, k, mark);
    else hipLaunchKernelGGL((conv_dw_split_kernel<G, 2>), grid, dim3(G::NT), 0, st, a, k, mark);
    APRNET_LAUNCH_CHECK("conv_dw_split_kernel");
    return 0;
}
// Partial sums of the weight gradient; a.xi / a.xi_ld: the output gradient in groups of four channels (prepare_split), a.x the features'
// planes, a.gw_part the slots of k.  *mark (cleared by the caller) is set where a sum is not finite.
int launch_conv_dw_split(int code, const ConvArgs<float>& a, const DwWork& k, int* mark, hipStream_t st) {
    switch (code) {
        case 333: return launch_dw_split<D333>(a, k, mark, st);
        case 155: return launch_dw_split<D155>(a, k, mark, st);
    }
    return fail(APRNET_ERR_UNSUPPORTED, "no matrix-core kernel for this stencil");
}

}  // namespace aprnet
