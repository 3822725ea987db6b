// Weight gradient of a stencil convolution for bfloat16 features grouped by eight channels, gfx950.
//
//   dW[s][co][ci][t] = sum over the output positions (columns) of  gY[co][column] * patch[ci][cell(column) + off(t)]
//
// As a matrix product per tap: M = 16 output channels, N = 16 input channels, K = the columns of a window, 32 per
// v_mfma_f32_16x16x32_bf16.  Both operands want eight values of ONE channel (consecutive columns) per lane, while a staged
// cell holds eight channels of one position (16 bytes, what a gathered item is).  ds_read_b64_tr_b16 turns that round
// on the way out of LDS: the sixteen lanes of a group each name 8 bytes (four channels of a column; every lane its own
// address, so the columns need not be neighbours), and lane n receives channel n of four columns.  Two such reads make an
// operand; a tap is a constant added to the address.
//
// A workgroup owns 16 input channels, 16 * NCO output channels and a contiguous range of windows of one stencil index; its
// eight waves are WT groups of taps x WK shares of the columns.  The sums stay in registers over all windows, the WK
// shares meet in LDS at the end, and every workgroup writes its sums to a slot of its own (added up in slot order by
// dw_g8_reduce_kernel).  Calls on one plan give the same bits; the lists of another plan of the same APR may hold a window's
// columns in another order (their places are taken with an atomic counter when the lists are built), and with it the sums.
//
// What bounds it: waiting.  1x5x5 64 -> 64 on 15.4 M particles, alone: the waves wait 62 % of their resident cycles
// (the gather and the three barriers of a window, which every one of its 4 x 2 channel blocks stages anew), LDS is busy
// 42 % of the launch (a third of that with bank conflicts), the matrix pipes 25 %.  The kernel before it read one channel per lane: eight 2-byte LDS reads per operand and a gather of
// 2-byte values from the channel planes: 24.2 ms, 5.9 ms here (3.15 TFLOP).
#include "conv_common.hpp"

namespace aprnet {

typedef float floatx4g __attribute__((ext_vector_type(4)));
typedef int intx4g __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8g __attribute__((ext_vector_type(8)));
typedef short shortx4g __attribute__((ext_vector_type(4)));
typedef short shortx8g __attribute__((ext_vector_type(8)));

struct DwG8Args {
    const bf16_t* xi; const bf16_t* ti; const bf16_t* gyi;     // [C / 8][count][8]: features, mean tree, output gradient
    int64_t xi_ld, ti_ld, gy_ld;                               // particles between two groups
    int64_t x_count, t_count, gy_count;
    int Cin, Cout, CinP, CoutP;                                // channels of the copies, and rounded up to the kernel's blocks
    const int4* win;
    const int* item_idx; const unsigned short* item_pos; const int* col_idx; const unsigned short* col_pos;
    float* part;                                               // [blocks][K][CoutP][CinP]
    int n_s;                                                   // stencil indices that have windows
    int s_of[MAX_LEVELS], win0[MAX_LEVELS], nwin[MAX_LEVELS];  // their index, first window and windows
    int blk0[MAX_LEVELS + 1];                                  // their first workgroup (blockIdx.x)
    int ci0, CinW;                                             // first of these channels in the layer, its input channels
};

constexpr int DWG_COLS = 256;             // columns whose output gradient is staged at a time
template <class G> struct DwG8Shape {
    static constexpr int WT = G::K > 16 ? 4 : 2, WK = G::NWAVE / WT;      // wave groups over taps x over columns
    static constexpr int TPW = (G::K + WT - 1) / WT;
    // cells per channel group: eight more than the rows need, so that the two groups of a read lie on different banks
    static constexpr int PS = G::NROW * G::RS + 8, GS = DWG_COLS + 8;
    static constexpr int IPT = (G::MAXITEM + G::NT - 1) / G::NT;
};

// four columns of one channel for this lane from LDS byte address `off` (see above)
__device__ __forceinline__ shortx4g lds_tr(const char* base, int off) {
    typedef __attribute__((address_space(3))) shortx4g lds_s4;
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(base + off));
}
__device__ __forceinline__ bf16x8g join8(shortx4g a, shortx4g b) {
    return __builtin_bit_cast(bf16x8g, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

template <class G, int NCO>
__global__ void __launch_bounds__(G::NT) __attribute__((amdgpu_waves_per_eu(4, 4)))
conv_dw_g8_kernel(const DwG8Args a) {
    typedef DwG8Shape<G> S;
    static_assert(G::RS == 64 && G::NT == 512, "cells of the plan's lists, eight waves");
    static_assert((G::K - 1) / (G::KX * G::KY) * G::RX * 64 * 16 < 65536, "tap offsets");
    __shared__ __attribute__((aligned(16))) uint4 patch[2 * S::PS];
    __shared__ __attribute__((aligned(16))) uint4 gyl[2 * NCO * S::GS];
    __shared__ int cpl[DWG_COLS];

    int si = 0;
    while (si + 1 < a.n_s && (int)blockIdx.x >= a.blk0[si + 1]) ++si;
    const int nblk = a.blk0[si + 1] - a.blk0[si], bi = (int)blockIdx.x - a.blk0[si];
    const int wb = a.win0[si] + (int)((int64_t)a.nwin[si] * bi / nblk), we = a.win0[si] + (int)((int64_t)a.nwin[si] * (bi + 1) / nblk);
    const int tid = threadIdx.x, lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wt = wave % S::WT, wk = wave / S::WT;
    const int q0 = 2 * blockIdx.y, nq = (a.Cin + 7) / 8;                 // first group of the input block
    const int p0 = 2 * NCO * blockIdx.z, np = (a.Cout + 7) / 8;          // first group of the output block

    int toff[S::TPW];
#pragma unroll
    for (int i = 0; i < S::TPW; ++i) {
        const int t = min(wt * S::TPW + i, G::K - 1);
        toff[i] = (((t / (G::KX * G::KY)) * G::RX + (t / G::KY) % G::KX) * G::RS + t % G::KY) * 16;
    }
    const int ntap = min(S::TPW, G::K - wt * S::TPW);
    const int lrow = ((lane >> 4) << 3) + ((lane & 15) >> 2);            // this lane's column within 32 (first read)
    const char* pl = reinterpret_cast<const char*>(patch) + ((lane & 3) >> 1) * (S::PS * 16) + (lane & 1) * 8;
    const char* gl = reinterpret_cast<const char*>(gyl) + ((lane & 3) >> 1) * (S::GS * 16) + (lane & 1) * 8 + lrow * 16;

    floatx4g acc[S::TPW][NCO];
#pragma unroll
    for (int i = 0; i < S::TPW; ++i)
#pragma unroll
        for (int h = 0; h < NCO; ++h)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][h][r] = 0.f;

    // descriptors: a group past the last one reads as zeros
    auto rsrc = [](const bf16_t* base, int64_t ld, int q, int nq_, int64_t count) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(base + (int64_t)q * ld * 8), 0, q < nq_ ? (int)(count * 16) : 0, 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t rx0 = rsrc(a.xi, a.xi_ld, q0, nq, a.x_count), rx1 = rsrc(a.xi, a.xi_ld, q0 + 1, nq, a.x_count);
    const __amdgpu_buffer_rsrc_t rt0 = rsrc(a.ti, a.ti_ld, q0, nq, a.t_count), rt1 = rsrc(a.ti, a.ti_ld, q0 + 1, nq, a.t_count);
    const bool two = q0 + 1 < nq;                                        // uniform
    const int gc = tid & (DWG_COLS - 1), gp = tid / DWG_COLS;            // output gradient: this thread's column, first group (+ 2 per step)

    // lists of a window (unconditional buffer loads: lanes past the end read zero), one window ahead of their use
    struct Slots { int idx[S::IPT]; int pos[S::IPT]; int cidx, cpos; };
    auto load_slots = [&](const int4 hd, Slots& s) {
        const int nitem = hd.y, nc = min(hd.w, DWG_COLS);
        const __amdgpu_buffer_rsrc_t ri = __builtin_amdgcn_make_buffer_rsrc(const_cast<int*>(a.item_idx + (unsigned)hd.x), 0, nitem * 4, 0x00020000);
        const __amdgpu_buffer_rsrc_t rp = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned short*>(a.item_pos + (unsigned)hd.x), 0, nitem * 2, 0x00020000);
        const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(const_cast<int*>(a.col_idx + (unsigned)hd.z), 0, nc * 4, 0x00020000);
        const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned short*>(a.col_pos + (unsigned)hd.z), 0, nc * 2, 0x00020000);
#pragma unroll
        for (int k = 0; k < S::IPT; ++k) {
            const int it = tid + k * G::NT;
            s.idx[k] = __builtin_amdgcn_raw_buffer_load_b32(ri, it * 4, 0, 0);
            s.pos[k] = (int)__builtin_amdgcn_raw_buffer_load_b16(rp, it * 2, 0, 0);
        }
        s.cidx = __builtin_amdgcn_raw_buffer_load_b32(rc, gc * 4, 0, 0);
        s.cpos = (int)__builtin_amdgcn_raw_buffer_load_b16(rq, gc * 2, 0, 0);
    };
    auto header = [&](int w) {
        const int4 h = a.win[w];
        return make_int4(__builtin_amdgcn_readfirstlane(h.x), __builtin_amdgcn_readfirstlane(h.y), __builtin_amdgcn_readfirstlane(h.z), __builtin_amdgcn_readfirstlane(h.w));
    };
    intx4g gv[NCO];
    auto load_gy = [&](int cidx, int ng) {
        const int off = (int)(gc < ng ? (unsigned)cidx * 16u : BUF_OOB);         // (unsigned: up to 2^28 particles)
#pragma unroll
        for (int h = 0; h < NCO; ++h) {
            const int q = p0 + gp + 2 * h;                              // wave-uniform
            gv[h] = __builtin_amdgcn_raw_buffer_load_b128(rsrc(a.gyi, a.gy_ld, q, np, a.gy_count), off, 0, 0);
        }
    };
    auto store_gy = [&](int cpos, int ng) {
#pragma unroll
        for (int h = 0; h < NCO; ++h)
            gyl[(gp + 2 * h) * S::GS + gc] = __builtin_bit_cast(uint4, gv[h]);
        if (tid < DWG_COLS) cpl[gc] = gc < ng ? ((cpos & (int)COL_CELL) - G::TAP0) * 16 : 0;
    };
    auto contract = [&](int ng) {
        const int nks = (ng + 31) >> 5;
        for (int ks = wk; ks < nks; ks += S::WK) {
            const int c0 = ks * 32;
            const int ca = cpl[c0 + lrow], cb = cpl[c0 + lrow + 4];
            bf16x8g av[NCO];
#pragma unroll
            for (int h = 0; h < NCO; ++h)
                av[h] = join8(lds_tr(gl, c0 * 16 + h * (2 * S::GS * 16)), lds_tr(gl, c0 * 16 + 64 + h * (2 * S::GS * 16)));
#pragma unroll
            for (int i = 0; i < S::TPW; ++i) {
                if (i >= ntap) break;                                    // wave-uniform
                const bf16x8g bv = join8(lds_tr(pl, ca + toff[i]), lds_tr(pl, cb + toff[i]));
#pragma unroll
                for (int h = 0; h < NCO; ++h) acc[i][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[h], bv, acc[i][h], 0, 0, 0);
            }
        }
    };

    if (wb < we) {
        int4 hd = header(wb);
        Slots sl;
        load_slots(hd, sl);
        for (int w = wb; w < we; ++w) {
            const int nitem = hd.y, nc = hd.w;
            const int4 hn = header(min(w + 1, we - 1));
            // values of this window's items and of its first columns
            intx4g v0[S::IPT], v1[S::IPT];
#pragma unroll
            for (int k = 0; k < S::IPT; ++k) {
                if (k * G::NT >= nitem) break;                          // uniform
                const int off = (int)(tid + k * G::NT < nitem ? (unsigned)sl.idx[k] * 16u : BUF_OOB);
                if (sl.pos[k] & (int)ITEM_TREE) {
                    v0[k] = __builtin_amdgcn_raw_buffer_load_b128(rt0, off, 0, 0);
                    if (two) v1[k] = __builtin_amdgcn_raw_buffer_load_b128(rt1, off, 0, 0);
                    asm volatile("" ::: "memory");                       // keeps the two branches apart (one load with a per-lane descriptor otherwise)
                } else {
                    v0[k] = __builtin_amdgcn_raw_buffer_load_b128(rx0, off, 0, 0);
                    if (two) v1[k] = __builtin_amdgcn_raw_buffer_load_b128(rx1, off, 0, 0);
                }
            }
            int ng = min(nc, DWG_COLS);
            load_gy(sl.cidx, ng);
            __syncthreads();                                             // the previous window's operands have been read
            for (int i = tid; i < (two ? 2 : 1) * S::PS; i += G::NT) patch[i] = make_uint4(0u, 0u, 0u, 0u);
            __syncthreads();
#pragma unroll
            for (int k = 0; k < S::IPT; ++k) {
                if (tid + k * G::NT >= nitem) break;
                const int cell = sl.pos[k] & (int)ITEM_CELL;
                const bool pair = (sl.pos[k] & (int)ITEM_PAIR) != 0;
                patch[cell] = __builtin_bit_cast(uint4, v0[k]);
                if (pair) patch[cell + 1] = __builtin_bit_cast(uint4, v0[k]);
                if (two) {
                    patch[S::PS + cell] = __builtin_bit_cast(uint4, v1[k]);
                    if (pair) patch[S::PS + cell + 1] = __builtin_bit_cast(uint4, v1[k]);
                }
            }
            store_gy(sl.cpos, ng);
            if (w + 1 < we) load_slots(hn, sl);                          // travels during the matrix phase
            __syncthreads();
            for (int g0 = 0;;) {
                g0 += DWG_COLS;
                const bool more = g0 < nc;
                int cidx = 0, cpos = 0, ngn = 0;
                if (more) {                                              // the next group of columns: lists, then values, during this group's products
                    ngn = min(nc - g0, DWG_COLS);
                    const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(const_cast<int*>(a.col_idx + (unsigned)hd.z + g0), 0, ngn * 4, 0x00020000);
                    const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned short*>(a.col_pos + (unsigned)hd.z + g0), 0, ngn * 2, 0x00020000);
                    cidx = __builtin_amdgcn_raw_buffer_load_b32(rc, gc * 4, 0, 0);
                    cpos = (int)__builtin_amdgcn_raw_buffer_load_b16(rq, gc * 2, 0, 0);
                    load_gy(cidx, ngn);
                }
                contract(ng);
                if (!more) break;
                __syncthreads();
                ng = ngn;
                store_gy(cpos, ng);
                __syncthreads();
            }
            hd = hn;
        }
    }

    // the shares of the columns: share 0 adds the others, in order, and writes the workgroup's slot
    float* red = reinterpret_cast<float*>(patch);
    static_assert((S::WK - 1) * S::WT * NCO * 4 * 64 * 4 <= 2 * S::PS * 16, "shares of one tap fit the patch");
    float* dst = a.part + (int64_t)blockIdx.x * G::K * a.CoutP * a.CinP;
#pragma unroll
    for (int i = 0; i < S::TPW; ++i) {
        __syncthreads();
        if (wk > 0)
#pragma unroll
            for (int h = 0; h < NCO; ++h)
#pragma unroll
                for (int r = 0; r < 4; ++r) red[((((wk - 1) * S::WT + wt) * NCO + h) * 4 + r) * 64 + lane] = acc[i][h][r];
        __syncthreads();
        if (wk == 0 && i < ntap) {
            const int t = wt * S::TPW + i;
#pragma unroll
            for (int h = 0; h < NCO; ++h)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float v = acc[i][h][r];
#pragma unroll
                    for (int k = 1; k < S::WK; ++k) v += red[((((k - 1) * S::WT + wt) * NCO + h) * 4 + r) * 64 + lane];
                    const int co = (blockIdx.z * NCO + h) * 16 + 4 * (lane >> 4) + r, ci = blockIdx.y * 16 + (lane & 15);
                    dst[((int64_t)t * a.CoutP + co) * a.CinP + ci] = v;
                }
        }
    }
}

// gw[s][co][ci][t] += sum of part[block][t][co][ci] over the blocks of stencil index s, in an order fixed by their number:
// wave w adds blocks w, w + 8, ... (eight loads in flight), the eight sums meet in LDS.
constexpr int DWG_RED_W = 8;
__global__ void __launch_bounds__(64 * DWG_RED_W)
dw_g8_reduce_kernel(const DwG8Args a, int K, float* __restrict__ gw) {
    __shared__ float sums[DWG_RED_W][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, si = blockIdx.y;
    const int64_t n = (int64_t)K * a.Cout * a.Cin, e = (int64_t)blockIdx.x * 64 + lane, ee = e < n ? e : n - 1;
    const int ci = (int)(ee % a.Cin), co = (int)(ee / a.Cin % a.Cout), t = (int)(ee / ((int64_t)a.Cin * a.Cout));
    const int64_t ld = (int64_t)K * a.CoutP * a.CinP;
    const float* src = a.part + (int64_t)a.blk0[si] * ld + ((int64_t)t * a.CoutP + co) * a.CinP + ci;
    const int nb = a.blk0[si + 1] - a.blk0[si];
    float s[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) s[i] = 0.f;
    int k = w;
    for (; k + 7 * DWG_RED_W < nb; k += 8 * DWG_RED_W)
#pragma unroll
        for (int i = 0; i < 8; ++i) s[i] += src[(int64_t)(k + i * DWG_RED_W) * ld];
    for (; k < nb; k += DWG_RED_W) s[0] += src[(int64_t)k * ld];
    sums[w][lane] = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
    __syncthreads();
    if (w == 0 && e < n) {
        float v = 0.f;
#pragma unroll
        for (int i = 0; i < DWG_RED_W; ++i) v += sums[i][lane];
        gw[(((int64_t)a.s_of[si] * a.Cout + co) * a.CinW + a.ci0 + ci) * K + t] += v;
    }
}

using DG333 = ConvGeom<3, 3, 3, 2, 4, 512>;
using DG133 = ConvGeom<1, 3, 3, 1, 8, 512>;
using DG155 = ConvGeom<1, 5, 5, 1, 8, 512>;

static int dwg_taps(int code) { return code == 333 ? 27 : code == 133 ? 9 : 25; }
static int64_t dwg_slot_bytes(int code, const DwG8Args& a) { return (int64_t)dwg_taps(code) * a.CinP * a.CoutP * (int64_t)sizeof(float); }
static int dwg_nco(int Cout) { return Cout <= 16 ? 1 : 2; }
// Workgroups of a launch: about two rounds of the 512 that the chip holds (windows differ in work), fewer for layers with
// several channel blocks, whose every window is visited once per block.
static int dwg_blocks_x(int Cin, int Cout) {
    const int per = ((Cin + 15) / 16) * ((Cout + 16 * dwg_nco(Cout) - 1) / (16 * dwg_nco(Cout)));
    return std::max(64, 1024 / per);
}
// Channels rounded up to the kernel's blocks and the workgroups of every stencil index (level Lc - s has index s, every level
// from S_exp - 1 on the last one), from the windows there are.  A workgroup's slot is as large as the gradient of one
// stencil index: 3x3x3 512 -> 512 has slots of 28 MB, so the slots are held to 512 MiB, or to one per stencil index where
// that is more.  Wide layers fill the chip with their channel blocks alone (512 of them at 512 -> 512): with 18 slots
// instead of 66 that layer on 95 k particles takes 6.65 instead of 7.38 ms; up to 256 -> 256 the limit does not bind.
static void dwg_table(int code, int Cin, int Cout, int S_exp, int Lc, const WinLists& wl, DwG8Args& a) {
    const int nco = dwg_nco(Cout);
    a.Cin = Cin; a.Cout = Cout;
    a.CinP = (Cin + 15) / 16 * 16; a.CoutP = (Cout + 16 * nco - 1) / (16 * nco) * 16 * nco;
    a.n_s = 0;
    for (int k = 0; k < wl.n_lv; ++k) {                    // finest level first: stencil indices ascend
        const int s = std::min(S_exp - 1, Lc - wl.lv_level[k]);
        const int w0 = wl.lv_first[k], w1 = k + 1 < wl.n_lv ? wl.lv_first[k + 1] : wl.n_win;
        if (a.n_s > 0 && a.s_of[a.n_s - 1] == s) { a.nwin[a.n_s - 1] = w1 - a.win0[a.n_s - 1]; continue; }
        a.s_of[a.n_s] = s; a.win0[a.n_s] = w0; a.nwin[a.n_s] = w1 - w0; ++a.n_s;
    }
    const int64_t slots = ((int64_t)512 << 20) / dwg_slot_bytes(code, a);
    const int64_t bx = std::min<int64_t>(dwg_blocks_x(Cin, Cout), std::max<int64_t>(0, slots - a.n_s));
    a.blk0[0] = 0;
    for (int k = 0; k < a.n_s; ++k)                        // (together at most bx + n_s)
        a.blk0[k + 1] = a.blk0[k] + (int)std::max<int64_t>(1, std::min<int64_t>(a.nwin[k], bx * a.nwin[k] / wl.n_win));
}
// (not monotonous in the channels: the workgroups are rounded down)
size_t conv_dw_g8_part_bytes(int code, int Cin, int Cout, int S_exp, int Lc, const WinLists& wl) {
    DwG8Args a{};
    dwg_table(code, Cin, Cout, S_exp, Lc, wl, a);
    return (size_t)a.blk0[a.n_s] * dwg_slot_bytes(code, a);
}

template <class G>
static int launch_dw_g8_g(const DwG8Args& a, float* gw, hipStream_t st) {
    dim3 grid((unsigned)a.blk0[a.n_s], (unsigned)(a.CinP / 16), 1);
    if (dwg_nco(a.Cout) == 1) { grid.z = a.CoutP / 16; hipLaunchKernelGGL((conv_dw_g8_kernel<G, 1>), grid, dim3(G::NT), 0, st, a); }
    else { grid.z = a.CoutP / 32; hipLaunchKernelGGL((conv_dw_g8_kernel<G, 2>), grid, dim3(G::NT), 0, st, a); }
    APRNET_LAUNCH_CHECK("conv_dw_g8_kernel");
    const int64_t n = (int64_t)G::K * a.Cout * a.Cin;
    hipLaunchKernelGGL(dw_g8_reduce_kernel, dim3((unsigned)((n + 63) / 64), (unsigned)a.n_s), dim3(64 * DWG_RED_W), 0, st, a, (int)G::K, gw);
    APRNET_LAUNCH_CHECK("dw_g8_reduce_kernel");
    return 0;
}

// gw (of CinW input channels) += weight gradient of the input channels ci0 .. ci0 + Cin - 1, which are those of xi and ti;
// xi / ti / gyi grouped copies, fewer than 2^28 particles (32-bit byte offsets); `part` holds part_bytes, at least
// conv_dw_g8_part_bytes of Cin channels.  One launch for all stencil indices plus one for the sums.
int launch_conv_dw_g8(int code, const bf16_t* xi, int64_t xi_ld, int64_t x_count, const bf16_t* ti, int64_t ti_ld, int64_t t_count,
                      const bf16_t* gyi, int64_t gy_ld, int64_t gy_count, int Cin, int ci0, int CinW, int Cout, int S_exp, int Lc,
                      const WinLists& wl, float* part, size_t part_bytes, float* gw, hipStream_t st) {
    if (wl.n_win <= 0) return 0;
    DwG8Args a{};
    a.xi = xi; a.xi_ld = xi_ld; a.x_count = x_count; a.ti = ti; a.ti_ld = ti_ld; a.t_count = t_count;
    a.gyi = gyi; a.gy_ld = gy_ld; a.gy_count = gy_count;
    dwg_table(code, Cin, Cout, S_exp, Lc, wl, a);
    if ((size_t)a.blk0[a.n_s] * dwg_slot_bytes(code, a) > part_bytes)
        return fail(APRNET_ERR_INVALID_ARGUMENT, "weight gradient: the buffer for partial sums is too small");
    a.ci0 = ci0; a.CinW = CinW;
    a.win = wl.d_win; a.item_idx = wl.d_item_idx; a.item_pos = wl.d_item_pos; a.col_idx = wl.d_col_idx; a.col_pos = wl.d_col_pos;
    a.part = part;
    switch (code) {
        case 333: return launch_dw_g8_g<DG333>(a, gw, st);
        case 133: return launch_dw_g8_g<DG133>(a, gw, st);
        case 155: return launch_dw_g8_g<DG155>(a, gw, st);
    }
    return fail(APRNET_ERR_UNSUPPORTED, "no matrix-core kernel for this stencil");
}

}  // namespace aprnet
