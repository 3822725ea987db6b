// Stencil convolution backward on the matrix cores (fp32 MFMA), gfx950: gradient of the weights.
// (The gradient of the input is the forward kernel run on the output gradient with the transposed,
// flipped stencil, conv_mfma.hip.)
//
//   dW[s][co][ci][t] = sum over output positions (columns) of  gY[co][col] * patch[ci][pos(col) + off(t)]
//
// is a GEMM with M = 32 output channels, N = taps (27 of the 32 columns of the tile are used) and the
// columns of the window as the contracted axis, one 32x32 accumulator per input channel:
//
//     v_mfma_f32_32x32x2_f32:  D[co][t] += A[co][k] * B[k][t],   k = two columns of the window
//       A: lane l supplies gY[co = l%32] of column k = l/32      (LDS image gyl, laid out so that the
//                                                                  read is linear in the lane index)
//       B: lane l supplies patch[ci][pos(column k = l/32) + off(t = l%32)]
//
// A block owns 16 input channels (four staged chunks of 4) and 32 output channels.  Wave w takes input
// channel w%4 of every chunk and half of the columns (w/4), so it holds four accumulators, and keeps them
// in registers while the (persistent) block walks over many windows of one stencil index (one launch
// for all of them, see DwWork); its sums go to slots of its own (see DW_CHAINS), which sum_slots.hpp adds up in a fixed order.  The patch rows are 67 words
// apart so that the 27 tap offsets of a B read fall into 27 different LDS banks.
#include "conv_common.hpp"
#include "dw_work.hpp"
#include "sum_slots.hpp"

namespace aprnet {

typedef float floatx16 __attribute__((ext_vector_type(16)));
int bf16_math();       // conv.hip: bfloat16 features multiply on the bfloat16 matrix instructions (default) or in fp32

// row strides that put the tap offsets of one B read into different banks: 67 for 3-wide, 69 for 5-wide rows
using W333M = ConvGeom<3, 3, 3, 2, 4, 512, 67>;
using W133M = ConvGeom<1, 3, 3, 1, 8, 512, 67>;
using W155M = ConvGeom<1, 5, 5, 1, 8, 512, 69>;
constexpr int DW_CIB = 4;          // input channels per staged chunk
constexpr int DW_NCH = 4;          // chunks per block
constexpr int DW_GB = 256;         // columns of gY staged at a time
constexpr int DW_KB = 8;          // MFMAs issued back to back between operand phases (16 would spill registers)
constexpr int DW_GLD = 33;         // words per column of gyl (32 output channels + 1 against bank conflicts)

// The windows of this workgroup in turn, window(lists, columns, items, tree items) for each; flush(s, first) after every chain[k] of them
// and after the last one.
template <class G, typename T, class Window, class Flush>
__device__ __forceinline__ void dw_walk(const ConvArgs<T>& a, const DwWork& wk, const int bx, Window window, Flush flush) {
    int si = 0;
    while (si + 1 < wk.n_s && bx >= wk.blk0[si + 1]) ++si;
    const int n_run = wk.n_run[si], len = wk.len[si], rem = wk.rem[si], win0 = wk.win0[si], step = wk.blk0[si + 1] - wk.blk0[si];
    const int chain = wk.chain[si], s = wk.s_of[si];
    int left = chain;
    bool first = true;
    for (int run = bx - wk.blk0[si]; run < n_run; run += step) {
        const int w0 = win0 + run * len + min(run, rem), w1 = w0 + len + (run < rem ? 1 : 0);
        for (int w = w0; w < w1; ++w) {
            const int4 hd = a.win[w];
            const int nitem = __builtin_amdgcn_readfirstlane(hd.y), nc = __builtin_amdgcn_readfirstlane(hd.w);
            const WindowLists gl{a.l_item_idx + (unsigned)hd.x, a.l_item_pos + (unsigned)hd.x, a.l_col_idx + (unsigned)hd.z, a.l_col_pos + (unsigned)hd.z};
            window(gl, nc, nitem, w >= wk.first_coarse);
            if (--left == 0 || (w + 1 == w1 && run + step >= n_run)) { flush(s, first); left = chain; first = false; }
        }
    }
}

// Lists of the plan carry patch cells for rows of 64 words; this kernel's rows are RS words apart.
template <class G> __device__ __forceinline__ unsigned restride(unsigned pos) {
    return (pos & ~ITEM_CELL) | (((pos & ITEM_CELL) >> 6) * G::RS + (pos & 63u));
}

// Output gradient of one group of up to DW_GB columns -> LDS (through `put`), and the patch cell of every column of the
// group -> cpl.  Wave w takes output channels co0 + w, co0 + w + NWAVE, ... (NCO of them) of 64 columns per batch.
// The loads come in two rounds for the whole group -- column indices and cells of all batches (unconditional buffer
// loads, lanes past the group read zero), then the gradient values, those of batch b + 1 issued before the LDS stores
// of batch b -- instead of five dependent round trips per batch: a load under `c < ng`, or under `idx >= 0`, followed
// by its use makes the compiler wait for memory on the spot.
template <typename T, class G, int NCO, bool LISTS, class Lists, class Put>
__device__ __forceinline__ void stage_gy_group(const ConvArgs<T>& a, const Lists& sh, int g0, int ng, int co0, int co_end, int wave,
                                               int lane, int* __restrict__ cpl, Put put) {
    constexpr int NBM = DW_GB / 64;
    const int nbatch = (ng + 63) >> 6;
    int idx[NBM], pos[NBM];
    if constexpr (LISTS) {
        const __amdgpu_buffer_rsrc_t ri = __builtin_amdgcn_make_buffer_rsrc(const_cast<int*>(sh.col_idx + g0), 0, ng * 4, 0x00020000);
        const __amdgpu_buffer_rsrc_t rp = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned short*>(sh.col_pos + g0), 0, ng * 2, 0x00020000);
#pragma unroll
        for (int b = 0; b < NBM; ++b) {
            idx[b] = __builtin_amdgcn_raw_buffer_load_b32(ri, (b * 64 + lane) * 4, 0, 0);
            pos[b] = (int)__builtin_amdgcn_raw_buffer_load_b16(rp, (b * 64 + lane) * 2, 0, 0);
        }
    } else {
#pragma unroll
        for (int b = 0; b < NBM; ++b) {
            const int c = b * 64 + lane;
            idx[b] = c < ng ? sh.col_idx[g0 + c] : 0;
            pos[b] = c < ng ? (int)sh.col_pos[g0 + c] : 0;
        }
    }
    if (wave == 0) {        // patch cell of every column of the group, as a word offset
#pragma unroll
        for (int b = 0; b < NBM; ++b) {
            if (b >= nbatch) break;
            const int c = b * 64 + lane;
            cpl[c] = c < ng ? (LISTS ? (int)restride<G>((unsigned)pos[b]) : pos[b]) : G::TAP0;
        }
    }
    T cur[NCO], nxt[NCO];
    auto load = [&](int b, T (&v)[NCO]) {
#pragma unroll
        for (int k = 0; k < NCO; ++k) {
            const int co = co0 + wave + k * G::NWAVE;
            // (a lane past the group reads element 0 of the plane; its value is replaced by zero below)
            v[k] = a.gy[(int64_t)min(co, co_end - 1) * a.ldy + idx[b]];
        }
    };
    load(0, cur);
#pragma unroll
    for (int b = 0; b < NBM; ++b) {
        if (b >= nbatch) break;
        if (b + 1 < nbatch) load(b + 1 < NBM ? b + 1 : b, nxt);
        const int c = b * 64 + lane;
#pragma unroll
        for (int k = 0; k < NCO; ++k) {
            const int co = wave + k * G::NWAVE;
            put(b, c, co, cur[k], c < ng && co0 + co < co_end);
        }
#pragma unroll
        for (int k = 0; k < NCO; ++k) cur[k] = nxt[k];
    }
}

// One window: its output gradient goes to gyl in groups of DW_GB columns; per group the four channel chunks of
// the block are staged one after the other (the loads of the next chunk are issued before the matrix phase of
// the current one) and contracted with the group's columns.
template <typename T, class G, int CIB, int NCH, bool LISTS, class Lists>
__device__ __forceinline__ void dw_window(const ConvArgs<T>& a, const Lists& sh, int nc, int nitem, bool tree_items,
                                          int cig0, int co0, int bl, int kh, int hi, int wave, int lane,
                                          float* __restrict__ patch, float* __restrict__ gyl, int* __restrict__ cpl,
                                          const float* ap, floatx16 (&acc)[NCH]) {
    for (int i = threadIdx.x; i < CIB * G::CH_STRIDE; i += G::NT) patch[i] = 0.f;     // once per window
    ItemRegs<G, T, CIB> R;
    fetch_slots<G, T, CIB>(sh, nitem, R);
    if constexpr (LISTS) {
#pragma unroll
        for (int k = 0; k < ItemRegs<G, T, CIB>::IPT; ++k)
            if (R.pos[k] != 0xffffu) R.pos[k] = (unsigned short)restride<G>(R.pos[k]);
    }
    load_values<G, T, CIB>(a, cig0, nitem, tree_items, R);
    for (int g0 = 0; g0 < nc; g0 += DW_GB) {
        const int ng = min(DW_GB, nc - g0), nbatch = (ng + 63) >> 6;
        // output gradient of this group of columns -> gyl; a wave reads 64 columns of one channel
        stage_gy_group<T, G, 32 / G::NWAVE, LISTS>(a, sh, g0, ng, co0, a.Cout, wave, lane, cpl,
            [&](int b, int, int co, T v, bool valid) {
                const int slot = b * 64 + 2 * (lane & 31) + (lane >> 5);
                gyl[slot * DW_GLD + co] = valid ? Num<T>::ld(v) : 0.f;
            });
#pragma unroll
        for (int q = 0; q < NCH; ++q) {
            __syncthreads();        // previous chunk's reads of the patch are done / gyl is written
            store_items<G, T, CIB>(R, nitem, patch);
            __syncthreads();
            if (q + 1 < NCH) load_values<G, T, CIB>(a, cig0 + (q + 1) * CIB, nitem, tree_items, R);
            else if (g0 + DW_GB < nc) load_values<G, T, CIB>(a, cig0, nitem, tree_items, R);     // next group starts over
#pragma unroll 1
            for (int b = 0; b < nbatch; ++b) {
                const float* apb = ap + (b * 64 + 32 * kh) * DW_GLD;
                // Three separate phases, kept apart by scheduling barriers: operand addresses (one LDS read of the
                // column's cell and one vector add each), then the operand reads, then DW_KB MFMAs back to back.  A
                // vector instruction between two fp32 MFMAs costs a pipeline switch each time.
                const int* cp = cpl + b * 64 + 32 * hi + 16 * kh;      // lanes of the upper half take column k + 32
#pragma unroll
                for (int h = 0; h < 16; h += DW_KB) {
                    int addr[DW_KB];
#pragma unroll
                    for (int k = 0; k < DW_KB; ++k) addr[k] = bl + cp[h + k];
                    __builtin_amdgcn_sched_barrier(0);
                    float av[DW_KB], bv[DW_KB];
#pragma unroll
                    for (int k = 0; k < DW_KB; ++k) { av[k] = apb[2 * (h + k) * DW_GLD]; bv[k] = patch[addr[k]]; }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int k = 0; k < DW_KB; ++k) acc[q] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[k], bv[k], acc[q], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        __syncthreads();            // gyl is rewritten by the next group, the patch by the next window
    }
}

// ---------------------------------------------------------------------------------------------------------
// Layers of at most 16 output channels (the finest stages of the networks): the 32-row instruction above would
// multiply 16 rows of zeros.  Here D is 16 output channels x 16 taps on v_mfma_f32_16x16x4_f32, two tap tiles per
// input channel (taps 0-15 and 16-31), four columns per instruction:
//     A: lane l supplies gY[co = l%16] of column l/16 of the four            (gyl16[column][co], 17 words per column:
//                                                                              conflict-free writes by column, reads
//                                                                              with a few two-way conflicts)
//     B: lane l supplies patch[ci][cell(column l/16) + off(t = l%16 + 16 * tile)]
// Twice the columns per matrix-pipe cycle of the 32x32x2 form for such layers; same staging, same work split
// (wave w: input channel w%4 of each chunk, half w/4 of every 64 columns).
typedef float floatx4d __attribute__((ext_vector_type(4)));
constexpr int DW_GLD16 = 17;

template <typename T, class G, int CIB, int NCH, bool LISTS, class Lists>
__device__ __forceinline__ void dw_window16(const ConvArgs<T>& a, const Lists& sh, int nc, int nitem, bool tree_items,
                                            int cig0, const int (&bl)[2], int kh, int wave, int lane,
                                            float* __restrict__ patch, float* __restrict__ gyl, int* __restrict__ cpl,
                                            floatx4d (&acc)[NCH][2]) {
    for (int i = threadIdx.x; i < CIB * G::CH_STRIDE; i += G::NT) patch[i] = 0.f;     // once per window
    ItemRegs<G, T, CIB> R;
    fetch_slots<G, T, CIB>(sh, nitem, R);
    if constexpr (LISTS) {
#pragma unroll
        for (int k = 0; k < ItemRegs<G, T, CIB>::IPT; ++k)
            if (R.pos[k] != 0xffffu) R.pos[k] = (unsigned short)restride<G>(R.pos[k]);
    }
    load_values<G, T, CIB>(a, cig0, nitem, tree_items, R);
    const int q4 = lane >> 4;                                   // which of the four columns of an instruction
    const float* ap = gyl + q4 * DW_GLD16 + (lane & 15);
    for (int g0 = 0; g0 < nc; g0 += DW_GB) {
        const int ng = min(DW_GB, nc - g0), nbatch = (ng + 63) >> 6;
        stage_gy_group<T, G, 16 / G::NWAVE, LISTS>(a, sh, g0, ng, 0, a.Cout, wave, lane, cpl,
            [&](int, int c, int co, T v, bool valid) { gyl[c * DW_GLD16 + co] = valid ? Num<T>::ld(v) : 0.f; });
#pragma unroll
        for (int q = 0; q < NCH; ++q) {
            __syncthreads();        // previous chunk's reads of the patch are done / gyl is written
            store_items<G, T, CIB>(R, nitem, patch);
            __syncthreads();
            if (q + 1 < NCH) load_values<G, T, CIB>(a, cig0 + (q + 1) * CIB, nitem, tree_items, R);
            else if (g0 + DW_GB < nc) load_values<G, T, CIB>(a, cig0, nitem, tree_items, R);     // next group starts over
#pragma unroll 1
            for (int b = 0; b < nbatch; ++b) {
                const int c0 = b * 64 + 32 * kh;                 // this wave's 32 columns of the batch
                if (c0 >= ng) break;                             // wave-uniform: nothing but padding left
                const int* cp = cpl + c0 + q4;
                const float* apb = ap + c0 * DW_GLD16;
                int cell[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) cell[k] = cp[4 * k];
                __builtin_amdgcn_sched_barrier(0);
                float av[8], b0[8], b1[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) { av[k] = apb[4 * k * DW_GLD16]; b0[k] = patch[bl[0] + cell[k]]; b1[k] = patch[bl[1] + cell[k]]; }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    acc[q][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[k], b0[k], acc[q][0], 0, 0, 0);
                    acc[q][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[k], b1[k], acc[q][1], 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __syncthreads();            // gyl is rewritten by the next group, the patch by the next window
    }
}

template <typename T, class G, int CIB, int NCH, bool LISTS>
__device__ __forceinline__ void dw16_block(const ConvArgs<T>& a, const DwWork& wk, const int s_arg, const int bx, const int by) {
    static_assert(G::NWAVE == 8 && CIB == 4, "wave w owns input channel w%4 and column half w/4");
    __shared__ float patch[CIB * G::CH_STRIDE];
    __shared__ float gyl[DW_GB * DW_GLD16];
    __shared__ int cpl[DW_GB];

    const int cig0 = by * (CIB * NCH);
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int cil = wave & 3, kh = wave >> 2;
    int bl[2];
#pragma unroll
    for (int tile = 0; tile < 2; ++tile) {
        const int t = (lane & 15) + 16 * tile;
        const int tt = t < G::K ? t : 0;
        const int toff = ((tt / (G::KX * G::KY)) * G::RX + (tt / G::KY) % G::KX) * G::RS + (tt % G::KY);
        bl[tile] = cil * G::CH_STRIDE - G::TAP0 + toff;       // B operand: + cell of the column
    }
    floatx4d acc[NCH][2];
#pragma unroll
    for (int q = 0; q < NCH; ++q)
#pragma unroll
        for (int tile = 0; tile < 2; ++tile)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[q][tile][r] = 0.f;

    // the sums so far to this workgroup's slot of its column half (first: they start it)
    auto flush = [&](const int s, const bool first) {
        int l = lane;
        asm volatile("" : "+v"(l));         // addresses formed per call, not kept (and spilled) across the window loop
        const DwSlot slot(a, bx, 0, kh, 16, G::K, s);
#pragma unroll
        for (int q = 0; q < NCH; ++q)
#pragma unroll
            for (int tile = 0; tile < 2; ++tile)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (cig0 + q * CIB + cil < a.Cin) slot.add(4 * (l >> 4) + r, cig0 + q * CIB + cil, (l & 15) + 16 * tile, acc[q][tile][r], first);
                    acc[q][tile][r] = 0.f;
                }
    };
    if constexpr (LISTS) {
        dw_walk<G>(a, wk, bx, [&](const WindowLists& gl, int nc, int nitem, bool tree_items) {
            dw_window16<T, G, CIB, NCH, true>(a, gl, nc, nitem, tree_items, cig0, bl, kh, wave, lane, patch, gyl, cpl, acc);
        }, flush);
    } else {
        for (int ti = blockIdx.x; ti < a.n_tiles; ti += gridDim.x) {
            const ConvTile tile = a.tiles[ti];
            const int L = tile.level;
            const bool tree_items = L < a.Lc;
            __shared__ ConvShared<G> sh;
            const int yn = a.apr.y_num[L];
            const bool out_tree = (L == a.Lc) && (L < a.apr.level_max);
            __syncthreads();
            open_segments<G, T>(a, L, tile.z0, tile.x0, sh);
            __syncthreads();
            for (int y0 = 0; y0 < yn; y0 += G::TY) {
                scan_window<G, T>(a, L, y0, out_tree, sh);
                __syncthreads();
                const int nc = __builtin_amdgcn_readfirstlane(sh.ncol), nitem = __builtin_amdgcn_readfirstlane(sh.nitem);
                if (nc > 0) dw_window16<T, G, CIB, NCH, false>(a, sh, nc, nitem, tree_items, cig0, bl, kh, wave, lane, patch, gyl, cpl, acc);
                __syncthreads();
                close_window<G>(sh);
                __syncthreads();
            }
        }
        flush(s_arg, true);
    }
}

// ---------------------------------------------------------------------------------------------------------
// bfloat16 features and output gradient: the same contraction on v_mfma_f32_32x32x16_bf16 (16 columns per
// instruction, fp32 accumulation).  Both operands are bfloat16 values as loaded, so the products are the exact
// ones the fp32 kernel forms; only the order of the fp32 sums differs.
//     A: lane l supplies gY[co = l%32] of columns 8*(l/32) .. +7 of a group of 16: one 16-byte read from
//        gyl16[co][column] (rows DW_LDG16 apart)
//     B: lane l supplies patch16[ci][cell(column) + off(t = l%32)] of the same 8 columns: 8 two-byte reads
// An instruction does the work of eight of the fp32 ones, so the loop is bound by its LDS reads.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
constexpr int DW_LDG16 = DW_GB + 8;            // 16-byte aligned rows, 4 banks apart

template <class G, int CIB, int NCH, bool LISTS, class Lists>
__device__ __forceinline__ void dw_window_bf16(const ConvArgs<bf16_t>& a, const Lists& sh, int nc, int nitem, bool tree_items,
                                               int cig0, int co0, int bl, int kh, int hi, int wave, int lane,
                                               unsigned short* __restrict__ patch, unsigned short* __restrict__ gyl,
                                               int* __restrict__ cpl, floatx16 (&acc)[NCH]) {
    for (int i = threadIdx.x; i < CIB * G::CH_STRIDE / 2; i += G::NT) reinterpret_cast<unsigned*>(patch)[i] = 0u;   // once per window
    ItemRegs<G, bf16_t, CIB> R;
    fetch_slots<G, bf16_t, CIB>(sh, nitem, R);
    if constexpr (LISTS) {
#pragma unroll
        for (int k = 0; k < ItemRegs<G, bf16_t, CIB>::IPT; ++k)
            if (R.pos[k] != 0xffffu) R.pos[k] = (unsigned short)restride<G>(R.pos[k]);
    }
    load_values<G, bf16_t, CIB>(a, cig0, nitem, tree_items, R);
    for (int g0 = 0; g0 < nc; g0 += DW_GB) {
        const int ng = min(DW_GB, nc - g0), nbatch = (ng + 63) >> 6;
        stage_gy_group<bf16_t, G, 32 / G::NWAVE, LISTS>(a, sh, g0, ng, co0, a.Cout, wave, lane, cpl,
            [&](int, int c, int co, bf16_t v, bool valid) { gyl[co * DW_LDG16 + c] = valid ? v.bits : (unsigned short)0; });
#pragma unroll
        for (int q = 0; q < NCH; ++q) {
            __syncthreads();        // previous chunk's reads of the patch are done / gyl is written
#pragma unroll
            for (int k = 0; k < ItemRegs<G, bf16_t, CIB>::IPT; ++k) {
                if (k * G::NT >= nitem) break;       // wave-uniform
                if (R.pos[k] == 0xffffu) continue;
                unsigned short* cell = patch + (R.pos[k] & ITEM_CELL);
#pragma unroll
                for (int c = 0; c < CIB; ++c) {
                    const unsigned short v = (unsigned short)R.v[k][c];
                    cell[c * G::CH_STRIDE] = v;
                    if (R.pos[k] & ITEM_PAIR) cell[c * G::CH_STRIDE + 1] = v;
                }
            }
            __syncthreads();
            if (q + 1 < NCH) load_values<G, bf16_t, CIB>(a, cig0 + (q + 1) * CIB, nitem, tree_items, R);
            else if (g0 + DW_GB < nc) load_values<G, bf16_t, CIB>(a, cig0, nitem, tree_items, R);     // next group starts over
#pragma unroll 1
            for (int b = 0; b < nbatch; ++b) {
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const int c0 = b * 64 + 32 * kh + 16 * s;           // first of this instruction's 16 columns
                    if (c0 >= ng) break;                                // wave-uniform: nothing but padding left
                    const int4 ca = *reinterpret_cast<const int4*>(cpl + c0 + 8 * hi);
                    const int4 cb = *reinterpret_cast<const int4*>(cpl + c0 + 8 * hi + 4);
                    const int cell[8] = {ca.x, ca.y, ca.z, ca.w, cb.x, cb.y, cb.z, cb.w};
                    unsigned w[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        w[j] = (unsigned)patch[bl + cell[2 * j]] | ((unsigned)patch[bl + cell[2 * j + 1]] << 16);
                    const uint4 av = *reinterpret_cast<const uint4*>(gyl + (lane & 31) * DW_LDG16 + c0 + 8 * hi);
                    const uint4 bv = make_uint4(w[0], w[1], w[2], w[3]);
                    acc[q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, av), __builtin_bit_cast(bf16x8, bv),
                                                                     acc[q], 0, 0, 0);
                }
            }
        }
        __syncthreads();            // gyl is rewritten by the next group, the patch by the next window
    }
}

template <class G, int CIB, int NCH, bool LISTS>
__global__ void __launch_bounds__(G::NT) __attribute__((amdgpu_waves_per_eu(4, 4)))
conv_dw_bf16_kernel(const ConvArgs<bf16_t> a, const DwWork wk, const int s_arg) {
    static_assert(G::NWAVE == 8 && CIB == 4, "wave w owns input channel w%4 and column half w/4");
    static_assert(G::CH_STRIDE % 2 == 0 && DW_LDG16 % 8 == 0, "dword fill of the patch, 16-byte rows of gyl");
    __shared__ __attribute__((aligned(16))) unsigned short patch[CIB * G::CH_STRIDE];
    __shared__ __attribute__((aligned(16))) unsigned short gyl[32 * DW_LDG16];
    __shared__ __attribute__((aligned(16))) int cpl[DW_GB];

    const int cig0 = blockIdx.y * (CIB * NCH), co0 = blockIdx.z * 32;
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int cil = wave & 3, kh = wave >> 2;
    const int t = lane & 31, hi = lane >> 5;
    const int tt = t < G::K ? t : 0;
    const int toff = ((tt / (G::KX * G::KY)) * G::RX + (tt / G::KY) % G::KX) * G::RS + (tt % G::KY);
    const int bl = cil * G::CH_STRIDE - G::TAP0 + toff;       // B operand: + cell of the column

    floatx16 acc[NCH];
#pragma unroll
    for (int q = 0; q < NCH; ++q)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[q][r] = 0.f;

    // the sums so far to this workgroup's slot of its column half (first: they start it)
    auto flush = [&](const int s, const bool first) {
        int l = lane;
        asm volatile("" : "+v"(l));         // addresses formed per call, not kept (and spilled) across the window loop
        const DwSlot slot(a, blockIdx.x, co0, kh, 32, G::K, s);
#pragma unroll
        for (int q = 0; q < NCH; ++q)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                if (cig0 + q * CIB + cil < a.Cin) slot.add(4 * (l >> 5) + 8 * (r >> 2) + (r & 3), cig0 + q * CIB + cil, l & 31, acc[q][r], first);
                acc[q][r] = 0.f;
            }
    };
    if constexpr (LISTS) {
        dw_walk<G>(a, wk, blockIdx.x, [&](const WindowLists& gl, int nc, int nitem, bool tree_items) {
            dw_window_bf16<G, CIB, NCH, true>(a, gl, nc, nitem, tree_items, cig0, co0, bl, kh, hi, wave, lane, patch, gyl, cpl, acc);
        }, flush);
    } else {
        for (int ti = blockIdx.x; ti < a.n_tiles; ti += gridDim.x) {
            const ConvTile tile = a.tiles[ti];
            const int L = tile.level;
            const bool tree_items = L < a.Lc;
            __shared__ ConvShared<G> sh;
            const int yn = a.apr.y_num[L];
            const bool out_tree = (L == a.Lc) && (L < a.apr.level_max);
            __syncthreads();
            open_segments<G, bf16_t>(a, L, tile.z0, tile.x0, sh);
            __syncthreads();
            for (int y0 = 0; y0 < yn; y0 += G::TY) {
                scan_window<G, bf16_t>(a, L, y0, out_tree, sh);
                __syncthreads();
                const int nc = __builtin_amdgcn_readfirstlane(sh.ncol), nitem = __builtin_amdgcn_readfirstlane(sh.nitem);
                if (nc > 0) dw_window_bf16<G, CIB, NCH, false>(a, sh, nc, nitem, tree_items, cig0, co0, bl, kh, hi, wave, lane, patch, gyl, cpl, acc);
                __syncthreads();
                close_window<G>(sh);
                __syncthreads();
            }
        }
        flush(s_arg, true);
    }
}

// T: storage type of the features and of the output gradient (float, or bfloat16 widened to fp32 on load).
// LISTS: the windows come from the plan's lists; otherwise the block scans the access arrays.
template <typename T, class G, int CIB, int NCH, bool LISTS>
__device__ __forceinline__ void dw_block(const ConvArgs<T>& a, const DwWork& wk, const int s_arg, const int bx, const int by, const int bz) {
    static_assert(G::NWAVE == 8 && CIB == 4, "wave w owns input channel w%4 and column half w/4");
    __shared__ float patch[CIB * G::CH_STRIDE];
    __shared__ float gyl[DW_GB * DW_GLD];
    __shared__ int cpl[DW_GB];

    const int cig0 = by * (CIB * NCH), co0 = bz * 32;
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int cil = wave & 3, kh = wave >> 2;
    const int t = lane & 31, hi = lane >> 5;
    const int tt = t < G::K ? t : 0;
    const int toff = ((tt / (G::KX * G::KY)) * G::RX + (tt / G::KY) % G::KX) * G::RS + (tt % G::KY);
    const int bl = cil * G::CH_STRIDE - G::TAP0 + toff;       // B operand: + cell of the column
    const float* ap = gyl + lane + hi;                        // A operand: + (64 * batch + 2 * kk) * DW_GLD

    floatx16 acc[NCH];
#pragma unroll
    for (int q = 0; q < NCH; ++q)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[q][r] = 0.f;

    // the sums so far to this workgroup's slot of its column half (first: they start it)
    auto flush = [&](const int s, const bool first) {
        int l = lane;
        asm volatile("" : "+v"(l));         // addresses formed per call, not kept (and spilled) across the window loop
        const DwSlot slot(a, bx, co0, kh, 32, G::K, s);
#pragma unroll
        for (int q = 0; q < NCH; ++q)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                if (cig0 + q * CIB + cil < a.Cin) slot.add(4 * (l >> 5) + 8 * (r >> 2) + (r & 3), cig0 + q * CIB + cil, l & 31, acc[q][r], first);
                acc[q][r] = 0.f;
            }
    };
    if constexpr (LISTS) {
        dw_walk<G>(a, wk, bx, [&](const WindowLists& gl, int nc, int nitem, bool tree_items) {
            dw_window<T, G, CIB, NCH, true>(a, gl, nc, nitem, tree_items, cig0, co0, bl, kh, hi, wave, lane, patch, gyl, cpl, ap, acc);
        }, flush);
    } else {
        for (int ti = blockIdx.x; ti < a.n_tiles; ti += gridDim.x) {
            const ConvTile tile = a.tiles[ti];
            const int L = tile.level;
            const bool tree_items = L < a.Lc;
            __shared__ ConvShared<G> sh;
            const int yn = a.apr.y_num[L];
            const bool out_tree = (L == a.Lc) && (L < a.apr.level_max);
            __syncthreads();
            open_segments<G, T>(a, L, tile.z0, tile.x0, sh);
            __syncthreads();
            for (int y0 = 0; y0 < yn; y0 += G::TY) {
                scan_window<G, T>(a, L, y0, out_tree, sh);
                __syncthreads();
                const int nc = __builtin_amdgcn_readfirstlane(sh.ncol), nitem = __builtin_amdgcn_readfirstlane(sh.nitem);
                if (nc > 0) dw_window<T, G, CIB, NCH, false>(a, sh, nc, nitem, tree_items, cig0, co0, bl, kh, hi, wave, lane, patch, gyl, cpl, ap, acc);
                __syncthreads();
                close_window<G>(sh);
                __syncthreads();
            }
        }
        flush(s_arg, true);
    }
}

template <typename T, class G, int CIB, int NCH, bool LISTS>
__global__ void __launch_bounds__(G::NT) __attribute__((amdgpu_waves_per_eu(4, 4)))
conv_dw16_mfma_kernel(const ConvArgs<T> a, const DwWork wk, const int s_arg) {
    dw16_block<T, G, CIB, NCH, LISTS>(a, wk, s_arg, blockIdx.x, blockIdx.y);
}
template <typename T, class G, int CIB, int NCH, bool LISTS>
__global__ void __launch_bounds__(G::NT) __attribute__((amdgpu_waves_per_eu(4, 4)))
conv_dw_mfma_kernel(const ConvArgs<T> a, const DwWork wk, const int s_arg) {
    dw_block<T, G, CIB, NCH, LISTS>(a, wk, s_arg, blockIdx.x, blockIdx.y, blockIdx.z);
}
// The blocks (nx, ny, nz) of one of the two again, where the products of bfloat16 pieces did not come out finite (*a.redo,
// conv_dw_split.hip).  Few workgroups, which end at once otherwise: as many as there are blocks, up to 16,000 with 128 channels each way,
// they took longer to launch than the pieces gained.
template <class G, int CIB, int NCH, bool M16>
__global__ void __launch_bounds__(G::NT) __attribute__((amdgpu_waves_per_eu(4, 4)))
conv_dw_redo_kernel(const ConvArgs<float> a, const DwWork wk, const int nx, const int ny, const int nz) {
    if (*a.redo == 0) return;
    for (int u = blockIdx.x; u < nx * ny * nz; u += gridDim.x) {          // uniform
        if constexpr (M16) dw16_block<float, G, CIB, NCH, true>(a, wk, 0, u % nx, u / nx);
        else dw_block<float, G, CIB, NCH, true>(a, wk, 0, u % nx, u / nx % ny, u / nx / ny);
        __syncthreads();
    }
}

static int dw_taps(int code) { return code == 333 ? 27 : code == 133 ? 9 : 25; }
// a narrow input (the first layer of a network) fits one chunk: no staging and products of empty chunks
static int dw_chunks(int Cin) { return Cin <= DW_CIB ? 1 : DW_NCH; }
// Slots for partial sums: two for each of `blocks` workgroups along grid.x, within 512 MiB, but 16 workgroups at least.
static int dw_slot_cap(int code, int Cout, int Cin, int blocks) {
    const int64_t cap = ((int64_t)512 << 20) / (8 * (int64_t)Cout * Cin * dw_taps(code));
    return (int)std::max<int64_t>(16, std::min<int64_t>(blocks, cap));
}
// Workgroups along grid.x of a launch on lists: the 512 that the chip holds, two rounds of them for layers of one channel block.
static int dw_blocks_x(int code, int Cout, int Cin) {
    const int nci = DW_CIB * dw_chunks(Cin), per = ((Cin + nci - 1) / nci) * ((Cout + 31) / 32);
    return dw_slot_cap(code, Cout, Cin, std::max(512, 1024 / per));
}
// Windows whose products a workgroup adds up in registers before the sums go to its slots: the relative error of a sum of n products
// of either sign grows with the root of the additions that one accumulator sees.  A chain ends after a 512th of the stencil index's
// windows (of fewer where the slots are, see above), but not before DW_SHORT windows: the few windows of a coarse level in chains of one
// cost 3 to 10 % for nothing, since their gradient's error is below that of the finest level's all the same.
// 64 -> 64 channels on 2.8 M particles, error against 64 bits 0.85e-6, 9.7 ms, with 128 workgroups and chains to their end 1.95e-6, 9.9 ms;
// on 320 k 0.34e-6, 1.54 ms (0.63e-6, 1.38); 128 -> 128 on 320 k 0.52e-6, 4.95 ms (0.87e-6, 4.75); 32 -> 32 on 9.8 M 1.38e-6, 8.95 ms
// (1.66e-6, 8.75); 16 -> 16 on 9.8 M 1.14e-6, 3.19 ms (1.15e-6, 3.20).  Read back, added and stored instead of added by atomic
// operations that nobody waits for, 64 -> 64 took 11.5 and 1.73 ms.
constexpr int DW_CHAINS = 512, DW_SHORT = 4;
// Neighbouring windows of a run, where there are that many per workgroup: they read the same lines along y.  64 -> 64 channels on 320 k
// particles 1.54 -> 1.47 ms, 32 -> 32 0.47 -> 0.45 ms; runs of 16, whose windows are dense or sparse together, 32 -> 32 on 9.8 M 9.0 -> 9.7 ms.
constexpr int DW_RUN = 4;
// A window without a column costs a workgroup about what 256 columns cost it.  By windows alone the finest level's workgroups, whose windows
// are fuller, were the last to end: backward pass of 1x5x5 64 -> 64 on bfloat16
// planes, 15.4 M particles, 29.0 -> 28.3 ms (32.3 with 128 workgroups), 32 -> 32 on 2.8 M 2.83 -> 2.72 ms.
constexpr int DW_WINDOW_COST = 256;
// The stencil indices that have windows, and a share of the workgroups for each: one, and of the others by the cost of its windows.
DwWork dw_work(int code, int Cout, int Cin, int S_exp, int Lc, const WinLists& wl) {
    DwWork k{};
    k.first_coarse = (wl.n_lv > 0 && wl.lv_level[0] == Lc) ? (wl.n_lv > 1 ? wl.lv_first[1] : wl.n_win) : 0;
    int64_t cost[MAX_LEVELS + 1] = {}, total = 0;
    for (int i = 0; i < wl.n_lv; ++i) {                    // finest level first: stencil indices ascend
        const int s = std::min(S_exp - 1, Lc - wl.lv_level[i]);
        const int w0 = wl.lv_first[i], w1 = i + 1 < wl.n_lv ? wl.lv_first[i + 1] : wl.n_win;
        if (k.n_s == 0 || k.s_of[k.n_s - 1] != s) { k.s_of[k.n_s] = s; k.win0[k.n_s] = w0; ++k.n_s; }
        k.nwin[k.n_s - 1] = w1 - k.win0[k.n_s - 1];
        const int64_t c = wl.lv_cols[i] + (int64_t)DW_WINDOW_COST * (w1 - w0);
        cost[k.n_s - 1] += c; total += c;
    }
    const int chains = dw_slot_cap(code, Cout, Cin, DW_CHAINS), longest = (*std::max_element(k.nwin, k.nwin + k.n_s) + chains - 1) / chains;
    const int64_t more = std::max(0, dw_blocks_x(code, Cout, Cin) - k.n_s);
    for (int i = 0; i < k.n_s; ++i) {
        const int nb = (int)std::min<int64_t>(k.nwin[i], 1 + more * cost[i] / total);
        k.blk0[i + 1] = k.blk0[i] + nb;
        k.n_run[i] = nb * std::max(1, k.nwin[i] / (nb * DW_RUN));              // at most nwin: no run is empty
        k.len[i] = k.nwin[i] / k.n_run[i]; k.rem[i] = k.nwin[i] % k.n_run[i];
        k.chain[i] = std::max((k.nwin[i] + chains - 1) / chains, std::min(DW_SHORT, longest));
    }
    return k;
}
// wl null: the kernels scan
size_t conv_dw_partial_bytes(int code, int Cout, int Cin, int S_exp, int Lc, const WinLists* wl) {
    const int blocks = wl ? [&] { const DwWork k = dw_work(code, Cout, Cin, S_exp, Lc, *wl); return k.blk0[k.n_s]; }() : dw_slot_cap(code, Cout, Cin, DW_CHAINS);
    return (size_t)(2 * blocks) * Cout * Cin * dw_taps(code) * sizeof(float);
}

template <typename T, class G, bool LISTS>
static int launch_dw_kernel(const ConvArgs<T>& a, const DwWork& k, int s, int blocks, hipStream_t st) {
    const int nch = dw_chunks(a.Cin);
    dim3 grid((unsigned)blocks, (unsigned)((a.Cin + DW_CIB * nch - 1) / (DW_CIB * nch)), (unsigned)((a.Cout + 31) / 32));
    if constexpr (std::is_same<T, float>::value && LISTS && G::K != 9) {
        if (a.redo) {
            const int nx = (int)grid.x, ny = (int)grid.y, nz = (int)grid.z;
            const dim3 few((unsigned)std::min<int64_t>((int64_t)nx * ny * nz, 512));
#define APRNET_REDO(N, M16) hipLaunchKernelGGL((conv_dw_redo_kernel<G, DW_CIB, N, M16>), few, dim3(G::NT), 0, st, a, k, nx, ny, nz)
            if (a.Cout <= 16) { if (nch == 1) APRNET_REDO(1, true); else APRNET_REDO(DW_NCH, true); }
            else { if (nch == 1) APRNET_REDO(1, false); else APRNET_REDO(DW_NCH, false); }
#undef APRNET_REDO
            APRNET_LAUNCH_CHECK("conv_dw_redo_kernel");
            return 0;
        }
    }
    if constexpr (std::is_same<T, bf16_t>::value) {
        if (bf16_math()) {      // bfloat16 matrix instructions; the fp32 ones below when those are asked for
            if (nch == 1) hipLaunchKernelGGL((conv_dw_bf16_kernel<G, DW_CIB, 1, LISTS>), grid, dim3(G::NT), 0, st, a, k, s);
            else hipLaunchKernelGGL((conv_dw_bf16_kernel<G, DW_CIB, DW_NCH, LISTS>), grid, dim3(G::NT), 0, st, a, k, s);
            APRNET_LAUNCH_CHECK("conv_dw_bf16_kernel");
            return 0;
        }
    }
    if (a.Cout <= 16) {         // 16-row form
        if (nch == 1) hipLaunchKernelGGL((conv_dw16_mfma_kernel<T, G, DW_CIB, 1, LISTS>), grid, dim3(G::NT), 0, st, a, k, s);
        else hipLaunchKernelGGL((conv_dw16_mfma_kernel<T, G, DW_CIB, DW_NCH, LISTS>), grid, dim3(G::NT), 0, st, a, k, s);
        APRNET_LAUNCH_CHECK("conv_dw16_mfma_kernel");
        return 0;
    }
    if (nch == 1) hipLaunchKernelGGL((conv_dw_mfma_kernel<T, G, DW_CIB, 1, LISTS>), grid, dim3(G::NT), 0, st, a, k, s);
    else hipLaunchKernelGGL((conv_dw_mfma_kernel<T, G, DW_CIB, DW_NCH, LISTS>), grid, dim3(G::NT), 0, st, a, k, s);
    APRNET_LAUNCH_CHECK("conv_dw_mfma_kernel");
    return 0;
}

// Weight gradient; a.gw is accumulated into (the caller zeroes it).  The partial sums of a launch are added up in slot order
// (every slot of the grid is written in full).
template <typename T, class G>
static int launch_dw(const ConvArgs<T>& a0, const TileList& tl, const WinLists* wl, int level_min, hipStream_t st) {
    const int code = G::KZ * 100 + G::KX * 10 + G::KY;
    const int64_t n_el = (int64_t)a0.Cout * a0.Cin * G::K;
    if (a0.win_level && wl) {
        if (wl->n_win <= 0) return 0;
        const DwWork k = dw_work(code, a0.Cout, a0.Cin, a0.S_exp, a0.Lc, *wl);
        if (int rc = launch_dw_kernel<T, G, true>(a0, k, 0, k.blk0[k.n_s], st)) return rc;
        if (!a0.gw_part) return 0;
        SlotGroups g{};
        g.n = k.n_s;
        for (int i = 0; i < k.n_s; ++i) { g.first[i] = 2 * k.blk0[i]; g.out[i] = k.s_of[i]; }
        g.first[k.n_s] = 2 * k.blk0[k.n_s];
        return launch_sum_slot_groups((const float*)a0.gw_part, a0.gw_part_ld, g, n_el, (float*)a0.gw, st, a0.redo);
    }
    // scanning kernels: one launch per stencil index, level Lc - s for s < S_exp - 1, every coarser level for the last one
    // (adjacent in the tile list, which is sorted finest level first)
    for (int s = 0; s < a0.S_exp; ++s) {
        const int l_hi = a0.Lc - s, l_lo = (s == a0.S_exp - 1) ? level_min : l_hi;
        if (l_hi < level_min) break;
        int n = 0;
        for (int l = l_lo; l <= l_hi; ++l) n += tl.level_count[l];
        if (n == 0) continue;
        ConvArgs<T> a = a0;
        a.tiles = tl.d_tiles + tl.level_begin[l_hi]; a.n_tiles = n;
        const int blocks = std::min(n, a.gw_part ? dw_slot_cap(code, a.Cout, a.Cin, DW_CHAINS) : DW_CHAINS);
        if (int rc = launch_dw_kernel<T, G, false>(a, DwWork{}, s, blocks, st)) return rc;
        if (a.gw_part)
            if (int rc = launch_sum_slots((const float*)a.gw_part, a.gw_part_ld, 2 * blocks, n_el, (float*)a.gw + (int64_t)s * n_el, st)) return rc;
    }
    return 0;
}

template <typename T>
static int launch_dw_code(int code, const ConvArgs<T>& a, const TileList& tl, const WinLists* wl, int level_min, hipStream_t st) {
    switch (code) {
        case 333: return launch_dw<T, W333M>(a, tl, wl, level_min, st);
        case 133: return launch_dw<T, W133M>(a, tl, wl, level_min, st);
        case 155: return launch_dw<T, W155M>(a, tl, wl, level_min, st);
    }
    return fail(APRNET_ERR_UNSUPPORTED, "no matrix-core kernel for this stencil");
}
int launch_conv_dw_mfma(int code, const ConvArgs<float>& a, const TileList& tl, const WinLists* wl, int level_min, hipStream_t st) {
    return launch_dw_code<float>(code, a, tl, wl, level_min, st);
}
int launch_conv_dw_mfma(int code, const ConvArgs<bf16_t>& a, const TileList& tl, const WinLists* wl, int level_min, hipStream_t st) {
    return launch_dw_code<bf16_t>(code, a, tl, wl, level_min, st);
}

}  // namespace aprnet
