// Stencil convolution of fp32 features on the bfloat16 matrix instructions, gfx950: every fp32 operand as three bfloat16
// pieces.
//
// An fp32 value is the exact sum of three bfloat16 numbers: x = x1 + x2 + x3 with x1 = bf16(x), x2 = bf16(x - x1),
// x3 = x - x1 - x2 (8 significant bits each, round to nearest even).  Of the nine products of two such sums the six that
// reach 2^-24 of the whole are formed, x1 w1, x1 w2, x2 w1, x2 w2, x1 w3, x3 w1: a product of two bfloat16 numbers is
// exact in fp32, what is left out is below 2^-25 of |x w|, half of one rounding of an fp32 product, and all sums are fp32.
// v_mfma_f32_16x16x32_bf16 does 16 times the multiply-adds per cycle of v_mfma_f32_16x16x4_f32, so six products per
// multiply-add leave a factor of 2.7, and the bfloat16 instructions do not occupy the vector ALU the staging needs.
//
// A chunk of four input channels lies in LDS as three patches of 8 bytes per cell, one per piece; the 32 k of an instruction are
// 4 pairs of taps x 4 channels, so both operands are pieces as they lie there and a step of eight taps takes six instructions.  (With
// 16-byte cells {x1, x2} and weights {w1, w1}, {w2, w2}, {w3, w1} a step of four taps takes three, one eighth fewer over
// the 27 taps, but the doubled weights cost 24 register moves per step and wave: 10.1 against 9.1 ms for 32 -> 32 channels
// on 23 M particles, with the windows of one row group that the lists held then.)  Values come from the caller's planes (input gradient: from a copy of the output gradient in groups of four
// channels, see load_values_split); a value is split when it is written to LDS.  Lists, work split and epilogue are those of the fp32 kernel (conv_mfma.hip).
//
// Measured against the fp32 instructions (3x3x3, whole forward pass, tree fill included): 23 M particles, 32 -> 32 channels 9.1 ms (11.0), of which
// this kernel 8.3; 1 M, 32 -> 32 0.40 (0.52), 64 -> 64 1.40 (1.78); 320 k, 16 -> 16 0.075 (0.085), 64 -> 64 0.46 (0.64).  1x5x5 64 -> 64 on 23 M
// 31.4 (38.4).  Pairs of times further down were taken when a variant was tried, each pair on one state of the kernel and of the lists.
// Input gradient, whole backward pass with the weight gradient (conv_dw_split.hip): 1 M particles, 32 -> 32 channels 1.33 (1.84), 16 -> 16 0.48
// (0.72); the fp32 kernel scans the access arrays and stages box sums, this one reads lists kept with the plan.
// Bound by the barriers around the matrix phases and the LDS reads of the operands.
// Error against 64 bits (2-norm): 0.31 to 0.33 of the fp32 instructions' with N(0, 1) features, 0.31 to 0.35 with those after a ReLU, below theirs
// also where few products are not zero, but for a single one (1.02; see split_window).
//
// Infinities: where x or w is infinite the pieces of the other operand decide the result (infinity times a zero piece is
// NaN), and values of 2^111 and more, or sums of 2^95 and more, are infinite for these kernels (see SPLIT_SCALE).  Where a result comes
// out infinite or NaN its window and block of outputs are marked, and the fp32 instructions compute what is marked again (conv_mfma16_redo_kernel; as a call
// inside this kernel a second pass cost registers: 16 -> 16 channels on 23 M particles 3.47 instead of 3.26 ms then); an
// input gradient that holds one is made again from the start by the fp32 kernel.  Small values keep all their bits: features of 1e-37
// come out with 0.4 of the fp32 instructions' error (split without SPLIT_SCALE, 510 times that error).
#include "pieces.hpp"

namespace aprnet {

typedef float floatx4s __attribute__((ext_vector_type(4)));
typedef int intx4s __attribute__((ext_vector_type(4)));
// The 32 k of an instruction are 4 pairs of taps x 4 channels: lane group g = lane / 16 supplies pair 4 step + g.  Pairs are
// neighbours along y where the stencil's rows have them (dy 0 and 1, dy 2 and 3), the last taps of the rows among themselves.
// An LDS read of 8 bytes per lane goes out for two lane groups at a time, sixteen neighbouring cells each (256 bytes, every bank
// once) if the two groups' cells do not fall on the same banks: the order below was searched for that (27 taps: 10 of 16
// reads without conflict, in index order 2; 16 -> 16 on 23 M particles 3.27 -> 3.09 ms).  -1: no tap, zero weights.
template <int K> struct SplitTaps;
template <> struct SplitTaps<27> {
    static constexpr int STEPS = 4;
    static constexpr signed char tap[32] = {20, 26, 18, 19, 24, 25, 12, 13, 11, 2, 0, 1, 15, 16, 17, 14, 5, -1, 3, 4, 23, 8, 6, 7, 9, 10, -1, -1, 21, 22, -1, -1};
};
template <> struct SplitTaps<25> {
    static constexpr int STEPS = 4;
    static constexpr signed char tap[32] = {-1, -1, 7, 8, 0, 1, 2, 3, 17, 18, 15, 16, 12, 13, 10, 11, 22, 23, 20, 21, 14, 19, 4, -1, 24, 9, -1, -1, -1, -1, 5, 6};
};
template <class G> constexpr int split_steps() { return SplitTaps<G::K>::STEPS; }

constexpr int PREP_TB = 256;

// packed[s][cb][q][step][piece][h][lane] (16 bytes: two taps of four channels), cb = block of 16 * COH output channels, q = chunk
// of four contracted channels.  Cm / Ck: channels on the M axis / contracted; with `transposed` the image is that of the
// input gradient's stencil (channel axes swapped, taps reversed).  The marks of the launch are cleared on the way.
template <int K>
__device__ __forceinline__ void pack_weights_split(const float* __restrict__ w, int S_exp, int Cm, int Ck, int COH, int transposed, uint4* __restrict__ out,
                                                   int* __restrict__ marks, unsigned block, unsigned blocks) {
    constexpr int nstep = SplitTaps<K>::STEPS;
    const int Cout = transposed ? Ck : Cm, Cin = transposed ? Cm : Ck;
    for (unsigned i = block * PREP_TB + threadIdx.x; i < SPLIT_MARKS; i += blocks * PREP_TB) marks[i] = 0;
    const int ncb = (Cm + 16 * COH - 1) / (16 * COH), nq = (Ck + SP_CIB - 1) / SP_CIB;
    const unsigned n = (unsigned)S_exp * ncb * nq * nstep * COH * 64;          // (the host checks that it fits)
    for (unsigned e = block * PREP_TB + threadIdx.x; e < n; e += blocks * PREP_TB) {
        unsigned r = e;
        const int lane = (int)(r % 64u); r /= 64u;
        const int h = (int)(r % (unsigned)COH); r /= (unsigned)COH;
        const int step = (int)(r % (unsigned)nstep); r /= (unsigned)nstep;
        const int q = (int)(r % (unsigned)nq); r /= (unsigned)nq;
        const int cb = (int)(r % (unsigned)ncb); r /= (unsigned)ncb;
        const int s = (int)r;
        const int cm = (cb * COH + h) * 16 + (lane & 15);
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int t = SplitTaps<K>::tap[2 * (4 * step + (lane >> 4)) + (j >> 2)], ck = q * SP_CIB + (j & 3);
            v[j] = 0.f;
            if (t >= 0 && cm < Cm && ck < Ck)
                v[j] = SPLIT_SCALE * (transposed ? w[(((int64_t)s * Cout + ck) * Cin + cm) * K + (K - 1 - t)] : w[(((int64_t)s * Cout + cm) * Cin + ck) * K + t]);
        }
        uint4 p[3];
        split_pair(v[0], v[1], p[0].x, p[1].x, p[2].x);
        split_pair(v[2], v[3], p[0].y, p[1].y, p[2].y);
        split_pair(v[4], v[5], p[0].z, p[1].z, p[2].z);
        split_pair(v[6], v[7], p[0].w, p[1].w, p[2].w);
        const unsigned base = (((s * ncb + cb) * nq + q) * nstep + step) * 3u;
#pragma unroll
        for (int k = 0; k < 3; ++k) out[((base + k) * COH + h) * 64 + lane] = p[k];
    }
}

// ---- output gradient in groups of four channels: [C / 4][count][4] --------------------------------------------
// out[q][i][c] = SPLIT_SCALE * channel 4 q + c of element i; channels past C are zeros.  A streaming pass (8 bytes per value), four
// elements per thread, all reads issued before the first is used.
constexpr int IG_E = 4;
__device__ __forceinline__ void group4(const float* __restrict__ x, int64_t ldx, int C, int64_t count, float4* __restrict__ out, unsigned block, int q) {
    constexpr int IG_TB = PREP_TB;
    const int64_t i0 = (int64_t)block * (IG_TB * IG_E) + threadIdx.x;
    float v[SP_CIB][IG_E];
#pragma unroll
    for (int c = 0; c < SP_CIB; ++c) {
        const float* p = x + (int64_t)min(q * SP_CIB + c, C - 1) * ldx;
#pragma unroll
        for (int e = 0; e < IG_E; ++e) v[c][e] = p[min(i0 + e * IG_TB, count - 1)];
    }
#pragma unroll
    for (int c = 0; c < SP_CIB; ++c)
        if (q * SP_CIB + c >= C) {                  // uniform
#pragma unroll
            for (int e = 0; e < IG_E; ++e) v[c][e] = 0.f;
        }
    float4* dst = out + (int64_t)q * count;
#pragma unroll
    for (int e = 0; e < IG_E; ++e)
        if (i0 + e * IG_TB < count)
            dst[i0 + e * IG_TB] = make_float4(SPLIT_SCALE * v[0][e], SPLIT_SCALE * v[1][e], SPLIT_SCALE * v[2][e], SPLIT_SCALE * v[3][e]);
}

// What the convolution reads, in one launch: the first blocks pack the weights and clear the marks, the others copy the output gradient (nbx
// blocks per group of channels).
template <int K>
__global__ void __launch_bounds__(PREP_TB)
split_prepare_kernel(const float* __restrict__ w, int S_exp, int Cm, int Ck, int COH, int transposed, uint4* __restrict__ image,
                     int* __restrict__ marks, unsigned nb_pack, const float* __restrict__ x, int64_t ldx, int64_t count, float4* __restrict__ out, unsigned nbx) {
    unsigned b = blockIdx.x;
    if (b < nb_pack) { pack_weights_split<K>(w, S_exp, Cm, Ck, COH, transposed, image, marks, b, nb_pack); return; }
    b -= nb_pack;
    group4(x, ldx, Ck, count, out, b % nbx, (int)(b / nbx));
}

template <class G> struct SplitItems : ItemRegs16<G, (G::MAXITEM + G::NT - 1) / G::NT> {
    static constexpr int IPT = (G::MAXITEM + G::NT - 1) / G::NT;
};
// Forward: from the caller's channel planes, four loads per item, every plane at a scalar offset from the first one of the chunk, so that features
// and tree take one descriptor each.  (One 16-byte load per item from copies in groups of four channels, made by a pass of 8 bytes per value:
// 32 -> 32 channels on 23 M particles 9.5 instead of 8.7 ms, 16 -> 16 on 43 M 6.9 and 6.5, on 1 M 0.175 and 0.164, 64 -> 48 on 2 M 2.55 and 2.48.)
// A chunk that takes channels of both tensors, or rows of 2^28 values and more, has a descriptor per plane.
// Input gradient: from the copy of the output gradient, which the weight gradient reads too.
template <class G, int MODE>
__device__ __forceinline__ void load_values_split(const ConvArgs<float>& a, int q, int nitem, bool tree_items, SplitItems<G>& R) {
    if constexpr (MODE == 0) {
        const int c0 = q * SP_CIB, last = min(SP_CIB, a.Cin - c0) - 1;         // (a channel past the last one reads that one's plane; its weights are zero)
        const bool second = a.x2 != nullptr && c0 >= a.c_split;
        const float* xb = second ? a.x2 + (int64_t)(c0 - a.c_split) * a.ldx2 : a.x + (int64_t)c0 * a.ldx;
        const int64_t ld = second ? a.ldx2 : a.ldx;
        const bool both = a.x2 != nullptr && !second && c0 + last >= a.c_split;
        if (both || ld >= (1ll << 28) || a.ldt >= (1ll << 28)) {               // uniform
#pragma unroll
            for (int c = 0; c < SP_CIB; ++c) {
                const int ch = c0 + min(c, last);
                const bool s2 = a.x2 != nullptr && ch >= a.c_split;
                const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(s2 ? a.x2 + (int64_t)(ch - a.c_split) * a.ldx2 : a.x + (int64_t)ch * a.ldx),
                                                                                    0, (int)(unsigned)(a.x_count * 4), 0x00020000);
                const __amdgpu_buffer_rsrc_t rt = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.tree_data + (int64_t)ch * a.ldt), 0,
                                                                                    tree_items ? (int)(unsigned)(a.t_count * 4) : 0, 0x00020000);
#pragma unroll
                for (int k = 0; k < SplitItems<G>::IPT; ++k) {
                    if (k * G::NT >= nitem) break;          // wave-uniform
                    if (R.pos[k] != 0xffffu && (R.pos[k] & ITEM_TREE) != 0) {
                        R.v[k][c] = __builtin_amdgcn_raw_buffer_load_b32(rt, (int)R.off[k], 0, 0);
                        asm volatile("" ::: "memory");
                    } else R.v[k][c] = __builtin_amdgcn_raw_buffer_load_b32(rx, (int)R.off[k], 0, 0);
                }
            }
            return;
        }
        const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(xb), 0, (int)(unsigned)((last * ld + a.x_count) * 4), 0x00020000);
        const __amdgpu_buffer_rsrc_t rt = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.tree_data + (int64_t)c0 * a.ldt), 0,
                                                                            tree_items ? (int)(unsigned)((last * a.ldt + a.t_count) * 4) : 0, 0x00020000);
#pragma unroll
        for (int k = 0; k < SplitItems<G>::IPT; ++k) {
            if (k * G::NT >= nitem) break;                  // wave-uniform
            const bool item = R.pos[k] != 0xffffu;
            const int off = item ? (int)R.off[k] : 0;       // (no item: a value that is not stored)
            if (tree_items) {
                if (item && (R.pos[k] & ITEM_TREE) != 0) {
#pragma unroll
                    for (int c = 0; c < SP_CIB; ++c) R.v[k][c] = __builtin_amdgcn_raw_buffer_load_b32(rt, off, plane_offset(min(c, last), a.ldt), 0);
                    asm volatile("" ::: "memory");          // keeps the two branches from being merged into one load with a per-lane descriptor
                } else {
#pragma unroll
                    for (int c = 0; c < SP_CIB; ++c) R.v[k][c] = __builtin_amdgcn_raw_buffer_load_b32(rx, off, plane_offset(min(c, last), ld), 0);
                }
            } else {
#pragma unroll
                for (int c = 0; c < SP_CIB; ++c) R.v[k][c] = __builtin_amdgcn_raw_buffer_load_b32(rx, off, plane_offset(min(c, last), ld), 0);
            }
        }
        return;
    }
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.xi + (int64_t)q * a.xi_ld * SP_CIB), 0,
                                                                        (int)(a.x_count * 16), 0x00020000);
#pragma unroll
    for (int k = 0; k < SplitItems<G>::IPT; ++k) {
        if (k * G::NT >= nitem) break;                      // wave-uniform
        R.v[k] = __builtin_amdgcn_raw_buffer_load_b128(rx, (int)R.off[k], 0, 0);
    }
}
template <class G, int COH>
struct SplitShared {
    uint4 w[split_steps<G>() * 3 * COH * 64];
    uint2 patch[3][G::CH_STRIDE];  // the three pieces of four channels, 8 bytes per cell
    float bias[16 * COH];
    int2 toff[split_steps<G>() * 4];
};
template <class G, int COH, int MODE>
__device__ __forceinline__ void store_items_split(const SplitItems<G>& R, int nitem, SplitShared<G, COH>& sh) {
    constexpr float S = MODE == 0 ? SPLIT_SCALE : 1.f;         // (the copy is scaled)
#pragma unroll
    for (int k = 0; k < SplitItems<G>::IPT; ++k) {
        if (k * G::NT >= nitem) break;                  // wave-uniform
        if (R.pos[k] == 0xffffu) continue;
        uint2 p[3];
        split_pair(S * __builtin_bit_cast(float, (int)R.v[k][0]), S * __builtin_bit_cast(float, (int)R.v[k][1]), p[0].x, p[1].x, p[2].x);
        split_pair(S * __builtin_bit_cast(float, (int)R.v[k][2]), S * __builtin_bit_cast(float, (int)R.v[k][3]), p[0].y, p[1].y, p[2].y);
        const int c = R.pos[k] & ITEM_CELL;
#pragma unroll
        for (int i = 0; i < 3; ++i) sh.patch[i][c] = p[i];
        if (R.pos[k] & ITEM_PAIR) {
#pragma unroll
            for (int i = 0; i < 3; ++i) sh.patch[i][c + 1] = p[i];
        }
    }
}

// MODE 0: forward, results stored (plus bias).  MODE 1: input gradient on the plan's input-gradient lists (items = output
// gradient): the columns of a coarser particle are summed across lanes and the first one takes the sum along; a place that no
// other column adds to takes a plain store, the others (one more column at most) an atomic addition.
template <class G, int COH, int NB, int MODE>
__device__ __forceinline__ void split_window(const ConvArgs<float>& a, int co0, int nc, int nitem, bool tree_items, int first,
                                             const uint4* __restrict__ wl, const WindowLists& gl, int* __restrict__ mark, SplitShared<G, COH>& sh) {
    constexpr int NSTEP = split_steps<G>(), NBA = NB > 0 ? NB : 1;
    const int lane = lane_id();
    int cell[NBA];
    // unconditional loads (columns past the end read zero) that travel together with the list loads below
    const __amdgpu_buffer_rsrc_t rcp = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned short*>(gl.col_pos), 0, nc * 2, 0x00020000);
#pragma unroll
    for (int j = 0; j < NB; ++j) cell[j] = (int)__builtin_amdgcn_raw_buffer_load_b16(rcp, (((first + G::NWAVE * j) << 4) + (lane & 15)) * 2, 0, 0);
    // Sums of x1 w1, and of the five products below 2^-8 of it: the large ones are rounded once per step, like a chain of fp32
    // multiply-adds or less often.  (Error against 64 bits relative to the fp32 instructions', 3x3x3, 32 channels: 0.32 dense, 0.35 after a ReLU;
    // where weights are zero but 2, 9 or 27 of them 0.85, 0.54, 0.45; a single product 1.02, what is left out.  With the five summed per step and
    // added to the sum so far, a second rounding: 0.38, 0.44; 1.30, 1.20, 1.01.  32 -> 32 channels on 23 M particles 11.3 and 11.3 ms, 16 -> 16
    // on 43 M 9.1 and 9.1, 64 -> 64 on 8 M 18.9 and 18.9, 24 -> 32 on 4.9 M in sparse windows 1.98 and 1.94, 1x5x5 16 -> 16 on 2 M 0.63 and 0.95.)
    floatx4s acc[NBA][COH], low[NBA][COH];
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int h = 0; h < COH; ++h) acc[j][h] = low[j][h] = floatx4s{0.f, 0.f, 0.f, 0.f};

    constexpr int W16 = NSTEP * 3 * COH * 64;                    // 16-byte elements of a weight chunk
    constexpr int WPT = (W16 + G::NT - 1) / G::NT;
    SplitItems<G> R;
    intx4s wr[WPT];                    // unconditional buffer loads, see the fp32 kernel
    auto load_weights = [&](int q) {
        const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint4*>(wl + (int64_t)q * W16), 0, W16 * 16, 0x00020000);
#pragma unroll
        for (int k = 0; k < WPT; ++k) wr[k] = __builtin_amdgcn_raw_buffer_load_b128(rw, (int)(threadIdx.x + k * G::NT) * 16, 0, 0);
    };
    fetch_slots16<G, SplitItems<G>::IPT, false, MODE == 0 ? 4 : 16>(gl, nitem, R);
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const int col = ((first + G::NWAVE * j) << 4) + (lane & 15);
        cell[j] = col < nc ? ((cell[j] & (int)COL_CELL) - G::TAP0) * 8 : 0;
    }
    load_values_split<G, MODE>(a, 0, nitem, tree_items, R);
    // With 32 outputs a wave that holds two and more blocks of columns asks for the weights of a chunk in front of the barrier that ends the
    // chunk before it, whose operands no longer need registers then; a wave with one block has them to spare and asks together with the
    // values (64 -> 64 channels on 8 M particles 18.9, always in front of the barrier 19.1, always with the values 20.0), as do the 16 outputs.
    constexpr bool LATE = COH == 2 && NB >= 2;
    if constexpr (!LATE) load_weights(0);
    for (int i = threadIdx.x; i < 3 * G::CH_STRIDE / 2; i += G::NT) reinterpret_cast<uint4*>(sh.patch)[i] = make_uint4(0u, 0u, 0u, 0u);
    for (int ci0 = 0; ci0 < a.Cin; ci0 += SP_CIB) {
        if constexpr (LATE) load_weights(ci0 / SP_CIB);
        __syncthreads();
        store_items_split<G, COH, MODE>(R, nitem, sh);
#pragma unroll
        for (int k = 0; k < WPT; ++k) {
            const int i = threadIdx.x + k * G::NT;
            if (i < W16) reinterpret_cast<intx4s*>(sh.w)[i] = wr[k];
        }
        __syncthreads();
        if (ci0 + SP_CIB < a.Cin) {
            load_values_split<G, MODE>(a, ci0 / SP_CIB + 1, nitem, tree_items, R);
            if constexpr (!LATE) load_weights(ci0 / SP_CIB + 1);
        }
        if constexpr (NB > 0) {
            const uintx4s* wa = reinterpret_cast<const uintx4s*>(sh.w) + lane;
            const int2* to = sh.toff + (lane >> 4);
            constexpr int PL = G::CH_STRIDE * 8;                 // bytes of a piece's patch
            const char* p0 = reinterpret_cast<const char*>(sh.patch);
            // one step at a time where the weights of a step fill the registers (32 outputs); all of them with 16 outputs
            constexpr int UNROLL = COH == 1 ? NSTEP : 1;
#pragma unroll UNROLL
            for (int st = 0; st < NSTEP; ++st) {
                bf16x8s a1[COH], a2[COH], a3[COH];
#pragma unroll
                for (int h = 0; h < COH; ++h) {
                    a1[h] = __builtin_bit_cast(bf16x8s, wa[((st * 3 + 0) * COH + h) * 64]);
                    a2[h] = __builtin_bit_cast(bf16x8s, wa[((st * 3 + 1) * COH + h) * 64]);
                    a3[h] = __builtin_bit_cast(bf16x8s, wa[((st * 3 + 2) * COH + h) * 64]);
                }
                const int2 off = to[st * 4];
#pragma unroll
                for (int j = 0; j < NB; ++j) {
                    const char* qa = p0 + (cell[j] + off.x);
                    const char* qb = p0 + (cell[j] + off.y);
                    bf16x8s b[3];
#pragma unroll
                    for (int i = 0; i < 3; ++i) {
                        const uintx2s u = *reinterpret_cast<const uintx2s*>(qa + i * PL), v = *reinterpret_cast<const uintx2s*>(qb + i * PL);
                        b[i] = __builtin_bit_cast(bf16x8s, uintx4s{u.x, u.y, v.x, v.y});
                    }
#define APRNET_PRODUCT(C, A, B) _Pragma("unroll") for (int h = 0; h < COH; ++h) C[j][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[h], B, C[j][h], 0, 0, 0);
                    APRNET_PRODUCT(low, a3, b[0]) APRNET_PRODUCT(low, a1, b[2]) APRNET_PRODUCT(low, a2, b[1])
                    APRNET_PRODUCT(low, a2, b[0]) APRNET_PRODUCT(low, a1, b[1]) APRNET_PRODUCT(acc, a1, b[0])
#undef APRNET_PRODUCT
                }
            }
        }
    }
    if constexpr (NB > 0) {
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int h = 0; h < COH; ++h) acc[j][h] += low[j][h];
        const __amdgpu_buffer_rsrc_t rci = __builtin_amdgcn_make_buffer_rsrc(const_cast<int*>(gl.col_idx), 0, nc * 4, 0x00020000);
        int ocol[NB], cpos[NB];
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            const int col = ((first + G::NWAVE * j) << 4) + (lane & 15);
            ocol[j] = __builtin_amdgcn_raw_buffer_load_b32(rci, col * 4, 0, 0);
            cpos[j] = MODE == 1 ? (int)__builtin_amdgcn_raw_buffer_load_b16(rcp, col * 2, 0, 0) : 0;
        }
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            const int col = ((first + G::NWAVE * j) << 4) + (lane & 15);
            if constexpr (MODE == 1) {
                const bool boxed = (cpos[j] & (int)COL_BOX) != 0;
                if (__ballot(boxed)) {
#pragma unroll
                    for (int h = 0; h < COH; ++h)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const float s = dx_group_sum<G>(acc[j][h][r]);
                            acc[j][h][r] = boxed ? s : acc[j][h][r];
                        }
                }
                if (boxed && (lane & (dx_group<G>() - 1)) != 0) continue;
            }
            if (col >= nc) continue;
            float t = 0.f;              // stays 0 unless one of the sums is infinite or NaN
#pragma unroll
            for (int h = 0; h < COH; ++h)
#pragma unroll
                for (int r = 0; r < 4; ++r) t = fmaf(acc[j][h][r], 0.f, t);
            if (t != 0.f) {
                mark[0] = 1;
                if constexpr (MODE == 0) mark[split_mark(blockIdx.y * gridDim.x + blockIdx.x)] = 1;
            }
            const bool to_tree = (cpos[j] & (int)COL_TREE) != 0, sole = (cpos[j] & (int)COL_SOLE) != 0;
            float* dst = (MODE == 0 ? a.y : to_tree ? a.gtree : a.gx) + ocol[j];
            const int64_t ld = MODE == 0 ? a.ldy : to_tree ? a.ldgt : a.ldgx;
#pragma unroll
            for (int h = 0; h < COH; ++h)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int cl = h * 16 + 4 * (lane >> 4) + r;
                    if (co0 + cl >= a.Cout) continue;
                    float v = acc[j][h][r] * SPLIT_UNSCALE;
                    if constexpr (MODE == 0) {
                        v = fmaf(acc[j][h][r], SPLIT_UNSCALE, sh.bias[cl]);
                        if (a.relu) v = v < 0.f ? 0.f : v;
                        dst[(int64_t)(co0 + cl) * ld] = v;
                    } else if (sole) dst[(int64_t)(co0 + cl) * ld] = v;
                    else unsafeAtomicAdd(dst + (int64_t)(co0 + cl) * ld, v);
                }
        }
    }
}

// One window per workgroup, two workgroups per CU.  (Three with 80 registers, some of them spilled, took 3 to 10 % longer with 16 outputs on every
// APR; eight windows one after the other, 32 -> 32 channels on 23 M particles 10.05 instead of 9.84 ms.)
template <class G, int COH, int MODE>
__global__ void __launch_bounds__(G::NT) __attribute__((amdgpu_waves_per_eu(4, 4)))
conv_split_kernel(const ConvArgs<float> a) {
    constexpr int NBW = 4, NSTEP = split_steps<G>();
    static_assert((G::MAXCOL + 15) / 16 <= G::NWAVE * NBW, "a window must fit the accumulators of the block");
    static_assert(G::RS == 64, "the plan's lists carry cells of rows of 64");
    __shared__ SplitShared<G, COH> sh;
    const int4 hd = a.win[blockIdx.x];
    const int L = a.win_level[blockIdx.x];
    const int co0 = blockIdx.y * 16 * COH;
    const int s_idx = min(a.S_exp - 1, a.Lc - L);
    const int nq = (a.Cin + SP_CIB - 1) / SP_CIB;
    const uint4* __restrict__ wl = reinterpret_cast<const uint4*>(a.w) +
                                   ((int64_t)s_idx * gridDim.y + blockIdx.y) * nq * (NSTEP * 3 * COH * 64);
    const int wave = threadIdx.x >> 6;
    const bool tree_items = MODE == 0 && L < a.Lc;       // the output gradient has no tree part

    if (threadIdx.x < 16 * COH)
        sh.bias[threadIdx.x] = (MODE == 0 && a.bias && co0 + (int)threadIdx.x < a.Cout) ? a.bias[co0 + threadIdx.x] : 0.f;
    if (threadIdx.x < NSTEP * 4) {
        int o[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            int t = SplitTaps<G::K>::tap[2 * threadIdx.x + h];
            if (t < 0) t = max((int)SplitTaps<G::K>::tap[2 * (threadIdx.x ^ 1) + h], 0);       // no tap (zero weights): the other group's cells
            o[h] = (((t / (G::KX * G::KY)) * G::RX + (t / G::KY) % G::KX) * G::RS + t % G::KY) * 8;
        }
        sh.toff[threadIdx.x] = make_int2(o[0], o[1]);
    }
    __syncthreads();
    const int nitem = __builtin_amdgcn_readfirstlane(hd.y), nc = __builtin_amdgcn_readfirstlane(hd.w);
    const unsigned i0 = (unsigned)__builtin_amdgcn_readfirstlane(hd.x), c0 = (unsigned)__builtin_amdgcn_readfirstlane(hd.z);
    const WindowLists gl{a.l_item_idx + i0, a.l_item_pos + i0, a.l_col_idx + c0, a.l_col_pos + c0};
    const int nblk = (nc + 15) >> 4;
    const int first = (wave - (int)blockIdx.x) & (G::NWAVE - 1);
    const int nb = first < nblk ? (nblk - first + G::NWAVE - 1) / G::NWAVE : 0;
    switch (__builtin_amdgcn_readfirstlane(nb)) {
        case 0: split_window<G, COH, 0, MODE>(a, co0, nc, nitem, tree_items, first, wl, gl, a.redo, sh); break;
        case 1: split_window<G, COH, 1, MODE>(a, co0, nc, nitem, tree_items, first, wl, gl, a.redo, sh); break;
        case 2: split_window<G, COH, 2, MODE>(a, co0, nc, nitem, tree_items, first, wl, gl, a.redo, sh); break;
        case 3: split_window<G, COH, 3, MODE>(a, co0, nc, nitem, tree_items, first, wl, gl, a.redo, sh); break;
        default: split_window<G, COH, 4, MODE>(a, co0, nc, nitem, tree_items, first, wl, gl, a.redo, sh); break;
    }
}

using S333 = ConvGeom<3, 3, 3, 2, 4, 512, 64, 16>;
using S155 = ConvGeom<1, 5, 5, 1, 8, 512, 64, 16>;

static int split_coh(int Cm) { return Cm <= 16 ? 1 : 2; }
static int split_nstep(int code) { return code == 333 ? split_steps<S333>() : split_steps<S155>(); }

int launch_conv_redo(int code, const ConvArgs<float>& a, int n_win, hipStream_t st);        // conv_mfma.hip

template <class G, int MODE>
static int launch_split(const ConvArgs<float>& a, int n_win, hipStream_t st) {
    const int coh = split_coh(a.Cout), n_cb = (a.Cout + 16 * coh - 1) / (16 * coh);
    dim3 grid((unsigned)n_win, (unsigned)n_cb);
    if (coh == 1) hipLaunchKernelGGL((conv_split_kernel<G, 1, MODE>), grid, dim3(G::NT), 0, st, a);
    else hipLaunchKernelGGL((conv_split_kernel<G, 2, MODE>), grid, dim3(G::NT), 0, st, a);
    APRNET_LAUNCH_CHECK("conv_split_kernel");
    return 0;
}
// a.w, a.redo: what prepare_split made of the weights a.w_raw; a.win_level ... the forward lists of the plan
int launch_conv_split(int code, const ConvArgs<float>& a, int n_win, hipStream_t st) {
    int rc;
    switch (code) {
        case 333: rc = launch_split<S333, 0>(a, n_win, st); break;
        case 155: rc = launch_split<S155, 0>(a, n_win, st); break;
        default: rc = fail(APRNET_ERR_UNSUPPORTED, "no matrix-core kernel for this stencil");
    }
    return rc ? rc : launch_conv_redo(code, a, n_win, st);
}
// Input gradient: a.x / a.xi / a.Cin describe the output gradient, a.Cout the layer's input channels, a.w the transposed image,
// a.win_level ... the input-gradient lists of the plan without the particles on far faces.  a.redo[0] is set if a sum is not finite.
int launch_conv_dx_split(int code, const ConvArgs<float>& a, int n_win, hipStream_t st) {
    switch (code) {
        case 333: return launch_split<S333, 1>(a, n_win, st);
        case 155: return launch_split<S155, 1>(a, n_win, st);
    }
    return fail(APRNET_ERR_UNSUPPORTED, "no matrix-core kernel for this stencil");
}
size_t split_mark_bytes() { return SPLIT_MARKS * sizeof(int); }
// Cm: channels on the M axis of the kernel, Ck: contracted channels (forward: Cout, Cin; transposed: Cin, Cout)
size_t conv_packed_split_bytes(int code, int S_exp, int Cm, int Ck) {
    const int coh = split_coh(Cm);
    return (size_t)S_exp * ((Cm + 16 * coh - 1) / (16 * coh)) * ((Ck + SP_CIB - 1) / SP_CIB) * split_nstep(code) * 3 * coh * 64 * sizeof(uint4);
}
// Packed weights, cleared marks and (xi not null) a copy of x in groups of four channels, [(Ck + 3) / 4][nx][4].  Fewer than 2^28 elements
// and 2^32 threads (split_dx_bytes).
int prepare_split(int code, const float* w, int S_exp, int Cm, int Ck, bool transposed, void* packed, int* marks, const float* x, int64_t ldx, int64_t nx, float* xi,
                  hipStream_t st) {
    const size_t n = conv_packed_split_bytes(code, S_exp, Cm, Ck) / (3 * sizeof(uint4));
    const unsigned nb = (unsigned)std::min<size_t>((n + PREP_TB - 1) / PREP_TB, 2048), nq = (unsigned)(Ck + SP_CIB - 1) / SP_CIB;
    const unsigned nbx = xi ? (unsigned)((nx + PREP_TB * IG_E - 1) / (PREP_TB * IG_E)) : 0;
#define APRNET_PREP(K) hipLaunchKernelGGL(split_prepare_kernel<K>, dim3(nb + nq * nbx), dim3(PREP_TB), 0, st, w, S_exp, Cm, Ck, split_coh(Cm), \
                                          transposed ? 1 : 0, (uint4*)packed, marks, nb, x, ldx, nx, (float4*)xi, nbx)
    if (code == 333) APRNET_PREP(27); else APRNET_PREP(25);
#undef APRNET_PREP
    APRNET_LAUNCH_CHECK("split_prepare_kernel");
    return 0;
}

}  // namespace aprnet
