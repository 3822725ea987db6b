// Stencil convolution on APR particles, forward (VALU path): Convolution<kz,kx,ky>::forward
// (conv.hpp:55-195) for stencils 3x3x3, 1x3x3, 1x5x5 and 5x5x5, fp32 and fp64.
//
// Per window (see conv_common.hpp) the block loops over chunks of CIB input channels: zero the LDS
// patch, gather the chunk from the three sources, then every thread owns up to ITER output
// positions ("columns") and COB output channels in registers.  The taps of a column come from LDS,
// the weights are wave-uniform and are fetched through the scalar cache.  All input channels are
// reduced inside the block, so each output element is written exactly once: no atomics, and the
// result does not depend on scheduling.  As in the reference, the sum over the K taps of one input
// channel is formed first and then added to the running output (helpers.hpp:537-544).
#include "conv_common.hpp"

#include <atomic>
#include <cstdlib>

namespace aprnet {

template <typename T, class G, int CIB, int COB>
__global__ void __launch_bounds__(G::NT)
conv_fwd_kernel(const ConvArgs<T> a) {
    typedef typename Num<T>::acc A;          // bfloat16 features: fp32 patch, weights, products and sums
    __shared__ A patch[CIB * G::CH_STRIDE];
    __shared__ ConvShared<G> sh;

    const ConvTile tile = a.tiles[blockIdx.x];
    const int L = tile.level, z0 = tile.z0, x0 = tile.x0;
    const int co0 = blockIdx.y * COB;
    const int yn = a.apr.y_num[L];
    const int s_idx = min(a.S_exp - 1, a.Lc - L);
    const bool out_tree = (L == a.Lc) && (L < a.apr.level_max);
    const A* __restrict__ wl = a.w + (int64_t)s_idx * a.Cout * a.Cin * G::K;

    open_segments<G, T>(a, L, z0, x0, sh);
    __syncthreads();

    for (int y0 = 0; y0 < yn; y0 += G::TY) {
        scan_window<G, T>(a, L, y0, out_tree, sh);
        __syncthreads();
        const int nc = sh.ncol, nitem = sh.nitem;
        if (nc > 0) {
            A acc[G::ITER][COB];
#pragma unroll
            for (int it = 0; it < G::ITER; ++it)
#pragma unroll
                for (int co = 0; co < COB; ++co) acc[it][co] = 0;
            for (int i = threadIdx.x; i < CIB * G::CH_STRIDE; i += G::NT) patch[i] = 0;

            for (int ci0 = 0; ci0 < a.Cin; ci0 += CIB) {
                __syncthreads();
                stage_values<G, T, CIB>(a, ci0, nitem, L < a.Lc, sh, patch, std::bool_constant<true>{});
                __syncthreads();
#pragma unroll
                for (int it = 0; it < G::ITER; ++it) {
                    const int col = threadIdx.x + it * G::NT;
                    if (col >= nc) continue;
                    const A* p0 = patch + (int)sh.col_pos[col] - G::TAP0;
#pragma unroll 1
                    for (int c = 0; c < CIB; ++c) {
                        const int ci = ci0 + c;
                        if (ci >= a.Cin) break;
                        A v[G::K];
#pragma unroll
                        for (int sz = 0; sz < G::KZ; ++sz)
#pragma unroll
                            for (int sx = 0; sx < G::KX; ++sx)
#pragma unroll
                                for (int sy = 0; sy < G::KY; ++sy)
                                    v[(sz * G::KX + sx) * G::KY + sy] = p0[c * G::CH_STRIDE + (sz * G::RX + sx) * G::RS + sy];
#pragma unroll
                        for (int co = 0; co < COB; ++co) {
                            if (co0 + co >= a.Cout) break;
                            const A* __restrict__ wp = wl + ((int64_t)(co0 + co) * a.Cin + ci) * G::K;
                            A res = 0;
#pragma unroll
                            for (int t = 0; t < G::K; ++t) res += v[t] * wp[t];
                            acc[it][co] += res;
                        }
                    }
                }
            }
#pragma unroll
            for (int it = 0; it < G::ITER; ++it) {
                const int col = threadIdx.x + it * G::NT;
                if (col >= nc) continue;
                const int64_t o = sh.col_idx[col];
#pragma unroll
                for (int co = 0; co < COB; ++co)
                    if (co0 + co < a.Cout) {
                        A v = acc[it][co] + (a.bias ? a.bias[co0 + co] : (A)0);
                        if (a.relu) v = v < (A)0 ? (A)0 : v;
                        a.y[(int64_t)(co0 + co) * a.ldy + o] = Num<T>::st(v);
                    }
            }
        }
        __syncthreads();
        close_window<G>(sh);
        __syncthreads();
    }
}

// Optional timing of the dominant kernel with HIP events on the launch stream (aprnet_profile_*).
struct KernelTimer {
    bool enabled = false, armed = false;
    hipEvent_t start = nullptr, stop = nullptr;
};
static KernelTimer g_timer;

struct TimedLaunch {
    hipStream_t st;
    bool on;
    explicit TimedLaunch(hipStream_t s) : st(s), on(g_timer.enabled) {
        if (!on) return;
        if (!g_timer.start) { (void)hipEventCreate(&g_timer.start); (void)hipEventCreate(&g_timer.stop); }
        (void)hipEventRecord(g_timer.start, st);
    }
    ~TimedLaunch() { if (on) { (void)hipEventRecord(g_timer.stop, st); g_timer.armed = true; } }
};

template <typename T, class G, int CIB, int COB>
static int launch_fwd(const ConvArgs<T>& a, int n_tiles, hipStream_t st) {
    dim3 grid((unsigned)n_tiles, (unsigned)((a.Cout + COB - 1) / COB));
    TimedLaunch timed(st);
    hipLaunchKernelGGL((conv_fwd_kernel<T, G, CIB, COB>), grid, dim3(G::NT), 0, st, a);
    APRNET_LAUNCH_CHECK("conv_fwd_kernel");
    return 0;
}

// tile shapes: 3-D stencils 2 x 4 rows, 2-D stencils (kz == 1) 1 x 8 rows
using G333 = ConvGeom<3, 3, 3, 2, 4, 256>;
using G133 = ConvGeom<1, 3, 3, 1, 8, 256>;
using G155 = ConvGeom<1, 5, 5, 1, 8, 256>;
using G555 = ConvGeom<5, 5, 5, 2, 4, 256>;

template <typename T> struct Chunk;       // channels staged per pass so that the patch stays near 48 KB
template <> struct Chunk<float>  { static constexpr int c333 = 8, c133 = 16, c155 = 12, c555 = 4; };
template <> struct Chunk<double> { static constexpr int c333 = 4, c133 = 8,  c155 = 6,  c555 = 2; };

bool conv_mfma_supported(int code);
int launch_conv_mfma(int code, const ConvArgs<float>& a, int n_tiles, hipStream_t st);
int launch_conv_mfma(int code, const ConvArgs<bf16_t>& a, int n_tiles, hipStream_t st);
int launch_conv_mfma_bf16(int code, const ConvArgs<bf16_t>& a, int n_win, hipStream_t st);
size_t conv_packed_bf16_bytes(int code, int S_exp, int Cout, int Cin);
int pack_conv_weights_bf16(int code, const float* w, int S_exp, int Cout, int Cin, void* packed, hipStream_t st, bool transposed = false);
int interleave8_bf16(const bf16_t* x, int64_t ldx, const bf16_t* x2, int64_t ldx2, int c_split, int C, int64_t count, bf16_t* out,
                     hipStream_t st);
static std::atomic<int> g_bf16_math{1};      // bfloat16 features: 1 = bfloat16 matrix instructions, 0 = fp32 matrix instructions
static std::atomic<int> g_bf16_regroup{1};   // bfloat16 forward: 1 = stage from a copy of the input regrouped by 8 channels, 0 = from the channel planes
int fill_tree_for_conv(const aprnet_plan* p, int d, const bf16_t* x, int64_t ldx, int C, bf16_t* tree, int64_t ldt, hipStream_t st,
                       const NeedLists* need);
size_t conv_packed_floats(int code, int S_exp, int Cm, int Ck, bool transposed);
int pack_conv_weights(int code, const float* w, int S_exp, int Cm, int Ck, bool transposed, float* packed, hipStream_t st, const RedoClear* redo = nullptr);

size_t split_mark_bytes();
size_t conv_packed_split_bytes(int code, int S_exp, int Cm, int Ck);
int prepare_split(int code, const float* w, int S_exp, int Cm, int Ck, bool transposed, void* packed, int* marks, const float* x, int64_t ldx, int64_t nx, float* xi,
                  hipStream_t st);
int launch_conv_split(int code, const ConvArgs<float>& a, int n_win, hipStream_t st);
static std::atomic<int> g_f32_split{1};      // fp32 features: products of bfloat16 pieces (conv_split.hip) 1 = where faster, 2 = at any size, 0 = never
static std::atomic<int> g_dw_split{1};       // and their weight gradient (conv_dw_split.hip), likewise

bool conv_narrow_supported(int code, int Cin);
size_t conv_narrow_packed_floats(int code, int S_exp, int Cout, int Cin, bool bf16m);
bool conv_narrow_bf16_math(int code, int Cin);
int pack_conv_weights_narrow(int code, const float* w, int S_exp, int Cout, int Cin, float* packed, hipStream_t st, bool bf16m);
int launch_conv_narrow(int code, const ConvArgs<float>& a, const WinLists& wl, hipStream_t st);
int launch_conv_narrow(int code, const ConvArgs<bf16_t>& a, const WinLists& wl, hipStream_t st);
static std::atomic<int> g_big_addr{0};       // bfloat16 forward on grouped tensors: 1 = 64-bit addresses also where 32-bit offsets would do
static std::atomic<int> g_narrow{1};         // layers of 1 to 3 input channels: 1 = the bandwidth-shaped kernel (conv_narrow.hip), 0 = the general one
static std::atomic<int> g_conv_path{0};      // 0: matrix cores where available, 1: VALU kernels only
int conv_path() { return g_conv_path; }
int bf16_math();
int bf16_regroup();

static std::atomic<int> g_use_lists{1};      // 1: forward kernels take the window lists of the plan, 0: they scan per call
int bf16_math() { return g_bf16_math; }
int bf16_regroup() { return g_bf16_regroup; }
static std::atomic<int> g_bwd_overlap{1};    // backward: weight gradient on a second stream next to the input gradient
int backward_overlap() { return g_bwd_overlap; }
static std::atomic<int> g_wide{0};           // bfloat16 kernels on regrouped input: 64 outputs per workgroup (conv_mfma.hip, wide_outputs)
int conv_wide_mode() { return g_wide; }
static std::atomic<int> g_bwd_deterministic{1};   // backward: weight gradient summed in a fixed order (partial sums per workgroup) instead of atomics
int bwd_deterministic() { return g_bwd_deterministic; }

// Points the kernel at the plan's window lists (a.n_tiles: how many there are).  When the lists are switched off, or cannot be built (no device
// memory for them, too many entries), a.win_level stays null and the kernel scans the access arrays itself.
template <typename T>
static int set_lists(aprnet_plan* p, int d, int code, const TileList& tl, ConvArgs<T>& a, hipStream_t st, int dx = 0) {
    a.win_level = nullptr;
    if (!g_use_lists) return 0;
    WinLists wl;
    if (get_lists(p, d, code, tl, &wl, st, dx) != 0) { (void)hipGetLastError(); return 0; }
    if (wl.n_win == 0) return 0;
    a.n_tiles = wl.n_win;
    a.win_level = wl.d_level; a.win = wl.d_win;
    a.l_item_idx = wl.d_item_idx; a.l_item_pos = wl.d_item_pos; a.l_col_idx = wl.d_col_idx; a.l_col_pos = wl.d_col_pos;
    return 0;
}

int set_conv_lists(aprnet_plan* p, int d, int code, const TileList& tl, ConvArgs<float>& a, hipStream_t st) { return set_lists(p, d, code, tl, a, st); }
int set_conv_lists(aprnet_plan* p, int d, int code, const TileList& tl, ConvArgs<bf16_t>& a, hipStream_t st) { return set_lists(p, d, code, tl, a, st); }
// the input-gradient lists (tl: the tile list with a halo of one row)
int set_conv_dx_lists(aprnet_plan* p, int d, int code, const TileList& tl, ConvArgs<bf16_t>& a, hipStream_t st) { return set_lists(p, d, code, tl, a, st, 1); }
// without the particles on far faces
int set_conv_dx_lists(aprnet_plan* p, int d, int code, const TileList& tl, ConvArgs<float>& a, hipStream_t st) { return set_lists(p, d, code, tl, a, st, 2); }

// Channel-aware dispatch: a layer with 1 to 3 input channels is bound by memory (4 (Cin + Cout) bytes for 2 K Cin Cout
// flops per particle) and goes to the pipelined kernel of conv_narrow.hip, which needs the plan's window lists and a
// single input tensor.  *done tells whether the layer was taken.
template <typename T>
static int try_narrow(aprnet_plan* p, const ConvArgs<T>& a, int code, int d, const TileList& tl, hipStream_t st, bool* done) {
    if (!g_narrow || g_conv_path == 1 || !g_use_lists || a.x2 != nullptr || !conv_narrow_supported(code, a.Cin)) return 0;
    WinLists wl;
    if (get_lists(p, d, code, tl, &wl, st) != 0) { (void)hipGetLastError(); return 0; }
    *done = true;
    ScratchLease lease;
    // (bfloat16 features, one input channel, 3x3x3: the kernel's bfloat16 form and its image of the weights)
    const bool bf16m = std::is_same<T, bf16_t>::value && conv_narrow_bf16_math(code, a.Cin);
    if (int rc = lease.acquire(p, conv_narrow_packed_floats(code, a.S_exp, a.Cout, a.Cin, bf16m) * sizeof(float), st)) return rc;
    if (int rc = pack_conv_weights_narrow(code, (const float*)a.w, a.S_exp, a.Cout, a.Cin, (float*)p->d_scratch, st, bf16m)) return rc;
    ConvArgs<T> b = a;
    b.w = (const float*)p->d_scratch;
    b.win_level = wl.d_level; b.win = wl.d_win;
    b.l_item_idx = wl.d_item_idx; b.l_item_pos = wl.d_item_pos; b.l_col_idx = wl.d_col_idx; b.l_col_pos = wl.d_col_pos;
    TimedLaunch timed(st);
    return launch_conv_narrow(code, b, wl, st);
}

// Work space of the forward pass on products of bfloat16 pieces: packed weights and marks.  0: the layer does not take that path.
//  - fewer than SPLIT_MIN_CIN input channels.  The line was drawn when the kernel read copies of features and tree, whose cost these layers did not win
//    back (8 -> 16 channels 0.080 and 0.078 ms); without copies pieces are ahead there too, by less with 16 outputs (fp32 instructions and pieces, 3x3x3,
//    1 M particles: 4 -> 16 0.082 and 0.080 ms, 8 -> 16 0.113 and 0.106, 8 -> 32 0.168 and 0.137, 12 -> 32 0.224 and 0.170; 0.16 M: 8 -> 16 0.044 and
//    0.044, 8 -> 32 0.055 and 0.049), and so are input gradients of 4 to 12 outputs (1 M, whole backward pass, 16 -> 8 0.59 and 0.42, 32 -> 8 1.07 and
//    0.67).  It has not been moved since.
//  - 1x3x3: two steps of eight taps for nine.
//  - little work: one more launch than the fp32 kernel's, which also counts where the host is behind the device (3x3x3, pieces against
//    fp32; 16 outputs: 90 k particles x 16 channels 50 and 48 us, x 32 70 and 65, 160 k x 16 58 and 58, 320 k 78 and 90; 32 outputs: 12 k
//    x 16 34 and 36, x 32 43 and 49, 90 k 79 and 95; 64 outputs: 2 k x 64 62 and 74, 90 k 183 and 251 us).
//    1x5x5 gains about as much (16 -> 16 channels on 80 k 44 and 43 us, on 230 k 54 and 58; 64 -> 64 on 20 k 68 and 86, on 1 M 1.21 and 1.64 ms).
//  - values are reached with 32-bit offsets: fewer than 2^28 particles.
constexpr int SPLIT_MIN_CIN = 16;
static size_t split_align(size_t v) { return (v + 255) / 256 * 256; }
static size_t split_fwd_bytes(int code, int Cin, int S_exp, int Cout, int64_t nx, int64_t nt) {
    if (!g_f32_split || g_conv_path == 1 || (code != 333 && code != 155) || Cin < SPLIT_MIN_CIN || nx >= (1ll << 28) || nt >= (1ll << 28)) return 0;
    if (g_f32_split == 1 && (double)nx * Cin * ((Cout + 15) / 16 * 16) < (Cout <= 16 ? 1 << 26 : 1 << 23)) return 0;
    if (conv_packed_split_bytes(code, S_exp, Cout, Cin) / 48 >= (1u << 29)) return 0;               // elements the packing kernel counts in 32 bits
    return split_mark_bytes() + split_align(conv_packed_split_bytes(code, S_exp, Cout, Cin));
}

// The same of the input gradient: packed weights and the output gradient in groups of four channels.
// Next to a weight gradient on fp32 instructions, which bounds many of these calls, it gains less by it (whole backward pass, split against fp32:
// 3x3x3 16 -> 16 channels on 70 k particles 152 and 159 us, on 320 k 319 and 353; 32 -> 32 on 14 k 144 and 142, on 70 k 242
// and 266; 64 -> 64 on 14 k 212 and 220; 128 -> 128 on 2 k 218 and 278; 1x5x5 16 -> 16 on 14 k 139 and 119, on 70 k 142
// and 157, 64 -> 64 on 14 k 209 and 209).
// The first such pass of a plan also builds its window lists, 0.1 to 0.5 ms once per level delta: 16 -> 16 channels on 0.7 M particles 1.04
// and 0.79 ms (later passes 0.53 and 0.63), on 14 M 10.6 and 10.1 (8.6 and 9.1); 32 -> 32 on 0.7 M 1.83 and 1.85, on 14 M 24.5 and 25.8; 64 -> 64
// on 0.7 M 5.5 and 5.9.  Whether the lists are there decides nothing: the first pass and the later ones have the same bits.
size_t split_dx_bytes(int code, int Cin, int S_exp, int Cout, int64_t n) {
    if (!g_f32_split || !g_use_lists || g_conv_path == 1 || (code != 333 && code != 155) || Cout < SPLIT_MIN_CIN || n >= (1ll << 28)) return 0;
    if (g_f32_split == 1 && (double)n * Cout * ((Cin + 15) / 16 * 16) < 1 << 24) return 0;
    if (conv_packed_split_bytes(code, S_exp, Cin, Cout) / 48 >= (1u << 29)) return 0;
    if ((double)(Cout + 3) / 4 * n >= 1.6e10) return 0;
    return split_mark_bytes() + split_align(conv_packed_split_bytes(code, S_exp, Cin, Cout)) + (size_t)(Cout + 3) / 4 * (size_t)n * 16;
}

// The weight gradient is made of pieces too where the input gradient is (and reads its copy of the output gradient): faster from the
// smallest sizes on (backward pass, fp32 instructions against pieces: 3x3x3 64 -> 64 channels on 5 k particles 177 and 162 us, 128 -> 128
// on 5 k 470 and 383, 32 -> 32 on 42 k 200 and 168, 16 -> 16 on 90 k 173 and 153; 1x5x5 32 -> 32 on 20 k 209 and 184; large
// ones in conv_dw_split.hip).  "At any size" of the input gradient's switch leaves it where it is.  Eight planes of the features and of the tree are
// reached with 32-bit byte offsets: rows of fewer than 2^27 values.
bool split_dw(int Cin, int Cout, int64_t n, int64_t ldx, int64_t ldt) {
    if (!g_dw_split || ldx >= (1ll << 27) || ldt >= (1ll << 27)) return false;
    return g_dw_split == 2 || (double)n * Cout * ((Cin + 15) / 16 * 16) >= 1 << 24;
}

template <typename T> static int try_mfma(aprnet_plan*, const ConvArgs<T>&, int, int, const TileList&, int, hipStream_t, bool*, void*, int64_t) { return 0; }
template <> int try_mfma<float>(aprnet_plan* p, const ConvArgs<float>& a, int code, int d, const TileList& tl, int n_tiles,
                                hipStream_t st, bool* done, void* ws, int64_t ws_bytes) {
    if (g_conv_path == 1 || !conv_mfma_supported(code)) return 0;
    if (int rc = try_narrow<float>(p, a, code, d, tl, st, done)) return rc;
    if (*done) return 0;
    *done = true;
    ConvArgs<float> b = a;
    if (int rc = set_lists(p, d, code, tl, b, st)) return rc;
    const size_t need = b.win_level ? split_fwd_bytes(code, a.Cin, a.S_exp, a.Cout, a.x_count, a.t_count) : 0;
    if (need > 0 && ws && ws_bytes >= 0 && (size_t)ws_bytes >= need) {
        // products of bfloat16 pieces: weights and marks in the caller's work space
        char* image = (char*)ws + split_mark_bytes();
        if (int rc = prepare_split(code, a.w, a.S_exp, a.Cout, a.Cin, false, image, (int*)ws, nullptr, 0, 0, nullptr, st)) return rc;
        b.w_raw = a.w; b.w = (const float*)image; b.redo = (int*)ws;
        TimedLaunch timed(st);
        return launch_conv_split(code, b, b.n_tiles, st);
    }
    // plan-owned scratch for the re-laid-out weights, grown on demand
    ScratchLease lease;
    if (int rc = lease.acquire(p, conv_packed_floats(code, a.S_exp, a.Cout, a.Cin, false) * sizeof(float), st)) return rc;
    if (int rc = pack_conv_weights(code, a.w, a.S_exp, a.Cout, a.Cin, false, (float*)p->d_scratch, st)) return rc;
    b.w = (const float*)p->d_scratch;
    TimedLaunch timed(st);
    return launch_conv_mfma(code, b, b.win_level ? b.n_tiles : n_tiles, st);
}

int fill_tree_for_conv(const aprnet_plan* p, int d, const float* x, int64_t ldx, int C, float* tree, int64_t ldt, hipStream_t st,
                       const NeedLists* need);
int fill_tree_for_conv(const aprnet_plan* p, int d, const double* x, int64_t ldx, int C, double* tree, int64_t ldt, hipStream_t st,
                       const NeedLists* need);

// The tree nodes the forward kernels of this stencil read, for a fill that skips the others; null when the restricted
// fill is switched off or its lists cannot be had (no window lists, first call under stream capture, no memory): the
// caller then fills every node.  The kernels stage exactly what the window lists name, so either fill gives the same result.
static std::atomic<int> g_need_fill{1};      // 1: the tree fill before a forward convolution covers the nodes that are read, 0: all nodes
const NeedLists* needed_nodes(aprnet_plan* p, int d, int code, const TileList& tl, hipStream_t st, NeedLists* store) {
    if (!g_need_fill || !g_use_lists || g_conv_path == 1 || !conv_mfma_supported(code) || tl.n == 0) return nullptr;
    WinLists wl;
    if (get_lists(p, d, code, tl, &wl, st) != 0) { (void)hipGetLastError(); return nullptr; }
    if (get_need_lists(p, d, code, wl, store, st) != 0) { (void)hipGetLastError(); return nullptr; }
    return store;
}

// Optional parts of the fused forward entry points: a second input tensor whose C2 channels follow the Cin of x
// in the contraction, and a clamp at zero of the result.
template <typename T>
struct Fusion {
    const T* x2 = nullptr; int64_t ldx2 = 0; int C2 = 0; int relu = 0;
    const T* x2_coarse = nullptr; int64_t ld_coarse = 0;      // grouped bfloat16 only: what x2 was upsampled from
};
template <typename T>
static int read_fusion(const aprnet_conv_fusion* f, Fusion<T>* out) {
    *out = Fusion<T>{};
    if (!f) return 0;
    if (f->C2 < 0 || (f->C2 > 0 && !f->x2)) return fail(APRNET_ERR_INVALID_ARGUMENT, "conv_forward: second input without data");
    if (f->C2 > 0) { out->x2 = (const T*)f->x2; out->ldx2 = f->ldx2; out->C2 = f->C2; }
    if (f->C2 > 0 && f->x2_coarse) { out->x2_coarse = (const T*)f->x2_coarse; out->ld_coarse = f->ld_coarse; }
    out->relu = f->relu != 0;
    return 0;
}

template <typename T>
int conv_fwd(const aprnet_plan* cp, int d, int kz, int kx, int ky, const T* x, int64_t ldx, int C1, const T* w,
             int S_exp, int Cout, const T* bias, T* y, int64_t ldy, T* tree_ws, int64_t ldt, hipStream_t st,
             const Fusion<T>& fu = Fusion<T>{}, void* ws = nullptr, int64_t ws_bytes = 0) {
    aprnet_plan* p = const_cast<aprnet_plan*>(cp);
    if (int rc = check_level_delta(p, d, "conv_forward")) return rc;
    if (int rc = check_plane_size(p, d, sizeof(*x), "conv_forward")) return rc;
    if (int rc = check_rows(ldx, p->number_parts(d), "conv_forward", "input")) return rc;
    if (int rc = check_rows(ldy, p->number_parts(d), "conv_forward", "output")) return rc;
    if (fu.C2 > 0) if (int rc = check_rows(fu.ldx2, p->number_parts(d), "conv_forward", "second input")) return rc;
    const int Cin = C1 + fu.C2;
    if (C1 <= 0 || Cout <= 0 || S_exp <= 0) return fail(APRNET_ERR_INVALID_ARGUMENT, "conv_forward: empty channel / stencil count");
    const int code = kz * 100 + kx * 10 + ky;
    if (code != 333 && code != 133 && code != 155 && code != 555)
        return fail(APRNET_ERR_UNSUPPORTED, "conv_forward: stencil must be 333, 133, 155 or 555");
    const int64_t nt = p->tree_parts(d);
    if (nt > 0 && (!tree_ws || ldt < nt)) return fail(APRNET_ERR_INVALID_ARGUMENT, "conv_forward: tree work space too small");
    APRNET_HIP_CHECK(hipSetDevice(p->device));
    const bool flat = (kz == 1);
    TileList tl;
    if (int rc = get_tiles(p, d, flat ? 1 : 2, flat ? 8 : 4, &tl, st)) return rc;
    NeedLists need_store;
    const NeedLists* need = sizeof(T) == 4 ? needed_nodes(p, d, code, tl, st, &need_store) : nullptr;
    if (int rc = fill_tree_for_conv(p, d, x, ldx, C1, tree_ws, ldt, st, need)) return rc;
    if (fu.C2 > 0)
        if (int rc = fill_tree_for_conv(p, d, fu.x2, fu.ldx2, fu.C2, tree_ws + (int64_t)C1 * ldt, ldt, st, need)) return rc;
    if (tl.n == 0) return 0;
    ConvArgs<T> a{};
    a.apr = p->dapr; a.tree = p->dtree; a.tiles = tl.d_tiles;
    a.x = x; a.ldx = ldx; a.Cin = Cin; a.w = w; a.S_exp = S_exp; a.Cout = Cout; a.bias = bias; a.y = y; a.ldy = ldy;
    a.x2 = fu.x2; a.ldx2 = fu.ldx2; a.c_split = C1; a.relu = fu.relu;
    a.tree_data = tree_ws; a.ldt = ldt; a.Lc = p->lc(d); a.tree_off = p->tree_offset(a.Lc);
    a.x_count = p->number_parts(d); a.t_count = p->tree_parts(d);
    bool done = false;
    if (int rc = try_mfma<T>(p, a, code, d, tl, tl.n, st, &done, ws, ws_bytes)) return rc;
    if (done) return 0;
    // few output channels per thread keep the wave-uniform weights within the scalar register file;
    // wider layers run more blocks along grid.y (each re-stages its patch)
    switch (code) {
        case 333: return launch_fwd<T, G333, Chunk<T>::c333, 4>(a, tl.n, st);
        case 133: return launch_fwd<T, G133, Chunk<T>::c133, 4>(a, tl.n, st);
        case 155: return launch_fwd<T, G155, Chunk<T>::c155, 4>(a, tl.n, st);
        case 555: return launch_fwd<T, G555, Chunk<T>::c555, 4>(a, tl.n, st);
    }
    return 0;
}

// bfloat16 features, fp32 weights and bias, fp32 arithmetic: 3x3x3 on the matrix cores only
int conv_fwd_bf16(const aprnet_plan* cp, int d, int kz, int kx, int ky, const bf16_t* x, int64_t ldx, int C1, const float* w,
                  int S_exp, int Cout, const float* bias, bf16_t* y, int64_t ldy, bf16_t* tree_ws, int64_t ldt, hipStream_t st,
                  const Fusion<bf16_t>& fu = Fusion<bf16_t>{}) {
    aprnet_plan* p = const_cast<aprnet_plan*>(cp);
    if (int rc = check_level_delta(p, d, "conv_forward")) return rc;
    if (int rc = check_plane_size(p, d, sizeof(*x), "conv_forward")) return rc;
    if (int rc = check_rows(ldx, p->number_parts(d), "conv_forward", "input")) return rc;
    if (int rc = check_rows(ldy, p->number_parts(d), "conv_forward", "output")) return rc;
    if (fu.C2 > 0) if (int rc = check_rows(fu.ldx2, p->number_parts(d), "conv_forward", "second input")) return rc;
    const int Cin = C1 + fu.C2;
    if (C1 <= 0 || Cout <= 0 || S_exp <= 0) return fail(APRNET_ERR_INVALID_ARGUMENT, "conv_forward: empty channel / stencil count");
    const int code = kz * 100 + kx * 10 + ky;
    if (!conv_mfma_supported(code) && code != 555)
        return fail(APRNET_ERR_UNSUPPORTED, "conv_forward: bfloat16 features are supported for the 3x3x3, 1x3x3, 1x5x5 and 5x5x5 stencils");
    const int64_t nt = p->tree_parts(d);
    if (nt > 0 && (!tree_ws || ldt < nt)) return fail(APRNET_ERR_INVALID_ARGUMENT, "conv_forward: tree work space too small");
    APRNET_HIP_CHECK(hipSetDevice(p->device));
    TileList tl;
    if (int rc = get_tiles(p, d, kz == 1 ? 1 : 2, kz == 1 ? 8 : 4, &tl, st)) return rc;
    NeedLists need_store;
    const NeedLists* need = needed_nodes(p, d, code, tl, st, &need_store);
    if (tl.n == 0) return 0;
    auto fill_planes = [&]() -> int {
        if (int rc = fill_tree_for_conv(p, d, x, ldx, C1, tree_ws, ldt, st, need)) return rc;
        return fu.C2 > 0 ? fill_tree_for_conv(p, d, fu.x2, fu.ldx2, fu.C2, tree_ws + (int64_t)C1 * ldt, ldt, st, need) : 0;
    };
    ConvArgs<bf16_t> a{};
    if (code == 555) {
        if (int rc = fill_planes()) return rc;
        // no matrix-core kernel for this stencil: the vector-ALU kernel with fp32 patch, weights and sums
        a.apr = p->dapr; a.tree = p->dtree; a.tiles = tl.d_tiles;
        a.x = x; a.ldx = ldx; a.Cin = Cin; a.w = w; a.S_exp = S_exp; a.Cout = Cout; a.bias = bias;
        a.x2 = fu.x2; a.ldx2 = fu.ldx2; a.c_split = C1; a.relu = fu.relu;
        a.y = y; a.ldy = ldy; a.tree_data = tree_ws; a.ldt = ldt; a.Lc = p->lc(d); a.tree_off = p->tree_offset(a.Lc);
        a.x_count = p->number_parts(d); a.t_count = p->tree_parts(d);
        return launch_fwd<bf16_t, G555, Chunk<float>::c555, 4>(a, tl.n, st);
    }
    bool filled = false;
    if (conv_narrow_supported(code, Cin) && fu.C2 == 0) {
        // a narrow first layer on the pipelined kernel: one input channel of a 3x3x3 layer on the bfloat16 matrix
        // instruction (weights rounded to bfloat16, as below), otherwise fp32 products of the bfloat16 features
        ConvArgs<bf16_t> n{};
        n.apr = p->dapr; n.tree = p->dtree; n.tiles = tl.d_tiles;
        n.x = x; n.ldx = ldx; n.Cin = Cin; n.w = w; n.S_exp = S_exp; n.Cout = Cout; n.bias = bias; n.relu = fu.relu;
        n.y = y; n.ldy = ldy; n.tree_data = tree_ws; n.ldt = ldt; n.Lc = p->lc(d); n.tree_off = p->tree_offset(n.Lc);
        n.x_count = p->number_parts(d); n.t_count = p->tree_parts(d);
        bool done = false;
        if (int rc = fill_planes()) return rc;
        filled = true;
        if (int rc = try_narrow<bf16_t>(p, n, code, d, tl, st, &done)) return rc;
        if (done) return 0;
    }
    if (int rc = set_lists(p, d, code, tl, a, st)) return rc;
    const bool bf16_math = g_bf16_math && a.win_level;      // the bfloat16 contraction exists with window lists only
    const int64_t n_x = p->number_parts(d), n_t = p->tree_parts(d);
    ScratchLease lease;
    if (bf16_math) {
        // The input regrouped as [Cin / 8][count][8] behind the packed weights in the plan's scratch buffer, when its
        // 16-byte items stay addressable with 32-bit offsets and the copy stays below 32 GiB.
        // The mean tree is made of the regrouped features, in the tree work space: the same bits as a tree of the planes regrouped, with eight
        // channels per access and no pass over a copy (1x5x5 64 -> 64 on 15.4 M particles, forward and backward: 19.5 -> 18.3 ms; 3x3x3 16 -> 16
        // on 5.2 M, forward: 0.370 -> 0.333 ms).  A last group that is not full does not fit the work space: tree of the planes, regrouped behind
        // the features.
        const size_t wbytes = (conv_packed_bf16_bytes(code, S_exp, Cout, Cin) + 255) / 256 * 256;
        const bool tree_g8 = tree_ws_grouped(Cin, tree_ws);
        const size_t ng = (size_t)(Cin + 7) / 8, ibytes = ng * (size_t)(n_x + (tree_g8 ? 0 : n_t)) * 16;
        const bool regroup = bf16_regroup() && n_x < (1ll << 28) && n_t < (1ll << 28) && ng * (size_t)(n_x + n_t) * 16 <= ((size_t)32 << 30);
        if (int rc = lease.acquire(p, wbytes + (regroup ? ibytes : 0), st)) return rc;
        if (int rc = pack_conv_weights_bf16(code, w, S_exp, Cout, Cin, p->d_scratch, st)) return rc;
        if (regroup) {
            bf16_t* xi = (bf16_t*)((char*)p->d_scratch + wbytes);
            if (int rc = interleave8_bf16(x, ldx, fu.x2, fu.ldx2, C1, Cin, n_x, xi, st)) return rc;
            bf16_t* ti = tree_g8 ? tree_ws : xi + ng * (size_t)n_x * 8;
            if (tree_g8) {
                if (int rc = fill_tree_mean_g8(p, d, xi, n_x, Cin, ti, n_t, st, need)) return rc;
            } else {
                if (!filled) if (int rc = fill_planes()) return rc;
                if (int rc = interleave8_bf16(tree_ws, ldt, nullptr, 0, Cin, Cin, n_t, ti, st)) return rc;
            }
            filled = true;
            a.xi = xi; a.ti = ti; a.xi_ld = n_x; a.ti_ld = n_t;
        }
    } else {
        if (int rc = lease.acquire(p, conv_packed_floats(code, S_exp, Cout, Cin, false) * sizeof(float), st)) return rc;
        if (int rc = pack_conv_weights(code, w, S_exp, Cout, Cin, false, (float*)p->d_scratch, st)) return rc;
    }
    if (!filled) if (int rc = fill_planes()) return rc;
    if (!a.win_level) a.n_tiles = tl.n;
    a.apr = p->dapr; a.tree = p->dtree; a.tiles = tl.d_tiles;
    a.x = x; a.ldx = ldx; a.Cin = Cin; a.w = (const float*)p->d_scratch; a.S_exp = S_exp; a.Cout = Cout; a.bias = bias;
    a.x2 = fu.x2; a.ldx2 = fu.ldx2; a.c_split = C1; a.relu = fu.relu;
    a.y = y; a.ldy = ldy; a.tree_data = tree_ws; a.ldt = ldt; a.Lc = p->lc(d); a.tree_off = p->tree_offset(a.Lc);
    a.x_count = p->number_parts(d); a.t_count = p->tree_parts(d);
    TimedLaunch timed(st);
    return bf16_math ? launch_conv_mfma_bf16(code, a, a.n_tiles, st) : launch_conv_mfma(code, a, a.n_tiles, st);
}

// bfloat16 features with a layout per tensor: planes [C][ld] or groups of eight channels [C / 8][ld][8] (grouped.hip).
//   grouped input   Cin (and the channels of a second input) multiples of 8; tree_ws is grouped too; the kernel stages
//                   straight from the tensors, no regrouping pass
//   planes input    1 to 3 channels (the first layer of a network) on the pipelined kernel
//   grouped output  Cout a multiple of 8
int tree_of_upsampled_g8(const aprnet_plan* p, int d, const bf16_t* z, int64_t ldz, int C, bf16_t* tree, int64_t ldt, hipStream_t st,
                         const NeedLists* need);
// The 1x1x1 convolution that follows a layer inside its kernel (ConvArgs::head_w): out [C][ld] planes.
struct ConvHead { const float* w = nullptr; const float* bias = nullptr; int S = 0, C = 0; bf16_t* out = nullptr; int64_t ld = 0; };
int conv_fwd_bf16_layout(const aprnet_plan* cp, int d, int kz, int kx, int ky, const bf16_t* x, int64_t ldx, int C1, int x_g8, const float* w,
                         int S_exp, int Cout, const float* bias, bf16_t* y, int64_t ldy, int y_g8, bf16_t* tree_ws, int64_t ldt,
                         hipStream_t st, const Fusion<bf16_t>& fu, const ConvHead* head = nullptr, const void* packed = nullptr) {
    aprnet_plan* p = const_cast<aprnet_plan*>(cp);
    if (int rc = check_level_delta(p, d, "conv_forward")) return rc;
    if (int rc = check_plane_size(p, d, 2, "conv_forward")) return rc;           // the plane input of a first layer: 32-bit offsets
    if (int rc = check_rows(ldx, p->number_parts(d), "conv_forward", "input")) return rc;
    if (head) {
        if (!head->w || !head->out || head->S <= 0 || head->C <= 0)
            return fail(APRNET_ERR_INVALID_ARGUMENT, "conv_forward: head without weights or output");
        if (!x_g8 || Cout > 16 || head->C > 4)
            return fail(APRNET_ERR_UNSUPPORTED, "conv_forward: the fused head takes grouped input, at most 16 channels between "
                                                "the two convolutions and at most 4 outputs");
        if (int rc = check_rows(head->ld, p->number_parts(d), "conv_forward", "head output")) return rc;
    } else
    if (int rc = check_rows(ldy, p->number_parts(d), "conv_forward", "output")) return rc;
    if (fu.C2 > 0) if (int rc = check_rows(fu.ldx2, p->number_parts(d), "conv_forward", "second input")) return rc;
    const int Cin = C1 + fu.C2;
    if (C1 <= 0 || Cout <= 0 || S_exp <= 0) return fail(APRNET_ERR_INVALID_ARGUMENT, "conv_forward: empty channel / stencil count");
    const int code = kz * 100 + kx * 10 + ky;
    if (!conv_mfma_supported(code))
        return fail(APRNET_ERR_UNSUPPORTED, "conv_forward: bfloat16 features are supported for the 3x3x3, 1x3x3 and 1x5x5 stencils");
    if (y_g8 && Cout % 8) return fail(APRNET_ERR_INVALID_ARGUMENT, "conv_forward: a grouped output holds a multiple of eight channels");
    if (x_g8 && (C1 % 8 || fu.C2 % 8)) return fail(APRNET_ERR_INVALID_ARGUMENT, "conv_forward: grouped inputs hold multiples of eight channels");
    if (fu.x2_coarse && !x_g8) return fail(APRNET_ERR_UNSUPPORTED, "conv_forward: x2_coarse is taken with grouped inputs only");
    if (!x_g8 && (fu.C2 > 0 || !conv_narrow_supported(code, Cin)))
        return fail(APRNET_ERR_UNSUPPORTED, "conv_forward: a planes input with a grouped output is taken for 1 to 3 channels only");
    const int64_t nt = p->tree_parts(d);
    if (nt > 0 && (!tree_ws || ldt < nt)) return fail(APRNET_ERR_INVALID_ARGUMENT, "conv_forward: tree work space too small");
    APRNET_HIP_CHECK(hipSetDevice(p->device));
    TileList tl;
    if (int rc = get_tiles(p, d, kz == 1 ? 1 : 2, kz == 1 ? 8 : 4, &tl, st)) return rc;
    ConvArgs<bf16_t> a{};
    a.apr = p->dapr; a.tree = p->dtree; a.tiles = tl.d_tiles;
    a.x = x; a.ldx = ldx; a.Cin = Cin; a.w = w; a.S_exp = S_exp; a.Cout = Cout; a.bias = bias; a.relu = fu.relu;
    a.y = y; a.ldy = ldy; a.y_g8 = y_g8; a.tree_data = tree_ws; a.ldt = ldt; a.Lc = p->lc(d); a.tree_off = p->tree_offset(a.Lc);
    a.x_count = p->number_parts(d); a.t_count = nt; a.c_split = C1;
    if (head) {
        a.head_w = head->w; a.head_b = head->bias; a.head_S = head->S; a.head_C = head->C; a.head_y = head->out; a.head_ld = head->ld;
    }
    NeedLists need_store;
    const NeedLists* need = needed_nodes(p, d, code, tl, st, &need_store);
    if (!x_g8) {
        if (int rc = fill_tree_for_conv(p, d, x, ldx, C1, tree_ws, ldt, st, need)) return rc;
        if (tl.n == 0) return 0;
        bool done = false;
        if (int rc = try_narrow<bf16_t>(p, a, code, d, tl, st, &done)) return rc;
        return done ? 0 : fail(APRNET_ERR_UNSUPPORTED, "conv_forward: the window lists of the plan are not available");
    }
    if (int rc = fill_tree_mean_g8(p, d, x, ldx, C1, tree_ws, ldt, st, need)) return rc;
    if (fu.C2 > 0) {
        bf16_t* tree2 = tree_ws + (int64_t)(C1 / 8) * ldt * 8;
        if (fu.x2_coarse) { if (int rc = tree_of_upsampled_g8(p, d, fu.x2_coarse, fu.ld_coarse, fu.C2, tree2, ldt, st, need)) return rc; }
        else if (int rc = fill_tree_mean_g8(p, d, fu.x2, fu.ldx2, fu.C2, tree2, ldt, st, need)) return rc;
    }
    if (tl.n == 0) return 0;
    if (int rc = set_lists(p, d, code, tl, a, st)) return rc;
    if (!a.win_level) return fail(APRNET_ERR_UNSUPPORTED, "conv_forward: the window lists of the plan are not available");
    // An image of the weights that the caller keeps spares a launch of 6 to 13 us per layer (28 to 1792 small blocks, bound by their
    // start and by reads 27 floats apart), which is what 13 layers of a U-Net on 0.6 M particles spend 7 % of their time on.
    ScratchLease lease;
    if (!packed) {
        if (int rc = lease.acquire(p, conv_packed_bf16_bytes(code, S_exp, Cout, Cin), st)) return rc;
        if (int rc = pack_conv_weights_bf16(code, w, S_exp, Cout, Cin, p->d_scratch, st)) return rc;
    }
    a.w = (const float*)(packed ? packed : p->d_scratch);
    a.xi = x; a.xi_ld = ldx; a.xi2 = fu.C2 > 0 ? fu.x2 : nullptr; a.xi2_ld = fu.ldx2; a.ti = tree_ws; a.ti_ld = ldt;
    a.x = nullptr; a.x2 = nullptr; a.tree_data = nullptr;
    // 16-byte items: 32-bit byte offsets reach 2^28 elements of a group; beyond, the kernel takes 64-bit addresses
    a.big = g_big_addr || a.x_count >= (1ll << 28) || a.t_count >= (1ll << 28);
    TimedLaunch timed(st);
    return launch_conv_mfma_bf16(code, a, a.n_tiles, st);
}

int conv111_fwd_relu(const aprnet_plan*, int, const float*, int64_t, int, const float*, int, int, const float*, float*, int64_t, hipStream_t, int);
int conv111_fwd_relu(const aprnet_plan*, int, const double*, int64_t, int, const double*, int, int, const double*, double*, int64_t, hipStream_t, int);
int conv111_fwd_relu(const aprnet_plan*, int, const bf16_t*, int64_t, int, const float*, int, int, const float*, bf16_t*, int64_t, hipStream_t, int);

}  // namespace aprnet

using namespace aprnet;

extern "C" {
int aprnet_conv_fwd_bf16(const aprnet_plan* p, int d, int kz, int kx, int ky, const uint16_t* x, int64_t ldx, int Cin,
                         const float* w, int S_exp, int Cout, const float* bias, uint16_t* y, int64_t ldy, uint16_t* tree_ws,
                         int64_t ldt, void* st) {
    return conv_fwd_bf16(p, d, kz, kx, ky, (const bf16_t*)x, ldx, Cin, w, S_exp, Cout, bias, (bf16_t*)y, ldy, (bf16_t*)tree_ws,
                         ldt, (hipStream_t)st);
}
#define APRNET_FUSED_111(T)                                                                                              \
    if (kz == 1 && kx == 1 && ky == 1) {                                                                                 \
        if (fu.C2 > 0) return fail(APRNET_ERR_UNSUPPORTED, "conv_forward: the 1x1x1 convolution takes a single input");  \
        return conv111_fwd_relu(p, d, (const T*)x, ldx, Cin, w, S_exp, Cout, bias, (T*)y, ldy, (hipStream_t)st, fu.relu); \
    }
int aprnet_conv_fwd_fused_bf16(const aprnet_plan* p, int d, int kz, int kx, int ky, const uint16_t* x, int64_t ldx, int Cin,
                               const float* w, int S_exp, int Cout, const float* bias, uint16_t* y, int64_t ldy,
                               uint16_t* tree_ws, int64_t ldt, const aprnet_conv_fusion* fusion, void* st) {
    Fusion<bf16_t> fu;
    if (int rc = read_fusion(fusion, &fu)) return rc;
    APRNET_FUSED_111(bf16_t)
    return conv_fwd_bf16(p, d, kz, kx, ky, (const bf16_t*)x, ldx, Cin, w, S_exp, Cout, bias, (bf16_t*)y, ldy, (bf16_t*)tree_ws,
                         ldt, (hipStream_t)st, fu);
}
int aprnet_conv_fwd_fused_bf16l(const aprnet_plan* p, int d, int kz, int kx, int ky, const uint16_t* x, int64_t ldx, int Cin, int x_grouped,
                                const float* w, int S_exp, int Cout, const float* bias, uint16_t* y, int64_t ldy, int y_grouped,
                                uint16_t* tree_ws, int64_t ldt, const aprnet_conv_fusion* fusion, void* st) {
    Fusion<bf16_t> fu;
    if (int rc = read_fusion(fusion, &fu)) return rc;
    return conv_fwd_bf16_layout(p, d, kz, kx, ky, (const bf16_t*)x, ldx, Cin, x_grouped, w, S_exp, Cout, bias, (bf16_t*)y, ldy, y_grouped,
                                (bf16_t*)tree_ws, ldt, (hipStream_t)st, fu);
}
int aprnet_conv_fwd_head_bf16g(const aprnet_plan* p, int d, int kz, int kx, int ky, const uint16_t* x, int64_t ldx, int Cin,
                               const float* w, int S_exp, int Cout, const float* bias, uint16_t* tree_ws, int64_t ldt,
                               const aprnet_conv_fusion* fusion, const float* head_w, int head_S, int head_C, const float* head_bias,
                               uint16_t* out, int64_t ldo, void* st) {
    Fusion<bf16_t> fu;
    if (int rc = read_fusion(fusion, &fu)) return rc;
    ConvHead head;
    head.w = head_w; head.bias = head_bias; head.S = head_S; head.C = head_C; head.out = (bf16_t*)out; head.ld = ldo;
    return conv_fwd_bf16_layout(p, d, kz, kx, ky, (const bf16_t*)x, ldx, Cin, 1, w, S_exp, Cout, bias, nullptr, 0, 0,
                                (bf16_t*)tree_ws, ldt, (hipStream_t)st, fu, &head);
}
int64_t aprnet_conv_pack_bf16_bytes(int kz, int kx, int ky, int S_exp, int Cout, int Cin) {
    const int code = kz * 100 + kx * 10 + ky;
    return conv_mfma_supported(code) && S_exp > 0 && Cout > 0 && Cin > 0 ? (int64_t)conv_packed_bf16_bytes(code, S_exp, Cout, Cin) : 0;
}
int aprnet_conv_pack_bf16(int kz, int kx, int ky, const float* w, int S_exp, int Cout, int Cin, void* packed, void* st) {
    if (aprnet_conv_pack_bf16_bytes(kz, kx, ky, S_exp, Cout, Cin) == 0) return fail(APRNET_ERR_UNSUPPORTED, "conv_pack: stencil must be 333, 133 or 155, with channels");
    if (!w || !packed || ((uintptr_t)packed & 15) != 0) return fail(APRNET_ERR_INVALID_ARGUMENT, "conv_pack: no weights, or an image that is not aligned to 16 bytes");
    return pack_conv_weights_bf16(kz * 100 + kx * 10 + ky, w, S_exp, Cout, Cin, packed, (hipStream_t)st);
}
int aprnet_conv_fwd_packed_bf16l(const aprnet_plan* p, int d, int kz, int kx, int ky, const uint16_t* x, int64_t ldx, int Cin, int x_grouped,
                                 const float* w, const void* packed, int S_exp, int Cout, const float* bias, uint16_t* y, int64_t ldy,
                                 int y_grouped, uint16_t* tree_ws, int64_t ldt, const aprnet_conv_fusion* fusion, void* st) {
    Fusion<bf16_t> fu;
    if (int rc = read_fusion(fusion, &fu)) return rc;
    if (((uintptr_t)packed & 15) != 0) return fail(APRNET_ERR_INVALID_ARGUMENT, "conv_forward: the packed weights are not aligned to 16 bytes");
    return conv_fwd_bf16_layout(p, d, kz, kx, ky, (const bf16_t*)x, ldx, Cin, x_grouped, w, S_exp, Cout, bias, (bf16_t*)y, ldy, y_grouped,
                                (bf16_t*)tree_ws, ldt, (hipStream_t)st, fu, nullptr, packed);
}
int aprnet_conv_fwd_head_packed_bf16g(const aprnet_plan* p, int d, int kz, int kx, int ky, const uint16_t* x, int64_t ldx, int Cin,
                                      const float* w, const void* packed, int S_exp, int Cout, const float* bias, uint16_t* tree_ws, int64_t ldt,
                                      const aprnet_conv_fusion* fusion, const float* head_w, int head_S, int head_C, const float* head_bias,
                                      uint16_t* out, int64_t ldo, void* st) {
    Fusion<bf16_t> fu;
    if (int rc = read_fusion(fusion, &fu)) return rc;
    if (((uintptr_t)packed & 15) != 0) return fail(APRNET_ERR_INVALID_ARGUMENT, "conv_forward: the packed weights are not aligned to 16 bytes");
    ConvHead head;
    head.w = head_w; head.bias = head_bias; head.S = head_S; head.C = head_C; head.out = (bf16_t*)out; head.ld = ldo;
    return conv_fwd_bf16_layout(p, d, kz, kx, ky, (const bf16_t*)x, ldx, Cin, 1, w, S_exp, Cout, bias, nullptr, 0, 0,
                                (bf16_t*)tree_ws, ldt, (hipStream_t)st, fu, &head, packed);
}
int aprnet_conv_fwd_fused_f32(const aprnet_plan* p, int d, int kz, int kx, int ky, const float* x, int64_t ldx, int Cin,
                              const float* w, int S_exp, int Cout, const float* bias, float* y, int64_t ldy, float* tree_ws,
                              int64_t ldt, const aprnet_conv_fusion* fusion, void* st) {
    Fusion<float> fu;
    if (int rc = read_fusion(fusion, &fu)) return rc;
    APRNET_FUSED_111(float)
    return conv_fwd<float>(p, d, kz, kx, ky, x, ldx, Cin, w, S_exp, Cout, bias, y, ldy, tree_ws, ldt, (hipStream_t)st, fu);
}
int64_t aprnet_conv_ws_bytes_f32(const aprnet_plan* p, int d, int kz, int kx, int ky, int Cin, int S_exp, int Cout) {
    if (!p || d < 0 || d >= p->tree.level_max + 1 || Cin <= 0 || S_exp <= 0 || Cout <= 0) return 0;
    return (int64_t)split_fwd_bytes(kz * 100 + kx * 10 + ky, Cin, S_exp, Cout, p->number_parts(d), p->tree_parts(d));
}
int aprnet_conv_fwd_ws_f32(const aprnet_plan* p, int d, int kz, int kx, int ky, const float* x, int64_t ldx, int Cin,
                           const float* w, int S_exp, int Cout, const float* bias, float* y, int64_t ldy, float* tree_ws,
                           int64_t ldt, const aprnet_conv_fusion* fusion, void* ws, int64_t ws_bytes, void* st) {
    Fusion<float> fu;
    if (int rc = read_fusion(fusion, &fu)) return rc;
    APRNET_FUSED_111(float)
    if (((uintptr_t)ws & 15) != 0) return fail(APRNET_ERR_INVALID_ARGUMENT, "conv_forward: the work space is not aligned to 16 bytes");
    return conv_fwd<float>(p, d, kz, kx, ky, x, ldx, Cin, w, S_exp, Cout, bias, y, ldy, tree_ws, ldt, (hipStream_t)st, fu, ws, ws_bytes);
}
int aprnet_conv_fwd_fused_f64(const aprnet_plan* p, int d, int kz, int kx, int ky, const double* x, int64_t ldx, int Cin,
                              const double* w, int S_exp, int Cout, const double* bias, double* y, int64_t ldy, double* tree_ws,
                              int64_t ldt, const aprnet_conv_fusion* fusion, void* st) {
    Fusion<double> fu;
    if (int rc = read_fusion(fusion, &fu)) return rc;
    APRNET_FUSED_111(double)
    return conv_fwd<double>(p, d, kz, kx, ky, x, ldx, Cin, w, S_exp, Cout, bias, y, ldy, tree_ws, ldt, (hipStream_t)st, fu);
}
int aprnet_set_conv_path(int path) {
    // process-wide, so a caller that is not a test or a measurement has no business here: the switch answers only in a
    // process that asked for it through its environment before the first call
    static const bool testing = [] { const char* e = getenv("APRNET_TESTING"); return e && e[0] && !(e[0] == '0' && !e[1]); }();
    if (!testing)
        return fail(APRNET_ERR_UNSUPPORTED, "set_conv_path: the kernel-selection switch is for tests and measurements; "
                                            "it answers only when the process runs with APRNET_TESTING=1 in its environment");
    if (path == 2 || path == 3) { g_bf16_math = path == 2; return 0; }
    if (path == 4 || path == 5) { g_use_lists = path == 4; return 0; }
    if (path == 6 || path == 7) { g_bwd_overlap = path == 6; return 0; }
    if (path == 8 || path == 9) { g_bf16_regroup = path == 8; return 0; }
    if (path == 10 || path == 11) { g_bwd_deterministic = path == 10; return 0; }
    if (path == 12 || path == 13) { g_narrow = path == 12; return 0; }
    if (path == 14 || path == 15) { g_big_addr = path == 15; return 0; }
    if (path == 16 || path == 17) { g_need_fill = path == 16; return 0; }
    if (path >= 24 && path <= 26) { g_wide = path - 24; return 0; }
    if (path >= 21 && path <= 23) { g_dw_split = path == 21 ? 1 : path == 22 ? 0 : 2; return 0; }
    if (path >= 18 && path <= 20) { g_f32_split = path == 18 ? 1 : path == 19 ? 0 : 2; return 0; }
    if (path != 0 && path != 1)
        return fail(APRNET_ERR_INVALID_ARGUMENT, "set_conv_path: 0 (auto), 1 (VALU only), 2 / 3 (bfloat16 features: bfloat16 / fp32 "
                                                 "matrix math), 4 / 5 (forward: window lists of the plan / scan per call), 6 / 7 (backward on two streams / one), "
                                                 "8 / 9 (bfloat16 forward: regrouped copy of the input / channel planes), 10 / 11 (weight gradient: "
                                                 "fixed-order partial sums / atomic additions), 12 / 13 (1 to 3 input channels: pipelined kernel / general kernel), "
                                                 "14 / 15 (grouped bfloat16 forward: 32-bit offsets where they suffice / 64-bit addresses always), "
                                                 "16 / 17 (tree fill before a forward convolution: the nodes it reads / every node), "
                                                 "18 / 19 / 20 (fp32 features with a work space: products of bfloat16 pieces where faster / fp32 matrix instructions / pieces at any size), "
                                                 "21 / 22 / 23 (the same for the weight gradient beside an input gradient on pieces), "
                                                 "24 / 25 / 26 (bfloat16, flat stencils, more than 32 outputs: 64 per workgroup where that is faster / always / never)");
    g_conv_path = path;
    return 0;
}
int aprnet_profile_enable(int on) { g_timer.enabled = on != 0; g_timer.armed = false; return 0; }
float aprnet_profile_last_ms(void) {
    if (!g_timer.armed) return -1.0f;
    float ms = -1.0f;
    if (hipEventSynchronize(g_timer.stop) != hipSuccess) return -1.0f;
    if (hipEventElapsedTime(&ms, g_timer.start, g_timer.stop) != hipSuccess) return -1.0f;
    return ms;
}
int aprnet_conv_fwd_f32(const aprnet_plan* p, int d, int kz, int kx, int ky, const float* x, int64_t ldx, int Cin,
                        const float* w, int S_exp, int Cout, const float* bias, float* y, int64_t ldy, float* tree_ws,
                        int64_t ldt, void* st) {
    return conv_fwd<float>(p, d, kz, kx, ky, x, ldx, Cin, w, S_exp, Cout, bias, y, ldy, tree_ws, ldt, (hipStream_t)st);
}
int aprnet_conv_fwd_f64(const aprnet_plan* p, int d, int kz, int kx, int ky, const double* x, int64_t ldx, int Cin,
                        const double* w, int S_exp, int Cout, const double* bias, double* y, int64_t ldy, double* tree_ws,
                        int64_t ldt, void* st) {
    return conv_fwd<double>(p, d, kz, kx, ky, x, ldx, Cin, w, S_exp, Cout, bias, y, ldy, tree_ws, ldt, (hipStream_t)st);
}
}
