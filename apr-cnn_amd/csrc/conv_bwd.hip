// Stencil convolution, backward: Convolution<kz,kx,ky>::backward (conv.hpp:261-481 with
// helpers.hpp:423-478, 578-704).  Two kernels over the same tiles / windows as the forward pass.
//
// grad_input.  Per window and chunk of input channels every thread owns one output position and
// forms its K tap gradients  g[c][t] = sum_co dO[co] * w[co][c][t]  (weights wave-uniform), adds
// them into an LDS gradient patch (LDS atomics: neighbouring outputs overlap), and the patch is then
// flushed along the three gather sources - the exact transpose of the forward gather, including the
// two cells of a coarser particle.  Halo rows belong to neighbouring tiles as well, so the flush uses
// global floating-point atomics; tree cells of levels < Lc go to the tree-gradient buffer that
// fill_tree_mean_backward afterwards pushes down to the particles.
//
// grad_weights.  dW[s][co][ci][t] = sum over outputs of dO[co] * tap[ci][t].  A thread owns one
// (co, ci) pair and keeps its K sums in registers while the (persistent) block walks over many
// tiles; dO and the patch are staged in LDS.  Sums are flushed with one atomic per element when the
// stencil index changes and at the end.
#include "dw_work.hpp"

#include <functional>

namespace aprnet {

// Streaming passes over the rows of the work space: a thread handles STREAM_V consecutive values with 16-byte accesses
// (element-aligned: rows start wherever the leading dimension puts them), STREAM_R times a block's width apart, all loads
// of a thread ahead of its first store.
constexpr int STREAM_TB = 256, STREAM_V = 4, STREAM_R = 4, STREAM_BLOCK = STREAM_TB * STREAM_V * STREAM_R;

// Bound by the stores.  One 4-byte store per lane and turn of a grid-stride loop filled the two
// work spaces of 64 channels (5.2 GB) in 1.69 ms; that and round_to_bf16_kernel below: 1x5x5 64 -> 64 forward and backward
// on 15.4 M particles 25.9 -> 24.7 ms, training step on 5.5 M particles 21.4 -> 20.8 ms.
template <typename T>
__global__ void __launch_bounds__(STREAM_TB) fill_kernel(T* __restrict__ p, int64_t ld, int64_t n, T v) {
    constexpr int V = 16 / sizeof(T);
    typedef T vec __attribute__((ext_vector_type(V), aligned(sizeof(T))));
    T* row = p + (int64_t)blockIdx.y * ld;
    vec w;
#pragma unroll
    for (int e = 0; e < V; ++e) w[e] = v;
#pragma unroll
    for (int r = 0; r < STREAM_R; ++r) {
        const int64_t i = ((int64_t)blockIdx.x * STREAM_R + r) * (STREAM_TB * V) + threadIdx.x * V;
        if (i + V <= n) *reinterpret_cast<vec*>(row + i) = w;
        else
            for (int64_t k = i; k < n; ++k) row[k] = v;
    }
}

template <typename T>
static void fill2d(T* p, int64_t ld, int64_t n, int rows, T v, hipStream_t st) {
    if (n <= 0 || rows <= 0) return;
    constexpr int64_t per = STREAM_TB * (16 / sizeof(T)) * STREAM_R;
    hipLaunchKernelGGL(fill_kernel<T>, dim3((unsigned)((n + per - 1) / per), (unsigned)rows), dim3(STREAM_TB), 0, st, p, ld, n, v);
}

// Transpose of stage_values: add the gradient patch back to its sources, item by item.
template <class G, typename T, int CIB>
__device__ __forceinline__ void flush_values(const ConvArgs<T>& a, int ci0, int nitem, const ConvShared<G>& sh,
                                             const T* gpatch) {
    for (int it = threadIdx.x; it < nitem; it += G::NT) {
        const unsigned pos = sh.item_pos[it];
        const int64_t idx = sh.item_idx[it];
        T* base = (pos & ITEM_TREE) ? a.gtree + idx : a.gx + idx;
        const int64_t ld = (pos & ITEM_TREE) ? a.ldgt : a.ldgx;
        const T* cell = gpatch + (pos & ITEM_CELL);
#pragma unroll
        for (int c = 0; c < CIB; ++c) {
            if (ci0 + c >= a.Cin) break;
            T v = cell[c * G::CH_STRIDE];
            if (pos & ITEM_PAIR) v += cell[c * G::CH_STRIDE + 1];
            if (v != (T)0) atomicAdd(base + (int64_t)(ci0 + c) * ld, v);
        }
    }
}

template <typename T, class G, int CIB, int COBLK>
__global__ void __launch_bounds__(G::NT)
conv_bwd_dx_kernel(const ConvArgs<T> a) {
    static_assert(G::ITER == 1, "one output position per thread");
    __shared__ T gpatch[CIB * G::CH_STRIDE];
    __shared__ T dOs[COBLK * G::MAXCOL];
    __shared__ ConvShared<G> sh;

    const ConvTile tile = a.tiles[blockIdx.x];
    const int L = tile.level, z0 = tile.z0, x0 = tile.x0;
    const int ci0 = blockIdx.y * CIB;
    const int yn = a.apr.y_num[L];
    const int s_idx = min(a.S_exp - 1, a.Lc - L);
    const bool out_tree = (L == a.Lc) && (L < a.apr.level_max);
    const T* __restrict__ wl = a.w + (int64_t)s_idx * a.Cout * a.Cin * G::K;

    open_segments<G, T>(a, L, z0, x0, sh);
    __syncthreads();

    for (int y0 = 0; y0 < yn; y0 += G::TY) {
        scan_window<G, T>(a, L, y0, out_tree, sh);
        __syncthreads();
        const int nc = sh.ncol, nitem = sh.nitem;
        if (nc > 0) {
            for (int i = threadIdx.x; i < CIB * G::CH_STRIDE; i += G::NT) gpatch[i] = 0;
            T g[CIB][G::K];
#pragma unroll
            for (int c = 0; c < CIB; ++c)
#pragma unroll
                for (int t = 0; t < G::K; ++t) g[c][t] = 0;
            const int col = threadIdx.x;
            for (int co0 = 0; co0 < a.Cout; co0 += COBLK) {
                __syncthreads();
                const int nco = min(COBLK, a.Cout - co0);
                for (int i = threadIdx.x; i < nco * nc; i += G::NT) {
                    const int co = i / nc, cc = i - co * nc;
                    dOs[co * G::MAXCOL + cc] = a.gy[(int64_t)(co0 + co) * a.ldy + sh.col_idx[cc]];
                }
                __syncthreads();
                if (col < nc) {
#pragma unroll 1
                    for (int co = 0; co < nco; ++co) {
                        const T dO = dOs[co * G::MAXCOL + col];
#pragma unroll
                        for (int c = 0; c < CIB; ++c) {
                            if (ci0 + c >= a.Cin) break;
                            const T* __restrict__ wp = wl + ((int64_t)(co0 + co) * a.Cin + ci0 + c) * G::K;
#pragma unroll
                            for (int t = 0; t < G::K; ++t) g[c][t] += dO * wp[t];
                        }
                    }
                }
            }
            if (col < nc) {
                T* p0 = gpatch + (int)sh.col_pos[col] - G::TAP0;
#pragma unroll
                for (int c = 0; c < CIB; ++c)
#pragma unroll
                    for (int sz = 0; sz < G::KZ; ++sz)
#pragma unroll
                        for (int sx = 0; sx < G::KX; ++sx)
#pragma unroll
                            for (int sy = 0; sy < G::KY; ++sy)
                                atomicAdd(&p0[c * G::CH_STRIDE + (sz * G::RX + sx) * G::RS + sy],
                                          g[c][(sz * G::KX + sx) * G::KY + sy]);
            }
            __syncthreads();
            flush_values<G, T, CIB>(a, ci0, nitem, sh, gpatch);
        }
        __syncthreads();
        close_window<G>(sh);
        __syncthreads();
    }
}

template <typename T, class G, int CIB, int COB>
__global__ void __launch_bounds__(G::NT)
conv_bwd_dw_kernel(const ConvArgs<T> a) {
    static_assert(CIB * COB <= G::NT, "one thread per (co, ci) pair");
    constexpr int DOS_LD = COB + 1;
    __shared__ T patch[CIB * G::CH_STRIDE];
    __shared__ T dOs[G::MAXCOL * DOS_LD];
    __shared__ ConvShared<G> sh;

    const int ci0 = blockIdx.y * CIB, co0 = blockIdx.z * COB;
    const int pco = threadIdx.x % COB, pc = threadIdx.x / COB;
    const bool worker = threadIdx.x < CIB * COB && (co0 + pco) < a.Cout && (ci0 + pc) < a.Cin;
    T acc[G::K];
#pragma unroll
    for (int t = 0; t < G::K; ++t) acc[t] = 0;
    int cur_s = -1;

    auto flush = [&](int s_idx) {
        if (!worker || s_idx < 0) return;
        T* dst = a.gw + (((int64_t)s_idx * a.Cout + co0 + pco) * a.Cin + ci0 + pc) * G::K;
#pragma unroll
        for (int t = 0; t < G::K; ++t) { if (acc[t] != (T)0) atomicAdd(dst + t, acc[t]); acc[t] = 0; }
    };

    for (int ti = blockIdx.x; ti < a.n_tiles; ti += gridDim.x) {
        const ConvTile tile = a.tiles[ti];
        const int L = tile.level, z0 = tile.z0, x0 = tile.x0;
        const int yn = a.apr.y_num[L];
        const int s_idx = min(a.S_exp - 1, a.Lc - L);
        const bool out_tree = (L == a.Lc) && (L < a.apr.level_max);
        if (s_idx != cur_s) { flush(cur_s); cur_s = s_idx; }

        __syncthreads();
        open_segments<G, T>(a, L, z0, x0, sh);
        __syncthreads();

        for (int y0 = 0; y0 < yn; y0 += G::TY) {
            scan_window<G, T>(a, L, y0, out_tree, sh);
            __syncthreads();
            const int nc = sh.ncol, nitem = sh.nitem;
            if (nc > 0) {
                for (int i = threadIdx.x; i < CIB * G::CH_STRIDE; i += G::NT) patch[i] = 0;
                const int nco = min(COB, a.Cout - co0);
                for (int i = threadIdx.x; i < nco * nc; i += G::NT) {
                    const int co = i / nc, cc = i - co * nc;
                    dOs[cc * DOS_LD + co] = a.gy[(int64_t)(co0 + co) * a.ldy + sh.col_idx[cc]];
                }
                __syncthreads();
                stage_values<G, T, CIB>(a, ci0, nitem, L < a.Lc, sh, patch);
                __syncthreads();
                if (worker) {
                    const T* pch = patch + pc * G::CH_STRIDE - G::TAP0;
                    for (int col = 0; col < nc; ++col) {
                        const T dO = dOs[col * DOS_LD + pco];
                        const T* p0 = pch + (int)sh.col_pos[col];
#pragma unroll
                        for (int sz = 0; sz < G::KZ; ++sz)
#pragma unroll
                            for (int sx = 0; sx < G::KX; ++sx)
#pragma unroll
                                for (int sy = 0; sy < G::KY; ++sy)
                                    acc[(sz * G::KX + sx) * G::KY + sy] += dO * p0[(sz * G::RX + sx) * G::RS + sy];
                    }
                }
            }
            __syncthreads();
            close_window<G>(sh);
            __syncthreads();
        }
    }
    flush(cur_s);
}

// geometries: 512 threads for grad_input (one output position per thread), 256 for grad_weights
using X333 = ConvGeom<3, 3, 3, 2, 4, 512>;
using X133 = ConvGeom<1, 3, 3, 1, 8, 512>;
using X155 = ConvGeom<1, 5, 5, 1, 8, 512>;
using X555 = ConvGeom<5, 5, 5, 2, 4, 512>;
using W333 = ConvGeom<3, 3, 3, 2, 4, 256>;
using W133 = ConvGeom<1, 3, 3, 1, 8, 256>;
using W155 = ConvGeom<1, 5, 5, 1, 8, 256>;
using W555 = ConvGeom<5, 5, 5, 2, 4, 256>;

int fill_tree_for_conv(const aprnet_plan* p, int d, const float* x, int64_t ldx, int C, float* tree, int64_t ldt, hipStream_t st, const NeedLists* need);
int fill_tree_for_conv(const aprnet_plan* p, int d, const double* x, int64_t ldx, int C, double* tree, int64_t ldt, hipStream_t st, const NeedLists* need);
int fill_tree_bwd_for_conv(const aprnet_plan* p, int d, float* gx, int64_t ldx, int C, float* gt, int64_t ldt, hipStream_t st, const NeedLists* need);
int fill_tree_bwd_for_conv(const aprnet_plan* p, int d, double* gx, int64_t ldx, int C, double* gt, int64_t ldt, hipStream_t st, const NeedLists* need);

template <typename T, class GX, int XCIB, class GW, int WCIB, int WCOB>
static int launch_bwd(ConvArgs<T>& a, hipStream_t st) {
    constexpr int COBLK = 8;
    if (a.gx) {
        dim3 gx((unsigned)a.n_tiles, (unsigned)((a.Cin + XCIB - 1) / XCIB));
        hipLaunchKernelGGL((conv_bwd_dx_kernel<T, GX, XCIB, COBLK>), gx, dim3(GX::NT), 0, st, a);
        APRNET_LAUNCH_CHECK("conv_bwd_dx_kernel");
    }
    dim3 gw((unsigned)std::min(a.n_tiles, 512), (unsigned)((a.Cin + WCIB - 1) / WCIB), (unsigned)((a.Cout + WCOB - 1) / WCOB));
    hipLaunchKernelGGL((conv_bwd_dw_kernel<T, GW, WCIB, WCOB>), gw, dim3(GW::NT), 0, st, a);
    APRNET_LAUNCH_CHECK("conv_bwd_dw_kernel");
    return 0;
}

// matrix-core kernels (conv_mfma.hip, conv_bwd_mfma.hip)
bool conv_mfma_supported(int code);
int launch_conv_dx_mfma(int code, const ConvArgs<float>& a, int n_tiles, hipStream_t st);
int launch_conv_dw_mfma(int code, const ConvArgs<float>& a, const TileList& tl, const WinLists* wl, int level_min, hipStream_t st);
int launch_conv_dx_mfma(int code, const ConvArgs<bf16_t>& a, int n_tiles, hipStream_t st);
int launch_conv_dw_mfma(int code, const ConvArgs<bf16_t>& a, const TileList& tl, const WinLists* wl, int level_min, hipStream_t st);
int fill_tree_for_conv(const aprnet_plan* p, int d, const bf16_t* x, int64_t ldx, int C, bf16_t* tree, int64_t ldt, hipStream_t st, const NeedLists* need);
size_t conv_packed_floats(int code, int S_exp, int Cm, int Ck, bool transposed);
int pack_conv_weights(int code, const float* w, int S_exp, int Cm, int Ck, bool transposed, float* packed, hipStream_t st, const RedoClear* redo = nullptr);
int conv_path();
// the tree nodes the forward window lists name, null: fill every node (conv.hip)
const NeedLists* needed_nodes(aprnet_plan* p, int d, int code, const TileList& tl, hipStream_t st, NeedLists* store);
// points a at the plan's window lists (conv.hip); leaves a.win_level null when they are off or unavailable
int set_conv_lists(aprnet_plan* p, int d, int code, const TileList& tl, ConvArgs<float>& a, hipStream_t st);
int set_conv_lists(aprnet_plan* p, int d, int code, const TileList& tl, ConvArgs<bf16_t>& a, hipStream_t st);
int set_conv_dx_lists(aprnet_plan* p, int d, int code, const TileList& tl, ConvArgs<bf16_t>& a, hipStream_t st);
int set_conv_dx_lists(aprnet_plan* p, int d, int code, const TileList& tl, ConvArgs<float>& a, hipStream_t st);
size_t split_dx_bytes(int code, int Cin, int S_exp, int Cout, int64_t n);
bool split_dw(int Cin, int Cout, int64_t n, int64_t ldx, int64_t ldt);
size_t split_mark_bytes();
size_t conv_packed_split_bytes(int code, int S_exp, int Cm, int Ck);
int prepare_split(int code, const float* w, int S_exp, int Cm, int Ck, bool transposed, void* packed, int* marks, const float* x, int64_t ldx, int64_t nx, float* xi,
                  hipStream_t st);
int launch_conv_dx_split(int code, const ConvArgs<float>& a, int n_win, hipStream_t st);
int launch_conv_dw_split(int code, const ConvArgs<float>& a, const DwWork& k, int* mark, hipStream_t st);
int launch_conv_dx_mfma_bf16(int code, const ConvArgs<bf16_t>& a, int n_win, hipStream_t st);
size_t conv_packed_bf16_bytes(int code, int S_exp, int Cout, int Cin);
int pack_conv_weights_bf16(int code, const float* w, int S_exp, int Cout, int Cin, void* packed, hipStream_t st, bool transposed);
int interleave8_bf16(const bf16_t* x, int64_t ldx, const bf16_t* x2, int64_t ldx2, int c_split, int C, int64_t count, bf16_t* out,
                     hipStream_t st);
int get_parents(aprnet_plan* p, hipStream_t st);
int finish_grouped_gradient(const aprnet_plan* p, int d, const float* gx4, int64_t ldx, int C, float* gt4, int64_t ldt, bf16_t* gx, int64_t ldgx,
                            const NeedLists* need, hipStream_t st);
int bf16_regroup();
int bf16_math();
int bwd_deterministic();
int launch_face_dx(const FaceLists& fl, const float* gy, int64_t ldy, const float* w, int S_exp, int Cout, int Cin, int K, int Lc,
                   float* gx, int64_t ldgx, hipStream_t st);
size_t conv_dw_g8_part_bytes(int code, int Cin, int Cout, int S_exp, int Lc, const WinLists& wl);
int launch_conv_dw_g8(int code, const bf16_t* xi, int64_t xi_ld, int64_t x_count, const bf16_t* ti, int64_t ti_ld, int64_t t_count,
                      const bf16_t* gyi, int64_t gy_ld, int64_t gy_count, int Cin, int ci0, int CinW, int Cout, int S_exp, int Lc,
                      const WinLists& wl, float* part, size_t part_bytes, float* gw, hipStream_t st);
size_t conv_dw_partial_bytes(int code, int Cout, int Cin, int S_exp, int Lc, const WinLists* wl);
// Points the weight-gradient kernels at their partial-sum slots, `off` bytes into the plan's scratch buffer (behind
// whatever the input gradient keeps there: the two run side by side).
template <typename T>
static void set_dw_partials(aprnet_plan* p, size_t off, int code, ConvArgs<T>& a) {
    a.gw_part = (float*)((char*)p->d_scratch + off);
    a.gw_part_ld = (int64_t)a.Cout * a.Cin * (code == 333 ? 27 : code == 133 ? 9 : 25);
}

// clear(finest): clears the input gradient and the tree's, with or without the places on the finest level
typedef std::function<void(bool)> ClearGradient;
template <typename T> static int try_mfma_bwd(aprnet_plan*, const ConvArgs<T>&, const TileList&, int, int, hipStream_t, bool*, void*, int64_t, const ClearGradient&) { return 0; }
static int fork_side(aprnet_plan* p, hipStream_t st, hipStream_t* side);
static int join_side(aprnet_plan* p, hipStream_t st, hipStream_t side);
// Joins the side stream on every way out of a backward call, also the failing ones: the caller's stream must not run
// ahead of a weight-gradient kernel that still reads the caller's tensors, and a capture must not end with an open fork.
struct SideJoin {
    aprnet_plan* p; hipStream_t st, side; bool open = true;
    SideJoin(aprnet_plan* p_, hipStream_t st_, hipStream_t side_) : p(p_), st(st_), side(side_) {}
    int join() { open = false; return join_side(p, st, side); }
    ~SideJoin() { if (open) (void)join_side(p, st, side); }
};
template <> int try_mfma_bwd<float>(aprnet_plan* p, const ConvArgs<float>& a, const TileList& tl, int code, int d, hipStream_t st, bool* done,
                                    void* ws, int64_t ws_bytes, const ClearGradient& clear) {
    if (conv_path() == 1 || !conv_mfma_supported(code)) return 0;
    *done = true;
    // weight gradient on the side stream (when there is an input gradient to run next to)
    ConvArgs<float> c = a;
    if (int rc = set_conv_lists(p, d, code, tl, c, st)) return rc;
    WinLists lists;
    const WinLists* wl = c.win_level && get_lists(p, d, code, tl, &lists, st) == 0 ? &lists : nullptr;
    if (!wl) c.win_level = nullptr;
    // everything that can allocate or fail on the host comes before the fork
    TileList near;
    FaceLists faces;
    const bool split_faces = a.gx && bwd_deterministic();
    if (a.gx) if (int rc = get_tiles(p, d, code == 333 ? 2 : 1, code == 333 ? 4 : 8, &near, st, 1)) return rc;
    if (split_faces) if (int rc = get_face_lists(p, d, code, &faces, st)) return rc;
    ConvArgs<float> e = a;          // input gradient on products of bfloat16 pieces: its lists
    const size_t need = split_faces && ws ? split_dx_bytes(code, a.Cin, a.S_exp, a.Cout, a.x_count) : 0;
    bool pieces = need > 0 && ws_bytes >= 0 && (size_t)ws_bytes >= need && near.n > 0;
    if (pieces) {
        if (int rc = set_conv_dx_lists(p, d, code, near, e, st)) return rc;
        pieces = e.win_level != nullptr;
    }
    const size_t wbytes = a.gx ? (conv_packed_floats(code, a.S_exp, a.Cin, a.Cout, true) * sizeof(float) + 255) / 256 * 256 : 0;
    const size_t pbytes = bwd_deterministic() ? conv_dw_partial_bytes(code, a.Cout, a.Cin, a.S_exp, a.Lc, wl) : 0;
    ScratchLease lease;          // before the join guard below: its hand-over event is recorded after the join
    if (wbytes + pbytes) if (int rc = lease.acquire(p, wbytes + pbytes, st)) return rc;
    if (pbytes) set_dw_partials(p, wbytes, code, c);
    clear(!pieces);
    // On products of bfloat16 pieces both halves read one copy of the output gradient in groups of four channels, and fp32 kernels
    // follow that do all of it again if a sum was not finite (conv_split.hip, conv_dw_split.hip).
    int* mark = nullptr;
    RedoClear redo{};
    if (pieces) {
        char* image = (char*)ws + split_mark_bytes();
        float* gi = (float*)(image + (conv_packed_split_bytes(code, a.S_exp, a.Cin, a.Cout) + 255) / 256 * 256);
        mark = (int*)ws;
        redo = RedoClear{mark, a.gx, a.ldgx, a.x_count, a.gtree, a.ldgt, a.t_count, a.Cin};
        if (int rc = prepare_split(code, a.w, a.S_exp, a.Cin, a.Cout, true, image, mark, a.gy, a.ldy, a.x_count, gi, st)) return rc;
        e.x = a.gy; e.ldx = a.ldy; e.Cin = a.Cout; e.Cout = a.Cin; e.w = (const float*)image; e.bias = nullptr; e.redo = mark;
        e.xi = gi; e.xi_ld = a.x_count;
    }
    const bool dw_pieces = pieces && wl && wl->n_win > 0 && split_dw(a.Cin, a.Cout, a.x_count, a.ldx, a.ldt);
    // Two kernels on pieces that each fill the chip run one after the other: beside each other they read more past the caches (3x3x3, 9.8 M
    // particles 32 -> 32 channels 12.6 and, on two streams, 13.8 ms, 16 -> 16 3.98 and 4.08; 1 M 64 -> 64 4.61 and 4.77, 16 -> 16 0.479
    // and 0.494; on 320 k, 32 -> 32 0.500 and 0.512, 64 -> 64 1.63 and 1.60; on 90 k 16 -> 16 0.140 and 0.134, 64 -> 64 0.670 and 0.627;
    // 1x5x5 1 M 16 -> 16 0.370 and 0.365, 3.9 M 64 -> 64 12.1 and 12.0).
    const bool in_turn = dw_pieces && code == 333 && a.x_count >= 1 << 20;
    hipStream_t side = st;
    if (a.gx && !in_turn) if (int rc = fork_side(p, st, &side)) return rc;
    SideJoin guard(p, st, side);
    if (dw_pieces) {
        c.xi = e.xi; c.xi_ld = e.xi_ld; c.redo = mark + 1;
        if (int rc = launch_conv_dw_split(code, c, dw_work(code, a.Cout, a.Cin, a.S_exp, a.Lc, *wl), mark + 1, side)) return rc;
    }
    if (int rc = launch_conv_dw_mfma(code, c, tl, wl, p->apr.level_min, side)) return rc;
    if (a.gx) {
        // input gradient: the forward kernel on the output gradient with the transposed, flipped stencil;
        // every row group within one row of an output takes part
        if (pieces) if (int rc = launch_conv_dx_split(code, e, e.n_tiles, st)) return rc;
        if (int rc = pack_conv_weights(code, a.w, a.S_exp, a.Cin, a.Cout, true, (float*)p->d_scratch, st, &redo)) return rc;
        ConvArgs<float> b = a;
        b.redo = mark;
        b.tiles = near.d_tiles; b.n_tiles = near.n;
        b.x = a.gy; b.ldx = a.ldy; b.Cin = a.Cout; b.Cout = a.Cin; b.w = (const float*)p->d_scratch; b.bias = nullptr;
        b.tree_data = nullptr; b.t_count = 0;
        b.dx_skip_faces = split_faces ? 1 : 0;
        if (near.n > 0) if (int rc = launch_conv_dx_mfma(code, b, near.n, st)) return rc;
        // coarser particles with cells outside their finer level: summed pair by pair in list order
        if (split_faces)
            if (int rc = launch_face_dx(faces, a.gy, a.ldy, a.w, a.S_exp, a.Cout, a.Cin, code == 333 ? 27 : code == 133 ? 9 : 25, a.Lc,
                                        a.gx, a.ldgx, st)) return rc;
    }
    return guard.join();
}

// Fork / join around the two halves of the backward pass: what follows fork() on the returned stream runs next to
// the caller's stream `st` until join().  Both kernels are bound by their matrix phases and the barriers between
// them at about half of the matrix peak, and read the same output gradient; side by side they fill each other's
// gaps.  Default priority, event based, so a caller may capture it into a graph.
int backward_overlap();
static int fork_side(aprnet_plan* p, hipStream_t st, hipStream_t* side) {
    *side = st;
    if (!backward_overlap()) return 0;
    if (!p->side) {
        if (int rc = side_stream_acquire(p->device, &p->side)) return rc;
        APRNET_HIP_CHECK(hipEventCreateWithFlags(&p->ev_fork, hipEventDisableTiming));
        APRNET_HIP_CHECK(hipEventCreateWithFlags(&p->ev_join, hipEventDisableTiming));
    }
    APRNET_HIP_CHECK(hipEventRecord(p->ev_fork, st));
    APRNET_HIP_CHECK(hipStreamWaitEvent(p->side, p->ev_fork, 0));
    *side = p->side;
    return 0;
}
static int join_side(aprnet_plan* p, hipStream_t st, hipStream_t side) {
    if (side == st) return 0;
    APRNET_HIP_CHECK(hipEventRecord(p->ev_join, side));
    APRNET_HIP_CHECK(hipStreamWaitEvent(st, p->ev_join, 0));
    return 0;
}

template <typename T>
int conv_bwd(const aprnet_plan* cp, int d, int kz, int kx, int ky, const T* x, int64_t ldx, int Cin, const T* w, int S_exp,
             int Cout, const T* gy, int64_t ldy, T* gx, int64_t ldgx, T* gw, T* tree_ws, int64_t ldt, T* gtree_ws,
             int64_t ldgt, hipStream_t st, void* ws = nullptr, int64_t ws_bytes = 0) {
    aprnet_plan* p = const_cast<aprnet_plan*>(cp);
    if (ws && ((uintptr_t)ws & 15) != 0) return fail(APRNET_ERR_INVALID_ARGUMENT, "conv_backward: the work space is not aligned to 16 bytes");
    if (int rc = check_level_delta(p, d, "conv_backward")) return rc;
    if (int rc = check_plane_size(p, d, sizeof(*x), "conv_backward")) return rc;
    if (int rc = check_rows(ldx, p->number_parts(d), "conv_backward", "input")) return rc;
    if (int rc = check_rows(ldy, p->number_parts(d), "conv_backward", "output gradient")) return rc;
    if (gx) if (int rc = check_rows(ldgx, p->number_parts(d), "conv_backward", "input gradient")) return rc;
    if (Cin <= 0 || Cout <= 0 || S_exp <= 0) return fail(APRNET_ERR_INVALID_ARGUMENT, "conv_backward: empty channel / stencil count");
    const int code = kz * 100 + kx * 10 + ky;
    if (code != 333 && code != 133 && code != 155 && code != 555)
        return fail(APRNET_ERR_UNSUPPORTED, "conv_backward: stencil must be 333, 133, 155 or 555");
    const int64_t nt = p->tree_parts(d);
    // gx == nullptr: the caller does not need the input gradient (first layer of a network); only gw is computed
    if (nt > 0 && (!tree_ws || ldt < nt || (gx && (!gtree_ws || ldgt < nt))))
        return fail(APRNET_ERR_INVALID_ARGUMENT, "conv_backward: tree work space too small");
    APRNET_HIP_CHECK(hipSetDevice(p->device));
    const bool flat = (kz == 1);
    TileList tl;
    if (int rc = get_tiles(p, d, flat ? 1 : 2, flat ? 8 : 4, &tl, st)) return rc;
    // the weight gradient on the matrix cores stages what the forward pass stages: the same tree nodes
    NeedLists need_store;
    const NeedLists* need = sizeof(T) == 4 ? needed_nodes(p, d, code, tl, st, &need_store) : nullptr;
    if (int rc = fill_tree_for_conv(p, d, x, ldx, Cin, tree_ws, ldt, st, need)) return rc;
    // (products of pieces write every place on the finest level, the last ones of a plane: see conv_bwd_bf16)
    auto clear = [&](bool finest) {
        if (!gx) return;
        fill2d<T>(gx, ldgx, finest ? p->number_parts(d) : p->apr.level_begin(p->lc(d)), Cin, (T)0, st);
        fill2d<T>(gtree_ws, ldgt, nt, Cin, (T)0, st);
    };
    if (tl.n > 0) {
        ConvArgs<T> a{};
        a.apr = p->dapr; a.tree = p->dtree; a.tiles = tl.d_tiles; a.n_tiles = tl.n;
        a.x = x; a.ldx = ldx; a.Cin = Cin; a.w = w; a.S_exp = S_exp; a.Cout = Cout;
        a.tree_data = tree_ws; a.ldt = ldt; a.Lc = p->lc(d); a.tree_off = p->tree_offset(a.Lc);
    a.x_count = p->number_parts(d); a.t_count = p->tree_parts(d);
        a.gy = gy; a.ldy = ldy; a.gx = gx; a.ldgx = ldgx; a.gtree = gtree_ws; a.ldgt = ldgt; a.gw = gw;
        constexpr bool f32 = sizeof(T) == 4;
        int rc = 0;
        bool done = false;
        if ((rc = try_mfma_bwd<T>(p, a, tl, code, d, st, &done, ws, ws_bytes, clear))) return rc;
        if (!done) clear(true);
        if (!done) switch (code) {
            case 333: rc = launch_bwd<T, X333, (f32 ? 4 : 2), W333, (f32 ? 8 : 4), (f32 ? 32 : 16)>(a, st); break;
            case 133: rc = launch_bwd<T, X133, (f32 ? 8 : 4), W133, (f32 ? 8 : 4), (f32 ? 32 : 16)>(a, st); break;
            case 155: rc = launch_bwd<T, X155, (f32 ? 4 : 2), W155, (f32 ? 8 : 4), (f32 ? 32 : 16)>(a, st); break;
            case 555: rc = launch_bwd<T, X555, 1, W555, (f32 ? 4 : 2), (f32 ? 32 : 16)>(a, st); break;
        }
        if (rc) return rc;
    } else clear(true);
    return gx ? fill_tree_bwd_for_conv(p, d, gx, ldgx, Cin, gtree_ws, ldgt, st, need) : 0;
}

// Bound by memory (6 bytes per value).  One value per lane and turn of a grid-stride loop took 1.47 ms
// for 64 channels of 15.4 M particles, 4.0 TB/s (gain: see fill_kernel).
__global__ void __launch_bounds__(STREAM_TB)
round_to_bf16_kernel(const float* __restrict__ src, int64_t lds, bf16_t* __restrict__ dst, int64_t ldd, int64_t n) {
    typedef float vecf __attribute__((ext_vector_type(STREAM_V), aligned(4)));
    typedef unsigned vech __attribute__((ext_vector_type(STREAM_V / 2), aligned(2)));
    const float* s = src + (int64_t)blockIdx.y * lds;
    bf16_t* d = dst + (int64_t)blockIdx.y * ldd;
    const int64_t i0 = (int64_t)blockIdx.x * STREAM_BLOCK + threadIdx.x * STREAM_V;
    if ((int64_t)(blockIdx.x + 1) * STREAM_BLOCK <= n) {                    // uniform
        vecf v[STREAM_R];
#pragma unroll
        for (int r = 0; r < STREAM_R; ++r) v[r] = *reinterpret_cast<const vecf*>(s + i0 + r * (STREAM_TB * STREAM_V));
#pragma unroll
        for (int r = 0; r < STREAM_R; ++r) {
            vech w;
#pragma unroll
            for (int e = 0; e < STREAM_V / 2; ++e)
                w[e] = (unsigned)float_to_bf16(v[r][2 * e]).bits | ((unsigned)float_to_bf16(v[r][2 * e + 1]).bits << 16);
            *reinterpret_cast<vech*>(d + i0 + r * (STREAM_TB * STREAM_V)) = w;
        }
        return;
    }
    for (int64_t i = (int64_t)blockIdx.x * STREAM_BLOCK + threadIdx.x; i < n; i += STREAM_TB) d[i] = float_to_bf16(s[i]);   // last block
}

// Input channels of the features and tree that the grouped weight gradient copies at a time (whole blocks of the kernel, 16
// channels).  The scratch buffer stays with the plan, so a program with a plan per APR pays for it on each: beside the
// output gradient's copy these may take what the forward pass of the layer has needed for its own copies anyway, plus
// 256 MiB; wider layers on larger APRs copy a part of their channels at a time, in equal parts.  Next to the input gradient,
// which fills the ends of the parts' launches, that costs no time (1x5x5 64 -> 64 on 15.4 M particles, four parts: 25.0 ->
// 24.4 ms forward and backward; 3x3x3 64 -> 64 on 23 M 38.3 -> 38.5 ms backward).  Without an input gradient it
// would (128 -> 64 on 5.4 M 9.9 -> 10.5 ms), and the call then has no fp32 work spaces, which are larger than the
// copies: all channels at once.
static int dw_copy_channels(int Cin, int64_t np, int64_t nt, size_t gybytes) {
    const size_t blk = (size_t)(np + nt) * 32, all = (size_t)((Cin + 7) / 8) * (size_t)(np + nt) * 16;
    const int nb = (Cin + 15) / 16;
    const size_t room = std::max(all, gybytes) - gybytes + ((size_t)256 << 20);
    const int most = (int)std::min<size_t>(nb, std::max<size_t>(1, room / std::max<size_t>(blk, 1)));
    const int parts = (nb + most - 1) / most;
    return 16 * ((nb + parts - 1) / parts);
}

// bfloat16 features and output gradient; weights, weight gradient and all accumulation in fp32 (the fp32
// matrix-core kernels with 16-bit loads).  gx32_ws [Cin][ldgx32] and gtree_ws [Cin][ldgt] are fp32 work space:
// the input gradient is accumulated there and rounded to bfloat16 at the end.
int conv_bwd_bf16(const aprnet_plan* cp, int d, int kz, int kx, int ky, const bf16_t* x, int64_t ldx, int Cin, const float* w,
                  int S_exp, int Cout, const bf16_t* gy, int64_t ldy, bf16_t* gx, int64_t ldgx, float* gw, bf16_t* tree_ws,
                  int64_t ldt, float* gx32_ws, int64_t ldgx32, float* gtree_ws, int64_t ldgt, hipStream_t st) {
    aprnet_plan* p = const_cast<aprnet_plan*>(cp);
    if (int rc = check_level_delta(p, d, "conv_backward")) return rc;
    if (int rc = check_plane_size(p, d, sizeof(float), "conv_backward")) return rc;
    if (int rc = check_rows(ldx, p->number_parts(d), "conv_backward", "input")) return rc;
    if (int rc = check_rows(ldy, p->number_parts(d), "conv_backward", "output gradient")) return rc;
    if (gx) if (int rc = check_rows(ldgx, p->number_parts(d), "conv_backward", "input gradient")) return rc;
    if (Cin <= 0 || Cout <= 0 || S_exp <= 0) return fail(APRNET_ERR_INVALID_ARGUMENT, "conv_backward: empty channel / stencil count");
    const int code = kz * 100 + kx * 10 + ky;
    if (!conv_mfma_supported(code))
        return fail(APRNET_ERR_UNSUPPORTED, "conv_backward: bfloat16 features are supported for the 3x3x3, 1x3x3 and 1x5x5 stencils");
    const int64_t nt = p->tree_parts(d), np = p->number_parts(d);
    if ((gx && (!gx32_ws || ldgx32 < np)) || (nt > 0 && (!tree_ws || ldt < nt || (gx && (!gtree_ws || ldgt < nt)))))
        return fail(APRNET_ERR_INVALID_ARGUMENT, "conv_backward: work space too small");
    APRNET_HIP_CHECK(hipSetDevice(p->device));
    const bool flat = (kz == 1);
    TileList tl, near;
    if (int rc = get_tiles(p, d, flat ? 1 : 2, flat ? 8 : 4, &tl, st)) return rc;
    NeedLists need_store;
    const NeedLists* nodes = needed_nodes(p, d, code, tl, st, &need_store);
    if (int rc = get_tiles(p, d, flat ? 1 : 2, flat ? 8 : 4, &near, st, 1)) return rc;
    bool g4 = false;                 // the work spaces hold groups of four channels (grad_groups.hip)
    if (tl.n > 0) {
        ConvArgs<bf16_t> a{};
        a.apr = p->dapr; a.tree = p->dtree; a.tiles = tl.d_tiles; a.n_tiles = tl.n;
        a.x = x; a.ldx = ldx; a.Cin = Cin; a.w = w; a.S_exp = S_exp; a.Cout = Cout;
        a.tree_data = tree_ws; a.ldt = ldt; a.Lc = p->lc(d); a.tree_off = p->tree_offset(a.Lc);
        a.x_count = np; a.t_count = nt;
        a.gy = gy; a.ldy = ldy; a.gx = gx32_ws; a.ldgx = ldgx32; a.gtree = gtree_ws; a.ldgt = ldgt; a.gw = gw;
        ConvArgs<bf16_t> b = a;
        b.tiles = near.d_tiles; b.n_tiles = near.n;
        b.x = gy; b.ldx = ldy; b.Cin = Cout; b.Cout = Cin; b.bias = nullptr;
        b.tree_data = nullptr; b.t_count = 0;
        // input gradient: bfloat16 products on the input-gradient lists of the plan when they are there, otherwise
        // (lists off or not buildable, fp32 products asked for) the scanning kernel with fp32 products
        if (!gx) near.n = 0;              // no input gradient asked for
        // weight gradient on the side stream, next to the input gradient
        if (int rc = set_conv_lists(p, d, code, tl, a, st)) return rc;
        // everything that can allocate or fail on the host comes before the fork
        if (near.n > 0 && bf16_math())
            if (int rc = set_conv_dx_lists(p, d, code, near, b, st)) return rc;
        // (the kernels with lists; other channel counts, tables that cannot be built: planes)
        g4 = near.n > 0 && b.win_level && Cin % 4 == 0 && (((uintptr_t)gx32_ws | (uintptr_t)gtree_ws) & 15) == 0 && get_parents(p, st) == 0;
        if (g4) {
            b.gx_g4 = 1; b.ldgx = np; b.ldgt = nt;
            // Places on the finest level, the last ones, are written by the one column they have (COL_SOLE): cleared are the others.
            fill2d<float>(gx32_ws, 4 * np, 4 * p->apr.level_begin(p->lc(d)), Cin / 4, 0.f, st);
            fill2d<float>(gtree_ws, 4 * nt, 4 * nt, Cin / 4, 0.f, st);
        }
        // Both halves stage from copies grouped by eight channels behind the packed weights in the scratch buffer: the output
        // gradient (read by both), the features and their tree (weight gradient).
        auto align = [](size_t v) { return (v + 255) / 256 * 256; };
        const size_t ngo = (size_t)(Cout + 7) / 8, ngi = (size_t)(Cin + 7) / 8;
        // the image of the weights that the input gradient below packs: fp32 ones where it has no lists (twice the bfloat16 size)
        const size_t wbytes = near.n == 0 ? 0 : align(b.win_level ? conv_packed_bf16_bytes(code, S_exp, Cin, Cout)
                                                                 : conv_packed_floats(code, S_exp, Cin, Cout, true) * sizeof(float));
        const size_t gybytes = align(ngo * (size_t)np * 16);
        const bool tree_g8 = tree_ws_grouped(Cin, tree_ws);          // the tree is made of the regrouped features, in its work space
        const int chunk = gx ? dw_copy_channels(Cin, np, tree_g8 ? 0 : nt, gybytes) : (Cin + 15) / 16 * 16;
        const size_t ngc = std::min<size_t>(ngi, chunk / 8), xbytes = align(ngc * (size_t)np * 16), tbytes = tree_g8 ? 0 : align(ngc * (size_t)nt * 16);
        const bool regroup = bf16_math() && bf16_regroup() && np < (1ll << 28) && nt < (1ll << 28);
        const bool regroup_gy = regroup && gybytes <= ((size_t)32 << 30);
        WinLists wl;
        const bool listed = a.win_level && get_lists(p, d, code, tl, &wl, st, false) == 0;
        if (!listed) a.win_level = nullptr;
        bool dw_g8 = regroup_gy && bwd_deterministic() && listed && gybytes + ngi * (size_t)(np + nt) * 16 <= ((size_t)48 << 30);
        const bool dx_g8 = near.n > 0 && b.win_level && regroup_gy;
        size_t need = 0, pbytes = 0;
        auto layout = [&]() {
            need = wbytes + (dw_g8 || dx_g8 ? gybytes : 0) + (dw_g8 ? xbytes + tbytes : 0);
            const int last = Cin - (Cin - 1) / chunk * chunk;              // channels of the last part
            pbytes = dw_g8 ? std::max(conv_dw_g8_part_bytes(code, std::min(Cin, chunk), Cout, S_exp, a.Lc, wl),
                                      conv_dw_g8_part_bytes(code, last, Cout, S_exp, a.Lc, wl)) : bwd_deterministic() ? conv_dw_partial_bytes(code, Cout, Cin, S_exp, a.Lc, listed ? &wl : nullptr) : 0;
            return need + pbytes;
        };
        ScratchLease lease;      // before the join guard below: its hand-over event is recorded after the join
        if (layout()) {
            int rc = lease.acquire(p, need + pbytes, st, dw_g8);
            if (rc && dw_g8) {   // no room for the copies, or a capture that may not grow the buffer: the kernel on channel planes
                (void)hipGetLastError();
                dw_g8 = false;
                rc = layout() ? lease.acquire(p, need + pbytes, st) : 0;
            }
            if (rc) return rc;
        }
        if (pbytes && !dw_g8) set_dw_partials(p, need, code, a);
        if (!dw_g8 || !tree_g8)
            if (int rc = fill_tree_for_conv(p, d, x, ldx, Cin, tree_ws, ldt, st, nodes)) return rc;
        if (gx && !g4) {
            fill2d<float>(gx32_ws, ldgx32, np, Cin, 0.f, st);
            fill2d<float>(gtree_ws, ldgt, nt, Cin, 0.f, st);
        }
        bf16_t* gyi = (bf16_t*)((char*)p->d_scratch + wbytes);
        if (dw_g8 || dx_g8) if (int rc = interleave8_bf16(gy, ldy, nullptr, 0, Cout, Cout, np, gyi, st)) return rc;
        // side by side at any size (in turn, forward and backward: 3x3x3 64 -> 64 channels on 1.2 M particles 2.03 instead of 2.12 ms, on 5.5 M 9.53
        // and 9.45, 1x5x5 64 -> 64 on 15.4 M 18.5 and 18.2)
        hipStream_t side = st;
        if (near.n > 0) if (int rc = fork_side(p, st, &side)) return rc;
        SideJoin guard(p, st, side);
        if (dw_g8) {
            bf16_t* xi = (bf16_t*)((char*)gyi + gybytes);
            for (int c0 = 0; c0 < Cin; c0 += chunk) {
                const int c = std::min(chunk, Cin - c0);
                if (int rc = interleave8_bf16(x + (int64_t)c0 * ldx, ldx, nullptr, 0, c, c, np, xi, side)) return rc;
                bf16_t* ti = tree_g8 ? tree_ws + (int64_t)c0 * nt : (bf16_t*)((char*)xi + xbytes);
                if (int rc = tree_g8 ? fill_tree_mean_g8(p, d, xi, np, c, ti, nt, side, nodes)
                                     : interleave8_bf16(tree_ws + (int64_t)c0 * ldt, ldt, nullptr, 0, c, c, nt, ti, side)) return rc;
                if (int rc = launch_conv_dw_g8(code, xi, np, np, ti, nt, nt, gyi, np, np, c, c0, Cin, Cout, S_exp, a.Lc, wl,
                                               (float*)((char*)p->d_scratch + need), pbytes, gw, side)) return rc;
            }
        } else if (int rc = launch_conv_dw_mfma(code, a, tl, listed ? &wl : nullptr, p->apr.level_min, side)) return rc;
        if (near.n > 0 && b.win_level) {
            if (int rc = pack_conv_weights_bf16(code, w, S_exp, Cin, Cout, p->d_scratch, st, true)) return rc;
            if (dx_g8) { b.xi = gyi; b.ti = nullptr; b.xi_ld = np; b.ti_ld = 0; }
            b.w = (const float*)p->d_scratch;
            if (int rc = launch_conv_dx_mfma_bf16(code, b, b.n_tiles, st)) return rc;
        } else if (near.n > 0) {
            if (int rc = pack_conv_weights(code, w, S_exp, Cin, Cout, true, (float*)p->d_scratch, st)) return rc;
            b.w = (const float*)p->d_scratch;
            b.win_level = nullptr;
            if (int rc = launch_conv_dx_mfma(code, b, near.n, st)) return rc;
        }
        if (int rc = guard.join()) return rc;
    } else if (gx) {
        fill2d<float>(gx32_ws, ldgx32, np, Cin, 0.f, st);
        fill2d<float>(gtree_ws, ldgt, nt, Cin, 0.f, st);
    }
    if (!gx) return 0;
    if (g4) return finish_grouped_gradient(p, d, gx32_ws, np, Cin, gtree_ws, nt, gx, ldgx, nodes, st);
    if (int rc = fill_tree_bwd_for_conv(p, d, gx32_ws, ldgx32, Cin, gtree_ws, ldgt, st, nodes)) return rc;
    if (np > 0) {
        dim3 grid((unsigned)((np + STREAM_BLOCK - 1) / STREAM_BLOCK), (unsigned)Cin);
        hipLaunchKernelGGL(round_to_bf16_kernel, grid, dim3(STREAM_TB), 0, st, gx32_ws, ldgx32, gx, ldgx, np);
        APRNET_LAUNCH_CHECK("round_to_bf16_kernel");
    }
    return 0;
}

}  // namespace aprnet

using namespace aprnet;
extern "C" {
int aprnet_conv_bwd_bf16(const aprnet_plan* p, int d, int kz, int kx, int ky, const uint16_t* x, int64_t ldx, int Cin,
                         const float* w, int S_exp, int Cout, const uint16_t* gy, int64_t ldy, uint16_t* gx, int64_t ldgx,
                         float* gw, uint16_t* tree_ws, int64_t ldt, float* gx32_ws, int64_t ldgx32, float* gtree_ws,
                         int64_t ldgt, void* st) {
    return conv_bwd_bf16(p, d, kz, kx, ky, (const bf16_t*)x, ldx, Cin, w, S_exp, Cout, (const bf16_t*)gy, ldy, (bf16_t*)gx, ldgx,
                         gw, (bf16_t*)tree_ws, ldt, gx32_ws, ldgx32, gtree_ws, ldgt, (hipStream_t)st);
}
int aprnet_conv_bwd_f32(const aprnet_plan* p, int d, int kz, int kx, int ky, const float* x, int64_t ldx, int Cin,
                        const float* w, int S_exp, int Cout, const float* gy, int64_t ldy, float* gx, int64_t ldgx,
                        float* gw, float* tree_ws, int64_t ldt, float* gtree_ws, int64_t ldgt, void* st) {
    return conv_bwd<float>(p, d, kz, kx, ky, x, ldx, Cin, w, S_exp, Cout, gy, ldy, gx, ldgx, gw, tree_ws, ldt, gtree_ws,
                           ldgt, (hipStream_t)st);
}
int64_t aprnet_conv_bwd_ws_bytes_f32(const aprnet_plan* p, int d, int kz, int kx, int ky, int Cin, int S_exp, int Cout) {
    if (!p || d < 0 || d >= p->tree.level_max + 1 || Cin <= 0 || S_exp <= 0 || Cout <= 0 || !bwd_deterministic()) return 0;
    return (int64_t)split_dx_bytes(kz * 100 + kx * 10 + ky, Cin, S_exp, Cout, p->number_parts(d));
}
int aprnet_conv_bwd_ws_f32(const aprnet_plan* p, int d, int kz, int kx, int ky, const float* x, int64_t ldx, int Cin,
                           const float* w, int S_exp, int Cout, const float* gy, int64_t ldy, float* gx, int64_t ldgx,
                           float* gw, float* tree_ws, int64_t ldt, float* gtree_ws, int64_t ldgt, void* ws, int64_t ws_bytes, void* st) {
    return conv_bwd<float>(p, d, kz, kx, ky, x, ldx, Cin, w, S_exp, Cout, gy, ldy, gx, ldgx, gw, tree_ws, ldt, gtree_ws,
                           ldgt, (hipStream_t)st, ws, ws_bytes);
}
int aprnet_conv_bwd_f64(const aprnet_plan* p, int d, int kz, int kx, int ky, const double* x, int64_t ldx, int Cin,
                        const double* w, int S_exp, int Cout, const double* gy, int64_t ldy, double* gx, int64_t ldgx,
                        double* gw, double* tree_ws, int64_t ldt, double* gtree_ws, int64_t ldgt, void* st) {
    return conv_bwd<double>(p, d, kz, kx, ky, x, ldx, Cin, w, S_exp, Cout, gy, ldy, gx, ldgx, gw, tree_ws, ldt, gtree_ws,
                            ldgt, (hipStream_t)st);
}
}
