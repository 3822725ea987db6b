// Window lists: what the convolution kernels stage and compute per window, built once per APR, level delta and
// stencil and kept in the plan.  A list entry is an index into the feature / tree vector plus a cell of the LDS
// patch, so the lists depend on the APR alone; every convolution call at that level delta reuses them and its
// kernel neither searches the access arrays nor keeps list bookkeeping in LDS.
//
// Windows are cut from a compressed y axis.  A row group (2 x 4 rows, 1 x 8 for flat stencils) of a sparse APR has outputs at a part
// of its y positions only, in thin shells around what is finely resolved: kept are the positions within the stencil's reach of an
// output, one after the other, and the kept positions of all row groups of a level behind each other, with as many empty cells between
// two groups as the stencil reaches.  Neighbours along y of an output are kept with it, so they are neighbours on the compressed
// axis too, and what lies next to the end of a run there is a position that no output occupies.  A window is up to 62 (60) cells of that axis
// and its halo, whatever row groups they come from; the kernels see cells only.
// The kernels are bound by what a window costs whether it is full or not (lists, round trips, weights, barriers).  Windows of
// 62 positions of one row group, as they were, held 173 outputs of 496 on average on the 23 M particles of a blob volume (134,000
// windows, now 60,200 of 385), 118 on a sparse light-sheet one of 43 M (366,000, now 121,000 of 355), 311 on a dense one of 52 M (167,000, now
// 121,000 of 428).  By the windows alone, whole passes: 3x3x3 of fp32 features 32 -> 32 on the first 11.6 -> 9.7 ms, 16 -> 16 on the second 9.1 -> 7.0, a
// bfloat16 U-Net on the third 58.4 -> 53.7.
//
// Three passes over the row groups: kept positions, then items and columns per window, then the lists; the host turns the counts into
// offsets in between.
#include "conv_common.hpp"

#include <cstring>

namespace aprnet {

struct ListArgs {
    AccessDev apr, tree;
    const ConvTile* tiles; int n_tiles;
    int Lc; int64_t tree_off;
    int skip_faces;                // input gradient: no columns for coarser particles that stick out of a far face
    int words;                     // 64-bit words of a row's bit map, for the longest rows
    int per_row;                   // a bit map per staged row fits LDS: items and columns are kept if an output lies in reach on three axes, not only along y
    int* n_cells;                  // [n_tiles] pass 0: kept positions of a row group
    const int* first_cell;         // [n_tiles] its first cell on the compressed axis of its level
    int win0[MAX_LEVELS + 1], nwin[MAX_LEVELS + 1];          // windows of a level
    int ty;                        // cells of a window without its halo
    int used_words;                // 64-bit words of the counters of a row group's windows
    int4* count;                   // [windows] pass 1: items, groups of columns (see dx_group), other columns
    const int* slot0;              // [n_tiles] first entry in `share` of a row group, which has one per window it stages a cell of,
    int4* share;                   // pass 1: the entries of other row groups before its own
    const int4* off;               // [windows] pass 2: first item, first column, groups of columns, 1 if the window is stored
    int* item_idx; unsigned short* item_pos; int* col_idx; unsigned short* col_pos;
};

// word u of a bit map (p the one before, n the one after it), dilated by hy to either side
__device__ __forceinline__ unsigned long long dilated(unsigned long long u, unsigned long long p, unsigned long long n, int hy) {
    unsigned long long k = u;
    for (int h = 1; h <= hy; ++h) k |= (u << h) | (u >> h) | (p >> (64 - h)) | (n << (64 - h));
    return k;
}

// DX: lists of the input gradient: items are the output positions of the staged rows, columns every cell of the centre rows that some
// source covers and an output reaches (the others' gradient is zero), those of a coarser particle in groups (dx_group).
// PASS 0 counts kept positions, 1 items and columns, 2 writes them.
template <class G, bool DX, int PASS>
__global__ void __launch_bounds__(G::NT)
build_lists_kernel(const ListArgs a) {
    extern __shared__ unsigned long long maps[];
    __shared__ int seg_b[G::NSEG], seg_e[G::NSEG];
    __shared__ int total;
    const ConvTile tile = a.tiles[blockIdx.x];
    const int L = tile.level, yn = a.apr.y_num[L], zn = a.apr.z_num[L], xn = a.apr.x_num[L];
    const bool out_tree = L == a.Lc && L < a.apr.level_max, tree_from_x = L == a.Lc;
    const int W = (yn + 63) >> 6, lane = lane_id(), wave = threadIdx.x >> 6;
    unsigned long long* keep = maps;                                     // [W] kept positions
    unsigned long long* any = maps + a.words;                            // [W] positions with an output in some row
    int* before = reinterpret_cast<int*>(maps + 2 * a.words);            // [W] kept positions in the words before
    int* used = reinterpret_cast<int*>(maps + 3 * a.words);              // [windows of the group][3] entries so far (pass 2: and those of other groups before them)
    unsigned long long* rows = maps + 3 * a.words + a.used_words;    // [NROW][W] outputs of a row (per_row)
    unsigned long long* reach = rows + G::NROW * a.words;                // [NROW][W] positions of a row with an output in reach (per_row)

    // ---- the rows of the group: particles of the level, of the coarser one, tree nodes
    for (int s = threadIdx.x; s < G::NSEG; s += G::NT) {
        const int r = s / 3, src = s - 3 * r, rz = r / G::RX, rx = r - rz * G::RX;
        const int z = tile.z0 - G::HZ + rz, x = tile.x0 - G::HX + rx;
        int b = 0, e = 0;
        if (z >= 0 && z < zn && x >= 0 && x < xn && (src == 0 || (src == 1 ? L > a.apr.level_min : L < a.apr.level_max))) {
            const AccessDev& acc = src == 2 ? a.tree : a.apr;
            const uint64_t row = src == 1 ? acc.row(L - 1, z >> 1, x >> 1) : acc.row(L, z, x);
            b = (int)acc.xz_end[row - 1]; e = (int)acc.xz_end[row];
        }
        seg_b[s] = b; seg_e[s] = e;
    }
    for (int i = threadIdx.x; i < W; i += G::NT) any[i] = 0;
    if (a.per_row) for (int i = threadIdx.x; i < G::NROW * W; i += G::NT) rows[i] = 0;
    __syncthreads();

    // ---- outputs (of the centre rows, DX: of all staged ones), and the positions within the stencil's reach of one along y
    auto centre = [](int r) { const int rz = r / G::RX, rx = r - rz * G::RX; return rz >= G::HZ && rz < G::HZ + G::TZ && rx >= G::HX && rx < G::HX + G::TX; };
    for (int s = wave; s < G::NSEG; s += G::NWAVE) {
        const int r = s / 3, src = s - 3 * r;
        if (!(src == 0 || (src == 2 && out_tree)) || !(DX || centre(r))) continue;
        const uint16_t* yv = src == 2 ? a.tree.y : a.apr.y;
        for (int i = seg_b[s] + lane; i < seg_e[s]; i += 64) {
            const int y = yv[i];
            atomicOr(&any[y >> 6], 1ull << (y & 63));
            if (a.per_row) atomicOr(&rows[r * W + (y >> 6)], 1ull << (y & 63));
        }
    }
    __syncthreads();
    for (int w = threadIdx.x; w < W; w += G::NT) {
        unsigned long long k = dilated(any[w], w > 0 ? any[w - 1] : 0, w + 1 < W ? any[w + 1] : 0, G::HY);
        // whole pairs 2y, 2y + 1, which a coarser particle covers; the added position has no output in reach and, like the last one of the run that
        // it lies next to on the compressed axis, none on it
        if (DX) k |= ((k & 0x5555555555555555ull) << 1) | ((k >> 1) & 0x5555555555555555ull);
        if (w == W - 1 && (yn & 63)) k &= ~0ull >> (64 - (yn & 63));
        keep[w] = k;
    }
    if (PASS > 0 && a.per_row)
        for (int i = threadIdx.x; i < G::NROW * W; i += G::NT) {
            const int r = i / W, w = i - r * W, rz = r / G::RX, rx = r - rz * G::RX;
            unsigned long long u = 0, p = 0, n = 0;
            for (int z2 = max(rz - G::HZ, 0); z2 <= min(rz + G::HZ, G::RZ - 1); ++z2)
                for (int x2 = max(rx - G::HX, 0); x2 <= min(rx + G::HX, G::RX - 1); ++x2) {
                    const unsigned long long* m = rows + (z2 * G::RX + x2) * W + w;
                    u |= m[0];
                    if (w > 0) p |= m[-1];
                    if (w + 1 < W) n |= m[1];
                }
            reach[i] = dilated(u, p, n, G::HY);
        }
    __syncthreads();
    if (wave == 0) {
        int sum = 0;
        for (int w0 = 0; w0 < W; w0 += 64) {
            const int n = w0 + lane < W ? __popcll(keep[w0 + lane]) : 0;
            int inc = n;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) { const int t = __shfl_up(inc, d); if (lane >= d) inc += t; }
            if (w0 + lane < W) before[w0 + lane] = sum + inc - n;
            sum += __shfl(inc, 63);
        }
        if (lane == 0) total = sum;
    }
    __syncthreads();
    if constexpr (PASS == 0) {
        if (threadIdx.x == 0) a.n_cells[blockIdx.x] = total;
        return;
    }
    const int first = a.first_cell[blockIdx.x], win0 = a.win0[L], nwin = a.nwin[L];
    auto kept = [&](int y) { return y >= 0 && y < yn && ((keep[y >> 6] >> (y & 63)) & 1ull) != 0; };
    auto cell_of = [&](int y) { return first + before[y >> 6] + __popcll(keep[y >> 6] & ((1ull << (y & 63)) - 1ull)); };
    // an output within the stencil's reach of position y of row r (whose position is kept)
    auto reached = [&](int r, int y) { return !a.per_row || ((reach[r * W + (y >> 6)] >> (y & 63)) & 1ull) != 0; };
    const int ty = a.ty, wf = max(first - G::HY, 0) / ty;        // first window that stages a cell of the group
    const int nw = total > 0 ? min((first + total - 1 + G::HY) / ty, nwin - 1) - wf + 1 : 0;
    int4* share = a.share + a.slot0[blockIdx.x];
    for (int i = threadIdx.x; i < nw; i += G::NT) {
        const int4 o = PASS == 2 ? share[i] : make_int4(0, 0, 0, 0);
        used[3 * i] = o.x; used[3 * i + 1] = o.y; used[3 * i + 2] = o.z;
    }
    __syncthreads();
    // One entry per lane with `has` to window w (of the level): place(number of the entry among those of `field` in that window)
    auto append = [&](bool has, int w, int field, auto place) {
        for (unsigned long long m = __ballot(has); m; m = __ballot(has)) {
            const int lead = __ffsll(m) - 1, wl = __shfl(w, lead);
            const unsigned long long mm = __ballot(has && w == wl);
            int base = 0;
            if (lane == lead) base = atomicAdd(&used[3 * (wl - wf) + field], __popcll(mm));
            if constexpr (PASS == 2) base = __shfl(base, lead);
            if (has && w == wl) {
                if constexpr (PASS == 2) place(win0 + wl, base + __popcll(mm & ((1ull << lane) - 1ull)));
                has = false;
            }
        }
    };
    // an item on cell c, and on c + 1 if it is a pair, for every window that stages one of the two
    auto item = [&](bool has, int r, int c, bool pair, int idx, unsigned flags) {
        const int lo = max(c - G::HY, 0) / ty, hi = min((c + (pair ? 1 : 0) + G::HY) / ty, nwin - 1), wy = ty + 2 * G::HY;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int w = lo + k, p = c - (w * ty - G::HY);
            const bool in = p >= 0 && p < wy, in2 = pair && p + 1 >= 0 && p + 1 < wy;
            append(has && w <= hi && (in || in2), w, 0, [&](int win, int n) {
                const int4 o = a.off[win];
                if (!o.w) return;
                a.item_idx[(size_t)(unsigned)o.x + n] = idx;
                a.item_pos[(size_t)(unsigned)o.x + n] = (unsigned short)((r * G::RS + (in ? p : p + 1)) | flags | (in && in2 ? ITEM_PAIR : 0u));
            });
        }
    };
    auto column = [&](bool has, int r, int c, int idx, unsigned flags) {
        const int w = c / ty;
        append(has, w, 2, [&](int win, int n) {
            const int4 o = a.off[win];
            if (!o.w) return;
            const size_t at = (size_t)(unsigned)o.y + (DX ? dx_group<G>() * o.z : 0) + n;
            a.col_idx[at] = idx;
            a.col_pos[at] = (unsigned short)((r * G::RS + c - w * ty + G::HY) | flags);
        });
    };
    for (int s = wave; s < G::NSEG; s += G::NWAVE) {
        const int r = s / 3, src = s - 3 * r, rz = r / G::RX, rx = r - rz * G::RX;
        const int z = tile.z0 - G::HZ + rz, x = tile.x0 - G::HX + rx;
        const bool mid = centre(r), is_out = src == 0 || (src == 2 && out_tree);
        const uint16_t* yv = src == 2 ? a.tree.y : a.apr.y;
        const int plus = src == 2 && tree_from_x ? (int)a.tree_off : 0;
        for (int i0 = seg_b[s]; i0 < seg_e[s]; i0 += 64) {                // wave-uniform
            const int i = i0 + lane;
            const bool valid = i < seg_e[s];
            const int y = valid ? (int)yv[i] : 0, ya = src == 1 ? 2 * y : y, yb = ya + 1;
            const bool ka = valid && kept(ya), kb = src == 1 && valid && kept(yb);
            const int ca = ka ? cell_of(ya) : 0, cb = kb ? cell_of(yb) : 0;
            if constexpr (!DX) {
                const bool need = (ka && reached(r, ya)) || (kb && reached(r, yb));
                item(need, r, ka ? ca : cb, ka && kb, i + plus, src == 2 && !tree_from_x ? ITEM_TREE : 0u);
                if (mid && is_out) column(valid, r, ca, i + plus, 0u);
            } else {
                if (is_out) item(valid, r, ca, false, i + plus, 0u);
                if (!mid) continue;
                if (src != 1) {
                    // a place is a centre cell of one window of its own level; further columns come from windows one level finer, which see
                    // it as a coarser particle: none above the finest level, none for a tree node
                    const bool to_tree = src == 2 && !tree_from_x;
                    column(ka && reached(r, ya), r, ca, i + plus, (to_tree ? COL_TREE : 0u) | (to_tree || tree_from_x ? COL_SOLE : 0u));
                    continue;
                }
                constexpr int N = dx_group<G>(), BOXZ = G::TZ >= 2 ? 2 : 1;         // a flat tile sees one z-slice of the coarser particle
                const bool rows_full = (BOXZ == 1 || (z | 1) < zn) && (x | 1) < xn;  // wave-uniform
                const bool first_row = (BOXZ == 1 || (z & 1) == 0) && (x & 1) == 0;
                const bool pooled = rows_full && yb < yn;
                if (rows_full && first_row) {
                    bool hit = false;
                    if (pooled && ka)
#pragma unroll
                        for (int k = 0; k < N; ++k) hit = hit || reached(r + (k >> 2) * G::RX + ((k >> 1) & 1), ya + (k & 1));
                    const int w = ca / ty;
                    append(hit, w, 1, [&](int win, int n) {
                        const int4 o = a.off[win];
                        if (!o.w) return;
#pragma unroll
                        for (int k = 0; k < N; ++k) {                     // cells in the order z, x, y
                            const size_t at = (size_t)(unsigned)o.y + N * n + k;
                            a.col_idx[at] = i;
                            a.col_pos[at] = (unsigned short)(((r + (k >> 2) * G::RX + ((k >> 1) & 1)) * G::RS + ca - w * ty + G::HY + (k & 1)) | COL_BOX);
                        }
                    });
                }
                if (!a.skip_faces) {
                    column(ka && !pooled && reached(r, ya), r, ca, i, 0u);
                    column(kb && !pooled && reached(r, yb), r, cb, i, 0u);
                }
            }
        }
    }
    if constexpr (PASS == 1) {
        __syncthreads();
        for (int i = threadIdx.x; i < nw; i += G::NT) {
            int* c = reinterpret_cast<int*>(a.count + win0 + wf + i);
            int o[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) o[k] = used[3 * i + k] ? atomicAdd(c + k, used[3 * i + k]) : 0;
            share[i] = make_int4(o[0], o[1], o[2], 0);
        }
    }
}

using L333 = ConvGeom<3, 3, 3, 2, 4, 512>;
using L133 = ConvGeom<1, 3, 3, 1, 8, 512>;
using L155 = ConvGeom<1, 5, 5, 1, 8, 512>;

static size_t list_lds(int words, int rows, int used_words) { return 8 * ((size_t)words * (3 + 2 * rows) + used_words); }
template <class G, bool DX>
static void launch_build(const ListArgs& a, int pass, hipStream_t st) {
    const size_t lds = list_lds(a.words, a.per_row ? G::NROW : 0, a.used_words);
    if (pass == 0) hipLaunchKernelGGL((build_lists_kernel<G, DX, 0>), dim3((unsigned)a.n_tiles), dim3(G::NT), lds, st, a);
    else if (pass == 1) hipLaunchKernelGGL((build_lists_kernel<G, DX, 1>), dim3((unsigned)a.n_tiles), dim3(G::NT), lds, st, a);
    else hipLaunchKernelGGL((build_lists_kernel<G, DX, 2>), dim3((unsigned)a.n_tiles), dim3(G::NT), lds, st, a);
}
static void launch_build_code(int code, const ListArgs& a, bool dx, int pass, hipStream_t st) {
    if (code == 333) { if (dx) launch_build<L333, true>(a, pass, st); else launch_build<L333, false>(a, pass, st); }
    else if (code == 133) { if (dx) launch_build<L133, true>(a, pass, st); else launch_build<L133, false>(a, pass, st); }
    else { if (dx) launch_build<L155, true>(a, pass, st); else launch_build<L155, false>(a, pass, st); }
}

void free_lists(WinLists& wl) {
    if (wl.d_block) (void)hipFree(wl.d_block);
    wl = WinLists{};
}

// Cells of a window without its halo: as many as the patch holds where that leaves a window for each of the 512 workgroups that the chip
// holds, fewer otherwise, an even number of them; one width for all levels of a list, by their cells together.  Training step on two APRs of 338 k particles, whose coarser level deltas had 5 to 370
// full windows, 11.5 -> 10.3 ms, group-normed fp32 U-Net on 2.7 M 5.31 -> 5.13.  (1024 windows 32 -> 32 channels on 320 k particles
// 0.176 instead of 0.165 ms, 2048 0.209; down to 14 cells the step 10.3, to 6 11.4 ms; widths of 62, 30 and 14 only 10.75.)
// One list serves layers of any width, and the line is drawn for few blocks of channels.  Kernels with many, whose workgroups fill the chip on fuller
// windows, pay for narrow ones: weight gradients without an input gradient on lists of 11 to 31 thousand cells, 64 -> 128 channels 1x5x5 on 0.04 M
// particles 365 us with full windows of one row group, 475 with these, 315 with full ones; 1 -> 16 on bfloat16 38, 44 and 38.  256 windows instead of
// 512 mend a third of these calls, the step above 10.1 instead of 10.3, but 16 and 32 outputs lose (U-Net on 2.7 M 5.10 and 5.22, 32 -> 32 on 0.16 M 0.095 and 0.101).
constexpr int WINDOWS_MIN = 512, CELLS_MIN = 22;
static int window_cells(int64_t n_cells, int HY) {
    const int widest = 64 - 2 * HY;
    return (int)std::max<int64_t>(CELLS_MIN, std::min<int64_t>(widest, n_cells / WINDOWS_MIN & ~(int64_t)1));
}

// Lists of the forward convolution at `level_delta` for stencil `code` (333, 133, 155); `tl` must be the tile list
// of the same stencil.  Built on first use (synchronises the stream and allocates), then served from the plan.
// dx: 1 = the lists of the input gradient instead, `tl` is then the tile list with a halo of one row; 2 = those without the
// particles that stick out of a far face (faces.hip sums these).
int get_lists(aprnet_plan* p, int level_delta, int code, const TileList& tl, WinLists* out, hipStream_t st, int dx) {
    auto key = std::make_pair(level_delta, code + 1000 * dx);
    auto it = p->lists.find(key);
    if (it != p->lists.end()) {
        *out = it->second;
        return it->second.unavailable ? fail(APRNET_ERR_UNSUPPORTED, "window lists are not available for this plan") : 0;
    }
    if (stream_is_capturing(st))
        return fail(APRNET_ERR_UNSUPPORTED, "window lists are built on the first call at a level delta (allocates and synchronises): "
                                            "run it once before capturing the stream");
    WinLists wl{};
    WinLists none{}; none.unavailable = true;
    p->lists[key] = none;             // replaced below when the build succeeds
    if (tl.n > 0) {
        const int HY = code == 155 ? 2 : 1, nrow = code == 333 ? L333::NROW : code == 133 ? L133::NROW : L155::NROW;
        const int group = dx ? (code == 333 ? dx_group<L333>() : dx_group<L133>()) : 0;
        ListArgs a{};
        a.apr = p->dapr; a.tree = p->dtree; a.tiles = tl.d_tiles; a.n_tiles = tl.n; a.Lc = p->lc(level_delta); a.tree_off = p->tree_offset(a.Lc);
        a.skip_faces = dx == 2 ? 1 : 0;
        a.words = (p->apr.y_num[a.Lc] + 63) / 64;              // (no level is longer)
        a.per_row = list_lds(a.words, nrow, 0) <= 48 * 1024;
        std::vector<void*> temps;                              // freed on every way out
        struct Free { std::vector<void*>& t; ~Free() { for (void* q : t) (void)hipFree(q); } } guard{temps};
        auto alloc = [&](void** q, size_t bytes) -> int { APRNET_HIP_CHECK(hipMalloc(q, std::max<size_t>(bytes, 16))); return 0; };
        auto temp = [&](void** q, size_t bytes) -> int { const int rc = alloc(q, bytes); if (!rc) temps.push_back(*q); return rc; };
        // kept positions of every row group -> its place on the compressed axis of its level, windows of the level
        int* d_tile = nullptr;                                 // [3][n_tiles]
        if (int rc = temp((void**)&d_tile, (size_t)tl.n * 3 * sizeof(int))) return rc;
        a.n_cells = d_tile;
        launch_build_code(code, a, dx != 0, 0, st);
        APRNET_LAUNCH_CHECK("build_lists_kernel (positions)");
        std::vector<int> cells(tl.n), place((size_t)2 * tl.n);
        APRNET_HIP_CHECK(hipStreamSynchronize(st));
        APRNET_HIP_CHECK(hipMemcpy(cells.data(), a.n_cells, (size_t)tl.n * sizeof(int), hipMemcpyDeviceToHost));
        int* first = place.data(), *slot0 = first + tl.n;
        int64_t nw = 0, nslot = 0, n_cells = 0;
        for (int t = 0; t < tl.n; ++t) n_cells += (cells[t] + HY + 1) & ~1;
        a.ty = window_cells(n_cells, HY);
        int most = 0;                                          // windows that stage a cell of one row group
        for (int l = MAX_LEVELS; l >= 0; --l) {                // tiles are sorted finest level first
            int64_t c = 0;
            for (int t = tl.level_begin[l]; t < tl.level_begin[l] + tl.level_count[l]; ++t) {
                first[t] = (int)c; slot0[t] = (int)nslot;
                c += (cells[t] + HY + 1) & ~1;                 // (even: pairs of cells stay in one window)
                const int n = (cells[t] + 2 * HY) / a.ty + 2;
                nslot += n; most = std::max(most, n);
                if (c >= INT32_MAX - 65536 || nslot >= INT32_MAX - 65536) return fail(APRNET_ERR_UNSUPPORTED, "window lists: more than 2^31 positions");
            }
            a.win0[l] = (int)nw; a.nwin[l] = (int)((c + a.ty - 1) / a.ty);
            nw += a.nwin[l];
        }
        a.used_words = (3 * most + 1) / 2;                     // (at most 65,536 positions in windows of 60: 13 KB; narrower ones of fewer cells)
        if (nw >= (int64_t)INT32_MAX) return fail(APRNET_ERR_UNSUPPORTED, "window lists: more than 2^31 windows");
        APRNET_HIP_CHECK(hipMemcpy(d_tile + tl.n, place.data(), place.size() * sizeof(int), hipMemcpyHostToDevice));
        a.first_cell = d_tile + tl.n; a.slot0 = d_tile + 2 * tl.n;
        // items and columns per window -> offsets; windows without an output (or, input gradient, without a column) are not stored
        std::vector<int4> cnt((size_t)nw, make_int4(0, 0, 0, 0)), off((size_t)nw), win;
        if (int rc = temp((void**)&a.count, (size_t)(2 * nw + nslot) * sizeof(int4))) return rc;
        int4* d_off = a.count + nw;
        a.share = d_off + nw;
        APRNET_HIP_CHECK(hipMemcpy(a.count, cnt.data(), (size_t)nw * sizeof(int4), hipMemcpyHostToDevice));
        launch_build_code(code, a, dx != 0, 1, st);
        APRNET_LAUNCH_CHECK("build_lists_kernel (count)");
        APRNET_HIP_CHECK(hipStreamSynchronize(st));
        APRNET_HIP_CHECK(hipMemcpy(cnt.data(), a.count, (size_t)nw * sizeof(int4), hipMemcpyDeviceToHost));
        int64_t ni = 0, nc = 0;
        for (int l = MAX_LEVELS; l >= 0; --l) {
            const int w_first = (int)win.size();
            const int64_t c_first = nc;
            for (int w = a.win0[l]; w < a.win0[l] + a.nwin[l]; ++w) {
                const int cols = group * cnt[w].y + cnt[w].z;
                off[w] = make_int4(0, 0, 0, 0);
                if (cols == 0 || cnt[w].x == 0) continue;
                off[w] = make_int4((int)(uint32_t)ni, (int)(uint32_t)nc, cnt[w].y, 1);
                win.push_back(make_int4((int)(uint32_t)ni, cnt[w].x, (int)(uint32_t)nc, cols));
                ni += cnt[w].x; nc += cols;
            }
            if ((int)win.size() == w_first) continue;
            wl.lv_first[wl.n_lv] = w_first; wl.lv_level[wl.n_lv] = l; wl.lv_cols[wl.n_lv] = nc - c_first;
            ++wl.n_lv;
        }
        if (ni >= (int64_t)UINT32_MAX || nc >= (int64_t)UINT32_MAX) return fail(APRNET_ERR_UNSUPPORTED, "window lists: more than 2^32 entries");
        wl.n_win = (int)win.size(); wl.n_items = ni; wl.n_cols = nc;
        std::vector<int> level;
        level.reserve(win.size());
        for (int k = 0; k < wl.n_lv; ++k) level.resize((size_t)(k + 1 < wl.n_lv ? wl.lv_first[k + 1] : wl.n_win), wl.lv_level[k]);
        // one allocation for all of it
        size_t at = 0;
        auto part = [&](size_t bytes) { const size_t o = at; at = (at + bytes + 255) / 256 * 256; return o; };
        const size_t o_win = part(win.size() * sizeof(int4)), o_level = part(level.size() * sizeof(int)), o_ii = part((size_t)ni * sizeof(int)),
                     o_ci = part((size_t)nc * sizeof(int)), o_ip = part((size_t)ni * sizeof(unsigned short)), o_cp = part((size_t)nc * sizeof(unsigned short));
        if (int rc = alloc(&wl.d_block, at)) return rc;
        char* base = (char*)wl.d_block;
        wl.d_win = (int4*)(base + o_win); wl.d_level = (int*)(base + o_level);
        wl.d_item_idx = (int*)(base + o_ii); wl.d_col_idx = (int*)(base + o_ci);
        wl.d_item_pos = (unsigned short*)(base + o_ip); wl.d_col_pos = (unsigned short*)(base + o_cp);
        std::vector<char> head(o_ii);                          // headers and levels, in one copy
        if (!win.empty()) {
            std::memcpy(head.data() + o_win, win.data(), win.size() * sizeof(int4));
            std::memcpy(head.data() + o_level, level.data(), level.size() * sizeof(int));
        }
        auto copy = [&](void* dst, const void* src, size_t bytes) -> int { if (bytes) APRNET_HIP_CHECK(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice)); return 0; };
        int rc = copy(wl.d_block, head.data(), head.size());
        if (!rc) rc = copy(d_off, off.data(), (size_t)nw * sizeof(int4));
        if (rc) { free_lists(wl); return rc; }
        a.off = d_off; a.item_idx = wl.d_item_idx; a.item_pos = wl.d_item_pos; a.col_idx = wl.d_col_idx; a.col_pos = wl.d_col_pos;
        launch_build_code(code, a, dx != 0, 2, st);
        hipError_t e = hipGetLastError();
        if (e == hipSuccess) e = hipStreamSynchronize(st);
        if (e != hipSuccess) { free_lists(wl); return fail(APRNET_ERR_HIP, std::string("build_lists_kernel (fill): ") + hipGetErrorString(e)); }
    }
    p->lists[key] = wl;
    *out = wl;
    return 0;
}

}  // namespace aprnet
