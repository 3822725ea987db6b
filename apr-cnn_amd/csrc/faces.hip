// Input gradient of the particles that stick out of the far faces of a level.
//
// A particle one level coarser than a tile fills the 2 x 2 x 2 cells it covers (helpers.hpp:381-399).  The input
// gradient kernels give such a particle ONE column that reads the box-summed output gradient (conv_mfma.hip) or add up
// the columns of its cells (conv_split.hip), which needs all eight cells to exist.  Where a level has an odd size, the particles on its far faces cover cells outside
// the image; the forward pass never read those cells (zero_boundary, helpers.hpp:481-502), so only the existing
// cells count.  There are few such particles (a 2-D set), and they are handled here, away from the main kernel,
// so that every element of the input gradient receives at most two atomic contributions there (same-level term and
// box term: the sum of two values onto zero does not depend on their order) and the gradient repeats bit for bit.
//
// Built once per plan, level delta and stencil on the host: for each such particle the output positions that read it and the
// taps through which they do (one cell, so one tap, each).  The kernel sums
//     gx[ci][p] += sum_co sum_tap w[s][co][ci][tap] * (sum of gy[co][out] over the outputs that read p through the tap)
// in an order that depends on the lists alone.
#include "common.hpp"

#include <algorithm>

namespace aprnet {

// index of the particle at (row, y) of an access, or -1
static int64_t find_in_row(const HostAccess& h, int l, int z, int x, int y) {
    const uint64_t row = h.row(l, z, x);
    const uint16_t* b = h.y.data() + h.xz_end[row - 1];
    const uint16_t* e = h.y.data() + h.xz_end[row];
    const uint16_t* it = std::lower_bound(b, e, (uint16_t)y);
    return (it != e && *it == (uint16_t)y) ? (int64_t)(it - h.y.data()) : -1;
}

int get_face_lists(aprnet_plan* p, int d, int code, FaceLists* out, hipStream_t st) {
    auto key = std::make_pair(d, code);
    auto it = p->faces.find(key);
    if (it != p->faces.end()) { *out = it->second; return 0; }
    if (stream_is_capturing(st))
        return fail(APRNET_ERR_UNSUPPORTED, "the first convolution backward at a level delta builds the plan's face lists "
                                            "(allocates and copies): run it once before capturing the stream");
    const HostAccess& apr = p->apr; const HostAccess& tree = p->tree;
    const int kz = code / 100, kx = (code / 10) % 10, ky = code % 10;
    const int hz = (kz - 1) / 2, hx = (kx - 1) / 2, hy = (ky - 1) / 2;
    const int Lc = p->lc(d);
    const int64_t tree_off = p->tree_offset(Lc);
    std::vector<int> part_idx, part_level, out_begin{0}, outs;
    std::vector<unsigned> taps;
    std::vector<std::pair<int, unsigned>> found;
    // l: level of the tile (of the outputs); the particles in question live on level l - 1
    for (int l = std::min(Lc, apr.level_max); l > apr.level_min; --l) {
        const int zn = apr.z_num[l], xn = apr.x_num[l], yn = apr.y_num[l];
        const int czn = apr.z_num[l - 1], cxn = apr.x_num[l - 1];
        const bool out_tree = (l == Lc) && (l < apr.level_max);
        const bool z_odd = (zn & 1) != 0, x_odd = (xn & 1) != 0, y_odd = (yn & 1) != 0;
        if (!z_odd && !x_odd && !y_odd) continue;
        for (int zc = 0; zc < czn; ++zc)
            for (int xc = 0; xc < cxn; ++xc) {
                const bool row_cut = (2 * zc + 1 >= zn && kz > 1) || 2 * xc + 1 >= xn;
                // 2-D stencils on flat tiles see the z slices of a coarser particle one by one: a missing slice is no cut
                if (!row_cut && !y_odd) continue;
                const uint64_t row = apr.row(l - 1, zc, xc);
                int64_t b = (int64_t)apr.xz_end[row - 1], e = (int64_t)apr.xz_end[row];
                if (b == e) continue;
                if (!row_cut) {                      // only the last particle of the row can stick out in y
                    if (2 * (int)apr.y[e - 1] + 1 < yn) continue;
                    b = e - 1;
                }
                for (int64_t i = b; i < e; ++i) {
                    const int yc = apr.y[i];
                    part_idx.push_back((int)i); part_level.push_back(l);
                    found.clear();
                    for (int dz = 0; dz < 2; ++dz)
                        for (int dx = 0; dx < 2; ++dx)
                            for (int dy = 0; dy < 2; ++dy) {
                                const int cz = 2 * zc + dz, cx = 2 * xc + dx, cy = 2 * yc + dy;
                                if (cz >= zn || cx >= xn || cy >= yn) continue;
                                for (int t = 0; t < kz * kx * ky; ++t) {
                                    const int sz = t / (kx * ky), sx = (t / ky) % kx, sy = t % ky;
                                    // the output at o reads cell o + (s - h) with tap t
                                    const int oz = cz - (sz - hz), ox = cx - (sx - hx), oy = cy - (sy - hy);
                                    if (oz < 0 || oz >= zn || ox < 0 || ox >= xn || oy < 0 || oy >= yn) continue;
                                    int64_t o = find_in_row(apr, l, oz, ox, oy);
                                    if (o < 0 && out_tree) {
                                        const int64_t tn = find_in_row(tree, l, oz, ox, oy);
                                        if (tn >= 0) o = tn + tree_off;
                                    }
                                    if (o < 0) continue;
                                    found.emplace_back((int)o, 1u << t);
                                }
                            }
                    std::sort(found.begin(), found.end());
                    for (size_t k = 0; k < found.size(); ++k)
                        if (k > 0 && found[k].first == found[k - 1].first) taps.back() |= found[k].second;
                        else { outs.push_back(found[k].first); taps.push_back(found[k].second); }
                    out_begin.push_back((int)outs.size());
                }
            }
        while (part_idx.size() % FACE_PB != 0) {         // a workgroup's particles use the same weights
            part_idx.push_back(-1); part_level.push_back(l); out_begin.push_back((int)outs.size());
        }
    }
    FaceLists fl{};
    fl.n_part = (int)part_idx.size();
    if (fl.n_part > 0) {
        auto upload = [&](void** dst, const void* src, size_t bytes) -> int {
            APRNET_HIP_CHECK(hipMalloc(dst, std::max<size_t>(bytes, 16)));
            if (bytes) APRNET_HIP_CHECK(hipMemcpy(*dst, src, bytes, hipMemcpyHostToDevice));
            return 0;
        };
        int rc = upload((void**)&fl.d_part_idx, part_idx.data(), part_idx.size() * 4);
        if (!rc) rc = upload((void**)&fl.d_part_level, part_level.data(), part_level.size() * 4);
        if (!rc) rc = upload((void**)&fl.d_out_begin, out_begin.data(), out_begin.size() * 4);
        if (!rc) rc = upload((void**)&fl.d_out, outs.data(), outs.size() * 4);
        if (!rc) rc = upload((void**)&fl.d_taps, taps.data(), taps.size() * 4);
        if (rc) { free_face_lists(fl); return rc; }
    }
    p->faces[key] = fl;
    *out = fl;
    return 0;
}

void free_face_lists(FaceLists& fl) {
    for (void* q : {(void*)fl.d_part_idx, (void*)fl.d_part_level, (void*)fl.d_out_begin, (void*)fl.d_out, (void*)fl.d_taps})
        if (q) (void)hipFree(q);
    fl = FaceLists{};
}

// Four particles per workgroup, 64 input channels (one per lane), chunks of 64 output channels.  One wave per particle adds up
// the output gradient by tap in LDS (lanes = output channels; one read per output, not per output and tap); then each wave takes a
// quarter of the chunk's output channels: the taps of 64 input channels lie next to each other in memory, so they are
// read in one stream into the wave's own piece of LDS and from there lane by lane (stride K, odd: no bank twice), and every weight
// serves four particles.  The quarters are added up in the order of the waves.
//
// One workgroup per particle and one thread per input channel, every product a read of its own from the weights (stride K), was a chain
// of outputs x taps x Cout loads: backward pass of 128 -> 128 channels on 2 k particles of an uneven volume 274 (1568) us, 64 -> 64 on
// 14 k 223 (622), on 70 k 539 (945), 16 -> 16 on 320 k 318 (386) us.
constexpr int FACE_CO = 64;
template <int K>
__global__ void __launch_bounds__(64 * FACE_PB)
face_dx_kernel(const FaceLists fl, const float* __restrict__ gy, int64_t ldy, const float* __restrict__ w, int S_exp, int Cout, int Cin,
               int Lc, float* __restrict__ gx, int64_t ldgx) {
    static_assert(FACE_PB == 4, "the sums of a tap and an output channel are one float4");
    __shared__ float4 sum[K * FACE_CO];                       // [tap][output channel], one component per particle
    __shared__ float stage[FACE_PB][64 * K];
    __shared__ unsigned used[FACE_PB];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int p0 = blockIdx.x * FACE_PB, ci0 = blockIdx.y * 64;
    const int ob = fl.d_out_begin[p0 + wave], oe = fl.d_out_begin[p0 + wave + 1];
    const int s = min(S_exp - 1, Lc - fl.d_part_level[p0]);
    const int nci = min(64, Cin - ci0);
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int c0 = 0; c0 < Cout; c0 += FACE_CO) {
        const int nco = min(FACE_CO, Cout - c0);
        for (int i = threadIdx.x; i < K * FACE_CO; i += 64 * FACE_PB) sum[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        __syncthreads();
        float* mine = reinterpret_cast<float*>(sum) + 4 * lane + wave;
        const float* col = gy + (int64_t)(c0 + min(lane, nco - 1)) * ldy;
        unsigned any = 0u;
        for (int k0 = ob; k0 < oe; k0 += 8) {
            float v[8];
            unsigned m[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int e = min(k0 + k, oe - 1);            // uniform
                v[k] = col[fl.d_out[e]];
                m[k] = k0 + k < oe ? fl.d_taps[e] : 0u;
            }
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                any |= m[k];
                for (unsigned b = m[k]; b != 0u; b &= b - 1u) mine[4 * FACE_CO * (__ffs(b) - 1)] += v[k];
            }
        }
        if (lane == 0) used[wave] = any;
        __syncthreads();
        for (int c = wave; c < nco; c += FACE_PB) {
            const float* wp = w + (((int64_t)s * Cout + c0 + c) * Cin + ci0) * K;
            float* st = stage[wave];
            float r[K];
#pragma unroll
            for (int t = 0; t < K; ++t) r[t] = t * 64 + lane < nci * K ? wp[t * 64 + lane] : 0.f;
#pragma unroll
            for (int t = 0; t < K; ++t) st[t * 64 + lane] = r[t];
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            float z = 0.f;                                    // stays 0 if the weights are finite
#pragma unroll
            for (int t = 0; t < K; ++t) { r[t] = st[lane * K + t]; z = fmaf(r[t], 0.f, z); }
            if (__ballot(z != 0.f) == 0) {
#pragma unroll
                for (int t = 0; t < K; ++t) {
                    const float4 g = sum[t * FACE_CO + c];
                    acc.x = fmaf(r[t], g.x, acc.x); acc.y = fmaf(r[t], g.y, acc.y); acc.z = fmaf(r[t], g.z, acc.z); acc.w = fmaf(r[t], g.w, acc.w);
                }
            } else {                                          // no product where a particle has no output for the tap
#pragma unroll
                for (int t = 0; t < K; ++t) {
                    const float4 g = sum[t * FACE_CO + c];
                    if ((used[0] >> t) & 1u) acc.x = fmaf(r[t], g.x, acc.x);
                    if ((used[1] >> t) & 1u) acc.y = fmaf(r[t], g.y, acc.y);
                    if ((used[2] >> t) & 1u) acc.z = fmaf(r[t], g.z, acc.z);
                    if ((used[3] >> t) & 1u) acc.w = fmaf(r[t], g.w, acc.w);
                }
            }
            __builtin_amdgcn_wave_barrier();                  // the next channel's weights come after these reads
        }
        __syncthreads();
    }
    sum[wave * 64 + lane] = acc;
    __syncthreads();
    const int o = fl.d_part_idx[p0 + wave];
    if (o < 0 || lane >= nci) return;
    const float* part = reinterpret_cast<const float*>(sum) + 4 * lane + wave;
    gx[(int64_t)(ci0 + lane) * ldgx + o] += ((part[0] + part[256]) + part[512]) + part[768];
}

// Adds the face terms to gx.  Runs after the main input-gradient kernel on the same stream.
int launch_face_dx(const FaceLists& fl, const float* gy, int64_t ldy, const float* w, int S_exp, int Cout, int Cin, int K, int Lc,
                   float* gx, int64_t ldgx, hipStream_t st) {
    if (fl.n_part == 0) return 0;
    dim3 grid((unsigned)(fl.n_part / FACE_PB), (unsigned)((Cin + 63) / 64));
#define APRNET_FACE(K) hipLaunchKernelGGL(face_dx_kernel<K>, grid, dim3(64 * FACE_PB), 0, st, fl, gy, ldy, w, S_exp, Cout, Cin, Lc, gx, ldgx)
    if (K == 27) APRNET_FACE(27); else if (K == 9) APRNET_FACE(9); else APRNET_FACE(25);
#undef APRNET_FACE
    APRNET_LAUNCH_CHECK("face_dx_kernel");
    return 0;
}

}  // namespace aprnet
