// fs_rows.hip -- multigrid smoothers with the tile in registers (gfx950).
//
// A workgroup's tile is 2 G columns wide and NG M rows high: NG = 64 NW / G groups of G lanes, group i holding rows
// i M .. i M + M - 1, a lane the columns 2 l and 2 l + 1 of each, with solution, conductances, rhs and 1/diagonal in
// registers for all sweeps.  A cell's vertical neighbours are the same lane's other rows, its horizontal ones the
// other column or the next lane (a DPP wavefront shift inside the multiply), so a sweep touches LDS only for the
// top and bottom row of each group: two reads and two writes per lane and half-sweep instead of five LDS accesses
// and an index per cell.  With two columns per lane a red-black half-sweep updates exactly one of them in every row
// (which one is known at compile time): no lane idles, and an update is nine VALU instructions.
// Every cell of the tile is updated in every sweep.  What lies outside the tile is taken as zero or stale, an
// error that moves one cell inwards per half-sweep (red-black) or sweep (Jacobi): after the sweeps the cells at
// least `halo` from the edge hold what global sweeps give, so only they are written.  Every tile evaluates the same
// expressions in the same order: the same values bit for bit.
// Cells outside the grid read the zero halo of the padded fields, so their weights and 1/diagonal are zero and
// they stay zero.
//
// What bounds it: VALU issue and latency on tiles that fit the chip once, HBM beyond.  Measured against the same
// smoothers on LDS tiles (per launch): red-black V(4) post-smoothing 2048^2 65.3 -> 25.7 us, 1920x1080 34.2 -> 15.5,
// 1024^2 18.1 -> 9.5, 256^2 5.9 -> 5.1; pre-smoothing + residual + restriction 2048^2 54.5 -> 27.9, 1920x1080
// 29.7 -> 15.9, 257x129 9.3 -> 5.8; Chebyshev with 8 sweeps post 2048^2 65.7 -> 37.2 (on a tile chosen for it; 42 to 48
// on those the tuner may keep from 3 sweeps), pre + restriction 71.1 -> 43.1, 257x129 9.7 -> 7.4 (about 2.3 us of
// each is the launch).
#include "fs_kernels.hpp"
#include "fs_mg_device.hpp"

#include <type_traits>

namespace fsim {

namespace {

enum RowsMode : int { kRowsPre = 0, kRowsPost = 1, kRowsPreRestrict = 2 };

// Cells between a tile's edge and what it writes: the smoothing halo and, where the residual is restricted, three more
// (taps reach two cells past the coarse tile's fine image, the operator one), rounded to even so that the tile keeps
// its colour parity.
__host__ __device__ constexpr int rows_halo(int jacobi, int nu) { return jacobi ? (nu + 1) & ~1 : 2 * nu; }
__host__ __device__ constexpr int rows_edge(int mode, int jacobi, int nu)
{
    return rows_halo(jacobi, nu) + (mode == kRowsPreRestrict ? 4 : 0);
}

template <int JACOBI, int MODE, int G, int NW, int M, class C, class V, class VC>
__device__ __forceinline__ void rows_tile(const LevelViewT<C, V>& L, int cur, const V* rhs, const double* shift,
    const SmoothWeights& wt, int nu, const CoarseLinkT<VC>& link, const LevelViewT<C, VC>& Cl, const AxisRestrict& rx,
    const AxisRestrict& ry, const int* status, int bx, int by)
{
    constexpr int NG = NW * 64 / G;   // lane groups, one above the other
    constexpr int LX = 2 * G, LY = NG * M;
    constexpr int RES = MODE == kRowsPreRestrict ? LY * LX : 1;
    constexpr int TAB = MODE == kRowsPreRestrict ? 256 : 1;
    static_assert(M % 2 == 0, "a group's first row keeps the tile's colour parity");
    // red-black: [colour][top, bottom][group][lane]; Jacobi: [buffer][top, bottom][group][column]
    constexpr int EX = JACOBI ? 2 * G : G;
    __shared__ float s_edge[2][2][NG][EX];
    __shared__ float s_res[RES];
    __shared__ int s_rxi[TAB], s_ryi[TAB];
    __shared__ float s_rxw[TAB], s_ryw[TAB];
    const int w = L.w, h = L.h, s = L.s;
    const int edge = rows_edge(MODE, JACOBI, nu);
    const int TX = LX - 2 * edge, TY = LY - 2 * edge;
    const int lane = threadIdx.x & (G - 1);
    const int group = G == 64 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : (int)threadIdx.x / G;
    const int x0 = bx * TX - edge, y0 = by * TY - edge;
    const int R0 = y0 + group * M;
    const int xa = x0 + 2 * lane;
    // Element index of a row's column pair.  Columns past the halo read the pair next to the grid: (-2, -1) is the
    // previous row's right halo and this row's left one, (w, w + 1) this row's right one and the next row's left
    // one, zeros all four; rows outside the grid read the first pair of the upper halo row.
    const int e = min(max(xa, -2), w) + 1;
    // (a whole wavefront per row keeps the row's part scalar and 64 bits wide; the others add it per lane in 32 bits,
    // which reaches every level of a grid of 2^28 cells, the most that fs_grid_create takes: padded, thin ones have the
    // most elements, 3 * 2^28)
    struct Index {
        size_t row;
        unsigned at;
    };
    auto index_of = [&](int r) {
        const int y = R0 + r;
        const bool in = y >= 0 && y < h;
        if constexpr (G == 64)
            return Index{in ? (size_t)(y + 1) * s - 1 : 0, in ? (unsigned)(e + 1) : 0u};
        return Index{0, in ? (unsigned)((y + 1) * s + e) : 0u};
    };
    auto two = [](auto* p, Index i, float (&v)[2]) {
        using T = std::remove_cv_t<std::remove_pointer_t<decltype(p)>>;
        const Pair<T> t = *(const Pair<T>*)((const char*)(p + i.row) + (size_t)(i.at * (unsigned)sizeof(T)));
        v[0] = ldv(t.a);
        v[1] = ldv(t.b);
    };
    float x[M][2], wr[M][2], wd[M][2], cb[M][2], wu[2];
    two(L.down, index_of(-1), wu);
#pragma unroll
    for (int r = 0; r < M; ++r) {
        const Index i = index_of(r);
        two(L.right, i, wr[r]);
        two(L.down, i, wd[r]);
        two(rhs, i, cb[r]);
        if (MODE == kRowsPost)
            two((const V*)L.sol[cur], i, x[r]);
        else
            x[r][0] = x[r][1] = 0.f;
    }
    if constexpr (MODE == kRowsPost) {
        // Bilinear prolongation of the coarse correction.  A coarse row is interpolated along x once for the
        // fine rows that use it: fine row f takes coarse rows f / 2 - 1 .. f / 2 + 1 only.
        constexpr int NH = M / 2 + 2;
        const int ch = (h + 1) >> 1;
        const int i0 = min(max(xa, 0), w - 1), i1 = min(max(xa + 1, 0), w - 1);
        const float wx[2] = {link.pxw[i0], link.pxw[i1]};
        const int a0[2] = {link.pxf[i0], link.pxf[i1]}, a1[2] = {link.pxs[i0], link.pxs[i1]};
        const int cr0 = (R0 >> 1) - 1;
        float wy[M];
        int first[M], second[M];
        if constexpr (G == 64) {   // one row table per wavefront: lane r holds row r's entries
            const int fc = min(max(R0 + (lane & (M - 1)), 0), h - 1);
            const float lw = link.pyw[fc];
            const int lf = link.pyf[fc] - cr0, ls = link.pys[fc] - cr0;
#pragma unroll
            for (int r = 0; r < M; ++r) {
                wy[r] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(lw), r));
                first[r] = __builtin_amdgcn_readlane(lf, r);
                second[r] = __builtin_amdgcn_readlane(ls, r);
            }
        } else {
#pragma unroll
            for (int r = 0; r < M; ++r) {
                const int fc = min(max(R0 + r, 0), h - 1);
                wy[r] = link.pyw[fc];
                first[r] = link.pyf[fc] - cr0;
                second[r] = link.pys[fc] - cr0;
            }
        }
        float hv[NH][2];
#pragma unroll
        for (int i = 0; i < NH; ++i) {
            const int row = (min(max(cr0 + i, -1), ch) + 1) * link.cs + 1;
            const VC* base = link.csol + (G == 64 ? row : 0);
            auto at = [&](int c) {
                return ldv(*(const VC*)((const char*)base + (size_t)((unsigned)(G == 64 ? c : row + c) * (unsigned)sizeof(VC))));
            };
#pragma unroll
            for (int j = 0; j < 2; ++j)
                hv[i][j] = (1.f - wx[j]) * at(a0[j]) + wx[j] * at(a1[j]);
        }
#pragma unroll
        for (int r = 0; r < M; ++r) {
            const int f = R0 + r;
            const bool in = f >= 0 && f < h;
            const bool fa = first[r] <= r / 2, sa = second[r] <= r / 2, sb = second[r] == r / 2 + 1;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const float a = fa ? hv[r / 2][j] : hv[r / 2 + 1][j];
                const float b = sa ? hv[r / 2][j] : sb ? hv[r / 2 + 1][j] : hv[r / 2 + 2][j];
                const float v = x[r][j] + ((1.f - wy[r]) * a + wy[r] * b);
                x[r][j] = in && xa + j >= 0 && xa + j < w ? v : 0.f;
            }
        }
    }
    const int CTX = TX >> 1, CTY = TY >> 1;   // coarse tile (kRowsPreRestrict)
    const int cx0 = bx * CTX, cy0 = by * CTY;
    if constexpr (MODE == kRowsPreRestrict) {
        // restriction tables of the coarse tile, relative to the fine tile; a missing tap has weight 0
        const int t = threadIdx.x;
        if (t < CTX + CTY) {
            const bool isx = t < CTX;
            const int e = isx ? t : t - CTX;
            const int c = (isx ? cx0 : cy0) + e, limit = isx ? Cl.w : Cl.h;
            const AxisRestrict& R = isx ? rx : ry;
            const int cc = min(c, limit - 1);
            const int n = c < limit ? R.count[cc] : 0;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const bool on = k < n;
                const int i = R.index[cc * 4 + k];
                const float v = R.weight[cc * 4 + k];
                (isx ? s_rxi : s_ryi)[e * 4 + k] = on ? i - (isx ? x0 : y0) : edge;
                (isx ? s_rxw : s_ryw)[e * 4 + k] = on ? v : 0.f;
            }
        }
    }
    if (status && *status != kRunning)
        return;
    float wl[M], inv[M][2];
    const double sh = shift ? *shift : 0.0;
#pragma unroll
    for (int r = 0; r < M; ++r) {
        wl[r] = from_left(wr[r][1]);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const float l = j ? wr[r][0] : wl[r], u = r ? wd[r - 1][j] : wu[j];
            inv[r][j] = inv_or_zero((l + wr[r][j]) + (u + wd[r][j]));
            if (shift)
                cb[r][j] = (float)((double)cb[r][j] - sh);
        }
    }
    const int above = max(group - 1, 0), below = min(group + 1, NG - 1);   // the tile's own edge: stale, never used
    float up[2] = {0.f, 0.f}, dn[2] = {0.f, 0.f};
    if constexpr (JACOBI) {
        auto publish = [&](int buf) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                s_edge[buf][0][group][2 * lane + j] = x[0][j];
                s_edge[buf][1][group][2 * lane + j] = x[M - 1][j];
            }
        };
        auto fetch = [&](int buf) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                up[j] = s_edge[buf][1][above][2 * lane + j];
                dn[j] = s_edge[buf][0][below][2 * lane + j];
            }
        };
        // a cell without conductance is zero from the start and stays zero
#pragma unroll
        for (int r = 0; r < M; ++r)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                x[r][j] = inv[r][j] > 0.f ? x[r][j] : 0.f;
                if (MODE != kRowsPost) {
                    const float v = wt.w[0] * cb[r][j] * inv[r][j];
                    x[r][j] = inv[r][j] > 0.f ? v : 0.f;
                }
            }
        constexpr int first = MODE == kRowsPost ? 0 : 1;
        publish(first);
        __syncthreads();
#pragma unroll 1
        for (int k = first; k < nu; ++k) {
            float wk = wt.w[0];   // uniform select: no dynamic indexing of the argument block
#pragma unroll
            for (int i = 1; i < kJacobiMaxSweeps; ++i)
                wk = k == i ? wt.w[i] : wk;
            fetch(k & 1);
#pragma unroll
            for (int r = 0; r < M; ++r) {
                const float c0 = x[r][0], c1 = x[r][1];
                const float n[2][2] = {{from_left(c1), c1}, {c0, from_right(c0)}};
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const float c = j ? c1 : c0;
                    const float l = j ? wr[r][0] : wl[r], u = r ? wd[r - 1][j] : wu[j];
                    const float nd = r + 1 < M ? x[r + 1][j] : dn[j];
                    const float product = (l * (c - n[j][0]) + wr[r][j] * (c - n[j][1])) +
                                          (u * (c - up[j]) + wd[r][j] * (c - nd));
                    x[r][j] = c + wk * (cb[r][j] - product) * inv[r][j];
                    up[j] = c;
                }
            }
            publish((k & 1) ^ 1);
            __syncthreads();
        }
        if (MODE == kRowsPreRestrict)
            fetch(nu & 1);
    } else {
        auto publish = [&](auto color) {
            constexpr int c = decltype(color)::value;
            s_edge[c][0][group][lane] = x[0][c];
            s_edge[c][1][group][lane] = x[M - 1][c ^ 1];
        };
        // One half-sweep of colour c: in row r the cell of column (c + r) & 1.
        auto half = [&](auto color, bool neighbours) {
            constexpr int c = decltype(color)::value;
            const float hu = s_edge[c ^ 1][1][above][lane], hd = s_edge[c ^ 1][0][below][lane];
#pragma unroll
            for (int r = 0; r < M; ++r) {
                const int j = (c + r) & 1;
                float v = cb[r][j];
                if (neighbours) {
                    const float n0 = j ? x[r][0] : from_left(x[r][1]);
                    const float n1 = j ? from_right(x[r][0]) : x[r][1];
                    const float n2 = r ? x[r - 1][j] : hu;
                    const float n3 = r + 1 < M ? x[r + 1][j] : hd;
                    const float a = j ? wr[r][0] : wl[r], u = r ? wd[r - 1][j] : wu[j];
                    v += (a * n0 + wr[r][j] * n1) + (u * n2 + wd[r][j] * n3);
                }
                x[r][j] = v * inv[r][j];
            }
            publish(color);
            __syncthreads();
        };
        constexpr std::integral_constant<int, 0> red{};
        constexpr std::integral_constant<int, 1> black{};
        if constexpr (MODE == kRowsPost) {   // reversed order
            publish(red);
            __syncthreads();
#pragma unroll 1
            for (int k = 0; k < nu; ++k) {
                half(black, true);
                half(red, true);
            }
        } else {
            half(red, false);
            half(black, true);
#pragma unroll 1
            for (int k = 1; k < nu; ++k) {
                half(red, true);
                half(black, true);
            }
        }
        if (MODE == kRowsPreRestrict) {
            // row 0's columns meet the row above in its colours' order: column j of an odd row has colour j ^ 1
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                up[j] = s_edge[j ^ 1][1][above][lane];
                dn[j] = s_edge[j][0][below][lane];
            }
        }
    }
    V* sol_out = L.sol[cur ^ 1];
    const bool lane_in = 2 * lane >= edge && 2 * lane < LX - edge;
#pragma unroll
    for (int r = 0; r < M; ++r) {
        const int ty = group * M + r, y = R0 + r;
        if (ty >= edge && ty < LY - edge && y < h && lane_in) {
            V* row = sol_out + (G == 64 ? (size_t)(y + 1) * s : 0);
            const unsigned at = (unsigned)(G == 64 ? xa + 1 : (y + 1) * s + xa + 1);
            char* q = (char*)row + (size_t)(at * (unsigned)sizeof(V));
            if (xa + 1 < w)
                *(Pair<V>*)q = Pair<V>{stv<V>(x[r][0]), stv<V>(x[r][1])};
            else if (xa < w)
                *(V*)q = stv<V>(x[r][0]);
        }
    }
    if constexpr (MODE == kRowsPreRestrict) {
        // of the solution as it is stored
        if constexpr (!std::is_same<V, float>::value) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
#pragma unroll
                for (int r = 0; r < M; ++r)
                    x[r][j] = ldv(stv<V>(x[r][j]));
                up[j] = ldv(stv<V>(up[j]));
                dn[j] = ldv(stv<V>(dn[j]));
            }
        }
        // residual of the whole tile (right where the restriction reads it), zero at cells without conductance
#pragma unroll
        for (int r = 0; r < M; ++r) {
            float res[2];
            const float n[2][2] = {{from_left(x[r][1]), x[r][1]}, {x[r][0], from_right(x[r][0])}};
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const float c = x[r][j];
                const float l = j ? wr[r][0] : wl[r], u = r ? wd[r - 1][j] : wu[j];
                const float nu_ = r ? x[r - 1][j] : up[j], nd = r + 1 < M ? x[r + 1][j] : dn[j];
                const float product = (l * (c - n[j][0]) + wr[r][j] * (c - n[j][1])) +
                                      (u * (c - nu_) + wd[r][j] * (c - nd));
                const bool active = (l + wr[r][j]) + (u + wd[r][j]) > 0.f;
                res[j] = active ? cb[r][j] - product : 0.f;
            }
            s_res[(group * M + r) * LX + 2 * lane] = res[0];
            s_res[(group * M + r) * LX + 2 * lane + 1] = res[1];
        }
        __syncthreads();
        const float inv_ctx = 1.0f / (float)CTX;
        for (int e = threadIdx.x; e < CTX * CTY; e += 64 * NW) {
            const int ly = (int)(((float)e + 0.5f) * inv_ctx), lx = e - ly * CTX;   // exact: e < 2^12
            const int X = cx0 + lx, Y = cy0 + ly;
            if (X >= Cl.w || Y >= Cl.h)
                continue;
            float tap[4][4];
#pragma unroll
            for (int iy = 0; iy < 4; ++iy) {
                const float* row = s_res + s_ryi[ly * 4 + iy] * LX;
#pragma unroll
                for (int ix = 0; ix < 4; ++ix)
                    tap[iy][ix] = row[s_rxi[lx * 4 + ix]];
            }
            float value = 0.f;
#pragma unroll
            for (int iy = 0; iy < 4; ++iy) {
                float horizontal = 0.f;
#pragma unroll
                for (int ix = 0; ix < 4; ++ix)
                    horizontal += s_rxw[lx * 4 + ix] * tap[iy][ix];
                value += s_ryw[ly * 4 + iy] * horizontal;
            }
            Cl.rhs[(Y + 1) * Cl.s + X + 1] = stv<VC>(value);
        }
    }
}

template <int JACOBI, int MODE, int G, int NW, int M, class C, class V, class VC>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(4)))
void k_rows(LevelViewT<C, V> L, int cur, const V* rhs, const double* shift, SmoothWeights wt, int nu,
    CoarseLinkT<VC> link, LevelViewT<C, VC> Cl, AxisRestrict rx, AxisRestrict ry, const int* status)
{
    constexpr int LX = 2 * G, LY = NW * 64 / G * M;
    const int edge = rows_edge(MODE, JACOBI, nu);
    const int TX = LX - 2 * edge, TY = LY - 2 * edge;
    int bx, by;
    xcd_tile((L.w + TX - 1) / TX, (L.h + TY - 1) / TY, bx, by);
    rows_tile<JACOBI, MODE, G, NW, M, C, V, VC>(L, cur, rhs, shift, wt, nu, link, Cl, rx, ry, status, bx, by);
}

// A tiled level of many grids in one launch: red-black on FP32 levels, 64 x 64 tiles on 512 threads.
constexpr int kBatchG = 32, kBatchNW = 8, kBatchM = 4;
template <int MODE>
__global__ __launch_bounds__(64 * kBatchNW) __attribute__((amdgpu_waves_per_eu(4)))
void k_rows_batch(const BatchItem* __restrict__ items, const int* __restrict__ item, const int* __restrict__ first, int level)
{
    const int i = item[blockIdx.x];
    const int local = (int)blockIdx.x - first[i];
    const BatchLevel B = items[i].lev[level];
    const PcgScalars* S = items[i].g.S;
    const int TX = 2 * kBatchG - 2 * rows_edge(MODE, 0, B.sweeps);
    const int columns = (B.L.w + TX - 1) / TX;
    const int row = local / columns;
    rows_tile<0, MODE, kBatchG, kBatchNW, kBatchM, float, float, float>(B.L, MODE == kRowsPost ? 1 : 0, B.L.rhs,
        level == 0 ? &S->r_mean : nullptr, SmoothWeights{}, B.sweeps, B.link, B.C, B.rx, B.ry, &S->status,
        local - row * columns, row);
}

template <int JACOBI, int MODE, class C, class V, class VC>
void launch_rows_mode(hipStream_t st, const LevelViewT<C, V>& L, int cur, const V* rhs, const double* shift,
    const SmoothWeights& wt, int nu, const CoarseLinkT<VC>& link, const LevelViewT<C, VC>& Cl, AxisRestrict rx,
    AxisRestrict ry, const int* status, int tile)
{
    const int edge = rows_edge(MODE, JACOBI, nu);
    const auto tiles = [&](int LX, int LY) {
        const int TX = LX - 2 * edge, TY = LY - 2 * edge;
        return ((L.w + TX - 1) / TX) * ((L.h + TY - 1) / TY);
    };
#define FS_ROWS(G, NW, M)                                                                                        \
    hipLaunchKernelGGL((k_rows<JACOBI, MODE, G, NW, M, C, V, VC>), dim3(tiles(2 * G, NW * 64 / G * M)), dim3(64 * NW), 0, \
        st, L, cur, rhs, shift, wt, nu, link, Cl, rx, ry, status)
    if constexpr (MODE == kRowsPreRestrict) {
        switch (tile) {
        case 0: FS_ROWS(64, 16, 8); break;
        case 1: FS_ROWS(64, 16, 4); break;
        case 2: FS_ROWS(32, 8, 4); break;
        case 3: FS_ROWS(32, 16, 2); break;
        case 4: FS_ROWS(16, 8, 2); break;
        default: FS_ROWS(16, 4, 2); break;
        }
    } else {
        switch (tile) {
        case 0: FS_ROWS(64, 8, 8); break;
        case 1: FS_ROWS(64, 16, 4); break;
        case 2: FS_ROWS(32, 8, 4); break;
        case 3: FS_ROWS(32, 16, 2); break;
        case 4: FS_ROWS(32, 4, 4); break;
        case 5: FS_ROWS(32, 8, 2); break;
        case 6: FS_ROWS(16, 4, 2); break;
        case 7: FS_ROWS(16, 4, 4); break;
        case 8: FS_ROWS(64, 8, 4); break;
        case 9: FS_ROWS(64, 16, 8); break;
        default: FS_ROWS(16, 8, 2); break;
        }
    }
#undef FS_ROWS
}

}  // namespace

int batch_level_blocks(const BatchLevel& level, bool post)
{
    const int edge = rows_edge(post ? kRowsPost : kRowsPreRestrict, 0, level.sweeps);
    const int TX = 2 * kBatchG - 2 * edge, TY = kBatchNW * 64 / kBatchG * kBatchM - 2 * edge;
    return ((level.L.w + TX - 1) / TX) * ((level.L.h + TY - 1) / TY);
}

void launch_batch_smooth(hipStream_t st, const BatchItem* items, const BatchPart& part, int level, bool post)
{
    if (part.blocks <= 0)
        return;
    if (post)
        hipLaunchKernelGGL(k_rows_batch<kRowsPost>, dim3(part.blocks), dim3(64 * kBatchNW), 0, st, items, part.item,
            part.first, level);
    else
        hipLaunchKernelGGL(k_rows_batch<kRowsPreRestrict>, dim3(part.blocks), dim3(64 * kBatchNW), 0, st, items, part.item,
            part.first, level);
}

template <class C, class V, class VC>
void launch_smooth(hipStream_t st, int jacobi, const LevelViewT<C, V>& L, int cur, const V* rhs,
    const double* shift, int pre, const SmoothWeights& wt, int nu, const CoarseLinkT<VC>& link, const int* status,
    int tile)
{
    const LevelViewT<C, VC> none{};
    const AxisRestrict r{};
    if constexpr (std::is_same<C, float>::value) {
        if (jacobi) {
            if (pre)
                launch_rows_mode<1, kRowsPre>(st, L, cur, rhs, shift, wt, nu, link, none, r, r, status, tile);
            else
                launch_rows_mode<1, kRowsPost>(st, L, cur, rhs, shift, wt, nu, link, none, r, r, status, tile);
            return;
        }
    }
    if (pre)
        launch_rows_mode<0, kRowsPre>(st, L, cur, rhs, shift, wt, nu, link, none, r, r, status, tile);
    else
        launch_rows_mode<0, kRowsPost>(st, L, cur, rhs, shift, wt, nu, link, none, r, r, status, tile);
}

template <class C, class V, class VC>
void launch_smooth_restrict(hipStream_t st, int jacobi, const LevelViewT<C, V>& L, int cur, const V* rhs,
    const double* shift, const SmoothWeights& wt, int nu, const LevelViewT<C, VC>& Cl, AxisRestrict rx, AxisRestrict ry,
    const int* status, int tile)
{
    const CoarseLinkT<VC> none{};
    if constexpr (std::is_same<C, float>::value) {
        if (jacobi) {
            launch_rows_mode<1, kRowsPreRestrict>(st, L, cur, rhs, shift, wt, nu, none, Cl, rx, ry, status, tile);
            return;
        }
    }
    launch_rows_mode<0, kRowsPreRestrict>(st, L, cur, rhs, shift, wt, nu, none, Cl, rx, ry, status, tile);
}

#define FS_ROWS_TYPES(C, V, VC)                                                                                   \
    template void launch_smooth<C, V, VC>(hipStream_t, int, const LevelViewT<C, V>&, int, const V*, const double*, \
        int, const SmoothWeights&, int, const CoarseLinkT<VC>&, const int*, int);                                 \
    template void launch_smooth_restrict<C, V, VC>(hipStream_t, int, const LevelViewT<C, V>&, int, const V*,        \
        const double*, const SmoothWeights&, int, const LevelViewT<C, VC>&, AxisRestrict, AxisRestrict, const int*, int);
FS_ROWS_TYPES(float, float, float)
FS_ROWS_TYPES(half16, float, float)
FS_ROWS_TYPES(bf16, float, float)
FS_ROWS_TYPES(bf16, float, bf16)
FS_ROWS_TYPES(bf16, bf16, bf16)
#undef FS_ROWS_TYPES

}  // namespace fsim
