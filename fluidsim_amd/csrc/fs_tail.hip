// fs_tail.hip -- the coarse end of a V-cycle in one workgroup, its levels in registers (gfx950).
//
// The levels of at most 4096 cells run one after another on one compute unit, so their time is a chain of barriers,
// LDS round trips and issue slots.  Here each level is held like fs_rows.hip holds a tile: thread t has columns 2 l and
// 2 l + 1 of M rows (lane l = t mod G of group t / G, G the power of two that covers the row's pairs), and a
// half-sweep exchanges only the groups' top and bottom rows through LDS.  Conductances go from memory straight to
// registers (all levels in one latency) and stay there for the whole cycle; levels that fit one wavefront need no
// workgroup barrier inside their sweeps; restriction sums along x in registers (lane shifts) and passes one value per
// row edge; the coarse inverse is applied column by column from LDS.  The expressions and the order of every sum are those
// of the kernels that keep the levels in LDS (tail_run): the same values bit for bit.
#include "fs_kernels.hpp"
#include "fs_mg_device.hpp"

#include <type_traits>

namespace fsim {

namespace {

// One level in registers.
template <int M> struct Held {
    float x[M][2], wr[M][2], wd[M][2], wu[2], wl[M], inv[M][2], cb[M][2];
};

constexpr int kTailMax = 1024;   // threads of the largest workgroup

constexpr int kTables = 512;     // entries of the levels' transfer tables

// LDS of the kernel.
struct TailShared {
    float edge[2][2][kTailMax];     // [colour][top, bottom][thread]
    float reach[2][kTailMax];       // the restriction's row sums: [top, bottom][thread]
    float field[kTailMax + 256];    // a coarse level's rhs (down) or solution (up), rows of width kernel-wide cells
    float inverse[64 * 64];         // the coarse inverse, column j at 64 j
    float4 table[kTables];          // transfer tables of the levels
};

struct Place {
    int lane, group, G;
    bool active;      // this wavefront holds cells of the level
    bool one;         // the level fits the first wavefront
};

template <int M> __device__ __forceinline__ Place place(const TailLevel& T)
{
    Place p;
    p.G = 1 << T.lanes;
    p.lane = threadIdx.x & (p.G - 1);
    p.group = threadIdx.x >> T.lanes;
    const int threads = ((T.h + M - 1) / M) << T.lanes;
    p.active = (int)(threadIdx.x & ~63u) < threads;
    p.one = threads <= 64;
    return p;
}

// Orders LDS traffic between the phases of a level: a workgroup barrier, or nothing but program order (LDS serves one
// wavefront's accesses in order) for a level of one wavefront.
__device__ __forceinline__ void level_barrier(bool one)
{
    if (one)
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    else
        __syncthreads();
}

// Element index of the thread's column pair in local row r of a padded field: past the last pair the zero halo pair
// (w, w + 1), outside the rows the first pair of the upper halo row.
template <int M> __device__ __forceinline__ int pair_index(const TailLevel& T, const Place& p, int r)
{
    const int y = p.group * M + r;
    return y >= 0 && y < T.h ? (y + 1) * T.s + min(2 * p.lane, T.w) + 1 : 0;
}

template <class T> __device__ __forceinline__ void load_two(const T* p, int i, float (&v)[2])
{
    const Pair<T> t = *(const Pair<T>*)(p + i);
    v[0] = ldv(t.a);
    v[1] = ldv(t.b);
}

// Issues the loads of a level's conductances (finish_level completes them).
template <int M> __device__ __forceinline__ void load_level(const TailLevel& T, Held<M>& v)
{
    const Place p = place<M>(T);
    load_two(T.down, pair_index<M>(T, p, -1), v.wu);
#pragma unroll
    for (int r = 0; r < M; ++r) {
        const int i = pair_index<M>(T, p, r);
        load_two(T.right, i, v.wr[r]);
        load_two(T.down, i, v.wd[r]);
    }
}

template <int M> __device__ __forceinline__ void finish_level(Held<M>& v)
{
#pragma unroll
    for (int r = 0; r < M; ++r) {
        // the first lane's left face is a wall: the previous group's last face or nothing, zero either way
        v.wl[r] = from_left(v.wr[r][1]);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const float l = j ? v.wr[r][0] : v.wl[r], u = r ? v.wd[r - 1][j] : v.wu[j];
            v.inv[r][j] = inv_or_zero((l + v.wr[r][j]) + (u + v.wd[r][j]));
        }
    }
}

// `sweeps` red-black sweeps, forward or (post-smoothing) reversed; FROM_ZERO: x starts at zero.
template <int M, bool POST> __device__ __forceinline__ void smooth(Held<M>& v, const Place& p, int sweeps, TailShared& S)
{
    const int t = threadIdx.x;
    const int above = max(t - p.G, 0), below = min(t + p.G, kTailMax - 1);
    auto publish = [&](auto color) {
        constexpr int c = decltype(color)::value;
        S.edge[c][0][t] = v.x[0][c];
        S.edge[c][1][t] = v.x[M - 1][c ^ 1];
    };
    auto half = [&](auto color, bool neighbours) {
        constexpr int c = decltype(color)::value;
        if (p.active) {
            const float hu = S.edge[c ^ 1][1][above], hd = S.edge[c ^ 1][0][below];
#pragma unroll
            for (int r = 0; r < M; ++r) {
                const int j = (c + r) & 1;
                float a = v.cb[r][j];
                if (neighbours) {
                    const float n0 = j ? v.x[r][0] : from_left(v.x[r][1]);
                    const float n1 = j ? from_right(v.x[r][0]) : v.x[r][1];
                    const float n2 = r ? v.x[r - 1][j] : hu;
                    const float n3 = r + 1 < M ? v.x[r + 1][j] : hd;
                    const float l = j ? v.wr[r][0] : v.wl[r], u = r ? v.wd[r - 1][j] : v.wu[j];
                    a += (l * n0 + v.wr[r][j] * n1) + (u * n2 + v.wd[r][j] * n3);
                }
                v.x[r][j] = a * v.inv[r][j];
            }
            publish(color);
        }
        level_barrier(p.one);
    };
    constexpr std::integral_constant<int, 0> red{};
    constexpr std::integral_constant<int, 1> black{};
    if (p.one && !p.active)
        return;
    if constexpr (POST) {
        if (p.active)
            publish(red);
        level_barrier(p.one);
#pragma unroll 1
        for (int k = 0; k < sweeps; ++k) {
            half(black, true);
            half(red, true);
        }
    } else {
        half(red, false);
        half(black, true);
#pragma unroll 1
        for (int k = 1; k < sweeps; ++k) {
            half(red, true);
            half(black, true);
        }
    }
}

// Residual of the level and its restriction into S.field (rows of T.cw).
template <int M> __device__ __forceinline__ void restrict_level(const TailLevel& T, Held<M>& v, const Place& p, TailShared& S)
{
    const int t = threadIdx.x;
    float h[M];
    const float4* tab = S.table + T.table;
    const int pairs = (T.w + 1) >> 1, rows = (T.h + 1) >> 1;
    if (p.active) {
        const float4 wx = tab[2 * min(p.lane, pairs - 1) + 1];
        const int above = max(t - p.G, 0), below = min(t + p.G, kTailMax - 1);
        float up[2], dn[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            up[j] = S.edge[j ^ 1][1][above];
            dn[j] = S.edge[j][0][below];
        }
#pragma unroll
        for (int r = 0; r < M; ++r) {
            float res[2];
            const float n[2][2] = {{from_left(v.x[r][1]), v.x[r][1]}, {v.x[r][0], from_right(v.x[r][0])}};
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const float c = v.x[r][j];
                const float l = j ? v.wr[r][0] : v.wl[r], u = r ? v.wd[r - 1][j] : v.wu[j];
                const float nu = r ? v.x[r - 1][j] : up[j], nd = r + 1 < M ? v.x[r + 1][j] : dn[j];
                const float product = (l * (c - n[j][0]) + v.wr[r][j] * (c - n[j][1])) +
                                      (u * (c - nu) + v.wd[r][j] * (c - nd));
                const bool active = (l + v.wr[r][j]) + (u + v.wd[r][j]) > 0.f;
                res[j] = active ? v.cb[r][j] - product : 0.f;
            }
            // fine columns 2 l - 1 .. 2 l + 2 onto coarse column l; a missing tap has weight 0
            h[r] = ((wx.x * from_left(res[1]) + wx.y * res[0]) + wx.z * res[1]) + wx.w * from_right(res[0]);
        }
        S.reach[0][t] = h[0];
        S.reach[1][t] = h[M - 1];
    }
    level_barrier(p.one);
    if (p.active) {
        const float hu = S.reach[1][max(t - p.G, 0)], hd = S.reach[0][min(t + p.G, kTailMax - 1)];
#pragma unroll
        for (int k = 0; k < M / 2; ++k) {
            const int Y = p.group * (M / 2) + k;
            const float4 wy = tab[2 * (pairs + min(Y, rows - 1)) + 1];
            const float first = k ? h[2 * k - 1] : hu;
            const float last = 2 * k + 2 < M ? h[2 * k + 2] : hd;
            const float value = ((wy.x * first + wy.y * h[2 * k]) + wy.z * h[2 * k + 1]) + wy.w * last;
            if (p.lane < T.cw && Y < T.ch)
                S.field[Y * T.cw + p.lane] = value;
        }
    }
    __syncthreads();
}

// Adds the prolonged coarse solution in S.field to x.
template <int M> __device__ __forceinline__ void prolong_level(const TailLevel& T, Held<M>& v, const Place& p, const TailShared& S)
{
    if (!p.active)
        return;
    const float4* tab = S.table + T.table;
    const int pairs = (T.w + 1) >> 1, rows = (T.h + 1) >> 1;
    const int l = min(p.lane, pairs - 1);
    const float4 tx = tab[2 * l];
    const int code = __float_as_int(tx.z);
    const int c0 = max(l - 1, 0), c2 = min(l + 1, T.cw - 1);
    constexpr int NH = M / 2 + 2;
    float hv[NH][2];
#pragma unroll
    for (int i = 0; i < NH; ++i) {
        const int Y = min(max(p.group * (M / 2) - 1 + i, 0), T.ch - 1);
        const float* q = S.field + Y * T.cw;
        const float a = q[c0], b = q[l], c = q[c2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const float w = j ? tx.y : tx.x;
            const int k = code >> (4 * j);
            const float first = k & 1 ? b : a;
            const float second = k & 4 ? c : k & 2 ? b : a;
            hv[i][j] = (1.f - w) * first + w * second;
        }
    }
#pragma unroll
    for (int k = 0; k < M / 2; ++k) {
        const int Y = p.group * (M / 2) + k;
        const float4 ty = tab[2 * (pairs + min(Y, rows - 1))];
        const int cy = __float_as_int(ty.z);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int r = 2 * k + i;
            const float w = i ? ty.y : ty.x;
            const int s = cy >> (4 * i);
            const bool in = p.group * M + r < T.h;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const float a = s & 1 ? hv[k + 1][j] : hv[k][j];
                const float b = s & 4 ? hv[k + 2][j] : s & 2 ? hv[k + 1][j] : hv[k][j];
                const float sum = v.x[r][j] + ((1.f - w) * a + w * b);
                v.x[r][j] = in && 2 * p.lane + j < T.w ? sum : 0.f;
            }
        }
    }
}

// The coarsest level (tail_coarse_solve's arithmetic): rhs in S.field, the solution left there.  One wavefront.
__device__ __forceinline__ void coarse_solve(const TailLevel& T, int n, TailShared& S)
{
    const int lane = threadIdx.x;
    const int cells = n + 1;
    const float b = lane < cells ? S.field[lane] : 0.f;
    const double mean = wave_sum((double)b) / cells;
    const float y = (float)((double)b - mean);
    // c = G y in the order j = 0 .. n - 1; y_j is held by lane j + 1
    float c = 0.f;
    for (int j0 = 0; j0 < n; j0 += 8) {
        float g[8];
#pragma unroll
        for (int q = 0; q < 8; ++q)
            g[q] = S.inverse[64 * min(j0 + q, 62) + lane];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const float yv = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(y), min(j0 + q, 62) + 1));
            c += g[q] * (j0 + q < n ? yv : 0.f);
        }
    }
    const double gauge = wave_sum(lane < n ? (double)c : 0.0) / cells;
    if (lane < n)
        S.field[lane + 1] = (float)((double)c - gauge);
    if (lane == 0)
        S.field[0] = (float)(-gauge);
}

// NL levels above the coarsest; ANY: up to NL, as many as D has.
template <int K, int NL, bool ANY> struct Cycle {
    // Level K's cycle; its rhs is in S.field for K > 0, its solution left in the registers.
    template <int M, class Deeper>
    static __device__ __forceinline__ void run(const TailDesc& D, Held<M>& v, Deeper& deeper, TailShared& S)
    {
        const TailLevel& T = D.lev[K];
        const Place p = place<M>(T);
        if constexpr (K > 0) {
#pragma unroll
            for (int r = 0; r < M; ++r)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const int x = 2 * p.lane + j, y = p.group * M + r;
                    v.cb[r][j] = x < T.w && y < T.h ? S.field[y * T.w + x] : 0.f;
                }
        }
#pragma unroll
        for (int r = 0; r < M; ++r)
            v.x[r][0] = v.x[r][1] = 0.f;
        smooth<M, false>(v, p, D.sweeps, S);
        if constexpr (K > 0)
            __syncthreads();   // S.field has been read
        restrict_level<M>(T, v, p, S);
        bool last = true;
        if constexpr (K + 1 < NL) {
            last = ANY && K + 2 >= D.levels;
            if (!last) {
                Cycle<K + 1, NL, ANY>::run(D, deeper[K], deeper, S);
                const TailLevel& C = D.lev[K + 1];
                const Place q = place<2>(C);
                __syncthreads();
#pragma unroll
                for (int r = 0; r < 2; ++r)
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const int x = 2 * q.lane + j, y = q.group * 2 + r;
                        if (x < C.w && y < C.h)
                            S.field[y * C.w + x] = deeper[K].x[r][j];
                    }
            }
        }
        if (last && threadIdx.x < 64)
            coarse_solve(D.lev[K + 1], D.coarse_n, S);
        __syncthreads();
        prolong_level<M>(T, v, p, S);
        smooth<M, true>(v, p, D.sweeps, S);
    }
};

template <int M, int NT, int NL, bool ANY, class TV>
__device__ __forceinline__ void tail_cycle(const TailDesc& D, const double* shift, const int* status, TailShared& S)
{
    const TailLevel& T = D.lev[0];
    const Place p = place<M>(T);
    Held<M> top;
    Held<2> deeper[NL > 1 ? NL - 1 : 1];
    load_level<M>(T, top);
#pragma unroll
    for (int r = 0; r < M; ++r)
        load_two((const TV*)D.top_rhs, pair_index<M>(T, p, r), top.cb[r]);
#pragma unroll
    for (int k = 0; k + 1 < NL; ++k)
        load_level<2>(D.lev[ANY ? min(k + 1, D.levels - 1) : k + 1], deeper[k]);
    constexpr int TG = (63 * 63 + NT - 1) / NT, TT = (kTables + NT - 1) / NT;
    const int n = D.coarse_n, nn = n * n;
    float gv[TG];
    float4 tv[TT];
#pragma unroll
    for (int k = 0; k < TG; ++k)
        gv[k] = D.ginv[min((int)threadIdx.x + k * NT, max(nn - 1, 0))];
#pragma unroll
    for (int k = 0; k < TT; ++k)
        tv[k] = D.pair_tables[min((int)threadIdx.x + k * NT, D.pair_table_n - 1)];
    if (status && *status != kRunning)
        return;
    // neighbours past a level's rows read zeros (or another level's finite values) with zero weights
    for (int i = threadIdx.x; i < kTailMax; i += NT) {
#pragma unroll
        for (int c = 0; c < 2; ++c)
            S.edge[c][0][i] = S.edge[c][1][i] = 0.f;
        S.reach[0][i] = S.reach[1][i] = 0.f;
    }
    const float inv_n = 1.0f / (float)max(n, 1);
#pragma unroll
    for (int k = 0; k < TG; ++k) {
        const int e = threadIdx.x + k * NT;
        const int i = (int)(((float)e + 0.5f) * inv_n), j = e - i * n;   // exact: e < 2^12
        if (e < nn)
            S.inverse[64 * j + i] = gv[k];
    }
    for (int e = threadIdx.x; e < 64 * 63; e += NT)
        if ((e & 63) >= n || (e >> 6) >= n)
            S.inverse[e] = 0.f;
#pragma unroll
    for (int k = 0; k < TT; ++k)
        if ((int)threadIdx.x + k * NT < D.pair_table_n)
            S.table[threadIdx.x + k * NT] = tv[k];
    finish_level<M>(top);
#pragma unroll
    for (int k = 0; k + 1 < NL; ++k)
        finish_level<2>(deeper[k]);
    if (shift) {
        const double sh = *shift;
#pragma unroll
        for (int r = 0; r < M; ++r)
#pragma unroll
            for (int j = 0; j < 2; ++j)
                top.cb[r][j] = (float)((double)top.cb[r][j] - sh);
    }
    __syncthreads();
    Cycle<0, NL, ANY>::run(D, top, deeper, S);
    TV* out = (TV*)D.top_sol;
#pragma unroll
    for (int r = 0; r < M; ++r) {
        const int y = p.group * M + r, x = 2 * p.lane;
        if (y < T.h && x < T.w) {
            TV* q = out + (y + 1) * T.s + x + 1;
            if (x + 1 < T.w)
                *(Pair<TV>*)q = Pair<TV>{stv<TV>(top.x[r][0]), stv<TV>(top.x[r][1])};
            else
                *q = stv<TV>(top.x[r][0]);
        }
    }
}

template <int M, int NT, int NL, class TV>
__global__ __launch_bounds__(NT) void k_tail(const TailDesc D, const double* shift, const int* status)
{
    __shared__ TailShared S;
    tail_cycle<M, NT, NL, false, TV>(D, shift, status, S);
}

// The tails of many grids, one workgroup each: 512 threads, eight rows per thread, whatever the shapes.
constexpr int kBatchThreads = 512;
__global__ __launch_bounds__(kBatchThreads) void k_tail_batch(const BatchItem* __restrict__ items,
    const int* __restrict__ list)
{
    __shared__ TailShared S;
    const BatchItem& I = items[list[blockIdx.x]];
    const double* shift = I.levels == 0 ? &I.g.S->r_mean : nullptr;
    tail_cycle<8, kBatchThreads, 4, true, float>(I.tail, shift, &I.g.S->status, S);
}

template <int M, int NT, class TV>
void launch_levels(hipStream_t st, const TailDesc& D, const double* shift, const int* status)
{
    switch (D.levels) {
    case 2: hipLaunchKernelGGL((k_tail<M, NT, 1, TV>), dim3(1), dim3(NT), 0, st, D, shift, status); break;
    case 3: hipLaunchKernelGGL((k_tail<M, NT, 2, TV>), dim3(1), dim3(NT), 0, st, D, shift, status); break;
    case 4: hipLaunchKernelGGL((k_tail<M, NT, 3, TV>), dim3(1), dim3(NT), 0, st, D, shift, status); break;
    default: hipLaunchKernelGGL((k_tail<M, NT, 4, TV>), dim3(1), dim3(NT), 0, st, D, shift, status); break;
    }
}

template <class TV> void launch_held(hipStream_t st, const TailDesc& D, const double* shift, const int* status)
{
    if (D.held_rows == 2)
        launch_levels<2, 1024, TV>(st, D, shift, status);
    else if (D.held_rows == 4)
        launch_levels<4, 768, TV>(st, D, shift, status);
    else
        launch_levels<8, 512, TV>(st, D, shift, status);
}

}  // namespace

void tail_hold(TailDesc& t)
{
    // A level's lanes: the power of two that covers its column pairs.
    const auto lanes = [](const TailLevel& T) {
        int b = 0;
        while ((1 << b) < (T.w + 1) / 2)
            ++b;
        return b;
    };
    const auto threads = [&](const TailLevel& T, int rows) { return ((T.h + rows - 1) / rows) << lanes(T); };
    t.held_rows = t.batch_rows = 0;
    if (t.levels < 2 || t.levels > 5)
        return;
    const auto fits = [&](int rows, int limit) {
        bool ok = t.lev[0].w <= 128 && threads(t.lev[0], rows) <= limit;
        int table = 0;
        for (int l = 0; l + 1 < t.levels; ++l) {
            ok = ok && (l == 0 || threads(t.lev[l], 2) <= limit);
            ok = ok && t.lev[l + 1].w * t.lev[l + 1].h <= kTailMax + 256;
            table += 2 * ((t.lev[l].w + 1) / 2 + (t.lev[l].h + 1) / 2);
        }
        return ok && table <= kTables;
    };
    t.held_rows = fits(2, 1024) ? 2 : fits(4, 768) ? 4 : fits(8, 512) ? 8 : 0;
    t.batch_rows = fits(8, kBatchThreads) ? 8 : 0;
    int at = 0;
    for (int l = 0; l < t.levels; ++l) {
        t.lev[l].lanes = lanes(t.lev[l]);
        t.lev[l].table = at;
        at += 2 * ((t.lev[l].w + 1) / 2 + (t.lev[l].h + 1) / 2);
    }
}

void launch_batch_tail(hipStream_t st, const BatchItem* items, const int* list, int n)
{
    if (n > 0)
        hipLaunchKernelGGL(k_tail_batch, dim3(n), dim3(kBatchThreads), 0, st, items, list);
}

void launch_held_tail(hipStream_t st, const TailDesc& desc, const double* shift, const int* status, int bf16_top)
{
    if (bf16_top)
        launch_held<bf16>(st, desc, shift, status);
    else
        launch_held<float>(st, desc, shift, status);
}

}  // namespace fsim
