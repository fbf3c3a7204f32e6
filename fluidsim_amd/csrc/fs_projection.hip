// fs_projection.hip -- the projection's kernels around the V-cycle (FluidGridCPU.cpp:1030-1205, 1728-1824).
//
// FP64 expressions (face weights, conductances, rhs, pressure, corrections) keep the reference's order with
// -ffp-contract=off, so they are bit-identical to it; the PCG vectors are FP32, every reduction FP64.
//
// Cell kernels use 64 x 16 tiles and 256 threads (four 64-wide wavefronts, one row segment each), so every wavefront
// touches 64 consecutive cells of a row: loads and stores coalesce.  Each kernel is a functor over one workgroup's
// part of one grid; a workgroup takes G tiles, one below the other: G = 1 spreads a small grid over the compute
// units, G = 4 keeps the number of partials that every consumer workgroup reads small on a large one (pcg_groups).
//
// What bounds them: a small grid's launch costs 2.3-4 us whatever it does, so phases share a launch wherever a
// workgroup can reduce the previous phase's partials for itself; a large grid's cost is its passes over memory.  Launches per
// projection besides the V-cycles: six to set up (they were fourteen) and four to close (six), five per iteration
// (nine).
#include "fs_kernels.hpp"

#include <math.h>

namespace fsim {

namespace {

constexpr int kTX = 64;
constexpr int kTY = 16;
constexpr int kNT = 256;

__device__ __forceinline__ double abs_or_inf(double v) { return isfinite(v) ? fabs(v) : INFINITY; }

// A workgroup's place in its grid's launch: column and row of its tile group, and the number of columns.
struct Block {
    int x, y, columns;
    __device__ __forceinline__ int id() const { return y * columns + x; }
};

// The four cells a thread owns in a 64 x 16 tile, as clamped (always valid) coordinates plus an
// in-range mask.  Kernels load through these unconditionally and predicate only the stores:
// a guarded load makes the compiler wait for it at the branch join, which serialises a thread's
// rows into one memory latency each.
struct Tile4 {
    int x, xc;
    int y[4], yc[4];
    int P[4];
    bool in[4];
};

__device__ __forceinline__ Tile4 tile4(const GridDev& g, int column, int row, int thread)
{
    Tile4 t;
    t.x = column * kTX + (thread & 63);
    t.xc = min(t.x, g.W - 1);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        t.y[k] = row * kTY + (thread >> 6) + 4 * k;
        t.yc[k] = min(t.y[k], g.H - 1);
        t.in[k] = t.x < g.W && t.y[k] < g.H;
        t.P[k] = pidx(t.xc, t.yc[k], g.s);
    }
    return t;
}
__device__ __forceinline__ Tile4 tile4(const GridDev& g, int column, int row)
{
    return tile4(g, column, row, threadIdx.x);
}

// ------------------------------------------------------------------------------------------
// Scalar block (kernels, so they are safe inside captured graphs).
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ void init_scalars(PcgScalars* S, double tol, int max_iterations, double rel_tol)
{
    PcgScalars z{};
    z.tol = tol;
    z.rel_tol = rel_tol;
    z.max_iterations = max_iterations;
    z.status = kRunning;
    z.restart = 1;
    *S = z;
}

__global__ void k_init_scalars(PcgScalars* S, double tol, int max_iterations, double rel_tol)
{
    if (threadIdx.x == 0 && blockIdx.x == 0)
        init_scalars(S, tol, max_iterations, rel_tol);
}

__global__ void k_merge_failure(const PcgScalars* from, PcgScalars* S)
{
    if (threadIdx.x == 0 && blockIdx.x == 0 && from->mg_failed) {
        S->mg_failed = 1;
        if (S->status == kRunning)
            S->status = kFailed;
    }
}

// ------------------------------------------------------------------------------------------
// Density (FluidGridCPU.cpp:1399-1423), the conductance of the face right of / below each cell 2 / (rho_a + rho_b)
// (:1154-1205; zero at walls and, with a solid mask, on every face that touches a solid cell), and the finest level's
// FP32 copies and 1/diagonal (Level::rebuildDiagonal, PressureMultigrid.cpp:104-117).  One launch where there were
// three: the tile's densities and those around it are summed once into LDS, and the faces left of and above a cell
// are formed again instead of read back.
// ------------------------------------------------------------------------------------------
template <bool SUM> struct Coefficients {
    template <int G> __device__ __forceinline__ void run(const GridDev& g, Block B) const
    {
        constexpr int LX = kTX + 2, LY = kTY + 2, LOADS = (LX * LY + kNT - 1) / kNT;
        __shared__ double s_rho[LY * LX];
        const int W = g.W, H = g.H;
        const size_t N = (size_t)W * H;
        const double inverse_cell_volume = 1.0 / (g.h * g.h);
        for (int group = 0; group < G; ++group) {
            const int row = B.y * G + group;
            if (group)
                __syncthreads();
            size_t at[LOADS];
            double rho[LOADS] = {};
#pragma unroll
            for (int it = 0; it < LOADS; ++it) {
                const int e = min((int)threadIdx.x + it * kNT, LX * LY - 1);
                const int ly = e / LX, lx = e - ly * LX;
                const int x = min(max(B.x * kTX - 1 + lx, 0), W - 1), y = min(max(row * kTY - 1 + ly, 0), H - 1);
                at[it] = (size_t)y * W + x;
            }
            // component by component, the loads of two together: a cell's components one after another left a thread
            // one load in flight (8 + 8 components at 1920 x 1080 cells: 298 us for a capillary force, 205 so; 300 x 200 61 and 44)
            auto add = [&](const double* mass, int n) {
                for (int k = 0; k < n; k += 2) {
                    double m[2][LOADS];
#pragma unroll
                    for (int j = 0; j < 2; ++j)
#pragma unroll
                        for (int it = 0; it < LOADS; ++it)
                            m[j][it] = mass[(size_t)min(k + j, n - 1) * N + at[it]];
#pragma unroll
                    for (int j = 0; j < 2; ++j)
#pragma unroll
                        for (int it = 0; it < LOADS; ++it)
                            rho[it] += k + j < n ? m[j][it] : 0.0;
                }
            };
            if constexpr (SUM) {
                add(g.lmass, g.nl);
                add(g.gmass, g.ng);
            }
#pragma unroll
            for (int it = 0; it < LOADS; ++it)
                s_rho[min((int)threadIdx.x + it * kNT, LX * LY - 1)] =
                    SUM ? rho[it] * inverse_cell_volume : g.density[at[it]];
            __syncthreads();
            const Tile4 T = tile4(g, B.x, row);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int e = ((threadIdx.x >> 6) + 4 * k + 1) * LX + (threadIdx.x & 63) + 1;
                const double c = s_rho[e];
                const int x = T.x, y = T.y[k];
                bool wl = x > 0, wr = x + 1 < W, wu = y > 0, wd = y + 1 < H;
                if (g.solid) {
                    const unsigned char* m = g.solid + (size_t)T.yc[k] * W;
                    const bool open = m[T.xc] == 0;
                    wl = wl && open && m[max(T.xc - 1, 0)] == 0;
                    wr = wr && open && m[min(T.xc + 1, W - 1)] == 0;
                    wu = wu && open && m[T.xc - (T.yc[k] > 0 ? W : 0)] == 0;
                    wd = wd && open && m[T.xc + (T.yc[k] + 1 < H ? W : 0)] == 0;
                }
                if (T.in[k]) {
                    const double rl = wl ? 2.0 / (s_rho[e - 1] + c) : 0.0, rr = wr ? 2.0 / (c + s_rho[e + 1]) : 0.0;
                    const double du = wu ? 2.0 / (s_rho[e - LX] + c) : 0.0, dd = wd ? 2.0 / (c + s_rho[e + LX]) : 0.0;
                    const int P = T.P[k];
                    if (SUM)
                        g.density[(size_t)y * W + x] = c;
                    g.right64[P] = rr;
                    g.down64[P] = dd;
                    level_diag_values(rl, rr, du, dd, g.invd32[P], g.right32[P], g.down32[P]);
                }
            }
        }
    }
};

// One level coarsened (PressureMultigrid.cpp:142-202) with its FP32 copies and 1/diagonal: the faces of a 64 x 4 tile,
// of the column left of it and of the row above it go through LDS.  A face is a chain of FP64 divisions, so each
// thread forms one cell's (taller tiles with several cells per thread took 17 us on 256^2 against 5).
constexpr int kCoarsenY = 4;
constexpr int kCoarsenThreads = 384;
__device__ __forceinline__ void coarsen_tile(const ChainLevel& L, int column, int row)
{
    constexpr int LX = kTX + 1, LY = kCoarsenY + 1;
    static_assert(LX * LY <= kCoarsenThreads, "one cell per thread");
    __shared__ double s_right[LY * LX], s_down[LY * LX];
    const int x0 = column * kTX - 1, y0 = row * kCoarsenY - 1;
    const int e = threadIdx.x;
    const int ly = e / LX, lx = e - ly * LX;
    const int x = x0 + lx, y = y0 + ly;
    const bool in = e < LX * LY && x >= 0 && x < L.cw && y >= 0 && y < L.ch;
    if (e < LX * LY) {
        double2 c = make_double2(0.0, 0.0);
        if (in)
            c = coarsen_cell(x, y, L.fw, L.fh, L.fcx, L.fcy, L.fright, L.fdown, L.cw, L.ch, L.ccx, L.ccy);
        s_right[e] = c.x;
        s_down[e] = c.y;
    }
    __syncthreads();
    if (in && lx > 0 && ly > 0) {
        const int i = pidx(x, y, L.cw + 2);
        L.cright[i] = s_right[e];
        L.cdown[i] = s_down[e];
        level_diag_values(s_right[e - 1], s_right[e], s_down[e - LX], s_down[e], L.invd32[i], L.right32[i],
            L.down32[i]);
    }
}

// One-dimensional: the tiles of a tall level are more than a launch has rows (65536).
__global__ __launch_bounds__(kCoarsenThreads) void k_coarsen(ChainLevel L)
{
    const int columns = (L.cw + kTX - 1) / kTX;
    const int row = (int)blockIdx.x / columns;
    coarsen_tile(L, (int)blockIdx.x - row * columns, row);
}

// ------------------------------------------------------------------------------------------
// Projection set-up (FluidGridCPU.cpp:1050-1090, :1728-1756), FP64.
// ------------------------------------------------------------------------------------------

// Zero wall velocities, form rhs = -div * h^2 / dt, sum it.
struct Rhs {
    template <int G> __device__ __forceinline__ void run(const GridDev& g, Block B) const
    {
        __shared__ double lds[kNT / 64];
        const int W = g.W, H = g.H;
        const double scale = g.h * g.h / g.dt;
        const int st = g.S->status;
        double sum[1] = {0.0};
#pragma unroll 1
        for (int group = 0; group < G; ++group) {
            const Tile4 T = tile4(g, B.x, B.y * G + group);
            const int x = T.x, xc = T.xc;
            double uL[4], uR[4], vT[4], vB[4];
            unsigned closed[4];   // solid mask: bit 0 left, 1 right, 2 top, 3 bottom face touches a solid cell
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int yc = T.yc[k];
                const double* hz = g.u + (size_t)yc * (W + 1);
                const double* vt = g.v + (size_t)yc * W;
                uL[k] = hz[xc];
                uR[k] = hz[xc + 1];
                vT[k] = vt[xc];
                vB[k] = vt[xc + W];
                closed[k] = 0u;
                if (g.solid) {
                    const unsigned char* m = g.solid + (size_t)yc * W;
                    const bool sc = m[xc] != 0;
                    closed[k] = (sc || m[max(xc - 1, 0)] ? 1u : 0u) | (sc || m[min(xc + 1, W - 1)] ? 2u : 0u) |
                                (sc || m[xc - (yc > 0 ? W : 0)] ? 4u : 0u) |
                                (sc || m[xc + (yc + 1 < H ? W : 0)] ? 8u : 0u);
                }
            }
            if (st != kRunning)
                return;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int y = T.y[k];
                if (T.in[k]) {
                    // walls are zeroed and read as zero (FluidGridCPU.cpp:1050-1061); faces touching a solid
                    // cell likewise (both cells of such a face write the same zero and neither reads it)
                    double* hz = g.u + (size_t)y * (W + 1);
                    double* vt = g.v + (size_t)y * W;
                    const bool cl = x == 0 || (closed[k] & 1u), cr = x + 1 == W || (closed[k] & 2u);
                    const bool ct = y == 0 || (closed[k] & 4u), cb = y + 1 == H || (closed[k] & 8u);
                    const double l = cl ? 0.0 : uL[k];
                    const double r = cr ? 0.0 : uR[k];
                    const double t = ct ? 0.0 : vT[k];
                    const double b = cb ? 0.0 : vB[k];
                    if (cl) hz[x] = 0.0;
                    if (cr) hz[x + 1] = 0.0;
                    if (ct) vt[x] = 0.0;
                    if (cb) vt[x + W] = 0.0;
                    const double du = r - l;
                    const double dv = b - t;
                    const double rhs = -(du + dv) / g.h * scale;
                    g.b[T.P[k]] = rhs;
                    sum[0] += rhs;
                }
            }
        }
        block_sums<kNT, 1>(sum, lds);
        if (threadIdx.x == 0)
            g.partials_ad[B.id()] = sum[0];
    }
};

// Remove the rhs mean and find max |rhs| (the early-out test of solvePressure); predictor p = 2 p - p_prev with the
// history shift, and the prediction's sum.
struct Predict {
    template <int G> __device__ __forceinline__ void run(const GridDev& g, Block B) const
    {
        __shared__ double lds[2 * kNT / 64];
        Partials<kNT, 1> total;
        total.load(g.fold_ad, g.fold_ad_n);
        const int st = g.S->status;
        double t[1];
        total.finish(g.fold_ad, g.fold_ad_n, t, lds);
        if (st != kRunning)
            return;
        const double mean = t[0] / ((double)g.W * g.H);
        if (B.id() == 0 && threadIdx.x == 0)
            g.S->b_mean = mean;
        double sum = 0.0, m = 0.0;
#pragma unroll 1
        for (int group = 0; group < G; ++group) {
            const Tile4 T = tile4(g, B.x, B.y * G + group);
            double bv[4], pv[4], qv[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                bv[k] = g.b[T.P[k]];
                pv[k] = g.p[T.P[k]];
                qv[k] = g.p_prev[T.P[k]];
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (T.in[k]) {
                    const double v = bv[k] - mean;
                    g.b[T.P[k]] = v;
                    m = fmax(m, abs_or_inf(v));
                    const double next = 2.0 * pv[k] - qv[k];
                    g.p[T.P[k]] = next;
                    g.p_prev[T.P[k]] = pv[k];
                    sum += next;
                }
            }
        }
        const double bs = block_sum<kNT>(sum, lds);
        const double bm = block_max<kNT>(m, lds);
        if (threadIdx.x == 0) {
            g.partials_up[2 * B.id()] = bs;
            g.partials_up[2 * B.id() + 1] = bm;
        }
    }
};

// What the prediction's partials (sum of p, max |b|) say: the residual tolerance and whether b is already below it
// (a divergence-free field needs no correction).
struct Outset {
    double p_mean, tol;
    bool zero;
};
__device__ __forceinline__ Outset outset(const GridDev& g, const double (&t)[2])
{
    Outset o;
    o.p_mean = t[0] / ((double)g.W * g.H);
    o.tol = g.S->rel_tol > 0.0 ? g.S->rel_tol * t[1] : g.S->tol;
    o.zero = t[1] <= o.tol;
    return o;
}

// True residual r = b - A (p - mean) of the predicted pressure, stored as the FP32 working residual.  The mean stays in p:
// the neighbours read it.
struct InitialResidual {
    template <int G> __device__ __forceinline__ void run(const GridDev& g, Block B) const
    {
        __shared__ double lds[2 * kNT / 64];
        Partials<kNT, 2, 1> up;
        up.load(g.fold_up, g.fold_up_n);
        const int st = g.S->status;
        double t[2];
        up.finish(g.fold_up, g.fold_up_n, t, lds);
        if (st != kRunning)
            return;
        const Outset o = outset(g, t);
        if (o.zero)
            return;
        const int s = g.s;
        double sum = 0.0, m = 0.0;
#pragma unroll 1
        for (int group = 0; group < G; ++group) {
            const Tile4 T = tile4(g, B.x, B.y * G + group);
            double r[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int i = T.P[k];
                auto at = [&](int j) { return g.p[j] - o.p_mean; };
                const double c = at(i);
                const double product = (g.right64[i - 1] * (c - at(i - 1)) + g.right64[i] * (c - at(i + 1))) +
                                       (g.down64[i - s] * (c - at(i - s)) + g.down64[i] * (c - at(i + s)));
                r[k] = g.b[i] - product;
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (T.in[k]) {
                    g.r[T.P[k]] = (float)r[k];
                    g.x[T.P[k]] = 0.0f;
                    sum += r[k];
                    m = fmax(m, fabs(r[k]));
                }
            }
        }
        const double bs = block_sum<kNT>(sum, lds);
        const double bm = block_max<kNT>(m, lds);
        if (threadIdx.x == 0) {
            g.partials_tr[2 * B.id()] = bs;
            g.partials_tr[2 * B.id() + 1] = bm;
        }
    }
};

// ------------------------------------------------------------------------------------------
// PCG loop (FluidGridCPU.cpp:1779-1819) with FP32 vectors and FP64 scalars.
// ------------------------------------------------------------------------------------------

// The direction of iteration c lives in d or d2 by the parity of c: the fused direction and operator kernel
// reads its neighbours' old values while other workgroups write new ones.
__device__ __forceinline__ float* direction_of(const GridDev& g, int c) { return c & 1 ? g.d2 : g.d; }

// The next direction from the r.z sums: every workgroup reduces the partials itself (same order, same
// value): beta = next / previous r.z (zero after a restart), or with FLEX the Polak-Ribiere
// -alpha (z - mean z).q / previous r.z.  Workgroup 0 records the new r.z in the next slot and stops the solve
// on a non-positive r.z (the budget stops it at the check).  Returns false when the solve stops.
template <bool FLEX>
__device__ __forceinline__ bool next_direction(const GridDev& g, const double (&t)[FLEX ? 5 : 3], bool first,
    float& mean, double& beta64)
{
    const double n = (double)g.W * g.H;
    const double zmean = t[0] / n;
    const double next = t[1] - zmean * t[2];
    const int c = g.S->iterations;
    double numerator = next;
    if constexpr (FLEX)
        numerator = -g.S->alpha * (t[3] - zmean * t[4]);
    beta64 = g.S->restart ? 0.0 : numerator / g.S->rz_slot[(c + 1) & 1];
    const bool stop = !isfinite(beta64) || !(c < g.S->max_iterations && next > 0.0 && isfinite(next));
    if (first && threadIdx.x == 0) {
        g.S->z_mean = zmean;
        g.S->beta = beta64;
        if (isfinite(beta64))
            g.S->rz_slot[c & 1] = next;
        if (stop)
            g.S->status = kStopped;
    }
    mean = (float)zmean;
    return !stop;
}

// d = (z - mean z) + beta d and q = A d (5-point, variable coefficient; walls have zero weight), d.q.
// One launch where there were two: it reads z and the old d once more around each tile (66 x 18 cells for 64 x 16,
// 66 x 66 for four) instead of writing d and reading it back, and a launch of a small grid costs about
// 4 us whatever it does.  A check that refreshed r left x to be folded into p: done here.
template <bool FLEX> struct DirectionAd {
    template <int G> __device__ __forceinline__ void run(const GridDev& g, Block B) const
    {
        constexpr int LX = kTX + 2, LY = kTY * G + 2;
        __shared__ double lds[5 * kNT / 64];
        __shared__ float s_d[LY * LX];
        const int s = g.s, W = g.W, H = g.H;
        const int x0 = B.x * kTX - 1, y0 = B.y * kTY * G - 1;
        constexpr int LOADS = (LX * LY + kNT - 1) / kNT;
        constexpr int NP = FLEX ? 5 : 3;
        Partials<kNT, NP> sums;
        sums.load(g.fold_rz, g.fold_rz_n);
        float zv[LOADS], dv[LOADS];
        int at[LOADS];
        // clamped to the zero halo: the values of cells outside the grid meet zero weights only
#pragma unroll
        for (int it = 0; it < LOADS; ++it) {
            const int e = min((int)threadIdx.x + it * kNT, LX * LY - 1);
            const int ly = e / LX, lx = e - ly * LX;
            at[it] = pidx(min(x0 + lx, W), min(y0 + ly, H), s);
            zv[it] = g.z[at[it]];
        }
        const int st = g.S->status;
        const int c = g.S->iterations;
        const float* d_old = direction_of(g, c + 1);
        float* d_new = direction_of(g, c);
#pragma unroll
        for (int it = 0; it < LOADS; ++it)
            dv[it] = d_old[at[it]];
        double t[NP];
        sums.finish(g.fold_rz, g.fold_rz_n, t, lds);
        if (st != kRunning)
            return;
        float mean;
        double beta64;
        if (!next_direction<FLEX>(g, t, B.id() == 0, mean, beta64))
            return;
        const float beta = (float)beta64;
#pragma unroll
        for (int it = 0; it < LOADS; ++it) {
            const int e = threadIdx.x + it * kNT;
            if (e < LX * LY) {
                const float zz = zv[it] - mean;
                s_d[e] = beta64 == 0.0 ? zz : zz + beta * dv[it];
            }
        }
        const bool fold = g.S->flush != 0;
        const double p_shift = g.S->p_shift;
        __syncthreads();
        double dot[1] = {0.0};
#pragma unroll
        for (int group = 0; group < G; ++group) {
            const Tile4 T = tile4(g, B.x, B.y * G + group);
            float dc[4], q[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int i = T.P[k];
                const float wl = g.right32[i - 1], wr = g.right32[i], wu = g.down32[i - s], wd = g.down32[i];
                const int e = (group * kTY + (threadIdx.x >> 6) + 4 * k + 1) * LX + (threadIdx.x & 63) + 1;
                dc[k] = s_d[e];
                const float dl = s_d[e - 1], dr = s_d[e + 1], du = s_d[e - LX], dd = s_d[e + LX];
                q[k] = (wl * (dc[k] - dl) + wr * (dc[k] - dr)) + (wu * (dc[k] - du) + wd * (dc[k] - dd));
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (T.in[k]) {
                    d_new[T.P[k]] = dc[k];
                    g.q[T.P[k]] = q[k];
                    dot[0] += (double)dc[k] * (double)q[k];
                }
            }
            if (fold) {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    if (T.in[k]) {
                        g.p[T.P[k]] = (g.p[T.P[k]] - p_shift) + (double)g.x[T.P[k]];
                        g.x[T.P[k]] = 0.0f;
                    }
                }
            }
        }
        block_sums<kNT, 1>(dot, lds);
        if (threadIdx.x == 0)
            g.partials_ad[B.id()] = dot[0];
    }
};

// x += alpha d ; r -= alpha q ; residual sum and max-norm.
// Every workgroup first reduces the operator's d.q partials itself (same order, same value) and forms
// alpha; workgroup 0 records it, clears the flags the previous direction consumed, and stops
// the solve on a non-positive d.q.
struct Update {
    template <int G> __device__ __forceinline__ void run(const GridDev& g, Block B) const
    {
        __shared__ double lds[2 * kNT / 64];
        Partials<kNT, 1> dot;
        dot.load(g.fold_ad, g.fold_ad_n);
        const int st = g.S->status;
        const int c = g.S->iterations;
        const float* d = direction_of(g, c);
        Tile4 T = tile4(g, B.x, B.y * G);
        float xv[4], dv[4], rv[4], qv[4];
        auto load = [&] {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int i = T.P[k];
                xv[k] = g.x[i];
                dv[k] = d[i];
                rv[k] = g.r[i];
                qv[k] = g.q[i];
            }
        };
        load();
        const double rz = g.S->rz_slot[c & 1];
        double dq[1];
        dot.finish(g.fold_ad, g.fold_ad_n, dq, lds);
        if (st != kRunning)
            return;
        bool stop = dq[0] <= 0.0 || !isfinite(dq[0]);
        const double alpha64 = stop ? 0.0 : rz / dq[0];
        stop = stop || !isfinite(alpha64);
        if (B.id() == 0 && threadIdx.x == 0) {
            g.S->dq = dq[0];
            g.S->alpha = alpha64;
            g.S->restart = 0;
            g.S->flush = 0;
            g.S->p_shift = 0.0;
            if (stop)
                g.S->status = kStopped;
        }
        if (stop)
            return;
        const float alpha = (float)alpha64;
        double sum = 0.0, m = 0.0;
#pragma unroll
        for (int group = 0; group < G; ++group) {
            if (group) {
                T = tile4(g, B.x, B.y * G + group);
                load();
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (T.in[k]) {
                    const int i = T.P[k];
                    g.x[i] = xv[k] + alpha * dv[k];
                    const float r = rv[k] - alpha * qv[k];
                    g.r[i] = r;
                    sum += (double)r;
                    m = fmax(m, (double)fabsf(r));
                }
            }
        }
        const double bs = block_sum<kNT>(sum, lds);
        const double bm = block_max<kNT>(m, lds);
        if (threadIdx.x == 0) {
            g.partials_up[2 * B.id()] = bs;
            g.partials_up[2 * B.id() + 1] = bm;
        }
    }
};

// What the update's residual (sum, max-norm) calls for: a check of the true residual when the recurrence
// reached the tolerance, or a refresh of r (replace) when it dropped far enough or ran long enough.
struct Recurrence {
    double rmax;
    bool verify, replace;
};
__device__ __forceinline__ Recurrence recurrence(const PcgScalars* S, const double (&t)[2])
{
    Recurrence c;
    c.rmax = isfinite(t[0]) ? t[1] : INFINITY;
    const bool done = c.rmax <= S->tol;
    c.replace = !done && (c.rmax <= kRefineDrop * S->window_rmax || (S->iterations + 1) % kReplaceEvery == 0);
    c.verify = done || c.replace;
    return c;
}

// r = b - A (p + x) of a thread's cells in FP64, and its sum and max-norm.
__device__ __forceinline__ void true_residual(const GridDev& g, const Tile4& T, double& sum, double& m)
{
    const int s = g.s;
    double r[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int i = T.P[k];
        auto at = [&](int j) { return g.p[j] + (double)g.x[j]; };
        const double c = at(i);
        const double product = (g.right64[i - 1] * (c - at(i - 1)) + g.right64[i] * (c - at(i + 1))) +
                               (g.down64[i - s] * (c - at(i - s)) + g.down64[i] * (c - at(i + s)));
        r[k] = g.b[i] - product;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if (T.in[k]) {
            g.r[T.P[k]] = (float)r[k];
            sum += r[k];
            m = fmax(m, fabs(r[k]));
        }
    }
}

// The check: every workgroup reduces the update's partials itself and, where they call for it, forms the FP64
// true residual b - A (p + x) as the new working residual.  p and x stay as they are (the neighbours read them):
// the next direction folds x into p.  The scalar block is written by the finish launch alone.
struct Check {
    template <int G> __device__ __forceinline__ void run(const GridDev& g, Block B) const
    {
        __shared__ double lds[2 * kNT / 64];
        const int st = g.S->status;
        double t[2];
        Partials<kNT, 2, 1>().all(g.fold_up, g.fold_up_n, t, lds);
        if (st != kRunning || !recurrence(g.S, t).verify)
            return;
        double sum = 0.0, m = 0.0;
#pragma unroll 1
        for (int group = 0; group < G; ++group)
            true_residual(g, tile4(g, B.x, B.y * G + group), sum, m);
        const double bs = block_sum<kNT>(sum, lds);
        const double bm = block_max<kNT>(m, lds);
        if (threadIdx.x == 0) {
            g.partials_tr[2 * B.id()] = bs;
            g.partials_tr[2 * B.id() + 1] = bm;
        }
    }
};

// sum z, r.z and sum r in one pass; r.(z - mean z) = r.z - mean z * sum r; then beta.
// FLEX (flexible CG, for a preconditioner that is not exactly linear): also sum z.q and q, from which
// the direction kernel forms the Polak-Ribiere beta z_new.(r_new - r_old) / r_old.z_old with
// r_new - r_old = -alpha q (Notay 2000).
template <bool FLEX> struct Rz {
    template <int G> __device__ __forceinline__ void run(const GridDev& g, Block B) const
    {
        constexpr int NP = FLEX ? 5 : 3;
        __shared__ double lds[NP * kNT / 64];
        const int st = g.S->status;
        double sums[NP] = {};
#pragma unroll
        for (int group = 0; group < G; ++group) {
            const Tile4 T = tile4(g, B.x, B.y * G + group);
            float zv[4], rv[4], qv[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                zv[k] = g.z[T.P[k]];
                rv[k] = g.r[T.P[k]];
                qv[k] = FLEX ? g.q[T.P[k]] : 0.f;
            }
            if (st != kRunning)
                return;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (T.in[k]) {
                    const double zz = (double)zv[k], rr = (double)rv[k];
                    sums[0] += zz;
                    sums[1] += rr * zz;
                    sums[2] += rr;
                    if constexpr (FLEX) {
                        sums[3] += zz * (double)qv[k];
                        sums[4] += (double)qv[k];
                    }
                }
            }
        }
        block_sums<kNT, NP>(sums, lds);
        if (threadIdx.x == 0)
#pragma unroll
            for (int c = 0; c < NP; ++c)
                g.partials[NP * B.id() + c] = sums[c];
    }
};

// Diagonal preconditioner z = (r - mean) / diag.
struct PrecondDiag {
    template <int G> __device__ __forceinline__ void run(const GridDev& g, Block B) const
    {
        const int st = g.S->status;
#pragma unroll 1
        for (int group = 0; group < G; ++group) {
            const Tile4 T = tile4(g, B.x, B.y * G + group);
            float rv[4], iv[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                rv[k] = g.r[T.P[k]];
                iv[k] = g.invd32[T.P[k]];
            }
            if (st != kRunning)
                return;
            const double mean = g.S->r_mean;
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (T.in[k])
                    g.zdiag[T.P[k]] = (float)(((double)rv[k] - mean) * (double)iv[k]);
        }
    }
};

// ------------------------------------------------------------------------------------------
// Closing phase, once the solve has stopped (a no-op while it runs: it may be queued behind iterations that do not
// finish the solve).  The pressure's final value is formed from p and x where it is needed and stored last, since the
// correction reads the neighbours' p and x.
// ------------------------------------------------------------------------------------------

// Pressure of a stopped solve before its mean is removed: zero for a divergence-free field.
struct Final {
    int st;
    double shift;
    __device__ __forceinline__ explicit Final(const GridDev& g) : st(g.S->status), shift(g.S->p_shift) {}
    __device__ __forceinline__ bool solved() const { return st == kConverged || st == kStopped; }
    __device__ __forceinline__ double at(const GridDev& g, int i) const
    {
        return st == kZeroRhs ? 0.0 : (g.p[i] - shift) + (double)g.x[i];
    }
};

struct FinalSum {
    template <int G> __device__ __forceinline__ void run(const GridDev& g, Block B) const
    {
        __shared__ double lds[kNT / 64];
        const Final F(g);
        double sum[1] = {0.0};
#pragma unroll 1
        for (int group = 0; group < G; ++group) {
            const Tile4 T = tile4(g, B.x, B.y * G + group);
            double v[4];
#pragma unroll
            for (int k = 0; k < 4; ++k)
                v[k] = F.at(g, T.P[k]);
            if (!F.solved())
                return;
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (T.in[k])
                    sum[0] += v[k];
        }
        block_sums<kNT, 1>(sum, lds);
        if (threadIdx.x == 0)
            g.partials_ad[B.id()] = sum[0];
    }
};

// u -= (dp/h) dt w_u ; v -= (dp/h) dt w_v (FluidGridCPU.cpp:1098-1118).  Each cell owns its left
// u face and its top v face.
struct CorrectVelocity {
    template <int G> __device__ __forceinline__ void run(const GridDev& g, Block B) const
    {
        __shared__ double lds[kNT / 64];
        const int W = g.W, s = g.s;
        Partials<kNT, 1> total;
        total.load(g.fold_ad, g.fold_ad_n);
        const Final F(g);
        double t[1];
        total.finish(g.fold_ad, g.fold_ad_n, t, lds);
        // a failed hierarchy leaves the velocity alone, a solve still running is corrected later
        if (F.st == kFailed || F.st == kRunning)
            return;
        const double mean = F.solved() ? t[0] / ((double)g.W * g.H) : 0.0;
        if (B.id() == 0 && threadIdx.x == 0)
            g.S->p_mean = mean;
        const double dt = g.dt;
#pragma unroll 1
        for (int group = 0; group < G; ++group) {
            const Tile4 T = tile4(g, B.x, B.y * G + group);
            const int x = T.x, xc = T.xc;
            double pc[4], pl[4], pu[4], wl[4], wu[4], uv[4], vv[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int P = T.P[k];
                pc[k] = F.at(g, P) - mean;
                pl[k] = F.at(g, P - 1) - mean;
                pu[k] = F.at(g, P - s) - mean;
                wl[k] = g.right64[P - 1];
                wu[k] = g.down64[P - s];
                uv[k] = g.u[(size_t)T.yc[k] * (W + 1) + xc];
                vv[k] = g.v[(size_t)T.yc[k] * W + xc];
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (!T.in[k])
                    continue;
                const int y = T.y[k];
                if (x >= 1)
                    g.u[(size_t)y * (W + 1) + x] = uv[k] - ((pc[k] - pl[k]) / g.h) * dt * wl[k];
                if (y >= 1)
                    g.v[(size_t)y * W + x] = vv[k] - ((pc[k] - pu[k]) / g.h) * dt * wu[k];
            }
        }
    }
};

// maxDivergence (FluidGridCPU.cpp:1126-1152): non-finite divergence reports infinity.
// CLOSE: closing a projection (only once the solve has stopped), it also stores the final pressure.
template <bool CLOSE> struct MaxDivergence {
    template <int G> __device__ __forceinline__ void run(const GridDev& g, Block B) const
    {
        __shared__ double lds[kNT / 64];
        const Final F(g);
        if (CLOSE && F.st == kRunning)
            return;
        const double mean = CLOSE && F.st != kFailed ? g.S->p_mean : 0.0;
        const int W = g.W;
        double m = 0.0;
#pragma unroll 1
        for (int group = 0; group < G; ++group) {
            const Tile4 T = tile4(g, B.x, B.y * G + group);
            double dv[4], p[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const double* hz = g.u + (size_t)T.yc[k] * (W + 1);
                const double* vt = g.v + (size_t)T.yc[k] * W;
                dv[k] = ((hz[T.xc + 1] - hz[T.xc]) + (vt[T.xc + W] - vt[T.xc])) / g.h;
                p[k] = CLOSE ? F.at(g, T.P[k]) - mean : 0.0;
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (T.in[k]) {
                    m = fmax(m, abs_or_inf(dv[k]));
                    if (CLOSE) {
                        g.p[T.P[k]] = p[k];
                        g.x[T.P[k]] = 0.0f;
                        if (F.st == kZeroRhs)
                            g.p_prev[T.P[k]] = 0.0;
                    }
                }
            }
        }
        const double bm = block_max<kNT>(m, lds);
        if (threadIdx.x == 0)
            g.partials_tr[B.id()] = bm;
    }
};

// ------------------------------------------------------------------------------------------
// Reduction finish: one workgroup reads the producer's per-block partials in block order and
// updates the scalar block.  Running it as its own launch keeps cross-XCD visibility at kernel
// boundaries instead of a device-scope fence in every producer block.
// ------------------------------------------------------------------------------------------
struct FinishSetup {
    __device__ __forceinline__ void run(const GridDev& g, int nb, double* lds) const
    {
        PcgScalars* S = g.S;
        if (S->status != kRunning)
            return;
        double t[2], e[2];
        Partials<kNT, 2, 1>().all(g.fold_up, g.fold_up_n, t, lds);
        Partials<kNT, 2, 1>().all(g.partials_tr, nb, e, lds);
        if (threadIdx.x != 0)
            return;
        const Outset o = outset(g, t);
        S->bmax = t[1];
        S->tol = o.tol;
        if (o.zero) {
            S->status = kZeroRhs;
            return;
        }
        const double maximum = isfinite(e[0]) ? e[1] : INFINITY;
        S->p_shift = o.p_mean;
        S->flush = 1;
        S->true_rmax = maximum;
        S->r_sum = e[0];
        S->rmax = maximum;
        S->initial_rmax = maximum;
        S->window_rmax = maximum;
        S->r_mean = e[0] / ((double)g.W * g.H);
        if (maximum <= S->tol || S->max_iterations == 0)
            S->status = kInitialOk;
    }
};

// The decision after an update: t its residual (sum, max-norm), e the true one's where it was formed.
__device__ __forceinline__ void decide(const GridDev& g, const Recurrence& c, const double (&t)[2], const double (&e)[2])
{
    PcgScalars* S = g.S;
    const double n = (double)g.W * g.H;
    S->iterations += 1;
    S->rmax = c.rmax;
    S->r_sum = t[0];
    S->r_mean = t[0] / n;
    if (c.verify) {
        const double maximum = isfinite(e[0]) ? e[1] : INFINITY;
        S->true_rmax = maximum;
        S->r_sum = e[0];
        S->flush = 1;
        if (maximum <= S->tol) {
            S->status = kConverged;
        } else {
            S->r_mean = e[0] / n;
            if (!c.replace || maximum > kDriftRatio * c.rmax) {
                S->restart = 1;
                S->restarts += 1;
            }
            S->rmax = maximum;
            S->window_rmax = maximum;
        }
    }
    // out of budget: the next direction would never be used
    if (S->status == kRunning && S->iterations >= S->max_iterations)
        S->status = kStopped;
}

// Check and decision of a small grid in one launch, four launches beside its V-cycle instead of five: one workgroup, a
// 256-thread group per tile, the sums in the order of the two launches.  61 x 47 (3 tiles) 6% per solve; with 16 tiles in
// four rounds a check on one compute unit costs what the launch saves (128 x 128: 4341 us against 4323), so only where
// one round takes them all.
constexpr int kSmallTiles = 4;
__global__ __launch_bounds__(kSmallTiles * kNT) void k_check_small(GridDev g, int columns, int tiles)
{
    __shared__ double lds[2][kSmallTiles * kNT / 64];
    const int lane = threadIdx.x & 63;
    const bool mine = lane < tiles;
    const int st = g.S->status;
    double t[2] = {mine ? load_partial(g.fold_up, 2 * lane) : 0.0, mine ? load_partial(g.fold_up, 2 * lane + 1) : 0.0};
    if (st != kRunning)
        return;
    t[0] = wave_sum(t[0]);
    t[1] = wave_max(t[1]);
    const Recurrence c = recurrence(g.S, t);
    __syncthreads();   // every wavefront has read the scalar block before decide() changes it
    double e[2] = {0.0, 0.0};
    if (c.verify) {   // the same in every thread
        const int thread = threadIdx.x & (kNT - 1), tile = threadIdx.x / kNT;
        double sum = 0.0, m = 0.0;
        if (tile < tiles)
            true_residual(g, tile4(g, tile % columns, tile / columns, thread), sum, m);
        sum = wave_sum(sum);
        m = wave_max(m);
        if (lane == 0) {
            lds[0][threadIdx.x >> 6] = sum;
            lds[1][threadIdx.x >> 6] = m;
        }
        __syncthreads();
        // lane k of the first wavefront collects tile k's sums
        if (threadIdx.x < kSmallTiles) {
#pragma unroll
            for (int i = 0; i < kNT / 64; ++i) {
                e[0] += lds[0][lane * (kNT / 64) + i];
                e[1] = fmax(e[1], lds[1][lane * (kNT / 64) + i]);
            }
        }
        if (threadIdx.x < 64) {
            e[0] = wave_sum(e[0]);
            e[1] = wave_max(e[1]);
        }
    }
    if (threadIdx.x == 0)
        decide(g, c, t, e);
}

// The update's residual norm; where it called for a check, the true residual's verdict as well.
struct FinishCheck {
    __device__ __forceinline__ void run(const GridDev& g, int nb, double* lds) const
    {
        PcgScalars* S = g.S;
        const int st = S->status;
        double t[2];
        Partials<kNT, 2, 1>().all(g.fold_up, g.fold_up_n, t, lds);
        if (st != kRunning)
            return;
        const Recurrence c = recurrence(S, t);
        __syncthreads();   // every wavefront has read the scalar block before decide() changes it
        double e[2] = {0.0, 0.0};
        if (c.verify)
            Partials<kNT, 2, 1>().all(g.partials_tr, nb, e, lds);
        if (threadIdx.x == 0)
            decide(g, c, t, e);
    }
};

template <bool CLOSE> struct FinishDivergence {
    __device__ __forceinline__ void run(const GridDev& g, int nb, double* lds) const
    {
        if (CLOSE && g.S->status == kRunning)
            return;
        const double t = finish_max<kNT>(g.partials_tr, nb, 1, 0, lds);
        if (threadIdx.x == 0)
            g.S->div_max = t;
    }
};

// ------------------------------------------------------------------------------------------
// launches: one grid
// ------------------------------------------------------------------------------------------
template <class Op, int G> __global__ __launch_bounds__(kNT) void k_cells(GridDev g)
{
    Op().template run<G>(g, Block{(int)blockIdx.x, (int)blockIdx.y, (int)gridDim.x});
}

template <class Op> __global__ __launch_bounds__(kNT) void k_finish(GridDev g, int nb)
{
    __shared__ double lds[2 * kNT / 64];
    Op().run(g, nb, lds);
}

// Large grids: one workgroup reduces the per-block partials (NC components, the first NSUM summed) into
// out[0 .. NC), in the order every consumer workgroup would otherwise repeat over all blocks.
template <int NC, int NSUM>
__global__ __launch_bounds__(kNT) void k_fold_partials(const double* partials, int nb, double* out)
{
    __shared__ double lds[NC * kNT / 64];
    double t[NC];
    Partials<kNT, NC, NSUM>().all(partials, nb, t, lds);
    if (threadIdx.x == 0)
#pragma unroll
        for (int c = 0; c < NC; ++c)
            out[c] = t[c];
}

// ------------------------------------------------------------------------------------------
// launches: many grids.  A small grid's kernel leaves most of the chip idle and costs its launch; one launch over
// the tiles of all of them costs little more than one grid's.
// ------------------------------------------------------------------------------------------
template <class Op> __global__ __launch_bounds__(kNT) void k_cells_batch(const BatchItem* __restrict__ items,
    const int* __restrict__ item, const int* __restrict__ first)
{
    const int i = item[blockIdx.x];
    const int local = (int)blockIdx.x - first[i];
    const GridDev g = items[i].g;
    const int columns = (g.W + kTX - 1) / kTX;
    const int row = local / columns;
    Op().template run<1>(g, Block{local - row * columns, row, columns});
}

template <class Op> __global__ __launch_bounds__(kNT) void k_finish_batch(const BatchItem* __restrict__ items,
    const int* __restrict__ list)
{
    __shared__ double lds[2 * kNT / 64];
    const GridDev g = items[list[blockIdx.x]].g;
    Op().run(g, g.fold_up_n, lds);
}

__global__ __launch_bounds__(kCoarsenThreads) void k_coarsen_batch(const BatchItem* __restrict__ items,
    const int* __restrict__ item, const int* __restrict__ first, int level)
{
    const int i = item[blockIdx.x];
    const int local = (int)blockIdx.x - first[i];
    const ChainLevel L = items[i].coarsen[level];
    const int columns = (L.cw + kTX - 1) / kTX;
    const int row = local / columns;
    coarsen_tile(L, local - row * columns, row);
}

__global__ void k_init_batch(const BatchItem* __restrict__ items, const int* __restrict__ list, int n)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) {
        const BatchItem& I = items[list[k]];
        init_scalars(I.g.S, I.tol, I.max_iterations, I.rel_tol);
    }
}

__global__ void k_scalars_batch(const BatchItem* __restrict__ items, const int* __restrict__ list, int n, PcgScalars* out)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n)
        out[k] = *items[list[k]].g.S;
}

template <class Op> void launch_cells_batch(hipStream_t st, const BatchItem* items, const BatchPart& part)
{
    if (part.blocks > 0)
        hipLaunchKernelGGL(k_cells_batch<Op>, dim3(part.blocks), dim3(kNT), 0, st, items, part.item, part.first);
}

template <class Op> void launch_finish_batch(hipStream_t st, const BatchItem* items, const int* list, int n)
{
    if (n > 0)
        hipLaunchKernelGGL(k_finish_batch<Op>, dim3(n), dim3(kNT), 0, st, items, list);
}

template <class Op> void launch_cells(hipStream_t st, const GridDev& g)
{
    const int G = pcg_groups(g.W, g.H);
    const dim3 grid((g.W + kTX - 1) / kTX, ((g.H + kTY - 1) / kTY + G - 1) / G);
    if (G == 1)
        hipLaunchKernelGGL((k_cells<Op, 1>), grid, dim3(kNT), 0, st, g);
    else
        hipLaunchKernelGGL((k_cells<Op, 4>), grid, dim3(kNT), 0, st, g);
}

template <class Op> void launch_finish(hipStream_t st, const GridDev& g)
{
    hipLaunchKernelGGL(k_finish<Op>, dim3(1), dim3(kNT), 0, st, g, pcg_blocks(g.W, g.H));
}

// Where the partials are reduced in place of every consumer: elsewhere `out` is the producer's own (a grid of one tile
// has a single partial as well).
template <int NC, int NSUM> void fold(hipStream_t st, const GridDev& g, const double* partials, double* out)
{
    if (out != partials)
        hipLaunchKernelGGL((k_fold_partials<NC, NSUM>), dim3(1), dim3(kNT), 0, st, partials, pcg_blocks(g.W, g.H), out);
}

}  // namespace

// Tiles per workgroup: a consumer workgroup reads every producer workgroup's partial, blocks^2 loads in all, which shows
// past about a thousand workgroups; four tiles each keep a 2048 x 2048 grid at 1024.  k_fold_partials takes over beyond.
// A single row of tiles leaves three of four empty: 100000 x 16 projects in 3190 us with four and 2970 with one, 60000 x 32
// (two rows) in 5190 and 5340.
int pcg_groups(int W, int H)
{
    const int rows = (H + kTY - 1) / kTY;
    return rows > 1 && (size_t)((W + kTX - 1) / kTX) * rows > 1024 ? 4 : 1;
}
int pcg_blocks(int W, int H)
{
    return ((W + kTX - 1) / kTX) * (((H + kTY - 1) / kTY + pcg_groups(W, H) - 1) / pcg_groups(W, H));
}

void launch_init_scalars(hipStream_t st, PcgScalars* S, double tol, int max_iterations, double rel_tol)
{
    hipLaunchKernelGGL(k_init_scalars, dim3(1), dim3(64), 0, st, S, tol, max_iterations, rel_tol);
}

void launch_merge_failure(hipStream_t st, const PcgScalars* from, PcgScalars* S)
{
    hipLaunchKernelGGL(k_merge_failure, dim3(1), dim3(64), 0, st, from, S);
}

// A tile's halo is a sixth of its cells, and their components are read again: past twelve components on a large grid the
// densities take a launch of their own (a capillary force with 20 + 20 components: 1920 x 1080 279 us against 305 in one
// launch, 8 + 8 199 against 205, 1024^2 161 against 166; a small grid's launch costs more than it saves, 300 x 200 53
// against 49).
void launch_coefficients(hipStream_t st, const GridDev& g)
{
    if (g.nl + g.ng > 12 && batch_cell_blocks(g.W, g.H) >= 1024) {
        launch_density(st, g);
        launch_cells<Coefficients<false>>(st, g);
    } else {
        launch_cells<Coefficients<true>>(st, g);
    }
}

void launch_coarsen(hipStream_t st, const ChainLevel& level)
{
    hipLaunchKernelGGL(k_coarsen, dim3(batch_coarsen_blocks(level)), dim3(kCoarsenThreads), 0, st, level);
}

void launch_project_setup(hipStream_t st, const GridDev& g)
{
    launch_cells<Rhs>(st, g);
    fold<1, 1>(st, g, g.partials_ad, g.fold_ad);
    launch_cells<Predict>(st, g);
    fold<2, 1>(st, g, g.partials_up, g.fold_up);
    launch_cells<InitialResidual>(st, g);
    launch_finish<FinishSetup>(st, g);
}

void launch_project_end(hipStream_t st, const GridDev& g)
{
    launch_cells<FinalSum>(st, g);
    fold<1, 1>(st, g, g.partials_ad, g.fold_ad);
    launch_cells<CorrectVelocity>(st, g);
    launch_cells<MaxDivergence<true>>(st, g);
    launch_finish<FinishDivergence<true>>(st, g);
}

// A tile per workgroup on every grid: only the finish reads the partials (1100 x 1050 cells 19.8 us, 20.4 with the
// solve's four).
void launch_max_divergence(hipStream_t st, const GridDev& g)
{
    const dim3 tiles((g.W + kTX - 1) / kTX, (g.H + kTY - 1) / kTY);
    hipLaunchKernelGGL((k_cells<MaxDivergence<false>, 1>), tiles, dim3(kNT), 0, st, g);
    hipLaunchKernelGGL(k_finish<FinishDivergence<false>>, dim3(1), dim3(kNT), 0, st, g, (int)(tiles.x * tiles.y));
}

void launch_pcg_direction_ad(hipStream_t st, const GridDev& g, int flexible)
{
    if (flexible)
        launch_cells<DirectionAd<true>>(st, g);
    else
        launch_cells<DirectionAd<false>>(st, g);
    fold<1, 1>(st, g, g.partials_ad, g.fold_ad);
}

void launch_pcg_update(hipStream_t st, const GridDev& g)
{
    launch_cells<Update>(st, g);
    fold<2, 1>(st, g, g.partials_up, g.fold_up);
}

void launch_pcg_check(hipStream_t st, const GridDev& g)
{
    const int columns = (g.W + kTX - 1) / kTX, tiles = columns * ((g.H + kTY - 1) / kTY);
    if (tiles <= kSmallTiles) {
        hipLaunchKernelGGL(k_check_small, dim3(1), dim3(kSmallTiles * kNT), 0, st, g, columns, tiles);
        return;
    }
    launch_cells<Check>(st, g);
    launch_finish<FinishCheck>(st, g);
}

void launch_pcg_rz(hipStream_t st, const GridDev& g, int flexible)
{
    if (flexible) {
        launch_cells<Rz<true>>(st, g);
        fold<5, 5>(st, g, g.partials, g.fold_rz);
    } else {
        launch_cells<Rz<false>>(st, g);
        fold<3, 3>(st, g, g.partials, g.fold_rz);
    }
}

void launch_precond_diag(hipStream_t st, const GridDev& g) { launch_cells<PrecondDiag>(st, g); }

int batch_cell_blocks(int W, int H) { return ((W + kTX - 1) / kTX) * ((H + kTY - 1) / kTY); }
int batch_coarsen_blocks(const ChainLevel& level)
{
    return ((level.cw + kTX - 1) / kTX) * ((level.ch + kCoarsenY - 1) / kCoarsenY);
}

void launch_batch_init(hipStream_t st, const BatchItem* items, const int* list, int n)
{
    if (n > 0)
        hipLaunchKernelGGL(k_init_batch, dim3((n + 63) / 64), dim3(64), 0, st, items, list, n);
}

void launch_batch_coefficients(hipStream_t st, const BatchItem* items, const BatchPart& part)
{
    launch_cells_batch<Coefficients<true>>(st, items, part);
}

void launch_batch_coarsen(hipStream_t st, const BatchItem* items, const BatchPart& part, int level)
{
    if (part.blocks > 0)
        hipLaunchKernelGGL(k_coarsen_batch, dim3(part.blocks), dim3(kCoarsenThreads), 0, st, items, part.item, part.first,
            level);
}

void launch_batch_setup(hipStream_t st, const BatchItem* items, const BatchPart& part, const int* list, int n)
{
    launch_cells_batch<Rhs>(st, items, part);
    launch_cells_batch<Predict>(st, items, part);
    launch_cells_batch<InitialResidual>(st, items, part);
    launch_finish_batch<FinishSetup>(st, items, list, n);
}

void launch_batch_step(hipStream_t st, const BatchItem* items, const BatchPart& part, const int* list, int n)
{
    launch_cells_batch<DirectionAd<false>>(st, items, part);
    launch_cells_batch<Update>(st, items, part);
    launch_cells_batch<Check>(st, items, part);
    launch_finish_batch<FinishCheck>(st, items, list, n);
}

void launch_batch_precond_diag(hipStream_t st, const BatchItem* items, const BatchPart& part)
{
    launch_cells_batch<PrecondDiag>(st, items, part);
}

void launch_batch_rz(hipStream_t st, const BatchItem* items, const BatchPart& part)
{
    launch_cells_batch<Rz<false>>(st, items, part);
}

void launch_batch_end(hipStream_t st, const BatchItem* items, const BatchPart& part, const int* list, int n)
{
    launch_cells_batch<FinalSum>(st, items, part);
    launch_cells_batch<CorrectVelocity>(st, items, part);
    launch_cells_batch<MaxDivergence<true>>(st, items, part);
    launch_finish_batch<FinishDivergence<true>>(st, items, list, n);
}

void launch_batch_scalars(hipStream_t st, const BatchItem* items, const int* list, int n, PcgScalars* out)
{
    if (n > 0)
        hipLaunchKernelGGL(k_scalars_batch, dim3((n + 63) / 64), dim3(64), 0, st, items, list, n, out);
}

}  // namespace fsim
