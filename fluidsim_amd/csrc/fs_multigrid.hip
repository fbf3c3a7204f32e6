// fs_multigrid.hip -- the multigrid preconditioner of PressureMultigrid.cpp on gfx950.
//
// A cycle's level smoothers are in fs_rows.hip: on the way down the sweeps, the residual and its
// transpose-of-bilinear restriction in one launch (or the restriction apart, k_res_restrict), on the way up
// the prolongation and the reversed sweeps in one.
// The deepest levels (up to 64 x 64, as LDS allows) and the coarse solve run in k_mg_tail, one
// 1024-thread workgroup with every array in LDS.  The pinned coarse system (PressureMultigrid.cpp:
// 300-384) is factored bit-exactly by k_coarse_factor, which also forms its inverse so the per-cycle
// coarse solve is a 63 x 63 matrix-vector product instead of two serial substitutions.
//
// Smoothers divide by the sum of the four face conductances formed in FP32 (one rcp); pre- and
// post-smoothing use the same diagonal, so the V-cycle stays symmetric.
#include "fs_kernels.hpp"
#include "fs_mg_device.hpp"

#include <math.h>

#include <algorithm>
#include <type_traits>

namespace fsim {

namespace {

constexpr int kNT = 256;

// ---------------------------------------------------------------------------------------------
// Residual + restriction (restrictResidual, PressureMultigrid.cpp:233-276).  A coarse tile of
// CTX x CTY cells gathers fine taps in [2c - 2, 2c + 3]; the fine residual is formed in LDS on
// that window (plus a one-cell ring of solution values).
// ---------------------------------------------------------------------------------------------
template <int CTX, int CTY, class C = float, class V = float, class VC = float>
__global__ __launch_bounds__(kNT) void k_res_restrict(LevelViewT<C, V> F, int cur, const V* rhs, const double* shift,
    LevelViewT<C, VC> Cl, AxisRestrict rx, AxisRestrict ry, const int* status)
{
    constexpr int LX = 2 * CTX + 6, LY = 2 * CTY + 6;
    __shared__ float s_sol[LY * LX];
    __shared__ float s_right[LY * LX];
    __shared__ float s_down[LY * LX];
    __shared__ float s_res[LY * LX];
    __shared__ int s_rxc[CTX], s_rxi[CTX * 4], s_ryc[CTY], s_ryi[CTY * 4];
    __shared__ float s_rxw[CTX * 4], s_ryw[CTY * 4];
    const int w = F.w, h = F.h, s = F.s;
    int bx, by;
    xcd_tile((Cl.w + CTX - 1) / CTX, (Cl.h + CTY - 1) / CTY, bx, by);
    const int cx0 = bx * CTX, cy0 = by * CTY;
    const int fx0 = 2 * cx0 - 3, fy0 = 2 * cy0 - 3;
    const V* sol = F.sol[cur];
    constexpr int NE = LX * LY;
    constexpr int LOADS = (NE + kNT - 1) / kNT;
    float vs[LOADS], vr[LOADS], vd[LOADS], vb[LOADS];
    bool vin[LOADS];
#pragma unroll
    for (int it = 0; it < LOADS; ++it) {
        const int e = threadIdx.x + it * kNT;
        const int ly = e / LX, lx = e - ly * LX;
        const int x = fx0 + lx, y = fy0 + ly;
        vin[it] = e < NE && x >= 0 && x < w && y >= 0 && y < h;
        const int P = (min(max(y, 0), h - 1) + 1) * s + (min(max(x, 0), w - 1) + 1);
        vs[it] = ldv(sol[P]);
        vr[it] = ldv(F.right[P]);
        vd[it] = ldv(F.down[P]);
        vb[it] = ldv(rhs[P]);
    }
    // restriction tables of this coarse tile (missing taps: weight 0 at a valid LDS cell)
    int tc[2], ti[2][4];
    float tw[2][4];
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        const int e = threadIdx.x - a * CTX;  // threads [0, CTX) take x, [CTX, CTX + CTY) take y
        const bool isx = a == 0;
        const int n_axis = isx ? CTX : CTY;
        const int c = (isx ? cx0 : cy0) + min(max(e, 0), n_axis - 1);
        const int limit = isx ? Cl.w : Cl.h;
        const AxisRestrict& R = isx ? rx : ry;
        const int cc = min(c, limit - 1);
        const int n = R.count[cc];
        tc[a] = c < limit ? n : 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            ti[a][k] = R.index[cc * 4 + k];
            tw[a][k] = R.weight[cc * 4 + k];
        }
    }
    if (status && *status != kRunning)
        return;
    const double sh = shift ? *shift : 0.0;
#pragma unroll
    for (int it = 0; it < LOADS; ++it) {
        const int e = threadIdx.x + it * kNT;
        if (e < NE) {
            s_sol[e] = vin[it] ? vs[it] : 0.f;
            s_right[e] = vin[it] ? vr[it] : 0.f;
            s_down[e] = vin[it] ? vd[it] : 0.f;
            s_res[e] = vin[it] ? (shift ? (float)((double)vb[it] - sh) : vb[it]) : 0.f;
        }
    }
    if (threadIdx.x < CTX) {
        const int e = threadIdx.x;
        s_rxc[e] = tc[0];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const bool on = k < tc[0];
            s_rxi[e * 4 + k] = on ? ti[0][k] - fx0 : 1;
            s_rxw[e * 4 + k] = on ? tw[0][k] : 0.f;
        }
    } else if (threadIdx.x < CTX + CTY) {
        const int e = threadIdx.x - CTX;
        s_ryc[e] = tc[1];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const bool on = k < tc[1];
            s_ryi[e * 4 + k] = on ? ti[1][k] - fy0 : 1;
            s_ryw[e * 4 + k] = on ? tw[1][k] : 0.f;
        }
    }
    __syncthreads();
    // residual in place of the rhs on the inner window
    for (int e = threadIdx.x; e < (LX - 2) * (LY - 2); e += kNT) {
        const int ly = 1 + e / (LX - 2), lx = 1 + e % (LX - 2);
        const int x = fx0 + lx, y = fy0 + ly;
        if (x < 0 || x >= w || y < 0 || y >= h)
            continue;
        const int i = ly * LX + lx;
        const float c = s_sol[i];
        const float product = (s_right[i - 1] * (c - s_sol[i - 1]) + s_right[i] * (c - s_sol[i + 1])) +
                              (s_down[i - LX] * (c - s_sol[i - LX]) + s_down[i] * (c - s_sol[i + LX]));
        // a cell without conductance (solid masks only) is not restricted: the V-cycle stays symmetric
        const bool active = (s_right[i - 1] + s_right[i]) + (s_down[i - LX] + s_down[i]) > 0.f;
        s_res[i] = active ? s_res[i] - product : 0.f;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < CTX * CTY; e += kNT) {
        const int ly = e / CTX, lx = e - ly * CTX;
        const int x = cx0 + lx, y = cy0 + ly;
        if (x >= Cl.w || y >= Cl.h)
            continue;
        // four taps per axis (missing taps carry weight 0 and a valid index): 16 independent reads
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
        Cl.rhs[(y + 1) * Cl.s + x + 1] = stv<VC>(value);
    }
}

// ---------------------------------------------------------------------------------------------
// Coarse factorisation (factorCoarsest, PressureMultigrid.cpp:300-345) and inverse.
// Right-looking updates applied column by column: every entry receives its subtractions in the
// same k order as the reference's row loop, so the factor is bit-identical to it.
// ---------------------------------------------------------------------------------------------
constexpr int kMaxCoarse = 63;
constexpr int kFactorThreads = 256;

__global__ __launch_bounds__(kFactorThreads) void k_coarse_factor(int w, int h, const double* right,
    const double* down, double* factor, float* ginv, int n, PcgScalars* S, int pin)
{
    __shared__ double a[kMaxCoarse * kMaxCoarse];   // Cholesky working matrix (lower triangle)
    __shared__ double m[kMaxCoarse * kMaxCoarse];   // Gauss-Jordan working matrix
    __shared__ double q[kMaxCoarse];
    __shared__ double assembled[kMaxCoarse];        // diagonal before elimination (pinning bound)
    __shared__ int failed;
    const int s = w + 2;
    const int tid = threadIdx.x;
    const int tc = tid & 63, tr = tid >> 6;
    constexpr int RSTEP = kFactorThreads / 64;
    for (int e = tid; e < n * n; e += kFactorThreads) {
        a[e] = 0.0;
        m[e] = 0.0;
    }
    if (tid == 0)
        failed = 0;
    __syncthreads();
    for (int cell = 1 + tid; cell <= n; cell += kFactorThreads) {
        const int x = cell % w, y = cell / w;
        const int i = (y + 1) * s + x + 1;
        const int row = cell - 1;
        const double diag = right[i - 1] + right[i] + down[i - s] + down[i];
        a[row * n + row] = diag;
        m[row * n + row] = diag;
        assembled[row] = diag;
        if (x > 0 && cell - 1 > 0) {
            a[row * n + row - 1] = -right[i - 1];
            m[row * n + row - 1] = -right[i - 1];
            m[(row - 1) * n + row] = -right[i - 1];
        }
        if (y > 0 && cell - w > 0) {
            a[row * n + row - w] = -down[i - s];
            m[row * n + row - w] = -down[i - s];
            m[(row - w) * n + row] = -down[i - s];
        }
    }
    __syncthreads();
    // Column k: pivot sqrt, quotients L[i][k] = a[i][k] / pivot into q (one barrier), then the trailing
    // update a[i][c] -= L[i][k] L[c][k] (second barrier).  Each entry still receives its subtractions
    // in increasing k, as the reference's row loop applies them.
    unsigned long long pinned = 0ull;   // the same in every thread
    for (int k = 0; k < n; ++k) {
        const double v = a[k * n + k];
        // a pinned unknown gets a zero column: the trailing update below then subtracts exact zeros
        const bool pin_k = pin && isfinite(v) && fabs(v) <= kPinRatio * assembled[k];
        if (!pin_k && (v <= 0.0 || !isfinite(v))) {
            if (tid == 0)
                failed = 1;
            break;
        }
        if (pin_k)
            pinned |= 1ull << k;
        const double pivot = pin_k ? 0.0 : sqrt(v);
        if (tid > k && tid < n) {
            const double l = pin_k ? 0.0 : a[tid * n + k] / pivot;
            a[tid * n + k] = l;
            q[tid] = l;
        }
        __syncthreads();
        if (tid == 0)
            a[k * n + k] = pivot;  // after the barrier: every thread has read the unfactored diagonal
        {
            // rows i = k+1+tr+4m; gather every operand first, then write (independent LDS accesses)
            const int c = k + 1 + tc;
            const int cc = min(c, n - 1);
            const double qc = q[cc];
            constexpr int M = (kMaxCoarse + RSTEP - 1) / RSTEP;
            double li[M], av[M];
#pragma unroll
            for (int mm = 0; mm < M; ++mm) {
                const int ic = min(k + 1 + tr + RSTEP * mm, n - 1);
                li[mm] = q[ic];
                av[mm] = a[ic * n + cc];
            }
#pragma unroll
            for (int mm = 0; mm < M; ++mm) {
                const int i = k + 1 + tr + RSTEP * mm;
                if (i < n && c <= i)
                    a[i * n + c] = av[mm] - li[mm] * qc;
            }
        }
        __syncthreads();
    }
    __syncthreads();
    if (failed) {
        if (tid == 0 && S) {
            S->mg_failed = 1;
            if (S->status == kRunning)
                S->status = kFailed;
        }
        return;
    }
    for (int e = tid; e < n * n; e += kFactorThreads) {
        const int r = e / n, c = e - r * n;
        factor[e] = c <= r && !((pinned >> r) & 1ull) ? a[e] : 0.0;
    }
    if (!ginv || pinned)
        return;   // the Gauss-Jordan inverse below assumes no pinned unknown (callers pass no ginv with pin)
    // In-place Gauss-Jordan inversion of the (SPD, so pivot-free) pinned matrix.
    for (int k = 0; k < n; ++k) {
        const double p = m[k * n + k];
        __syncthreads();  // every thread holds the pivot before row k is rewritten
        if (tid < n) {
            q[tid] = m[tid * n + k];
            m[k * n + tid] = tid == k ? 1.0 / p : m[k * n + tid] / p;
        }
        __syncthreads();
        {
            constexpr int M = (kMaxCoarse + RSTEP - 1) / RSTEP;
            const int tcc = min(tc, n - 1);
            const double pk = m[k * n + tcc];
            double fv[M], mv[M];
#pragma unroll
            for (int mm = 0; mm < M; ++mm) {
                const int ic = min(tr + RSTEP * mm, n - 1);
                fv[mm] = q[ic];
                mv[mm] = m[ic * n + tcc];
            }
#pragma unroll
            for (int mm = 0; mm < M; ++mm) {
                const int i = tr + RSTEP * mm;
                if (i < n && i != k && tc < n)
                    m[i * n + tc] = tc == k ? -fv[mm] / p : mv[mm] - fv[mm] * pk;
            }
        }
        __syncthreads();
    }
    for (int e = tid; e < n * n; e += kFactorThreads)
        ginv[e] = (float)m[e];
}

// ---------------------------------------------------------------------------------------------
// Inverse of the pinned coarse matrix for the per-cycle coarse solve (the hot path).  Goodnight's
// sweep operator, in place: the matrix lives in registers, column j in lane j and rows split over sixteen wavefronts
// (4 per wavefront, so that a step's row updates are a short chain).  A wavefront sweeps its four pivots on its own rows
// and broadcasts the four scaled pivot rows through LDS (double-buffered, one barrier); the others then apply
// them in the same order, the pivot column read inside each wavefront by lane.  Bound by the serial chain: 63 pivots
// are 16 barriers and 63 divisions, 28 us on 8 x 8 cells (37 with a barrier and every thread's checks per pivot and
// the entries assembled by one dependent load each).  Pivots are the Schur complement diagonals (the squared Cholesky
// pivots); a non-positive or non-finite one marks the hierarchy failed exactly where the Cholesky factorisation would.
// ---------------------------------------------------------------------------------------------
constexpr int kSweepRows = 4;     // rows per wavefront
constexpr int kSweepWaves = 16;   // kSweepWaves x kSweepRows >= kMaxCoarse

// v as held by lane k (k uniform across the wavefront).
__device__ __forceinline__ double lane_value(double v, int k)
{
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, k);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), k);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

__device__ __forceinline__ void coarse_inverse(int w, int h, const double* right, const double* down, float* ginv, int n,
    PcgScalars* S, int pin)
{
    __shared__ double rowbuf[2][kSweepRows][64];
    __shared__ int verdict[2];         // of a wavefront's pivots: bit r pinned, bit 8 + r failed
    __shared__ double assembled[64];   // diagonal before elimination (pinning bound)
    const int s = w + 2;
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // pinned matrix entry (i, j) of unknowns i, j (cells i + 1, j + 1)
    double a[kSweepRows];
    // every entry of column j is one of its cell's four conductances: one round of loads
    const int cj = lane + 1;
    const int yj = cj / w, xj = cj - yj * w;
    const int pj = (min(yj, h - 1) + 1) * s + xj + 1;
    const double cl = right[pj - 1], cr = right[pj], cu = down[pj - s], cd = down[pj];
#pragma unroll
    for (int r = 0; r < kSweepRows; ++r) {
        const int ci = wv * kSweepRows + r + 1;
        const int yi = ci / w, xi = ci - yi * w;
        double v = 0.0;
        if (ci == cj)
            v = cl + cr + cu + cd;
        else if (yi == yj && (xi - xj == 1 || xj - xi == 1))
            v = -(xi > xj ? cr : cl);
        else if (xi == xj && (yi - yj == 1 || yj - yi == 1))
            v = -(yi > yj ? cd : cu);
        a[r] = ci <= n && cj <= n ? v : 0.0;
        if (ci == cj && ci <= n)
            assembled[lane] = v;
    }
    bool failed = false;
    // Solid masks: an unknown whose Schur pivot vanishes is pinned -- never swept, and its row and
    // column of the inverse are zero (the swept block is then the inverse of the other unknowns' matrix)
    unsigned long long pinned = 0ull;   // the same in every thread
    if (pin)
        __syncthreads();   // assembled[]
    // a[] of one wavefront after the sweep of pivot k, whose scaled row is t; b, the pivot column, lies in lane k
    auto update = [&](int k, double t, int own) {
        const bool mine = lane == k;
#pragma unroll
        for (int r = 0; r < kSweepRows; ++r) {
            const double b = lane_value(a[r], k);
            const double base = mine ? 0.0 : a[r];
            a[r] = r == own ? t : base - b * t;
        }
    };
    for (int kb = 0; kb * kSweepRows < n && !failed; ++kb) {
        const int buf = kb & 1, k0 = kb * kSweepRows;
        if (wv == kb) {
            int code = 0;
#pragma unroll
            for (int r0 = 0; r0 < kSweepRows; ++r0) {
                const int k = k0 + r0;
                if (k >= n || code >> 8)
                    break;
                const double d = lane_value(a[r0], k);
                if (pin && isfinite(d) && fabs(d) <= kPinRatio * assembled[k]) {
                    code |= 1 << r0;
                    continue;
                }
                if (!(d > 0.0) || !isfinite(d)) {
                    code |= 256 << r0;
                    break;
                }
                // lane k's own entry of a scaled row becomes 1 / d
                const double inv_d = 1.0 / d;
                const double t = lane == k ? inv_d : a[r0] * inv_d;
                rowbuf[buf][r0][lane] = t;
                update(k, t, r0);
            }
            if (lane == 0)
                verdict[buf] = code;
        }
        __syncthreads();
        double t[kSweepRows];
#pragma unroll
        for (int r0 = 0; r0 < kSweepRows; ++r0)
            t[r0] = rowbuf[buf][r0][lane];
        const int code = __builtin_amdgcn_readfirstlane(verdict[buf]);
        failed = code >> 8 != 0;   // the same in every thread: the whole block leaves together
        pinned |= (unsigned long long)(code & 255) << k0;
        if (wv != kb && !failed) {
#pragma unroll
            for (int r0 = 0; r0 < kSweepRows; ++r0)
                if (k0 + r0 < n && !(code >> r0 & 1))
                    update(k0 + r0, t[r0], -1);
        }
    }
    if (failed) {
        if (threadIdx.x == 0 && S) {
            S->mg_failed = 1;
            if (S->status == kRunning)
                S->status = kFailed;
        }
        return;
    }
#pragma unroll
    for (int r = 0; r < kSweepRows; ++r) {
        const int i = wv * kSweepRows + r;
        if (i < n && lane < n)
            ginv[i * n + lane] = ((pinned >> i) & 1ull) || ((pinned >> lane) & 1ull) ? 0.f : (float)a[r];
    }
}

__global__ __launch_bounds__(64 * kSweepWaves) void k_coarse_inverse(int w, int h, const double* right,
    const double* down, float* ginv, int n, PcgScalars* S, int pin)
{
    coarse_inverse(w, h, right, down, ginv, n, S, pin);
}

// Coarse end of the hierarchy rebuild: each level's cells coarsened, then its diagonal and FP32 copies,
// each phase workgroup-strided and closed by a barrier (which also makes this workgroup's global
// writes visible to its next phase); then the coarse inverse.
__device__ __forceinline__ void coarse_chain(const ChainDesc& C, float* ginv, int n, PcgScalars* S, int pin)
{
    for (int l = 0; l < C.levels; ++l) {
        const ChainLevel& L = C.lev[l];
        const int cells = L.cw * L.ch;
        for (int t = threadIdx.x; t < cells; t += 64 * kSweepWaves) {
            const int y = t / L.cw, x = t - y * L.cw;
            const double2 c = coarsen_cell(x, y, L.fw, L.fh, L.fcx, L.fcy, L.fright, L.fdown, L.cw, L.ch, L.ccx, L.ccy);
            const int i = (y + 1) * (L.cw + 2) + x + 1;
            L.cright[i] = c.x;
            L.cdown[i] = c.y;
        }
        __syncthreads();
        const int s = L.cw + 2;
        for (int t = threadIdx.x; t < cells; t += 64 * kSweepWaves) {
            const int y = t / L.cw, x = t - y * L.cw;
            const int i = (y + 1) * s + x + 1;
            level_diag_values(L.cright[i - 1], L.cright[i], L.cdown[i - s], L.cdown[i], L.invd32[i], L.right32[i],
                L.down32[i]);
        }
        __syncthreads();
    }
    if (n > 0)
        coarse_inverse(C.w, C.h, C.right, C.down, ginv, n, S, pin);
}

__global__ __launch_bounds__(64 * kSweepWaves) void k_coarse_chain(const ChainDesc C, float* ginv, int n,
    PcgScalars* S, int pin)
{
    coarse_chain(C, ginv, n, S, pin);
}

// ---------------------------------------------------------------------------------------------
// Coarse tail: the deepest levels and the coarse solve in one workgroup.
// ---------------------------------------------------------------------------------------------
constexpr int kTailThreads = 1024;

struct TailArrays {
    float* right;
    float* down;
    float* rhs;
    float* sol;
    float* res;
    int* pxf; int* pxs; float* pxw;
    int* pyf; int* pys; float* pyw;
    int* rxc; int* rxi; float* rxw;
    int* ryc; int* ryi; float* ryw;
};

__device__ __forceinline__ TailArrays tail_arrays(float* lds, const TailLevel& T)
{
    TailArrays A;
    const int ps = T.s * (T.h + 2);
    float* p = lds + T.lds_arrays;
    A.right = p;
    A.down = p + ps;
    A.rhs = p + 2 * ps;
    A.sol = p + 3 * ps;
    A.res = p + 4 * ps;
    float* t = lds + T.lds_tables;
    A.pxf = (int*)t; t += T.w;
    A.pxs = (int*)t; t += T.w;
    A.pxw = t; t += T.w;
    A.pyf = (int*)t; t += T.h;
    A.pys = (int*)t; t += T.h;
    A.pyw = t; t += T.h;
    A.rxc = (int*)t; t += T.cw;
    A.rxi = (int*)t; t += 4 * T.cw;
    A.rxw = t; t += 4 * T.cw;
    A.ryc = (int*)t; t += T.ch;
    A.ryi = (int*)t; t += 4 * T.ch;
    A.ryw = t;
    return A;
}

// Tail loops: a thread owns at most ITER items of a level (ITER chosen per level from its size, so a
// small level does not execute the unrolled work of a large one), and a wavefront whose first item is
// past the end skips the loop body entirely.  Every LDS read goes through a clamped (valid) index and
// only the stores are predicated, so the reads of all items issue together.
constexpr int kTailIter = 4;   // at most 4 * 1024 items per phase (the tail selection guarantees it)

__device__ __forceinline__ bool wave_has_items(int items) { return (int)(threadIdx.x & ~63u) < items; }

// t / d for 0 <= t < 2^22 without an integer division: (t + 1/2) / d lies at least 1/(2d) from an
// integer, and the float product's error is below (t / d) 2^-22 < 1/(2d).
__device__ __forceinline__ int tail_div(int t, float inv_d) { return (int)(((float)t + 0.5f) * inv_d); }

// `sweeps` (uniform, 1..4) red-black sweeps of one tail level with each thread's cells, conductances, rhs
// and 1/diagonal held in registers across all the half-sweeps: a half-sweep is four LDS reads, one write
// and a barrier per item.
template <int ITER>
__device__ void tail_smooth4_n(const TailLevel& T, const TailArrays& A, int reverse, int from_zero, int sweeps)
{
    const int w = T.w, h = T.h, s = T.s;
    const int pairs = (w + 1) >> 1;
    const int items = pairs * h;
    const bool active = wave_has_items(items);
    const float inv_pairs = 1.0f / (float)pairs;
    int idx[2][ITER];
    bool on[2][ITER];
    float wl[2][ITER], wr[2][ITER], wu[2][ITER], wd[2][ITER], rb[2][ITER], inv[2][ITER];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
#pragma unroll
        for (int it = 0; it < ITER; ++it) {
            const int t = min((int)threadIdx.x + it * kTailThreads, items - 1);
            const int y = tail_div(t, inv_pairs);
            const int x = 2 * (t - y * pairs) + ((c ^ y) & 1);
            on[c][it] = active && (int)threadIdx.x + it * kTailThreads < items && x < w;
            const int i = (y + 1) * s + min(x, w - 1) + 1;
            idx[c][it] = i;
            wl[c][it] = A.right[i - 1];
            wr[c][it] = A.right[i];
            wu[c][it] = A.down[i - s];
            wd[c][it] = A.down[i];
            rb[c][it] = A.rhs[i];
        }
    }
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int it = 0; it < ITER; ++it)
            inv[c][it] = inv_or_zero((wl[c][it] + wr[c][it]) + (wu[c][it] + wd[c][it]));
    for (int k = 0; k < sweeps; ++k) {
        for (int pass = 0; pass < 2; ++pass) {
            const int color = reverse ? 1 - pass : pass;
            const bool neighbours = !(from_zero && k == 0 && pass == 0);
            if (active) {
                float v[ITER];
#pragma unroll
                for (int it = 0; it < ITER; ++it) {
                    const int i = idx[color][it];
                    float acc = rb[color][it];
                    const float n = (wl[color][it] * A.sol[i - 1] + wr[color][it] * A.sol[i + 1]) +
                                    (wu[color][it] * A.sol[i - s] + wd[color][it] * A.sol[i + s]);
                    if (neighbours)
                        acc += n;
                    v[it] = acc * inv[color][it];
                }
#pragma unroll
                for (int it = 0; it < ITER; ++it)
                    if (on[color][it])
                        A.sol[idx[color][it]] = v[it];
            }
            __syncthreads();
        }
    }
}

// `sweeps` sweeps (PressureMultigrid.cpp:204-231 applied four times in the reference's cycle); reverse =
// post-smoothing colour order.
__device__ void tail_smooth4(const TailLevel& T, const TailArrays& A, int reverse, int from_zero, int sweeps)
{
    const int items = ((T.w + 1) >> 1) * T.h;
    if (items <= kTailThreads)
        tail_smooth4_n<1>(T, A, reverse, from_zero, sweeps);
    else if (items <= 2 * kTailThreads)
        tail_smooth4_n<2>(T, A, reverse, from_zero, sweeps);
    else
        tail_smooth4_n<kTailIter>(T, A, reverse, from_zero, sweeps);
}

template <int ITER> __device__ void tail_residual_n(const TailLevel& T, const TailArrays& F)
{
    const int w = T.w, h = T.h, s = T.s;
    const int cells = w * h;
    if (!wave_has_items(cells))
        return;
    const float inv_w = 1.0f / (float)w;
    float rv[ITER];
    int idx[ITER];
    bool on[ITER];
#pragma unroll
    for (int it = 0; it < ITER; ++it) {
        const int e = min((int)threadIdx.x + it * kTailThreads, cells - 1);
        on[it] = (int)threadIdx.x + it * kTailThreads < cells;
        const int y = tail_div(e, inv_w), x = e - y * w;
        const int i = (y + 1) * s + x + 1;
        idx[it] = i;
        const float c = F.sol[i];
        const float product = (F.right[i - 1] * (c - F.sol[i - 1]) + F.right[i] * (c - F.sol[i + 1])) +
                              (F.down[i - s] * (c - F.sol[i - s]) + F.down[i] * (c - F.sol[i + s]));
        const bool active = (F.right[i - 1] + F.right[i]) + (F.down[i - s] + F.down[i]) > 0.f;
        rv[it] = active ? F.rhs[i] - product : 0.f;   // cells without conductance are not restricted
    }
#pragma unroll
    for (int it = 0; it < ITER; ++it)
        if (on[it])
            F.res[idx[it]] = rv[it];
}

template <int ITER> __device__ void tail_restrict_n(const TailLevel& T, const TailArrays& F, const TailLevel& Cn,
    const TailArrays& Cd)
{
    // missing taps carry weight 0 and index -1, which addresses the zero halo
    const int s = T.s;
    const int cells_c = Cn.w * Cn.h;
    if (!wave_has_items(cells_c))
        return;
    const float inv_cw = 1.0f / (float)Cn.w;
    float val[ITER];
    int dst[ITER];
#pragma unroll
    for (int it = 0; it < ITER; ++it) {
        const int e = min((int)threadIdx.x + it * kTailThreads, cells_c - 1);
        const int y = tail_div(e, inv_cw), x = e - y * Cn.w;
        float value = 0.f;
#pragma unroll
        for (int iy = 0; iy < 4; ++iy) {
            const float* row = F.res + (F.ryi[y * 4 + iy] + 1) * s + 1;
            float horizontal = 0.f;
#pragma unroll
            for (int ix = 0; ix < 4; ++ix)
                horizontal += F.rxw[x * 4 + ix] * row[F.rxi[x * 4 + ix]];
            value += F.ryw[y * 4 + iy] * horizontal;
        }
        val[it] = value;
        dst[it] = (y + 1) * Cn.s + x + 1;
    }
#pragma unroll
    for (int it = 0; it < ITER; ++it)
        if ((int)threadIdx.x + it * kTailThreads < cells_c)
            Cd.rhs[dst[it]] = val[it];
}

__device__ void tail_residual_restrict(const TailLevel& T, const TailArrays& F, const TailLevel& Cn,
    const TailArrays& Cd)
{
    const int cells = T.w * T.h;
    if (cells <= kTailThreads)
        tail_residual_n<1>(T, F);
    else if (cells <= 2 * kTailThreads)
        tail_residual_n<2>(T, F);
    else
        tail_residual_n<kTailIter>(T, F);
    __syncthreads();
    if (Cn.w * Cn.h <= kTailThreads)
        tail_restrict_n<1>(T, F, Cn, Cd);
    else
        tail_restrict_n<2>(T, F, Cn, Cd);
    __syncthreads();
}

template <int ITER> __device__ void tail_prolong_n(const TailLevel& T, const TailArrays& F, const TailLevel& Cn,
    const TailArrays& Cd)
{
    const int w = T.w, h = T.h;
    const int cells = w * h;
    if (!wave_has_items(cells))
        return;
    const float inv_w = 1.0f / (float)w;
    float add[ITER], cur[ITER];
    int idx[ITER];
    bool on[ITER];
#pragma unroll
    for (int it = 0; it < ITER; ++it) {
        const int e = min((int)threadIdx.x + it * kTailThreads, cells - 1);
        on[it] = (int)threadIdx.x + it * kTailThreads < cells;
        const int y = tail_div(e, inv_w), x = e - y * w;
        const float wy = F.pyw[y];
        const float* top = Cd.sol + (F.pyf[y] + 1) * Cn.s + 1;
        const float* bottom = Cd.sol + (F.pys[y] + 1) * Cn.s + 1;
        const int a0 = F.pxf[x], a1 = F.pxs[x];
        const float wx = F.pxw[x];
        const float a = (1.f - wx) * top[a0] + wx * top[a1];
        const float b = (1.f - wx) * bottom[a0] + wx * bottom[a1];
        add[it] = (1.f - wy) * a + wy * b;
        idx[it] = (y + 1) * T.s + x + 1;
        cur[it] = F.sol[idx[it]];
    }
#pragma unroll
    for (int it = 0; it < ITER; ++it)
        if (on[it])
            F.sol[idx[it]] = cur[it] + add[it];
}

__device__ void tail_prolong(const TailLevel& T, const TailArrays& F, const TailLevel& Cn, const TailArrays& Cd)
{
    const int cells = T.w * T.h;
    if (cells <= kTailThreads)
        tail_prolong_n<1>(T, F, Cn, Cd);
    else if (cells <= 2 * kTailThreads)
        tail_prolong_n<2>(T, F, Cn, Cd);
    else
        tail_prolong_n<kTailIter>(T, F, Cn, Cd);
    __syncthreads();
}

// solveCoarsest (PressureMultigrid.cpp:347-384): remove the rhs mean, solve the pinned system
// (here with its precomputed inverse), shift to a mean-zero gauge.  Wavefront 0, one lane per row;
// the caller orders the result for the other threads.
__device__ void tail_coarse_solve(const TailLevel& T, const TailArrays& A, const float* G, int n)
{
    const int lane = threadIdx.x;
    const int w = T.w, s = T.s;
    const int cells = n + 1;
    float b = 0.f;
    if (lane < cells)
        b = A.rhs[(lane / w + 1) * s + lane % w + 1];
    const double mean = wave_sum((double)b) / cells;
    // y_j = rhs(cell j + 1) - mean, held by lane j + 1
    const float y = (float)((double)b - mean);
    // c = G y in the order j = 0 .. n-1, eight terms at a time: their G loads and y reads (v_readlane of a
    // uniform lane, no LDS) issue before the additions
    float c = 0.f;
    const int grow = min(lane, max(n - 1, 0)) * n;
    for (int j0 = 0; j0 < n; j0 += 8) {
        float g[8], yv[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int j = min(j0 + q, n - 1);
            g[q] = G[grow + j];
            yv[q] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(y), j + 1));
        }
#pragma unroll
        for (int q = 0; q < 8; ++q)
            if (j0 + q < n && lane < n)
                c += g[q] * yv[q];
    }
    const double gauge = wave_sum(lane < n ? (double)c : 0.0) / cells;
    if (lane == 0)
        A.sol[s + 1] = (float)(-gauge);
    if (lane < n) {
        const int cell = lane + 1;
        A.sol[(cell / w + 1) * s + cell % w + 1] = (float)((double)c - gauge);
    }
}

// The tail V-cycle of one instance on a 1024-thread workgroup: stage every tail level, its transfer
// tables and the coarse inverse in `lds`, cycle, and write the first tail level's solution back.
// TV: storage of the first tail level's global rhs and solution (FP32, or bfloat16).
template <class TV = float> __device__ void tail_run(const TailDesc& D, const double* shift, const int* status,
    float* lds)
{
    const int nl = D.levels;
    // Flat index over every level's padded arrays; all loads issue before the LDS stores.  The level of an
    // element, its source pointers and its LDS slot are picked by comparisons against uniform level
    // offsets (no per-lane reads of the descriptor).
    constexpr int TL = 8;
    int start[kMaxTailLevels + 1];
    start[0] = 0;
#pragma unroll
    for (int k = 0; k < kMaxTailLevels; ++k)
        start[k + 1] = start[k] + (k < nl ? D.lev[k].s * (D.lev[k].h + 2) : 0);
    const int total = start[kMaxTailLevels];
    const TailLevel& T0 = D.lev[0];
    const float inv_s0 = 1.0f / (float)T0.s;
    float vr[TL], vd[TL], vb[TL];
    int slot[TL], size[TL];
    bool bin[TL];
#pragma unroll
    for (int it = 0; it < TL; ++it) {
        const int e0 = threadIdx.x + it * kTailThreads;
        const int e = min(e0, total - 1);
        const float* pr = T0.right;
        const float* pd = T0.down;
        int first = 0, lds_at = T0.lds_arrays, n_at = start[1];
#pragma unroll
        for (int k = 1; k < kMaxTailLevels; ++k) {
            if (k < nl && e >= start[k]) {
                pr = D.lev[k].right;
                pd = D.lev[k].down;
                first = start[k];
                lds_at = D.lev[k].lds_arrays;
                n_at = start[k + 1] - start[k];
            }
        }
        const int le = e - first;
        vr[it] = pr[le];
        vd[it] = pd[le];
        const int y = tail_div(e, inv_s0) - 1, x = e - (y + 1) * T0.s - 1;   // meaningful on level 0 only
        const bool interior0 = first == 0 && x >= 0 && x < T0.w && y >= 0 && y < T0.h;
        const float b = ldv(((const TV*)D.top_rhs)[min(e, start[1] - 1)]);
        vb[it] = interior0 ? b : 0.f;
        bin[it] = interior0;
        slot[it] = e0 < total ? lds_at + le : -1;
        size[it] = n_at;
    }
    // transfer tables (host-built, already in LDS layout) and the coarse inverse: flat copies with
    // clamped, unconditional loads, issued with the level loads above
    constexpr int TT = 2, TG = 4;
    unsigned tv[TT];
    float gv[TG];
    const int nn = D.coarse_n * D.coarse_n;
#pragma unroll
    for (int it = 0; it < TT; ++it)
        tv[it] = D.tables[min(threadIdx.x + it * kTailThreads, (unsigned)max(D.table_words - 1, 0))];
#pragma unroll
    for (int it = 0; it < TG; ++it)
        gv[it] = D.ginv[min(threadIdx.x + it * kTailThreads, (unsigned)max(nn - 1, 0))];
    if (status && *status != kRunning)
        return;
    const double sh = shift ? *shift : 0.0;
#pragma unroll
    for (int it = 0; it < TL; ++it) {
        if (slot[it] < 0)
            continue;
        float* p = lds + slot[it];
        const int ps = size[it];
        p[0] = vr[it];                 // right
        p[ps] = vd[it];                // down
        p[2 * ps] = (shift && bin[it]) ? (float)((double)vb[it] - sh) : vb[it];   // rhs
        p[3 * ps] = 0.f;               // sol
        p[4 * ps] = 0.f;               // res
    }
    {
        unsigned* tables = (unsigned*)(lds + D.lds_tables_base);
#pragma unroll
        for (int it = 0; it < TT; ++it) {
            const int e = threadIdx.x + it * kTailThreads;
            if (e < D.table_words)
                tables[e] = tv[it];
        }
        float* Gl = lds + D.lds_ginv;
#pragma unroll
        for (int it = 0; it < TG; ++it) {
            const int e = threadIdx.x + it * kTailThreads;
            if (e < nn)
                Gl[e] = gv[it];
        }
    }
    float* G = lds + D.lds_ginv;
    const int n = D.coarse_n;
    __syncthreads();
    for (int l = 0; l + 1 < nl; ++l) {
        const TailLevel& T = D.lev[l];
        const TailArrays A = tail_arrays(lds, T);
        tail_smooth4(T, A, 0, 1, D.sweeps);
        tail_residual_restrict(T, A, D.lev[l + 1], tail_arrays(lds, D.lev[l + 1]));
    }
    if (threadIdx.x < 64)
        tail_coarse_solve(D.lev[nl - 1], tail_arrays(lds, D.lev[nl - 1]), G, n);
    __syncthreads();
    for (int l = nl - 2; l >= 0; --l) {
        const TailLevel& T = D.lev[l];
        const TailArrays A = tail_arrays(lds, T);
        tail_prolong(T, A, D.lev[l + 1], tail_arrays(lds, D.lev[l + 1]));
        tail_smooth4(T, A, 1, 0, D.sweeps);
    }
    const TailArrays A0 = tail_arrays(lds, T0);
    const float inv_w0 = 1.0f / (float)T0.w;
    for (int e = threadIdx.x; e < T0.w * T0.h; e += kTailThreads) {
        const int y = tail_div(e, inv_w0), x = e - y * T0.w;
        const int i = (y + 1) * T0.s + x + 1;
        ((TV*)D.top_sol)[i] = stv<TV>(A0.sol[i]);
    }
}

template <class TV>
__global__ __launch_bounds__(kTailThreads) void k_mg_tail(const TailDesc D, const double* shift, const int* status)
{
    extern __shared__ float lds[];
    tail_run<TV>(D, shift, status, lds);
}

// Tails of many grids that fs_tail.hip's register layout does not take, one workgroup each.
__global__ __launch_bounds__(kTailThreads) void k_lds_tail_batch(const BatchItem* __restrict__ items,
    const int* __restrict__ list)
{
    extern __shared__ float lds[];
    const BatchItem& I = items[list[blockIdx.x]];
    tail_run<float>(I.tail, I.levels == 0 ? &I.g.S->r_mean : nullptr, &I.g.S->status, lds);
}

__global__ __launch_bounds__(64 * kSweepWaves) void k_chain_batch(const BatchItem* __restrict__ items,
    const int* __restrict__ list)
{
    const BatchItem& I = items[list[blockIdx.x]];
    coarse_chain(I.chain, I.ginv, I.coarse_n, I.g.S, I.pin);
}

}  // namespace

size_t tail_layout(TailDesc& t)
{
    int words = 0;
    for (int l = 0; l < t.levels; ++l) {
        TailLevel& T = t.lev[l];
        T.lds_arrays = words;
        words += 5 * T.s * (T.h + 2);
    }
    t.lds_ginv = words;
    words += t.coarse_n * t.coarse_n;
    t.lds_tables_base = words;
    int tw = 0;
    for (int l = 0; l < t.levels; ++l) {
        TailLevel& T = t.lev[l];
        T.lds_tables = words + tw;
        tw += 3 * T.w + 3 * T.h + 9 * T.cw + 9 * T.ch;
    }
    t.table_words = tw;
    words += tw;
    t.lds_words = words;
    return (size_t)words * 4;
}

bool tail_allow_lds(size_t bytes)
{
    return hipFuncSetAttribute((const void*)k_mg_tail<float>, hipFuncAttributeMaxDynamicSharedMemorySize,
               (int)bytes) == hipSuccess &&
           hipFuncSetAttribute((const void*)k_mg_tail<bf16>, hipFuncAttributeMaxDynamicSharedMemorySize,
               (int)bytes) == hipSuccess;
}

void launch_coarse_factor(hipStream_t st, int w, int h, const double* right64, const double* down64,
    double* factor, float* ginv, int n, PcgScalars* S, int pin)
{
    if (n <= 0)
        return;
    hipLaunchKernelGGL(k_coarse_factor, dim3(1), dim3(kFactorThreads), 0, st, w, h, right64, down64, factor, ginv, n,
        S, pin);
}

void launch_coarse_chain(hipStream_t st, const ChainDesc& chain, float* ginv, int n, PcgScalars* S, int pin)
{
    hipLaunchKernelGGL(k_coarse_chain, dim3(1), dim3(64 * kSweepWaves), 0, st, chain, ginv, n, S, pin);
}

void launch_coarse_inverse(hipStream_t st, int w, int h, const double* right64, const double* down64, float* ginv,
    int n, PcgScalars* S, int pin)
{
    if (n <= 0)
        return;
    hipLaunchKernelGGL(k_coarse_inverse, dim3(1), dim3(64 * kSweepWaves), 0, st, w, h, right64, down64, ginv, n, S,
        pin);
}

void launch_mg_tail(hipStream_t st, const TailDesc& desc, size_t lds_bytes, const double* shift, const int* status,
    int bf16_top)
{
    if (bf16_top)
        hipLaunchKernelGGL(k_mg_tail<bf16>, dim3(1), dim3(kTailThreads), lds_bytes, st, desc, shift, status);
    else
        hipLaunchKernelGGL(k_mg_tail<float>, dim3(1), dim3(kTailThreads), lds_bytes, st, desc, shift, status);
}

// ---- 16-bit multigrid levels ----
namespace {

template <class C>
__global__ __launch_bounds__(kNT) void k_level_pack(int w, int h, const double* right64, const double* down64,
    C* right, C* down)
{
    const int s = w + 2;
    const int n = s * (h + 2);
    for (int i = blockIdx.x * kNT + threadIdx.x; i < n; i += gridDim.x * kNT) {
        right[i] = stv<C>((float)right64[i]);
        down[i] = stv<C>((float)down64[i]);
    }
}

}  // namespace

template <class C> void launch_level_pack(hipStream_t st, int w, int h, const double* right64, const double* down64,
    C* right, C* down)
{
    const int n = (w + 2) * (h + 2);
    const int blocks = std::min((n + kNT - 1) / kNT, 4096);
    hipLaunchKernelGGL(k_level_pack<C>, dim3(blocks), dim3(kNT), 0, st, w, h, right64, down64, right, down);
}
template void launch_level_pack<half16>(hipStream_t, int, int, const double*, const double*, half16*, half16*);
template void launch_level_pack<bf16>(hipStream_t, int, int, const double*, const double*, bf16*, bf16*);

template <class C, class V, class VC>
void launch_res_restrict(hipStream_t st, const LevelViewT<C, V>& F, int cur, const V* rhs, const double* shift,
    const LevelViewT<C, VC>& Cl, AxisRestrict rx, AxisRestrict ry, const int* status, int variant)
{
#define FS_RRT(CX, CY)                                                                                        \
    hipLaunchKernelGGL((k_res_restrict<CX, CY, C, V, VC>), dim3(((Cl.w + CX - 1) / CX) * ((Cl.h + CY - 1) / CY)),  \
        dim3(kNT), 0, st, F, cur, rhs, shift, Cl, rx, ry, status)
    switch (variant) {
    case 1: FS_RRT(16, 16); break;
    case 2: FS_RRT(16, 8); break;
    case 3: FS_RRT(8, 8); break;
    default: FS_RRT(32, 16); break;
    }
#undef FS_RRT
}

#define FS_RESTRICT(C, V, VC)                                                                                  \
    template void launch_res_restrict<C, V, VC>(hipStream_t, const LevelViewT<C, V>&, int, const V*, const double*, \
        const LevelViewT<C, VC>&, AxisRestrict, AxisRestrict, const int*, int);
FS_RESTRICT(float, float, float)
FS_RESTRICT(half16, float, float)
FS_RESTRICT(bf16, float, float)
FS_RESTRICT(bf16, float, bf16)
FS_RESTRICT(bf16, bf16, bf16)
#undef FS_RESTRICT

bool batch_allow_lds(size_t bytes)
{
    return hipFuncSetAttribute((const void*)k_lds_tail_batch, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) ==
           hipSuccess;
}

void launch_batch_lds_tail(hipStream_t st, const BatchItem* items, const int* list, int n, size_t lds_bytes)
{
    if (n > 0)
        hipLaunchKernelGGL(k_lds_tail_batch, dim3(n), dim3(kTailThreads), lds_bytes, st, items, list);
}

void launch_batch_chain(hipStream_t st, const BatchItem* items, const int* list, int n)
{
    if (n > 0)
        hipLaunchKernelGGL(k_chain_batch, dim3(n), dim3(64 * kSweepWaves), 0, st, items, list);
}

}  // namespace fsim
