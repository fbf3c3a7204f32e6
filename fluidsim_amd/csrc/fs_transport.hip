// fs_transport.hip -- the reference's PLIC/VOF transport on gfx950, FP64.
//
// FluidGridCPU::advect (FluidGridCPU.cpp:362-463) splits each CFL substep into an X and a Y pass.
// Each pass is two launches here instead of the reference's six sweeps, both bound by HBM:
//   cells : MYC interface normal and line offset of the upwind donor (recomputed from its 3 x 3
//           fraction neighbourhood, FluidGridCPU.cpp:473-541), the liquid volume through the cell's near face
//           (liquidTransferX/Y, :759-833; the far face's comes from the neighbouring thread), the summed component
//           mass transfer (:1235-1305), every component's mass update, the new fraction and the new density
//           (advectComponents :1351-1397, :407-455, rebuildDensity :1399-1423); the X pass, which opens a substep, also
//           freezes the correction weights (:1307-1349) that the Y pass reads;
//   faces : momentum transfer of both velocity components and velocity recovery (advectMomentumX/Y
//           :560-712, recoverVelocity :714-757).
// Fractions, masses and transported velocities are double-buffered, which replaces the reference's in-place
// ordering ("finish all neighbour reads before changing any cell masses") with a pure gather.
//
// Every expression is evaluated in the reference's order with -ffp-contract=off, so on the same input
// the results are the reference's bit for bit.
#include "fs_kernels.hpp"

#include <math.h>

namespace fsim {

namespace {

constexpr int kNT = 256;   // 64 x 4 threads
constexpr int kBX = 64;
constexpr int kBY = 4;

__device__ __forceinline__ double dmin(double a, double b) { return b < a ? b : a; }   // std::min
__device__ __forceinline__ double dmax(double a, double b) { return a < b ? b : a; }   // std::max

// liquidArea (FluidGridCPU.cpp:93-133): area of {p : n.p <= offset} inside [x0,x1] x [y0,y1].
__device__ double liquid_area(double nx, double ny, double offset, double x0, double y0, double x1, double y1)
{
    const double width = x1 - x0;
    const double height = y1 - y0;
    const double area = width * height;
    const double min_projection = nx * (nx >= 0.0 ? x0 : x1) + ny * (ny >= 0.0 ? y0 : y1);
    const double cut = offset - min_projection;
    const double span_x = fabs(nx) * width;
    const double span_y = fabs(ny) * height;
    const double small_span = dmin(span_x, span_y);
    const double large_span = dmax(span_x, span_y);
    if (cut <= 0.0)
        return 0.0;
    if (cut >= small_span + large_span)
        return area;
    if (small_span == 0.0)
        return area * cut / large_span;
    if (cut < small_span)
        return area * cut * cut / (2.0 * small_span * large_span);
    if (cut < large_span)
        return area * (cut - 0.5 * small_span) / large_span;
    const double dry_cut = small_span + large_span - cut;
    return area * (1.0 - dry_cut * dry_cut / (2.0 * small_span * large_span));
}

// interfaceOffset (FluidGridCPU.cpp:135-167).
__device__ double interface_offset(double nx, double ny, double fraction)
{
    const double min_projection = dmin(nx, 0.0) + dmin(ny, 0.0);
    const double span_x = fabs(nx);
    const double span_y = fabs(ny);
    const double small_span = dmin(span_x, span_y);
    const double large_span = dmax(span_x, span_y);
    const double triangle_fraction = 0.5 * small_span / large_span;
    double cut;
    if (fraction < triangle_fraction)
        cut = sqrt(2.0 * small_span * large_span * fraction);
    else if (fraction <= 1.0 - triangle_fraction)
        cut = large_span * fraction + 0.5 * small_span;
    else
        cut = small_span + large_span - sqrt(2.0 * small_span * large_span * (1.0 - fraction));
    return min_projection + cut;
}

// interfaceNormal (FluidGridCPU.cpp:473-521): mixed Youngs-centred normal, neighbours clamped to the grid.
__device__ void interface_normal(const double* f, int W, int H, int x, int y, double& nx, double& ny)
{
    const int lx = max(x - 1, 0), rx = min(x + 1, W - 1);
    const double* above = f + (size_t)max(y - 1, 0) * W;
    const double* row = f + (size_t)y * W;
    const double* below = f + (size_t)min(y + 1, H - 1) * W;
    const double tl = above[lx], t = above[x], tr = above[rx];
    const double l = row[lx], r = row[rx];
    const double bl = below[lx], b = below[x], br = below[rx];
    const double left_sum = tl + l + bl;
    const double right_sum = tr + r + br;
    const double top_sum = tl + t + tr;
    const double bottom_sum = bl + b + br;
    double cx = 0.5 * (left_sum - right_sum), cy = 0.5 * (top_sum - bottom_sum);
    const double yx = left_sum + l - right_sum - r, yy = top_sum + t - bottom_sum - b;
    if (cx == 0.0 && cy == 0.0) {
        const bool none = yx == 0.0 && yy == 0.0;
        nx = none ? 1.0 : yx;
        ny = none ? 0.0 : yy;
        return;
    }
    bool youngs;
    if (fabs(cx) <= fabs(cy)) {
        cy = copysign(1.0, cy);
        youngs = fabs(yx) > fabs(cx * yy);
    } else {
        cx = copysign(1.0, cx);
        youngs = fabs(yy) > fabs(cy * yx);
    }
    nx = youngs ? yx : cx;
    ny = youngs ? yy : cy;
}

// componentMassTransfer (FluidGridCPU.cpp:543-551).
__device__ __forceinline__ double component_transfer(double volume_transfer, double donor_fraction, double donor_mass)
{
    return donor_fraction <= 0.0 ? 0.0 : donor_mass * (volume_transfer / donor_fraction);
}

// momentumTransfer (FluidGridCPU.cpp:553-558).
__device__ __forceinline__ double momentum_transfer(double mass_transfer, double before, double after)
{
    return mass_transfer * (mass_transfer >= 0.0 ? before : after);
}

// Scale of a pass: the caller's, or (first substep, queued before the host knows it) the one k_tr_outflow_finish left
// on the device; negative where the call is refused, and nothing may change.
__device__ __forceinline__ double pass_scale(const TransportDev& t, double scale) { return t.scale ? *t.scale : scale; }

// ------------------------------------------------------------------------------------------
// rebuildDensity and rebuildMomentum (FluidGridCPU.cpp:1399-1476) and the largest cell outflow (:366-386), one partial
// per 64 x 16 tile: each cell with its left and top face, and the far walls.
// ------------------------------------------------------------------------------------------
__global__ __launch_bounds__(kNT) void k_tr_begin(TransportDev t)
{
    constexpr int R = 4;   // rows per wavefront: a cell's density is summed once, for the row below and the next lane too
    __shared__ double lds[kNT / 64];
    const int W = t.W, H = t.H;
    const size_t N = (size_t)W * H;
    const int lane = threadIdx.x & 63;
    const int x = blockIdx.x * 64 + lane, xc = min(x, W - 1);
    const int y0 = blockIdx.y * 16 + (threadIdx.x >> 6) * R;
    // masses of rows y0 - 1 .. y0 + R - 1, and of the column left of the wavefront's
    double d[R + 1] = {}, edge[R] = {};
    size_t at[R + 1];
#pragma unroll
    for (int r = 0; r <= R; ++r)
        at[r] = (size_t)min(max(y0 + r - 1, 0), H - 1) * W;
    const int xl = max(xc - 1, 0);
    auto add = [&](const double* masses) {
#pragma unroll
        for (int r = 0; r <= R; ++r)
            d[r] += masses[at[r] + xc];
        if (lane == 0) {
#pragma unroll
            for (int r = 0; r < R; ++r)
                edge[r] += masses[at[r + 1] + xl];
        }
    };
    for (int k = 0; k < t.nl; ++k)
        add(t.lm + k * N);
    for (int k = 0; k < t.ng; ++k)
        add(t.gm + k * N);
#pragma unroll
    for (int r = 0; r <= R; ++r)
        d[r] *= t.icv;
#pragma unroll
    for (int r = 0; r < R; ++r)
        edge[r] *= t.icv;
    double m = 0.0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int y = y0 + r;
        const double here = d[r + 1];
        const double next = from_left(here);
        const double left = lane == 0 ? edge[r] : next;
        if (x >= W || y >= H)
            continue;
        const size_t cell = (size_t)y * W + x;
        const size_t fu = (size_t)y * (W + 1) + x, fv = cell;
        t.density[cell] = here;
        const double u = t.u[fu], un = t.u[fu + 1], v = t.v[fv], vn = t.v[fv + W];
        t.mom_u[fu] = x > 0 ? 0.5 * (left + here) * u : 0.0;
        t.nu_out[fu] = x > 0 ? u : 0.0;
        t.mom_v[fv] = y > 0 ? 0.5 * (d[r] + here) * v : 0.0;
        t.nv_out[fv] = y > 0 ? v : 0.0;
        if (x + 1 == W) {
            t.mom_u[fu + 1] = 0.0;
            t.nu_out[fu + 1] = 0.0;
        }
        if (y + 1 == H) {
            t.mom_v[fv + W] = 0.0;
            t.nv_out[fv + W] = 0.0;
        }
        m = dmax(m, dmax(un, 0.0) + dmax(-u, 0.0) + dmax(vn, 0.0) + dmax(-v, 0.0));
    }
    const double bm = block_max<kNT>(m, lds);
    if (threadIdx.x == 0)
        t.partials[blockIdx.y * gridDim.x + blockIdx.x] = bm;
}

// The largest outflow, for the host, and the first substep's scale, which the kernels queued behind this one read:
// no cell exports more than half its volume per substep (FluidGridCPU.cpp:388-389).
__global__ __launch_bounds__(kNT) void k_tr_outflow_finish(TransportDev t, int nb, double h, double dt,
    double max_substeps, double* host)
{
    __shared__ double lds[kNT / 64];
    const double m = finish_max<kNT>(t.partials, nb, 1, 0, lds);
    if (threadIdx.x == 0) {
        const double max_step = m > 0.0 ? 0.5 * h / m : dt;
        const bool refused = !(max_step > 0.0) || dt / max_step > max_substeps;
        *t.out = refused ? -1.0 : dmin(dt, max_step) / h;
        *host = m;
    }
}

// Liquid volume through the face behind (HORIZ: left of, else above) cell (x, y), which is no wall
// (liquidTransferX / liquidTransferY, FluidGridCPU.cpp:759-833); (dx, dy) is its upwind donor.
template <bool HORIZ>
__device__ __forceinline__ double liquid_transfer(const TransportDev& t, int dx, int dy, double speed, double fraction,
    double scale)
{
    if (speed == 0.0 || !(fraction > 0.0))
        return 0.0;
    const double volume_transfer = speed * scale;
    const double strip = fabs(volume_transfer);
    if (fraction >= 1.0)
        return volume_transfer;
    double nx, ny;
    interface_normal(t.f, t.W, t.H, dx, dy, nx, ny);
    const double offset = interface_offset(nx, ny, fraction);
    const double lo = speed > 0.0 ? 1.0 - strip : 0.0;
    const double hi = speed > 0.0 ? 1.0 : strip;
    const double area =
        HORIZ ? liquid_area(nx, ny, offset, lo, 0.0, hi, 1.0) : liquid_area(nx, ny, offset, 0.0, lo, 1.0, hi);
    const double floor_ = dmax(0.0, strip - (1.0 - fraction));
    const double ceil_ = dmin(strip, fraction);
    const double bounded = area < floor_ ? floor_ : (ceil_ < area ? ceil_ : area);  // std::clamp
    return speed > 0.0 ? bounded : -bounded;
}

// ------------------------------------------------------------------------------------------
// Pass, launch 1: a thread's near face and cell.  X: a wavefront holds 64 faces of a row and updates 63 cells, the far
// face's liquid coming from the next lane; Y: a workgroup holds 8 rows of 64 faces and updates 7, through LDS.  With
// the faces and the freezing of the weights in launches of their own every field was read twice: a substep of 700 x 500
// cells with 2 + 2 components moved 234 MB in 63 us in seven launches, now 162 MB in 47 us in four.
// ------------------------------------------------------------------------------------------
constexpr int kFaceRows = 8;

template <bool HORIZ>
__global__ __launch_bounds__(HORIZ ? kNT : 64 * kFaceRows) void k_tr_cells(TransportDev t, double scale_)
{
    __shared__ double s_lt[HORIZ ? 1 : kFaceRows][64];
    const int W = t.W, H = t.H;
    const size_t N = (size_t)W * H;
    const int lane = threadIdx.x & 63, row = threadIdx.x >> 6;
    const int x = HORIZ ? blockIdx.x * 63 + lane : blockIdx.x * 64 + lane;
    const int y = HORIZ ? blockIdx.y * kBY + row : blockIdx.y * (kFaceRows - 1) + row;
    const double scale = pass_scale(t, scale_);
    if (scale < 0.0)
        return;
    const bool cell = x < W && y < H;
    const size_t stride = HORIZ ? 1 : (size_t)W;
    const size_t i = cell ? (size_t)y * W + x : 0;
    const size_t before = HORIZ ? (size_t)y * (W + 1) + x : i;
    const double* flow = HORIZ ? t.u : t.v;
    const bool wall_before = HORIZ ? x == 0 : y == 0;
    double fb = 0.0, fa = 0.0, lt_b = 0.0, f = 0.0, frac_b = 0.0;
    size_t donor_b = i;
    if (cell) {
        fb = flow[before];
        fa = flow[before + stride];
        f = t.f[i];
        // upwind donors of the two faces (clamped to the cell itself at walls, where nothing moves)
        if (!wall_before && fb > 0.0)
            donor_b = i - stride;
        frac_b = t.f[donor_b];
        if (!wall_before) {
            const int back = donor_b != i;
            lt_b = liquid_transfer<HORIZ>(t, HORIZ ? x - back : x, HORIZ ? y : y - back, fb, frac_b, scale);
        }
    }
    double lt_a;
    bool own;
    if constexpr (HORIZ) {
        lt_a = from_right(lt_b);
        own = lane < 63;
    } else {
        s_lt[row][lane] = lt_b;
        __syncthreads();
        lt_a = s_lt[min(row + 1, kFaceRows - 1)][lane];
        own = row < kFaceRows - 1;
    }
    if (!own)
        return;
    if (!cell) {
        // the far wall
        if (HORIZ ? (x == W && y < H) : (y == H && x < W))
            t.mt[HORIZ ? before : (size_t)y * W + x] = 0.0;
        return;
    }
    const bool wall_after = HORIZ ? x + 1 == W : y + 1 == H;
    const size_t donor_a = (!wall_after && !(fa > 0.0)) ? i + stride : i;
    const double frac_a = t.f[donor_a];
    const double all_b = fb * scale, all_a = fa * scale;
    const double net_fluid = scale * (fa - fb);
    // freezeComponentCorrections (FluidGridCPU.cpp:1307-1349): only the weights of the cell's phase are kept, the
    // others are zero
    bool selected;
    double inverse_fraction = 0.0, correction = 0.0;
    if (HORIZ) {
        selected = f > 0.5;
        t.split[i] = (unsigned char)selected;
        inverse_fraction = 1.0 / (selected ? f : 1.0 - f);
    } else {
        selected = t.split[i] != 0;
    }
    double mt = 0.0, total = 0.0;
    // two components at a time, so that their loads travel together
    auto components = [&](int n, const double* m, double* out, double* weights, bool weighted, double volume_b,
                          double fraction_b, double volume_a, double fraction_a) {
        for (int k = 0; k < n; k += 2) {
            double here[2], from_b[2], from_a[2], weight[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const size_t c = min(k + j, n - 1) * N;
                here[j] = m[c + i];
                from_b[j] = m[c + donor_b];
                from_a[j] = m[c + donor_a];
                weight[j] = !HORIZ && weighted ? weights[c + i] : 0.0;
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                if (k + j >= n)
                    break;
                const size_t c = (k + j) * N + i;
                if (HORIZ) {
                    if (weighted)
                        weights[c] = weight[j] = here[j] * inverse_fraction;
                    correction += weight[j] * t.icv;
                }
                const double ct_b = wall_before ? 0.0 : component_transfer(volume_b, fraction_b, from_b[j]);
                const double ct_a = wall_after ? 0.0 : component_transfer(volume_a, fraction_a, from_a[j]);
                mt += ct_b * t.icv;
                const double mass = here[j] + (ct_b - ct_a + weight[j] * net_fluid);
                out[c] = mass;
                total += mass;
            }
        }
    };
    components(t.nl, t.lm, t.lm_out, t.lcw, selected, lt_b, frac_b, lt_a, frac_a);
    components(t.ng, t.gm, t.gm_out, t.gcw, !selected, all_b - lt_b, 1.0 - frac_b, all_a - lt_a, 1.0 - frac_a);
    if (HORIZ)
        t.mcw[i] = correction;
    t.mt[before] = mt;
    t.density[i] = total * t.icv;
    t.f_out[i] = f - (lt_a - lt_b) + (double)selected * net_fluid;
}

// ------------------------------------------------------------------------------------------
// Pass, launch 2: momentum transfer and velocity recovery of a cell's left and top face (and the far walls), which share
// the cell's transfers, density and correction.  Bound by memory: 36 MB in 11 us per pass of 700 x 500 cells, the rate at
// which a copy of that size runs.
// ------------------------------------------------------------------------------------------
template <bool HORIZ>
__device__ __forceinline__ double mass_correction(const TransportDev& t, int cx, int cy, double scale)
{
    // weight * scale * (flow out - flow in) of one cell along the pass's axis
    const size_t cell = (size_t)cy * t.W + cx;
    const double w = t.mcw[cell];
    if (HORIZ) {
        const size_t lf = (size_t)cy * (t.W + 1) + cx;
        return w * scale * (t.u[lf + 1] - t.u[lf]);
    }
    return w * scale * (t.v[cell + t.W] - t.v[cell]);
}

template <bool HORIZ>
__global__ __launch_bounds__(kNT) void k_tr_momentum(TransportDev t, double scale_)
{
    const int W = t.W, H = t.H;
    const int x = blockIdx.x * kBX + (threadIdx.x & 63);
    const int y = blockIdx.y * kBY + (threadIdx.x >> 6);
    const double scale = pass_scale(t, scale_);
    if (scale < 0.0)
        return;
    const size_t us = (size_t)W + 1;
    const size_t fu = (size_t)y * us + x, cell = (size_t)y * W + x;   // cell: also the v face above it
    if (y < H && (x == 0 || x == W)) {
        t.mom_u[fu] = 0.0;
        t.nu_out[fu] = 0.0;
    }
    if (x < W && (y == 0 || y == H)) {
        t.mom_v[cell] = 0.0;
        t.nv_out[cell] = 0.0;
    }
    if (x >= W || y >= H)
        return;
    const double correction_here = mass_correction<HORIZ>(t, x, y, scale);
    const double density_here = t.density[cell];
    if (x > 0) {
        double m_before, m_after;   // momentum entering through the near side, leaving through the far side
        if (HORIZ) {
            const double lm = 0.5 * (t.mt[fu - 1] + t.mt[fu]);
            const double rm = 0.5 * (t.mt[fu] + t.mt[fu + 1]);
            m_before = momentum_transfer(lm, t.nu_in[fu - 1], t.nu_in[fu]);
            m_after = momentum_transfer(rm, t.nu_in[fu], t.nu_in[fu + 1]);
        } else {
            const double tm = 0.5 * (t.mt[cell - 1] + t.mt[cell]);
            const double bm = 0.5 * (t.mt[cell - 1 + W] + t.mt[cell + W]);
            m_before = y > 0 ? momentum_transfer(tm, t.nu_in[fu - us], t.nu_in[fu]) : 0.0;
            m_after = y + 1 < H ? momentum_transfer(bm, t.nu_in[fu], t.nu_in[fu + us]) : 0.0;
        }
        const double correction = 0.5 * (mass_correction<HORIZ>(t, x - 1, y, scale) + correction_here);
        const double momentum = t.mom_u[fu] + (m_before - m_after + t.u[fu] * correction);
        t.mom_u[fu] = momentum;
        t.nu_out[fu] = momentum / (0.5 * (t.density[cell - 1] + density_here));
    }
    if (y > 0) {
        double m_before, m_after;
        if (HORIZ) {
            const double lm = 0.5 * (t.mt[fu - us] + t.mt[fu]);
            const double rm = 0.5 * (t.mt[fu - us + 1] + t.mt[fu + 1]);
            m_before = x > 0 ? momentum_transfer(lm, t.nv_in[cell - 1], t.nv_in[cell]) : 0.0;
            m_after = x + 1 < W ? momentum_transfer(rm, t.nv_in[cell], t.nv_in[cell + 1]) : 0.0;
        } else {
            const double tm = 0.5 * (t.mt[cell - W] + t.mt[cell]);
            const double bm = 0.5 * (t.mt[cell] + t.mt[cell + W]);
            m_before = momentum_transfer(tm, t.nv_in[cell - W], t.nv_in[cell]);
            m_after = momentum_transfer(bm, t.nv_in[cell], t.nv_in[cell + W]);
        }
        const double correction = 0.5 * (mass_correction<HORIZ>(t, x, y - 1, scale) + correction_here);
        const double momentum = t.mom_v[cell] + (m_before - m_after + t.v[cell] * correction);
        t.mom_v[cell] = momentum;
        t.nv_out[cell] = momentum / (0.5 * (t.density[cell - W] + density_here));
    }
}

inline dim3 face_grid(int W, int H)
{
    // covers both (W+1) x H and W x (H+1)
    return dim3((W + 1 + kBX - 1) / kBX, (H + 1 + kBY - 1) / kBY, 1);
}

}  // namespace

void launch_transport_begin(hipStream_t st, const TransportDev& t, double h, double dt, double max_substeps,
    double* host)
{
    const dim3 tiles((t.W + 63) / 64, (t.H + 15) / 16);
    hipLaunchKernelGGL(k_tr_begin, tiles, dim3(kNT), 0, st, t);
    hipLaunchKernelGGL(k_tr_outflow_finish, dim3(1), dim3(kNT), 0, st, t, (int)(tiles.x * tiles.y), h, dt, max_substeps,
        host);
}

void launch_transport_pass(hipStream_t st, const TransportDev& t, int horizontal, double scale)
{
    const dim3 mg = face_grid(t.W, t.H);
    if (horizontal) {
        const dim3 cg((t.W + 1 + 62) / 63, (t.H + kBY - 1) / kBY);
        hipLaunchKernelGGL(k_tr_cells<true>, cg, dim3(kNT), 0, st, t, scale);
        hipLaunchKernelGGL(k_tr_momentum<true>, mg, dim3(kNT), 0, st, t, scale);
    } else {
        const dim3 cg((t.W + 63) / 64, (t.H + 1 + kFaceRows - 2) / (kFaceRows - 1));
        hipLaunchKernelGGL(k_tr_cells<false>, cg, dim3(64 * kFaceRows), 0, st, t, scale);
        hipLaunchKernelGGL(k_tr_momentum<false>, mg, dim3(kNT), 0, st, t, scale);
    }
}

}  // namespace fsim
