// fs_kernels.hip -- hand-written HIP kernels for gfx950 (MI355X) around the projection: density, forces,
// semi-Lagrangian transport, colours, edits and copies.  FP64 expressions keep the reference's order
// (-ffp-contract=off).
#include "fs_kernels.hpp"

#include <algorithm>

#include <math.h>

namespace fsim {

namespace {

constexpr int kTX = 64;
constexpr int kTY = 16;
constexpr int kNT = 256;

inline dim3 cell_grid(int W, int H) { return dim3((W + kTX - 1) / kTX, (H + kTY - 1) / kTY); }
// Iterate the (up to) four cells this thread owns in the block's 64 x 16 tile.
#define FS_TILE_BEGIN(WIDTH, HEIGHT)                                                   \
    {                                                                                  \
        const int x = blockIdx.x * kTX + (threadIdx.x & 63);                           \
        for (int k_ = 0; k_ < 4; ++k_) {                                               \
            const int y = blockIdx.y * kTY + (threadIdx.x >> 6) + 4 * k_;              \
            if (x >= (WIDTH) || y >= (HEIGHT))                                         \
                continue;
#define FS_TILE_END \
        }           \
    }

// ------------------------------------------------------------------------------------------
// Density (FluidGridCPU.cpp:1399-1423), FP64, bit-exact.
// ------------------------------------------------------------------------------------------
__global__ __launch_bounds__(kNT) void k_density(GridDev g)
{
    const size_t N = (size_t)g.W * g.H;
    const double inverse_cell_volume = 1.0 / (g.h * g.h);
    for (size_t i = (size_t)blockIdx.x * kNT + threadIdx.x; i < N; i += (size_t)gridDim.x * kNT) {
        double total = 0.0;
        for (int k = 0; k < g.nl; ++k)
            total += g.lmass[(size_t)k * N + i];
        for (int k = 0; k < g.ng; ++k)
            total += g.gmass[(size_t)k * N + i];
        g.density[i] = total * inverse_cell_volume;
    }
}

// applyGravity (FluidGridCPU.cpp:988-996): interior v rows only.
__global__ __launch_bounds__(kNT) void k_gravity(double* v, int first, int last, double increment)
{
    for (int i = first + blockIdx.x * kNT + threadIdx.x; i < last; i += gridDim.x * kNT)
        v[i] += increment;
}

// addVortex (FluidGridCPU.cpp:998-1028).
__global__ __launch_bounds__(kNT) void k_add_vortex(GridDev g, double ox, double oy, double cx, double cy,
    double radius, double strength)
{
    const int W = g.W, H = g.H;
    const int nu = (W + 1) * H, nv = W * (H + 1);
    for (int t = blockIdx.x * kNT + threadIdx.x; t < nu + nv; t += gridDim.x * kNT) {
        if (t < nu) {
            const int x = t % (W + 1), y = t / (W + 1);
            const double px = ox + x * g.h, py = oy + (y + 0.5) * g.h;
            const double dx = px - cx, dy = py - cy;
            const double r2 = dx * dx + dy * dy;
            const double falloff = exp(-r2 / (2.0 * radius * radius));
            g.u[t] += -dy * strength * falloff;
        } else {
            const int e = t - nu;
            const int x = e % W, y = e / W;
            const double px = ox + (x + 0.5) * g.h, py = oy + y * g.h;
            const double dx = px - cx, dy = py - cy;
            const double r2 = dx * dx + dy * dy;
            const double falloff = exp(-r2 / (2.0 * radius * radius));
            g.v[e] += dx * strength * falloff;
        }
    }
}

// ---- semi-Lagrangian transport mode (build-defined; samples as FluidGridCPU::sampleVelocity) ----
// Bound by FP64 issue (six divisions and 15 interpolations a face): std::lerp and std::clamp are written for what holds
// here, and an element's row comes from a multiplication instead of divisions.  A call on 1024^2 cells 103 -> 71 us,
// 2 x 100000 51 -> 33.  (Workgroups of 64 x 4 elements need no row at all, but leave lanes idle on narrow grids: 76
// and 320 us.)

// n / d of 0 <= n < 2^31 as one multiplication: with 2^(s-1) < d <= 2^s, magic = ceil(2^(31+s) / d) is too large by
// less than 2^s / d parts in 2^(31+s), which is less than 1 / d after the multiplication by n.
struct Divisor {
    unsigned magic;
    int shift;
    explicit Divisor(unsigned d)
    {
        int s = 0;
        while ((1u << s) < d)
            ++s;
        shift = 31 + s;
        magic = (unsigned)((((unsigned long long)1 << shift) + d - 1) / d);
    }
    __device__ __forceinline__ int of(unsigned n) const { return (int)(((unsigned long long)n * magic) >> shift); }
};

// std::lerp for 0 <= t < 1 (its exact ends beyond that cannot occur).
__device__ __forceinline__ double lerp_std(double a, double b, double t)
{
    const double x = a + t * (b - a);
    const double bounded = b > a ? fmin(x, b) : fmax(x, b);
    const bool mixed = (a <= 0 && b >= 0) || (a >= 0 && b <= 0);
    return mixed ? t * b + (1 - t) * a : bounded;
}

// A non-finite sample position (non-finite velocity) reads cell 0 instead of an undefined index: fmax drops a NaN.
__device__ double sample_scalar(const double* data, int width, int height, double x, double y)
{
    x = fmin(fmax(x, 0.0), (double)(width - 1));
    y = fmin(fmax(y, 0.0), (double)(height - 1));
    const int x0 = (int)x, y0 = (int)y;
    const int x1 = min(x0 + 1, width - 1), y1 = min(y0 + 1, height - 1);
    const double tx = x - x0, ty = y - y0;
    const double a = lerp_std(data[y0 * width + x0], data[y0 * width + x1], tx);
    const double b = lerp_std(data[y1 * width + x0], data[y1 * width + x1], tx);
    return lerp_std(a, b, ty);
}

__device__ __forceinline__ void sample_velocity(const GridDev& g, double ox, double oy, double px, double py,
    double* vx, double* vy)
{
    const double x = (px - ox) / g.h;
    const double y = (py - oy) / g.h;
    *vx = sample_scalar(g.u, g.W + 1, g.H, x, y - 0.5);
    *vy = sample_scalar(g.v, g.W, g.H + 1, x - 0.5, y);
}

__device__ __forceinline__ void backtrace(const GridDev& g, double ox, double oy, double px, double py, double dt,
    double* sx, double* sy)
{
    double vx, vy;
    sample_velocity(g, ox, oy, px, py, &vx, &vy);
    const double mx = px - 0.5 * dt * vx, my = py - 0.5 * dt * vy;
    sample_velocity(g, ox, oy, mx, my, &vx, &vy);
    *sx = px - dt * vx;
    *sy = py - dt * vy;
}

__global__ __launch_bounds__(kNT) void k_sl_faces(GridDev g, double ox, double oy, double dt, Divisor u_row,
    Divisor v_row, double* nu, double* nv)
{
    const int W = g.W, H = g.H;
    const int t = blockIdx.x * kNT + threadIdx.x;
    double value = 0.0, sx, sy;
    if (blockIdx.y == 0) {
        const int y = u_row.of(t), x = t - y * (W + 1);
        if (y >= H)
            return;
        if (x >= 1 && x < W) {
            backtrace(g, ox, oy, ox + x * g.h, oy + (y + 0.5) * g.h, dt, &sx, &sy);
            value = sample_scalar(g.u, W + 1, H, (sx - ox) / g.h, (sy - oy) / g.h - 0.5);
        }
        nu[t] = value;
    } else {
        const int y = v_row.of(t), x = t - y * W;
        if (y > H)
            return;
        if (y >= 1 && y < H) {
            backtrace(g, ox, oy, ox + (x + 0.5) * g.h, oy + y * g.h, dt, &sx, &sy);
            value = sample_scalar(g.v, W, H + 1, (sx - ox) / g.h - 0.5, (sy - oy) / g.h);
        }
        nv[t] = value;
    }
}

// Cell-centred scalars (fraction, every component mass) share one backtrace per cell.
__global__ __launch_bounds__(kNT) void k_sl_cells(GridDev g, double ox, double oy, double dt, Divisor row,
    double* fraction, double* lmass, double* gmass)
{
    const int W = g.W, H = g.H;
    const size_t N = (size_t)W * H;
    const int i = blockIdx.x * kNT + threadIdx.x;
    const int y = row.of(i), x = i - y * W;
    if (y >= H)
        return;
    double sx, sy;
    backtrace(g, ox, oy, ox + (x + 0.5) * g.h, oy + (y + 0.5) * g.h, dt, &sx, &sy);
    const double fx = (sx - ox) / g.h - 0.5, fy = (sy - oy) / g.h - 0.5;
    fraction[i] = sample_scalar(g.fraction, W, H, fx, fy);
    for (int k = 0; k < g.nl; ++k)
        lmass[(size_t)k * N + i] = sample_scalar(g.lmass + (size_t)k * N, W, H, fx, fy);
    for (int k = 0; k < g.ng; ++k)
        gmass[(size_t)k * N + i] = sample_scalar(g.gmass + (size_t)k * N, W, H, fx, fy);
}

__global__ __launch_bounds__(kNT) void k_pad_copy(const double* src, double* dst, int W, int H, int to_padded)
{
    const int s = W + 2;
    FS_TILE_BEGIN(W, H)
    if (to_padded)
        dst[pidx(x, y, s)] = src[(size_t)y * W + x];
    else
        dst[(size_t)y * W + x] = src[pidx(x, y, s)];
    FS_TILE_END
}

// Several FP64 device-to-device copies in one launch (blockIdx.y selects the copy).
__global__ __launch_bounds__(kNT) void k_copy_many(CopyList list)
{
    const CopyList::Item it = list.item[blockIdx.y];
    for (size_t i = (size_t)blockIdx.x * kNT + threadIdx.x; i < it.n; i += (size_t)gridDim.x * kNT)
        it.dst[i] = it.src[i];
}

__global__ void k_copy_f32(const float* src, float* dst, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

// writeColorPixels (FluidGridCPU.cpp:1826-1860): per cell, RGBA with the component colours weighted by
// their volume fractions mass / (density h^2), in the reference's precision and order (FP64 fraction,
// each channel term rounded to FP32 and summed in FP32, liquid components before gas components).
__global__ __launch_bounds__(kNT) void k_color(GridDev g, ColorTable t, int alpha_from_fraction, float4* out)
{
    const size_t N = (size_t)g.W * g.H;
    const double cell_volume = g.h * g.h;
    for (size_t i = (size_t)blockIdx.x * kNT + threadIdx.x; i < N; i += (size_t)gridDim.x * kNT) {
        float4 px = make_float4(0.0f, 0.0f, 0.0f, alpha_from_fraction ? (float)g.fraction[i] : 1.0f);
        for (int k = 0; k < g.nl + g.ng; ++k) {
            const double mass = k < g.nl ? g.lmass[(size_t)k * N + i] : g.gmass[(size_t)(k - g.nl) * N + i];
            const double volume_fraction = mass / (t.density[k] * cell_volume);
            px.x += (float)(volume_fraction * (double)t.rgb[k][0]);
            px.y += (float)(volume_fraction * (double)t.rgb[k][1]);
            px.z += (float)(volume_fraction * (double)t.rgb[k][2]);
        }
        out[i] = px;
    }
}

// commitEdits (FluidGridCPU.cpp:253-284) for resolved, duplicate-free cells: the cell becomes pure liquid
// or pure gas holding one component's mass, every other component's mass zero.
__global__ __launch_bounds__(kNT) void k_commit_edits(GridDev g, const EditCell* cells, int n)
{
    const size_t N = (size_t)g.W * g.H;
    for (int e = blockIdx.x * kNT + threadIdx.x; e < n; e += gridDim.x * kNT) {
        const EditCell c = cells[e];
        const size_t i = (size_t)c.y * g.W + c.x;
        const bool liquid = c.component < g.nl;
        g.fraction[i] = liquid ? 1.0 : 0.0;
        for (int k = 0; k < g.nl; ++k)
            g.lmass[(size_t)k * N + i] = k == c.component ? c.mass : 0.0;
        for (int k = 0; k < g.ng; ++k)
            g.gmass[(size_t)k * N + i] = g.nl + k == c.component ? c.mass : 0.0;
    }
}

inline unsigned linear_blocks(size_t n)
{
    size_t b = (n + kNT - 1) / kNT;
    if (b > 8192)
        b = 8192;
    return (unsigned)(b ? b : 1);
}

}  // namespace

// ------------------------------------------------------------------------------------------
// launchers
// ------------------------------------------------------------------------------------------

void launch_density(hipStream_t st, const GridDev& g)
{
    hipLaunchKernelGGL(k_density, dim3(linear_blocks((size_t)g.W * g.H)), dim3(kNT), 0, st, g);
}

void launch_color(hipStream_t st, const GridDev& g, const ColorTable& t, int alpha_from_fraction, float* rgba)
{
    hipLaunchKernelGGL(k_color, dim3(linear_blocks((size_t)g.W * g.H)), dim3(kNT), 0, st, g, t, alpha_from_fraction,
        (float4*)rgba);
}

void launch_commit_edits(hipStream_t st, const GridDev& g, const EditCell* cells, int n)
{
    if (n > 0)
        hipLaunchKernelGGL(k_commit_edits, dim3(linear_blocks((size_t)n)), dim3(kNT), 0, st, g, cells, n);
}

void launch_gravity(hipStream_t st, const GridDev& g, double gy, double dt)
{
    const int first = g.W, last = g.W * g.H;
    if (last <= first)
        return;
    hipLaunchKernelGGL(k_gravity, dim3(linear_blocks((size_t)(last - first))), dim3(kNT), 0, st, g.v, first, last,
        gy * dt);
}

void launch_add_vortex(hipStream_t st, const GridDev& g, double ox, double oy, double cx, double cy, double radius,
    double strength)
{
    const size_t n = (size_t)(g.W + 1) * g.H + (size_t)g.W * (g.H + 1);
    hipLaunchKernelGGL(k_add_vortex, dim3(linear_blocks(n)), dim3(kNT), 0, st, g, ox, oy, cx, cy, radius, strength);
}

void launch_semi_lagrangian(hipStream_t st, const GridDev& g, double ox, double oy, double dt, double* new_u,
    double* new_v, double* new_fraction, double* new_lmass, double* new_gmass)
{
    const auto blocks = [](size_t n) { return (unsigned)((n + kNT - 1) / kNT); };
    const size_t nu = (size_t)(g.W + 1) * g.H, nv = (size_t)g.W * (g.H + 1);
    hipLaunchKernelGGL(k_sl_faces, dim3(blocks(std::max(nu, nv)), 2), dim3(kNT), 0, st, g, ox, oy, dt,
        Divisor((unsigned)g.W + 1), Divisor((unsigned)g.W), new_u, new_v);
    hipLaunchKernelGGL(k_sl_cells, dim3(blocks((size_t)g.W * g.H)), dim3(kNT), 0, st, g, ox, oy, dt,
        Divisor((unsigned)g.W), new_fraction, new_lmass, new_gmass);
}

void launch_pad_copy(hipStream_t st, const double* src, double* dst, int W, int H, int to_padded)
{
    hipLaunchKernelGGL(k_pad_copy, cell_grid(W, H), dim3(kNT), 0, st, src, dst, W, H, to_padded);
}

void launch_copy_many(hipStream_t st, const CopyList& list)
{
    if (list.count <= 0)
        return;
    size_t most = 0;
    for (int k = 0; k < list.count; ++k)
        most = std::max(most, list.item[k].n);
    if (most == 0)
        return;
    const unsigned bx = (unsigned)std::min<size_t>((most + kNT - 1) / kNT, 2048);
    hipLaunchKernelGGL(k_copy_many, dim3(bx, list.count), dim3(kNT), 0, st, list);
}

void launch_copy_f32(hipStream_t st, const float* src, float* dst, size_t n)
{
    hipLaunchKernelGGL(k_copy_f32, dim3(linear_blocks(n)), dim3(kNT), 0, st, src, dst, n);
}

}  // namespace fsim
