// fs_viscosity_rows.hpp -- kernels of the implicit viscosity solve with their slots in registers (gfx950).
//
// A wavefront's 64 lanes are 64 neighbouring slot columns, each lane holding R rows of its column: coefficients,
// rhs, diagonal and velocity stay in registers through all sweeps of a launch.  A slot's horizontal neighbours come
// from the next lane (a DPP wavefront shift), its vertical ones from the same lane's other rows; only the first and
// last row of each wavefront pass through LDS.  Each shear stress is evaluated once per vertex (the smoothers on LDS
// tiles evaluated every one three times) and no sweep computes an index.
// Every slot of the tile is updated in every sweep; what lies outside it reads as zero, an error that moves one
// slot inwards per sweep, so the slots at least `halo` from the tile's edge hold what sweeps over the whole field give
// and only they are written.  Outside the field the velocity is zero: what a slot there contributes is
// multiplied by a vertex viscosity of zero.
//
// Measured against LDS-tile smoothers with separate residual, restriction, reduction, direction and update launches:
// an iteration of a solve on 641 x 363 170 -> 67 us (23 launches -> 12), on 1594 x 837 with four Chebyshev sweeps
// 400 -> 185, on 2048^2 545 -> 248, set-up included.
#pragma once

namespace fsim {

namespace {

// Element (row y, column x) of a slot field, clamped: the row's part is uniform in a wavefront.
template <class T> __device__ __forceinline__ T* slot_row(T* p, int w, int h, int y)
{
    return p + (size_t)min(max(y, 0), h) * (w + 1);
}

// The coefficients of R rows of a column: cell viscosity of rows -1 .. R - 1 and of the column to the left, vertex
// viscosity of rows 0 .. R, face masses, and which of the faces are unknowns.
template <int R> struct VisRows {
    float mu[R + 1];
    float left[R];
    float vert[R + 1];
    float mx[R], my[R];
    bool lane_u, lane_v;
    int y0, h;

    __device__ __forceinline__ bool u(int r) const { return lane_u && y0 + r >= 0 && y0 + r < h; }
    __device__ __forceinline__ bool v(int r) const { return lane_v && y0 + r > 0 && y0 + r < h; }

    __device__ __forceinline__ void load(const VLev& L, int x, int y)
    {
        y0 = y;
        h = L.h;
        lane_u = x > 0 && x < L.w;
        lane_v = x >= 0 && x < L.w;
        const int xc = min(max(x, 0), L.w);
        mu[0] = slot_row(L.coef, L.w, L.h, y - 1)[xc].x;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float4 c = slot_row(L.coef, L.w, L.h, y + r)[xc];
            mu[r + 1] = c.x;
            vert[r] = c.y;
            mx[r] = c.z;
            my[r] = c.w;
        }
        vert[R] = slot_row(L.coef, L.w, L.h, y + R)[xc].y;
#pragma unroll
        for (int r = 0; r < R; ++r)
            left[r] = from_left(mu[r + 1]);
    }

    // diagonal (ViscosityKernels.h:17-24)
    __device__ __forceinline__ float2 diagonal(int r, float dt) const
    {
        return make_float2(mx[r] + dt * (2.0f * (mu[r + 1] + left[r]) + vert[r] + vert[r + 1]),
            my[r] + dt * (2.0f * (mu[r + 1] + mu[r]) + vert[r] + from_right(vert[r])));
    }

    // product (ViscosityKernels.h:53-57), M s + dt K s, of rows 0 .. R - 1 (valid faces only), with the rows
    // above and below.
    __device__ __forceinline__ void product(const float2 (&s)[R], float2 up, float2 dn, float dt, float2 (&q)[R]) const
    {
        float t[R + 1];   // shear of rows 0 .. R
#pragma unroll
        for (int r = 0; r <= R; ++r) {
            const float2 c = r < R ? s[r < R ? r : 0] : dn;
            const float above = r ? s[r ? r - 1 : 0].x : up.x;
            t[r] = vert[r] * ((c.x - above) + (c.y - from_left(c.y)));
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float2 c = s[r];
            const float va = r ? s[r ? r - 1 : 0].y : up.y;
            const float vb = r + 1 < R ? s[r + 1 < R ? r + 1 : 0].y : dn.y;
            const float nu = 2.0f * (left[r] * (c.x - from_left(c.x)) + mu[r + 1] * (c.x - from_right(c.x)));
            const float nv = 2.0f * (mu[r] * (c.y - va) + mu[r + 1] * (c.y - vb));
            const float ku = nu + (t[r] - t[r + 1]);
            const float kv = nv + (t[r] - from_right(t[r]));
            q[r] = make_float2(mx[r] * c.x + dt * ku, my[r] * c.y + dt * kv);
        }
    }
};

// First and last rows of a workgroup's wavefronts, exchanged through LDS: publish, barrier, fetch; two buffers in
// turn, so one barrier per exchange.
template <int NW, int R> struct VisEdges {
    float2 row[2][NW][2][64];

    __device__ __forceinline__ void exchange(int buf, int wave, int lane, const float2 (&s)[R], float2& up, float2& dn)
    {
        row[buf][wave][0][lane] = s[0];
        row[buf][wave][1][lane] = s[R - 1];
        __syncthreads();
        up = row[buf][max(wave - 1, 0)][1][lane];        // the tile's own edge: stale, never used
        dn = row[buf][min(wave + 1, NW - 1)][0][lane];
    }
};

template <int R> __device__ __forceinline__ void vis_sweep(const VisRows<R>& c, float2 (&s)[R], const float2 (&b)[R],
    const float2 (&d)[R], float2 up, float2 dn, float dt, float wk)
{
    float2 q[R];
    c.product(s, up, dn, dt, q);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float vx = s[r].x + wk * (b[r].x - q[r].x) / d[r].x;
        const float vy = s[r].y + wk * (b[r].y - q[r].y) / d[r].y;
        s[r] = make_float2(c.u(r) ? vx : 0.0f, c.v(r) ? vy : 0.0f);
    }
}

// What the finest level's descent does on top of smoothing: the step of length alpha that the previous iteration
// left pending, r - alpha q for the rhs and x + alpha d for the iterate.
struct VisStep {
    const float2* r;   // residual before the step
    float2* r_new;
    const float2* q;
    const float2* d;
    float2* x;
};

__device__ __forceinline__ bool step_pending(const VisScalars* S) { return S->pending != 0 && S->restart == 0; }

// One level's way down (ViscosityKernels.h:187-236, 318-357): NS sweeps from zero, residual and transpose
// restriction in one launch.  Bound by VALU issue and HBM about equally on levels of a million slots (1594 x 837, NS 4:
// 27 us for 72 bytes a slot on the finest level), by the latency of one tile on small ones (4.6 us, 2.3 of it the
// launch).
template <int NS, int NW, int R, bool TOP>
__global__ __launch_bounds__(NW * 64) void k_vis_down(VLev L, VLev C, VisStep io, const VisScalars* S, VisSmooth M,
    int gx, int gy)
{
    constexpr int HALO = NS + 2;   // one ring per sweep, one for the residual, one for the restriction's taps
    constexpr int OX = 64 - 2 * HALO, OY = NW * R - 2 * HALO;
    static_assert(OY > 0 && R % 2 == 0 && HALO % 2 == 0, "tiles start on coarse slots");
    __shared__ VisEdges<NW, R> edges;
    __shared__ float2 res[NW * R][64];
    int bx, by;
    xcd_tile(gx, gy, bx, by);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int x = bx * OX - HALO + lane, y0 = by * OY - HALO + wave * R;
    const int w = L.w, h = L.h;
    VisRows<R> c;
    c.load(L, x, y0);
    float2 b[R], s[R], d[R];
    const int xc = min(max(x, 0), w);
    const float2* rhs = TOP ? io.r : (const float2*)L.b;
#pragma unroll
    for (int r = 0; r < R; ++r)
        b[r] = slot_row(rhs, w, h, y0 + r)[xc];
    float2 q[R];
    if (TOP) {
#pragma unroll
        for (int r = 0; r < R; ++r)
            q[r] = slot_row(io.q, w, h, y0 + r)[xc];
    }
    if (stopped(S))
        return;
    const float dt = S->dt;
    const bool own_x = lane >= HALO && lane < 64 - HALO && x <= w;
    auto own = [&](int r) {
        const int ty = wave * R + r;
        return own_x && ty >= HALO && ty < HALO + OY && y0 + r <= h;
    };
    if (TOP) {
        const bool apply = step_pending(S);
        const float alpha = (float)S->alpha;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (apply)
                b[r] = make_float2(b[r].x - alpha * q[r].x, b[r].y - alpha * q[r].y);
            if (own(r)) {
                const size_t i = (size_t)(y0 + r) * (w + 1) + x;
                io.r_new[i] = b[r];
                if (apply) {
                    const float2 dd = io.d[i], xx = io.x[i];
                    io.x[i] = make_float2(xx.x + alpha * dd.x, xx.y + alpha * dd.y);
                }
            }
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        d[r] = c.diagonal(r, dt);
        const float vx = M.w[0] * b[r].x / d[r].x, vy = M.w[0] * b[r].y / d[r].y;
        s[r] = make_float2(c.u(r) ? vx : 0.0f, c.v(r) ? vy : 0.0f);
    }
    float2 up, dn;
#pragma unroll
    for (int k = 1; k < NS; ++k) {
        edges.exchange(k & 1, wave, lane, s, up, dn);
        vis_sweep(c, s, b, d, up, dn, dt, M.w[k]);
    }
    edges.exchange(NS & 1, wave, lane, s, up, dn);
    c.product(s, up, dn, dt, q);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if (own(r))
            L.x[(size_t)(y0 + r) * (w + 1) + x] = s[r];
        res[wave * R + r][lane] = make_float2(c.u(r) ? b[r].x - q[r].x : 0.0f, c.v(r) ? b[r].y - q[r].y : 0.0f);
    }
    __syncthreads();
    // Restriction, the transpose of the face-location bilinear prolongation: along the face's own axis weights
    // 1/2, 1, 1/2, across it 1/4, 3/4, 3/4, 1/4, where a tap beyond the outermost coarse face folds onto it.
    constexpr int CX = OX / 2, CY = OY / 2;
    for (int e = threadIdx.x; e < CX * CY; e += NW * 64) {
        const int ex = e % CX, ey = e / CX;
        const int X = bx * CX + ex, Y = by * CY + ey;
        if (X > C.w || Y > C.h)
            continue;
        const int fx = HALO + 2 * ex, fy = HALO + 2 * ey;
        const float across_x[4] = {0.25f, X == 0 ? 1.0f : 0.75f, X == C.w - 1 ? 1.0f : 0.75f, 0.25f};
        const float across_y[4] = {0.25f, Y == 0 ? 1.0f : 0.75f, Y == C.h - 1 ? 1.0f : 0.75f, 0.25f};
        const float along[3] = {0.5f, 1.0f, 0.5f};
        float2 v = make_float2(0.0f, 0.0f);
#pragma unroll
        for (int dy = -1; dy <= 2; ++dy)
#pragma unroll
            for (int dx = -1; dx <= 1; ++dx)
                v.x += along[dx + 1] * across_y[dy + 1] * res[fy + dy][fx + dx].x;
#pragma unroll
        for (int dy = -1; dy <= 1; ++dy)
#pragma unroll
            for (int dx = -1; dx <= 2; ++dx)
                v.y += across_x[dx + 1] * along[dy + 1] * res[fy + dy][fx + dx].y;
        C.b[(size_t)Y * (C.w + 1) + X] =
            make_float2(X > 0 && X < C.w && Y < C.h ? v.x : 0.0f, Y > 0 && Y < C.h && X < C.w ? v.y : 0.0f);
    }
}

// F.x + P C.x of R rows of a column (ViscosityKernels.h:286-316, 359-391); y0 is even, so the coarse rows and
// weights of each row are known.
template <int R> __device__ __forceinline__ void vis_prolong(const VisRows<R>& c, const float2* cx, int cw, int ch,
    int x, int y0, float2 (&s)[R])
{
    const int k = x >> 1, base = y0 >> 1;
    const bool odd = x & 1;
    // columns of u: k, k + 1; of v: one to the left of them where x is even
    const int u0 = min(max(k, 0), cw), u1 = min(max(k + 1, 0), cw);
    const int kv = odd ? k : k - 1;
    const int v0 = min(max(kv, 0), cw - 1), v1 = min(max(kv + 1, 0), cw - 1);
    const float ux1 = odd ? 0.5f : 0.0f, ux0 = 1.0f - ux1;
    const float vx1 = odd ? 0.25f : 0.75f, vx0 = 1.0f - vx1;
    float a[R / 2 + 2][2], b[R / 2 + 1][2];
#pragma unroll
    for (int i = 0; i < R / 2 + 2; ++i) {
        const float2* row = cx + (size_t)min(max(base - 1 + i, 0), ch - 1) * (cw + 1);
        a[i][0] = row[u0].x;
        a[i][1] = row[u1].x;
    }
#pragma unroll
    for (int i = 0; i < R / 2 + 1; ++i) {
        const float2* row = cx + (size_t)min(max(base + i, 0), ch) * (cw + 1);
        b[i][0] = row[v0].y;
        b[i][1] = row[v1].y;
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int i = (r + 1) / 2;   // u: rows base - 1 + i and the next, 1/4 + 3/4 or 3/4 + 1/4
        const float uy1 = (r & 1) ? 0.25f : 0.75f, uy0 = 1.0f - uy1;
        float vx = s[r].x, vy = s[r].y;
        vx += ux0 * uy0 * a[i][0];
        vx += ux1 * uy0 * a[i][1];
        vx += ux0 * uy1 * a[i + 1][0];
        vx += ux1 * uy1 * a[i + 1][1];
        const int j = r / 2;         // v: row base + j alone, or half of it and half of the next
        const float vy1 = (r & 1) ? 0.5f : 0.0f, vy0 = 1.0f - vy1;
        vy += vx0 * vy0 * b[j][0];
        vy += vx1 * vy0 * b[j][1];
        if (r & 1) {
            vy += vx0 * vy1 * b[j + 1][0];
            vy += vx1 * vy1 * b[j + 1][1];
        }
        s[r] = make_float2(c.u(r) ? vx : 0.0f, c.v(r) ? vy : 0.0f);
    }
}

// r . z and r M^-1 r of a slot into (a, b, bad) (mode 1 of ViscosityKernels.h:395-470): a slot with a non-finite term adds
// nothing and raises the flag.
__device__ __forceinline__ void add_rz(float mx, float my, float2 r, float2 z, double (&v)[3])
{
    const double a = (double)r.x * z.x + (double)r.y * z.y;
    const double b = (double)r.x / mx * r.x + (double)r.y / my * r.y;
    const bool ok = isfinite(a) && isfinite(b);
    v[0] += ok ? a : 0.0;
    v[1] += ok ? b : 0.0;
    v[2] += ok ? 0.0 : 1.0;
}

// One level's way up: prolongation and NS sweeps (the weights in reverse), into L.xn; on the finest level also the
// partial sums of r . z and r M^-1 r.
template <int NS, int NW, int R, bool TOP>
__global__ __launch_bounds__(NW * 64) void k_vis_up(VLev L, VLev C, const float2* cx, const float2* rhs,
    const VisScalars* S, VisSmooth M, int gx, int gy, double* partials)
{
    constexpr int HALO = NS;
    constexpr int OX = 64 - 2 * HALO, OY = NW * R - 2 * HALO;
    static_assert(OY > 0 && R % 2 == 0 && HALO % 2 == 0, "tiles start on coarse slots");
    __shared__ VisEdges<NW, R> edges;
    __shared__ double lds[3 * NW];
    int bx, by;
    xcd_tile(gx, gy, bx, by);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int x = bx * OX - HALO + lane, y0 = by * OY - HALO + wave * R;
    const int w = L.w, h = L.h;
    VisRows<R> c;
    c.load(L, x, y0);
    float2 b[R], s[R], d[R];
    const int xc = min(max(x, 0), w);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        b[r] = slot_row(rhs, w, h, y0 + r)[xc];
        s[r] = slot_row((const float2*)L.x, w, h, y0 + r)[xc];
    }
    vis_prolong(c, cx, C.w, C.h, x, y0, s);
    if (stopped(S))
        return;
    const float dt = S->dt;
#pragma unroll
    for (int r = 0; r < R; ++r)
        d[r] = c.diagonal(r, dt);
    float2 up, dn;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        edges.exchange(k & 1, wave, lane, s, up, dn);
        vis_sweep(c, s, b, d, up, dn, dt, M.w[NS - 1 - k]);
    }
    double sums[3] = {0.0, 0.0, 0.0};
    const bool own_x = lane >= HALO && lane < 64 - HALO && x <= w;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int ty = wave * R + r;
        if (own_x && ty >= HALO && ty < HALO + OY && y0 + r <= h) {
            L.xn[(size_t)(y0 + r) * (w + 1) + x] = s[r];
            if (TOP)
                add_rz(c.mx[r], c.my[r], b[r], s[r], sums);
        }
    }
    if (TOP) {
        block_sums<NW * 64, 3>(sums, lds);
        if (threadIdx.x == 0) {
#pragma unroll
            for (int i = 0; i < 3; ++i)
                partials[3 * blockIdx.x + i] = sums[i];
        }
    }
}

// Operator kernels: each wavefront takes 62 columns of R rows with the ring around them, no exchange.
enum VisApplyMode : int { kVisDirection = 0, kVisTruthOf, kVisInitialOf };

struct VisApply {
    const float2* z;       // direction: preconditioned residual
    const float2* d;       // last direction
    float2* d_new;
    float2* q;             // direction: A d; truth: the recomputed residual; initial: the rhs
    float2* x;             // iterate
    float2* v0;
    const double* u64;     // initial: the velocity
    const double* v64;
    float dt;              // initial
};

// direction (d = z + beta d, q = A d, d . q), recomputed residual M v0 - A (x + alpha d) and its norm, or the set-up
// (v0, x = v0, r = M v0 - A v0 and the sums of mode 0), by MODE.  Bound by HBM on large grids, by latency below.
template <int MODE, int R>
__global__ __launch_bounds__(kVT) void k_vis_apply(VLev L, VisApply io, const VisScalars* S, int gx, int gy,
    double* partials)
{
    constexpr int NC = MODE == kVisInitialOf ? 4 : 2;
    __shared__ double lds[NC * (kVT / 64)];
    int bx, by;
    xcd_tile(gx, gy, bx, by);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int x = bx * 62 - 1 + lane, y0 = (by * (kVT / 64) + wave) * R;
    const int w = L.w, h = L.h;
    const int xc = min(max(x, 0), w);
    VisRows<R> c;
    c.load(L, x, y0);
    float2 s[R], up, dn, start[R];
    auto rows = [&](auto get) {
        up = get(-1);
        dn = get(R);
#pragma unroll
        for (int r = 0; r < R; ++r)
            s[r] = get(r);
    };
    float dt;
    if constexpr (MODE == kVisInitialOf) {
        dt = io.dt;
        rows([&](int r) {
            const int y = y0 + r;
            const float su = (float)io.u64[(size_t)min(max(y, 0), h - 1) * (w + 1) + xc];
            const float sv = (float)io.v64[(size_t)min(max(y, 0), h) * w + min(xc, w - 1)];
            return make_float2(c.u(r) ? su : 0.0f, c.v(r) ? sv : 0.0f);
        });
    } else {
        float2 last[R + 2], now[R + 2];
        const float2* base = MODE == kVisDirection ? io.z : (const float2*)io.x;
#pragma unroll
        for (int r = 0; r < R + 2; ++r) {
            now[r] = slot_row(base, w, h, y0 + r - 1)[xc];
            last[r] = slot_row(io.d, w, h, y0 + r - 1)[xc];
        }
        if (MODE == kVisTruthOf) {
#pragma unroll
            for (int r = 0; r < R; ++r)
                start[r] = slot_row((const float2*)io.v0, w, h, y0 + r)[xc];
        }
        if (MODE == kVisDirection ? stopped(S) : S->done != 0)
            return;
        dt = S->dt;
        const bool add = MODE == kVisDirection ? S->steps > 0 : step_pending(S);
        const float f = (float)(MODE == kVisDirection ? S->beta : S->alpha);
        rows([&](int r) {
            const float2 a = now[r + 1], b = last[r + 1];
            // faces that are no unknowns hold zeros; so does what lies outside the field
            const bool in = x >= 0 && x <= w && y0 + r >= 0 && y0 + r <= h;
            return make_float2(in ? (add ? a.x + f * b.x : a.x) : 0.0f, in ? (add ? a.y + f * b.y : a.y) : 0.0f);
        });
    }
    float2 q[R];
    c.product(s, up, dn, dt, q);
    double sums[NC] = {};
    const bool own_x = lane >= 1 && lane < 63 && x <= w;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if (!own_x || y0 + r > h)
            continue;
        const size_t i = (size_t)(y0 + r) * (w + 1) + x;
        const bool vu = c.u(r), vv = c.v(r);
        if constexpr (MODE == kVisDirection) {
            const float2 out = make_float2(vu ? q[r].x : 0.0f, vv ? q[r].y : 0.0f);
            io.d_new[i] = s[r];
            io.q[i] = out;
            const double a = (double)s[r].x * out.x + (double)s[r].y * out.y;
            const bool ok = isfinite(a);
            sums[0] += ok ? a : 0.0;
            sums[1] += ok ? 0.0 : 1.0;
        } else {
            const float2 v0 = MODE == kVisTruthOf ? start[r] : s[r];
            const float2 out =
                make_float2(vu ? c.mx[r] * v0.x - q[r].x : 0.0f, vv ? c.my[r] * v0.y - q[r].y : 0.0f);
            io.q[i] = out;
            const double a = (double)out.x / c.mx[r] * out.x + (double)out.y / c.my[r] * out.y;
            if constexpr (MODE == kVisTruthOf) {
                const bool ok = isfinite(a);
                sums[0] += ok ? a : 0.0;
                sums[1] += ok ? 0.0 : 1.0;
            } else {
                io.v0[i] = s[r];
                io.x[i] = s[r];
                const double b = (double)c.mx[r] * s[r].x * s[r].x + (double)c.my[r] * s[r].y * s[r].y;
                const double m = (double)c.mx[r] + (double)c.my[r];
                const bool ok = isfinite(a) && isfinite(b) && isfinite(m);
                sums[0] += ok ? a : 0.0;
                sums[1] += ok ? b : 0.0;
                sums[2] += ok ? m : 0.0;
                sums[3] += ok ? 0.0 : 1.0;
            }
        }
    }
    block_sums<kVT, NC>(sums, lds);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int i = 0; i < NC; ++i)
            partials[NC * blockIdx.x + i] = sums[i];
    }
}

// The coarse end of a V-cycle in one workgroup, a slot of every level per thread: coefficients, rhs, diagonal and
// solution of up to kVisTailLevels levels stay in the slot's thread, only velocities and residuals pass through LDS
// (where every slot's neighbours lie).
// Bound by the chain of about 40 dependent LDS exchanges: 14.9 us per cycle on levels of 42 x 24, 22 x 13, 12 x 7
// and 7 x 4 slots, where the same sweeps on levels in global memory took 48.
constexpr int kVisTailSlots = 1024;
constexpr int kVisTailLevels = 4;

struct VisTail {
    VLev lev[kVisTailLevels];
    VisSmooth M;
};

struct VisSlot {
    float mu, left, up, vert, vdn, vrt, mx, my;
    float2 diag;
    int xy;                      // slot position, x | y << 16
    int l, r, u, d;              // LDS indices of the neighbours (clamped into the field)
    bool in, vu, vv;

    __device__ __forceinline__ int x() const { return xy & 0xffff; }
    __device__ __forceinline__ int y() const { return xy >> 16; }

    // Slot e of a level of w x h cells with the coefficients at `coef`.
    __device__ __forceinline__ void init(int w, int h, const float4* coef, int e, float dt)
    {
        const int st = w + 1;
        in = e < st * (h + 1);
        const int i = in ? e : 0;
        const int y = i / st, x = i - y * st;
        xy = x | y << 16;
        l = i - (x > 0 ? 1 : 0);
        r = i + (x < w ? 1 : 0);
        u = y > 0 ? i - st : i;
        d = y < h ? i + st : i;
        const float4 c = coef[i];
        mu = c.x;
        vert = c.y;
        mx = c.z;
        my = c.w;
        left = coef[l].x;
        up = coef[u].x;
        vdn = coef[d].y;
        vrt = coef[r].y;
        vu = in && x > 0 && x < w && y < h;
        vv = in && y > 0 && y < h && x < w;
        diag = make_float2(mx + dt * (2.0f * (mu + left) + vert + vdn), my + dt * (2.0f * (mu + up) + vert + vrt));
    }

    __device__ __forceinline__ float2 product(const float2* s, int e, float2 c, float dt) const
    {
        const float2 sl = s[l], sr = s[r], su = s[u], sd = s[d], sld = s[d + l - e], sru = s[u + r - e];
        const float t = vert * ((c.x - su.x) + (c.y - sl.y));
        const float td = vdn * ((sd.x - c.x) + (sd.y - sld.y));
        const float tr = vrt * ((sr.x - sru.x) + (sr.y - c.y));
        const float nu = 2.0f * (left * (c.x - sl.x) + mu * (c.x - sr.x));
        const float nv = 2.0f * (up * (c.y - su.y) + mu * (c.y - sd.y));
        return make_float2(mx * c.x + dt * (nu + (t - td)), my * c.y + dt * (nv + (t - tr)));
    }

    __device__ __forceinline__ float2 sweep(const float2* s, int e, float2 c, float2 b, float dt,
        float wk) const
    {
        const float2 q = product(s, e, c, dt);
        const float vx = c.x + wk * (b.x - q.x) / diag.x, vy = c.y + wk * (b.y - q.y) / diag.y;
        return make_float2(vu ? vx : 0.0f, vv ? vy : 0.0f);
    }
};

// Restriction of the residuals at `res` (fine slots, w x h) to a coarse slot, as in k_vis_down.
__device__ __forceinline__ float2 restrict_slot(const float2* res, int w, int h, int cw, int ch, const VisSlot& c)
{
    const int X = c.x(), Y = c.y();
    const float across_x[4] = {0.25f, X == 0 ? 1.0f : 0.75f, X == cw - 1 ? 1.0f : 0.75f, 0.25f};
    const float across_y[4] = {0.25f, Y == 0 ? 1.0f : 0.75f, Y == ch - 1 ? 1.0f : 0.75f, 0.25f};
    const float along[3] = {0.5f, 1.0f, 0.5f};
    float2 v = make_float2(0.0f, 0.0f);
    auto at = [&](int x, int y) {
        const float2 r = res[min(max(y, 0), h) * (w + 1) + min(max(x, 0), w)];
        const bool in = x >= 0 && y >= 0 && x <= w && y <= h;
        return make_float2(in ? r.x : 0.0f, in ? r.y : 0.0f);
    };
#pragma unroll
    for (int dy = -1; dy <= 2; ++dy)
#pragma unroll
        for (int dx = -1; dx <= 1; ++dx)
            v.x += along[dx + 1] * across_y[dy + 1] * at(2 * X + dx, 2 * Y + dy).x;
#pragma unroll
    for (int dy = -1; dy <= 1; ++dy)
#pragma unroll
        for (int dx = -1; dx <= 2; ++dx)
            v.y += across_x[dx + 1] * along[dy + 1] * at(2 * X + dx, 2 * Y + dy).y;
    return make_float2(c.vu ? v.x : 0.0f, c.vv ? v.y : 0.0f);
}

// s + P c of a fine slot, c the coarse solution (cw x ch slots) in LDS.
__device__ __forceinline__ float2 prolong_slot(const VisSlot& f, float2 s, const float2* c, int cw, int ch)
{
    const int st = cw + 1;
    const bool ox = f.x() & 1, oy = f.y() & 1;
    const int k = f.x() >> 1, j = f.y() >> 1;
    const float ux[2] = {ox ? 0.5f : 1.0f, ox ? 0.5f : 0.0f}, uy[2] = {oy ? 0.75f : 0.25f, oy ? 0.25f : 0.75f};
    const float vx[2] = {ox ? 0.75f : 0.25f, ox ? 0.25f : 0.75f}, vy[2] = {oy ? 0.5f : 1.0f, oy ? 0.5f : 0.0f};
    const int ju = oy ? j : j - 1, kv = ox ? k : k - 1;
#pragma unroll
    for (int dy = 0; dy < 2; ++dy)
#pragma unroll
        for (int dx = 0; dx < 2; ++dx) {
            s.x += ux[dx] * uy[dy] * c[min(max(ju + dy, 0), ch - 1) * st + min(k + dx, cw)].x;
            s.y += vx[dx] * vy[dy] * c[min(j + dy, ch) * st + min(max(kv + dx, 0), cw - 1)].y;
        }
    return make_float2(f.vu ? s.x : 0.0f, f.vv ? s.y : 0.0f);
}

template <int NL>
__global__ __launch_bounds__(kVisTailSlots) void k_vis_tail(VisTail T, const float2* rhs, const VisScalars* S)
{
    // per level two buffers of velocities; a level below the first has at most half its slots and one column or row
    constexpr int kSlots[4] = {1024, 544, 320, 192};
    constexpr int kOffset[4] = {0, 2 * 1024, 2 * (1024 + 544), 2 * (1024 + 544 + 320)};
    __shared__ float2 lds[2 * (1024 + 544 + 320 + 192)];
    const float dt = S->dt;
    const int e = threadIdx.x;
    VisSlot slot[NL];
    float2 b[NL], x[NL];
    b[0] = rhs[min(e, (T.lev[0].w + 1) * (T.lev[0].h + 1) - 1)];
#pragma unroll
    for (int l = 0; l < NL; ++l)
        slot[l].init(T.lev[l].w, T.lev[l].h, T.lev[l].coef, e, dt);
    if (stopped(S))
        return;
#pragma unroll
    for (int l = 0; l + 1 < NL; ++l) {
        auto buf = [&](int i) { return lds + kOffset[l] + i * kSlots[l]; };
        const VisSlot& c = slot[l];
        const float vx = T.M.w[0] * b[l].x / c.diag.x, vy = T.M.w[0] * b[l].y / c.diag.y;
        x[l] = make_float2(c.vu ? vx : 0.0f, c.vv ? vy : 0.0f);
        for (int k = 1; k <= T.M.sweeps; ++k) {   // an even count: the last sweep's values lie in buf(1)
            if (c.in)
                buf((k - 1) & 1)[e] = x[l];
            __syncthreads();
            if (k < T.M.sweeps) {
                if (c.in)
                    x[l] = c.sweep(buf((k - 1) & 1), e, x[l], b[l], dt, T.M.w[k]);
            }
        }
        if (c.in) {
            const float2 q = c.product(buf(1), e, x[l], dt);
            buf(0)[e] = make_float2(c.vu ? b[l].x - q.x : 0.0f, c.vv ? b[l].y - q.y : 0.0f);
        }
        __syncthreads();
        const VLev &F = T.lev[l], &C = T.lev[l + 1];
        if (slot[l + 1].in)
            b[l + 1] = restrict_slot(buf(0), F.w, F.h, C.w, C.h, slot[l + 1]);
    }
    // the coarsest level: 16 sweeps from zero (ViscosityKernels.h:242-282), the last one's values in buffer 0
    {
        auto buf = [&](int i) { return lds + kOffset[NL - 1] + i * kSlots[NL - 1]; };
        const VisSlot& c = slot[NL - 1];
        float2 v = make_float2(0.0f, 0.0f);
        for (int k = 0; k < 16; ++k) {
            if (c.in)
                buf(k & 1)[e] = v;
            __syncthreads();
            if (c.in)
                v = c.sweep(buf(k & 1), e, v, b[NL - 1], dt, 0.5f);
        }
        if (c.in) {
            if (NL == 1)
                T.lev[0].x[e] = v;
            else
                buf(0)[e] = v;
        }
    }
#pragma unroll
    for (int l = NL - 2; l >= 0; --l) {
        __syncthreads();
        auto buf = [&](int i) { return lds + kOffset[l] + i * kSlots[l]; };
        const VisSlot& c = slot[l];
        if (c.in)
            x[l] = prolong_slot(c, x[l], lds + kOffset[l + 1], T.lev[l + 1].w, T.lev[l + 1].h);
        for (int k = 0; k < T.M.sweeps; ++k) {
            if (c.in)
                buf(k & 1)[e] = x[l];
            __syncthreads();
            if (c.in)
                x[l] = c.sweep(buf(k & 1), e, x[l], b[l], dt, T.M.w[T.M.sweeps - 1 - k]);
        }
        if (c.in) {
            if (l == 0)
                T.lev[0].x[e] = x[0];
            else
                buf(0)[e] = x[l];
        }
    }
}

}  // namespace

}  // namespace fsim
