// kx_eikonal.hip -- first-arrival traveltimes by fast sweeping
// (include/kirchx.h: kx_eikonal).
//
// Replaces the scikit-fmm calls of Kirchhoff._traveltime_table's eikonal
// mode (pylops/waveeqprocessing/kirchhoff.py:609-638): for every source
// cell, the traveltime (or, with unit slowness, the distance) from the zero
// contour of phi = -1 at that cell and +1 elsewhere.
//
// Method (Zhao 2005, fast sweeping): Godunov upwind updates of |grad T| = s,
// swept over the grid in the 4 (2D) or 8 (3D) diagonal orderings, repeated
// until no value changes: first-order updates to convergence, then (order
// 2, scikit-fmm's default order) second-order one-sided differences where
// the two upwind cells are monotone, lowering values until they converge.  Within one sweep every cell
// of an anti-diagonal ix' + iy' + iz' = d (primed: index counted along the
// sweep's direction) depends only on the diagonals before it, so one launch
// updates a whole diagonal for every source at once.  Cells within two
// cells of the source (per axis) start at the straight-ray time from the
// contour -- a diamond through the half-way points to the neighbouring cell
// centres, where phi interpolates to zero -- and stay fixed.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <vector>

#include "kirchx.h"

extern "C" int kx_solver_fail(int code, const char *msg);

namespace {

constexpr double kBig = 1e30;
// a workgroup is kEikSrc sources (one wave, adjacent in memory) x
// kEikCells cells
constexpr int kEikSrc = 64;
constexpr int kEikCells = 4;
constexpr int kEikBlock = kEikSrc * kEikCells;
constexpr int kInitRadius = 2;

int efail(int code, const char *fmt, ...)
{
    char buf[480];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    return kx_solver_fail(code, buf);
}

struct EikArgs {
    int nx, ny, nz;
    double hx, hy, hz;
    int three;     // 1 in 3D
    int n;         // sources
    int64_t ni;
};

// One axis of the upwind update: upwind value a (the smaller neighbour,
// kBig when there is none), difference base b and step g, so that the
// one-sided derivative is (t - b) / g.  First order: b = a, g = h.  Second
// order, where the second cell on the upwind side is known and not above
// the first: (3t - 4a + a2) / (2h), i.e. b = (4a - a2) / 3, g = 2h / 3.
struct Axis {
    double a, b, g;
};

// l1, l2: the neighbours one and two cells below on the axis, r1, r2 above
// (kBig outside the grid).
__device__ __forceinline__ Axis axis_terms(double l1, double l2, double r1, double r2, double h,
                                           int order)
{
    const bool low = l1 <= r1;
    const double a1 = low ? l1 : r1, a2 = low ? l2 : r2;
    Axis x{a1, a1, h};
    if (order == 2 && a1 < kBig && a2 < kBig && a2 <= a1) {
        x.b = fma(4.0, a1, -a2) / 3.0;
        x.g = (2.0 / 3.0) * h;
    }
    return x;
}

__device__ __forceinline__ Axis axis_terms(const double *Ts, int64_t c, int i, int n,
                                           int64_t stride, double h, int order)
{
    return axis_terms(i > 0 ? Ts[c - stride] : kBig, i > 1 ? Ts[c - 2 * stride] : kBig,
                      i < n - 1 ? Ts[c + stride] : kBig, i < n - 2 ? Ts[c + 2 * stride] : kBig, h,
                      order);
}

__device__ __forceinline__ void order_axes(Axis &u, Axis &v)
{
    if (v.a < u.a) {
        const Axis t = u;
        u = v;
        v = t;
    }
}

// Godunov update: the largest t with sum_k ((t - b_k) / g_k)^2 = s^2 over
// the axes whose upwind value a_k lies below t, taken in increasing a_k.
// *ok is cleared when a quadratic has no real root (possible only with
// second-order terms).
__device__ __forceinline__ double solve_upwind(Axis x0, Axis x1, Axis x2, double s, int three,
                                               bool *ok)
{
    order_axes(x0, x1);
    if (three) {
        order_axes(x1, x2);
        order_axes(x0, x1);
    }
    // (sums of products fused by hand: solve2 rounds the same way)
    *ok = true;
    double t = fma(s, x0.g, x0.b);
    if (t > x1.a) {
        const double w0 = 1.0 / (x0.g * x0.g), w1 = 1.0 / (x1.g * x1.g);
        double A = w0 + w1;
        double B = fma(x1.b, w1, x0.b * w0);
        double C = fma(x1.b * x1.b, w1, fma(x0.b * x0.b, w0, -(s * s)));
        double D = fma(B, B, -(A * C));
        *ok = D >= 0.0;
        t = (B + sqrt(fmax(D, 0.0))) / A;
        if (three && t > x2.a) {
            const double w2 = 1.0 / (x2.g * x2.g);
            A += w2;
            B = fma(x2.b, w2, B);
            C = fma(x2.b * x2.b, w2, C);
            D = fma(B, B, -(A * C));
            *ok = *ok && D >= 0.0;
            t = (B + sqrt(fmax(D, 0.0))) / A;
        }
    }
    return t;
}

// The cell's update; with a quadratic without a root, its first-order one.
__device__ __forceinline__ double cell_update(const EikArgs &g, const Axis &ax, const Axis &ay,
                                              const Axis &az, double sl)
{
    bool ok;
    // axes in the order x, z, y (the third only in 3D)
    double t = solve_upwind(ax, az, ay, sl, g.three, &ok);
    if (!ok) {
        const Axis fx = {ax.a, ax.a, g.hx}, fy = {ay.a, ay.a, g.hy}, fz = {az.a, az.a, g.hz};
        t = solve_upwind(fx, fz, fy, sl, g.three, &ok);
    }
    return t;
}

// Straight-ray time from the contour of the source cell (sx, sy, sz) to cell
// (ix, iy, iz) inside the fixed box, kBig elsewhere.
__device__ __forceinline__ double start_value(const EikArgs &g, const double *__restrict__ slow,
                                              int ix, int iy, int iz, int sx, int sy, int sz)
{
    if (abs(ix - sx) > kInitRadius || abs(iy - sy) > kInitRadius || abs(iz - sz) > kInitRadius)
        return kBig;
    const double dx = (ix - sx) * g.hx, dy = (iy - sy) * g.hy, dz = (iz - sz) * g.hz;
    const double rho = sqrt(dx * dx + dy * dy + dz * dz);
    // the contour in this direction lies at rho / S
    const double S = 2.0 * (fabs(dx) / g.hx + fabs(dz) / g.hz + (g.three ? fabs(dy) / g.hy : 0.0));
    const int64_t c = ((int64_t)iy * g.nx + ix) * g.nz + iz;
    const int64_t cs = ((int64_t)sy * g.nx + sx) * g.nz + sz;
    const double sl = 0.5 * (slow[c] + slow[cs]);
    return S > 0.0 ? sl * rho * fmax(0.0, 1.0 - 1.0 / S) : 0.0;
}

// T = start_value.  One thread per (cell, source); T[c * n + s].
__global__ __launch_bounds__(kEikBlock) void eik_init_kernel(EikArgs g,
                                                             const double *__restrict__ slow,
                                                             const int *__restrict__ src,
                                                             double *__restrict__ T)
{
    const int s = blockIdx.y * kEikSrc + threadIdx.x;
    const int64_t c = (int64_t)blockIdx.x * kEikCells + threadIdx.y;
    if (c >= g.ni || s >= g.n)
        return;
    const int iz = (int)(c % g.nz);
    const int ix = (int)((c / g.nz) % g.nx);
    const int iy = (int)(c / ((int64_t)g.nz * g.nx));
    T[c * g.n + s] =
        start_value(g, slow, ix, iy, iz, src[3 * s], src[3 * s + 1], src[3 * s + 2]);
}

// One anti-diagonal d of one sweep direction (dx, dy, dz = +1 / -1), every
// source: thread (pair, source) with pair = (ix' - ixlo) * ny + iy'.  The
// cells of a diagonal are never adjacent in memory, so the tables are
// point-major (T[c * n + s]) and the lanes of a wave take adjacent sources
// of one cell: every load and store is one contiguous 512-byte row.
// order 2 takes second-order terms where they apply and falls back to the
// first-order update of the cell when a quadratic has no root.
__global__ __launch_bounds__(kEikBlock) void eik_sweep_kernel(EikArgs g,
                                                              const double *__restrict__ slow,
                                                              const int *__restrict__ src,
                                                              double *__restrict__ T, int d,
                                                              int dx, int dy, int dz, int ixlo,
                                                              int nix, int order, int *changed)
{
    const int s = blockIdx.y * kEikSrc + threadIdx.x;
    const int64_t pair = (int64_t)blockIdx.x * kEikCells + threadIdx.y;
    if (pair >= (int64_t)nix * g.ny || s >= g.n)
        return;
    const int px = ixlo + (int)(pair / g.ny);
    const int py = (int)(pair % g.ny);
    const int pz = d - px - py;
    if (pz < 0 || pz >= g.nz)
        return;
    const int ix = dx > 0 ? px : g.nx - 1 - px;
    const int iy = dy > 0 ? py : g.ny - 1 - py;
    const int iz = dz > 0 ? pz : g.nz - 1 - pz;
    const int sx = src[3 * s], sy = src[3 * s + 1], sz = src[3 * s + 2];
    if (abs(ix - sx) <= kInitRadius && abs(iy - sy) <= kInitRadius &&
        abs(iz - sz) <= kInitRadius)
        return;  // fixed
    const int64_t c = ((int64_t)iy * g.nx + ix) * g.nz + iz;
    const int64_t e = c * g.n + s;
    const int64_t szs = g.n, sxs = (int64_t)g.nz * g.n, sys = (int64_t)g.nx * g.nz * g.n;
    const double sl = slow[c];
    const Axis ax = axis_terms(T, e, ix, g.nx, sxs, g.hx, order);
    const Axis az = axis_terms(T, e, iz, g.nz, szs, g.hz, order);
    Axis ay = {kBig, kBig, g.hy};
    if (g.three)
        ay = axis_terms(T, e, iy, g.ny, sys, g.hy, order);
    const double t = cell_update(g, ax, ay, az, sl);
    const double old = T[e];
    if (t < old) {
        T[e] = t;
        if (old - t > 1e-13 * t)
            *changed = 1;
    }
}

// All sweeps of one source of a 2D grid in one workgroup, every source in one
// launch.  (One launch per anti-diagonal: 301x151 with 21 + 101 tables, 18040
// launches of 3.4 us, 61 ms; here 5.3 ms.)  What bounds it is the chain of
// steps: about 1250 clocks each, a barrier, an exchange through LDS and the
// dependent double arithmetic of one update, whatever the number of tables
// (one workgroup each, 122 on 256 CUs).
// Lane i holds column i of the shorter axis (np <= 1024 columns) and walks
// along the other one; at step d of a sweep it updates cell w = d - p of its
// column, p its place in the sweep's direction: the cells of step d are one
// anti-diagonal, updated from the same values and in the same order as
// eik_sweep_kernel's.  A column's values arrive kAhead steps ahead in
// registers; neighbouring columns exchange theirs through LDS: the value
// just updated (read by lane p + 1 at the next step and p + 2 at the one
// after) and the old ones one and two cells ahead (read by lanes p - 1 and
// p - 2).  One barrier per step.  A source stops when its own round changes
// nothing.  W[s][cell] in the grid's order; stat: [phase - 1] the most rounds
// of a source, [2] set when one did not converge.
constexpr int kAhead = 8;
constexpr int kSweepThreads = 1024;

// x / 3 as a division rounds it, in three operations: the product with the
// rounded reciprocal, corrected by its fused residual (Markstein's correction
// of a quotient; |x| well inside the normal range: times, and 1e30 for none).
__device__ __forceinline__ double third(double x)
{
    const double r = 1.0 / 3.0, q = x * r;
    return fma(fma(-3.0, q, x), r, q);
}

// axis_terms and solve_upwind for two axes whose steps and their inverse
// squares (first and second order) are known: the divisions a step would
// otherwise wait for.
struct Step {
    double g1, g2, w1, w2;
};
__device__ __forceinline__ Step make_step(double h)
{
    const double g2 = (2.0 / 3.0) * h;
    return {h, g2, 1.0 / (h * h), 1.0 / (g2 * g2)};
}
struct Axis2 {
    double a, b, g, w;
};
__device__ __forceinline__ Axis2 axis2(double l1, double l2, double r1, double r2, const Step &h,
                                       bool second)
{
    const bool low = l1 <= r1;
    const double a1 = low ? l1 : r1, a2 = low ? l2 : r2;
    const bool use = second && a1 < kBig && a2 < kBig && a2 <= a1;
    return {a1, use ? third(fma(4.0, a1, -a2)) : a1, use ? h.g2 : h.g1, use ? h.w2 : h.w1};
}
__device__ __forceinline__ double solve2(const Axis2 &x, const Axis2 &z, double s, bool *ok)
{
    const bool swap = z.a < x.a;  // the upwind axis first
    const double a1 = swap ? x.a : z.a;
    const double b0 = swap ? z.b : x.b, b1 = swap ? x.b : z.b;
    const double w0 = swap ? z.w : x.w, w1 = swap ? x.w : z.w;
    const double t1 = fma(s, swap ? z.g : x.g, b0);
    const double A = w0 + w1;
    const double B = fma(b1, w1, b0 * w0);
    const double C = fma(b1 * b1, w1, fma(b0 * b0, w0, -(s * s)));
    const double D = fma(B, B, -(A * C));
    const double t2 = (B + sqrt(fmax(D, 0.0))) / A;
    *ok = !(t1 > a1) || D >= 0.0;
    return t1 > a1 ? t2 : t1;
}

__device__ __forceinline__ void step_barrier()
{
    // LDS only: the loads ahead and the stores stay in flight
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

__global__ __launch_bounds__(kSweepThreads) void eik_sweep2d_kernel(EikArgs g,
                                                                    const double *__restrict__ slow,
                                                                    const int *__restrict__ src,
                                                                    double *W, int walk_x,
                                                                    int max_iter, int order,
                                                                    int *__restrict__ stat)
{
    extern __shared__ double eik_lds[];
    const int np = walk_x ? g.nz : g.nx, nw = walk_x ? g.nx : g.nz;
    const int sp = walk_x ? 1 : g.nz, sw = walk_x ? g.nz : 1;
    const int row = np + 4;          // two cells of kBig at either end
    double *fresh = eik_lds;         // [4][row] updated values of the last steps
    double *next1 = fresh + 4 * row; // [2][row] old values one cell ahead
    double *next2 = next1 + 2 * row; // [2][row] two cells ahead
    const int s = blockIdx.x, i = threadIdx.x;
    const bool lane_on = i < np;
    const int ic = min(i, np - 1);
    const int sx = src[3 * s], sz = src[3 * s + 2];
    double *Tc = W + (int64_t)s * g.ni + (int64_t)ic * sp;
    const double *sc = slow + (int64_t)ic * sp;
    const int cp = walk_x ? sz : sx, cw = walk_x ? sx : sz;  // the source's column and cell
    const bool near = abs(ic - cp) <= kInitRadius;
    const Step hp = make_step(walk_x ? g.hz : g.hx), hw = make_step(walk_x ? g.hx : g.hz);

    if (lane_on)
        for (int w = 0; w < nw; ++w)
            Tc[(int64_t)w * sw] = walk_x ? start_value(g, slow, w, 0, i, sx, 0, sz)
                                         : start_value(g, slow, i, 0, w, sx, 0, sz);
    for (int phase = 1; phase <= order; ++phase) {
        int it = 0, changed = 1;
        while (changed && it < max_iter) {
            ++it;
            changed = 0;
            for (int q = 0; q < 4; ++q) {
                const int dx = (q & 1) ? -1 : 1, dz = (q & 2) ? -1 : 1;
                const int dp = walk_x ? dz : dx, dw = walk_x ? dx : dz;
                const int p = dp > 0 ? ic : np - 1 - ic;
                // cell w of the sweep lies at (dw > 0 ? w : nw - 1 - w)
                auto at = [&](int w) -> int64_t {
                    const int c = min(max(w, 0), nw - 1);
                    return (int64_t)(dw > 0 ? c : nw - 1 - c) * sw;
                };
                auto inside = [&](int w) { return (unsigned)w < (unsigned)nw; };
                __syncthreads();  // the last sweep's exchanges are read
                for (int k = i; k < 8 * row; k += blockDim.x)
                    eik_lds[k] = kBig;
                double old[kAhead], sl[kAhead];
#pragma unroll
                for (int k = 0; k < kAhead; ++k) {
                    old[k] = Tc[at(k - p)];
                    sl[k] = sc[at(k - p)];
                }
                __syncthreads();
                if (lane_on) {
                    next1[i + 2] = inside(1 - p) ? old[1] : kBig;
                    next2[i + 2] = inside(2 - p) ? old[2] : kBig;
                }
                step_barrier();
                double n1 = kBig, n2 = kBig;  // this column's last two updated values
                const int nd = np + nw - 1;
                for (int d0 = 0; d0 < nd; d0 += kAhead) {
#pragma unroll
                    for (int u = 0; u < kAhead; ++u) {
                        const int d = d0 + u, w = d - p;
                        const bool on = lane_on && inside(w);
                        // (lanes without a cell compute and drop a value)
                        const double pa = fresh[((d - 1) & 3) * row + ic + 2 - dp];
                        const double pb = fresh[((d - 2) & 3) * row + ic + 2 - 2 * dp];
                        const double na = next1[(d & 1) * row + ic + 2 + dp];
                        const double nb = next2[(d & 1) * row + ic + 2 + 2 * dp];
                        const double oa = inside(w + 1) ? old[(u + 1) % kAhead] : kBig;
                        const double ob = inside(w + 2) ? old[(u + 2) % kAhead] : kBig;
                        auto update = [&](bool second, bool *ok) {
                            const Axis2 vp = dp > 0 ? axis2(pa, pb, na, nb, hp, second)
                                                    : axis2(na, nb, pa, pb, hp, second);
                            const Axis2 vw = dw > 0 ? axis2(n1, n2, oa, ob, hw, second)
                                                    : axis2(oa, ob, n1, n2, hw, second);
                            return walk_x ? solve2(vw, vp, sl[u], ok) : solve2(vp, vw, sl[u], ok);
                        };
                        bool ok;
                        double t = update(phase == 2, &ok);
                        if (__builtin_expect(!ok, 0))
                            t = update(false, &ok);
                        const double o = old[u];
                        const int phys = dw > 0 ? w : nw - 1 - w;
                        const bool fixed = near && abs(phys - cw) <= kInitRadius;
                        double v = kBig;
                        if (on) {
                            v = o;
                            if (!fixed && t < o) {
                                v = t;
                                Tc[at(w)] = t;
                                changed |= o - t > 1e-13 * t;
                            }
                        }
                        n2 = n1;
                        n1 = v;
                        if (lane_on) {
                            fresh[(d & 3) * row + i + 2] = v;
                            next1[((d + 1) & 1) * row + i + 2] =
                                inside(w + 2) ? old[(u + 2) % kAhead] : kBig;
                            next2[((d + 1) & 1) * row + i + 2] =
                                inside(w + 3) ? old[(u + 3) % kAhead] : kBig;
                        }
                        old[u] = Tc[at(w + kAhead)];
                        sl[u] = sc[at(w + kAhead)];
                        step_barrier();
                    }
                }
            }
            changed = __syncthreads_or(changed);
        }
        if (i == 0) {
            atomicMax(&stat[phase - 1], it);
            if (changed)
                stat[2] = 1;
        }
    }
}

// T[c * stride + s] = W[s * ni + c] for n tables, 32 x 32 elements per
// workgroup.
constexpr int kTr = 32;
__global__ __launch_bounds__(256) void eik_transpose_kernel(const double *__restrict__ W,
                                                            int64_t ni, int n, int stride,
                                                            double *__restrict__ T)
{
    __shared__ double tile[kTr][kTr + 1];
    const int64_t c0 = (int64_t)blockIdx.x * kTr;
    const int s0 = blockIdx.y * kTr, x = threadIdx.x & (kTr - 1), y0 = threadIdx.x / kTr;
    for (int y = y0; y < kTr; y += 256 / kTr)
        if (s0 + y < n && c0 + x < ni)
            tile[y][x] = W[(int64_t)(s0 + y) * ni + c0 + x];
    __syncthreads();
    for (int y = y0; y < kTr; y += 256 / kTr)
        if (s0 + x < n && c0 + y < ni)
            T[(c0 + y) * stride + s0 + x] = tile[x][y];
}

// Whether a grid's sweeps run in one launch: 2D, the shorter axis one lane
// per column.
bool one_launch(int ndims, int nx, int nz, int n)
{
    return ndims == 2 && nx > 0 && nz > 0 && n > 0 && std::min(nx, nz) <= kSweepThreads;
}

// Sources whose sweeps can run at once, one workgroup each: more of them take
// turns, in the same workspace, at no cost (200x200 with 2000 sources 30.3 ms
// in groups of 512, 32.8 in one; but 301x151 with 600, which all run at once,
// 14.5 and 9.8 ms).
int sweep_sources(int nx, int nz)
{
    const int threads = (std::min(nx, nz) + 63) & ~63;
    return 256 * (2048 / threads);  // waves of the chip's 256 CUs
}

}  // namespace

extern "C" int64_t kx_eikonal_work_bytes(int32_t ndims, int32_t nx, int32_t ny, int32_t nz,
                                         int32_t n)
{
    (void)ny;
    if (!one_launch(ndims, nx, nz, n))
        return 0;
    return (int64_t)nx * nz * std::min(n, sweep_sources(nx, nz)) * 8 + 64;
}

extern "C" int kx_eikonal(int32_t ndims, int32_t nx, int32_t ny, int32_t nz, double hx, double hy,
                          double hz, const double *slow, int32_t n, const int32_t *src, double *T,
                          int32_t max_iter, int32_t order, int32_t *flag, int32_t *iters,
                          void *stream)
{
    return kx_eikonal_ws(ndims, nx, ny, nz, hx, hy, hz, slow, n, src, T, max_iter, order, flag,
                         iters, nullptr, 0, stream);
}

extern "C" int kx_eikonal_ws(int32_t ndims, int32_t nx, int32_t ny, int32_t nz, double hx,
                             double hy, double hz, const double *slow, int32_t n,
                             const int32_t *src, double *T, int32_t max_iter, int32_t order,
                             int32_t *flag, int32_t *iters, void *work, int64_t work_bytes,
                             void *stream)
{
    if (ndims != 2 && ndims != 3)
        return efail(KX_EINVAL, "eikonal: ndims must be 2 or 3");
    if (ndims == 2)
        ny = 1;
    if (order != 1 && order != 2)
        return efail(KX_EINVAL, "eikonal: order must be 1 or 2");
    if (nx <= 0 || ny <= 0 || nz <= 0 || n <= 0 || n > (1 << 22) || max_iter <= 0)
        return efail(KX_ESHAPE, "eikonal: bad sizes (nx=%d ny=%d nz=%d n=%d)", nx, ny, nz, n);
    if (!(hx > 0) || !(hz > 0) || (ndims == 3 && !(hy > 0)))
        return efail(KX_EINVAL, "eikonal: spacings must be positive");
    if (!slow || !src || !T || !flag)
        return efail(KX_EINVAL, "eikonal: NULL buffer");
    EikArgs g;
    g.nx = nx;
    g.ny = ny;
    g.nz = nz;
    g.hx = hx;
    g.hy = ndims == 3 ? hy : 1.0;
    g.hz = hz;
    g.three = ndims == 3;
    g.n = n;
    g.ni = (int64_t)nx * ny * nz;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    // the kernels index the slowness at each source cell: check the cells
    // on the host before any launch
    std::vector<int32_t> hs((size_t)3 * n);
    hipError_t e = hipMemcpyAsync(hs.data(), src, hs.size() * sizeof(int32_t),
                                  hipMemcpyDeviceToHost, st);
    if (e == hipSuccess)
        e = hipStreamSynchronize(st);
    if (e != hipSuccess)
        return efail((int)e, "eikonal: %s", hipGetErrorString(e));
    for (int32_t k = 0; k < n; ++k) {
        const int32_t sx = hs[3 * k], sy = hs[3 * k + 1], sz = hs[3 * k + 2];
        if (sx < 0 || sx >= nx || sy < 0 || sy >= ny || sz < 0 || sz >= nz)
            return efail(KX_ESHAPE, "eikonal: source %d at cell (%d, %d, %d) outside the "
                         "%d x %d x %d grid", k, sx, sy, sz, nx, ny, nz);
    }
    const int64_t least = kx_eikonal_work_bytes(ndims, nx, ny, nz, 1);
    if (least > 0 && work != nullptr && work_bytes >= least) {
        // as many sources at a time as the workspace holds
        const int at_once =
            (int)std::min<int64_t>(std::min(n, sweep_sources(nx, nz)), (work_bytes - 64) / (g.ni * 8));
        double *W = static_cast<double *>(work);
        int32_t *stat = reinterpret_cast<int32_t *>(W + g.ni * at_once), h[3] = {0, 0, 0};
        e = hipMemsetAsync(stat, 0, sizeof(h), st);
        if (e != hipSuccess)
            return efail((int)e, "eikonal: %s", hipGetErrorString(e));
        const int walk_x = nx > nz, np = std::min(nx, nz);
        const size_t lds = (size_t)8 * (np + 4) * sizeof(double);
        if (lds > 64 * 1024) {
            e = hipFuncSetAttribute(reinterpret_cast<const void *>(&eik_sweep2d_kernel),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            if (e != hipSuccess)
                return efail((int)e, "eikonal: %s", hipGetErrorString(e));
        }
        for (int s0 = 0; s0 < n; s0 += at_once) {
            const int ns = std::min(at_once, n - s0);
            hipLaunchKernelGGL(eik_sweep2d_kernel, dim3((unsigned)ns), dim3((np + 63) & ~63), lds,
                               st, g, slow, src + 3 * (int64_t)s0, W, walk_x, max_iter, order,
                               stat);
            hipLaunchKernelGGL(eik_transpose_kernel,
                               dim3((unsigned)((g.ni + kTr - 1) / kTr),
                                    (unsigned)((ns + kTr - 1) / kTr)),
                               dim3(256), 0, st, W, g.ni, ns, n, T + s0);
            e = hipGetLastError();
            if (e != hipSuccess)
                return efail((int)e, "eikonal sweeps: %s", hipGetErrorString(e));
        }
        e = hipMemcpyAsync(h, stat, sizeof(h), hipMemcpyDeviceToHost, st);
        if (e == hipSuccess)
            e = hipStreamSynchronize(st);
        if (e != hipSuccess)
            return efail((int)e, "eikonal: %s", hipGetErrorString(e));
        if (iters) {
            iters[0] = h[0] + h[1];
            iters[1] = !h[2];
        }
        return KX_OK;
    }
    const int64_t nb = (g.ni + kEikCells - 1) / kEikCells;
    const unsigned nsb = (unsigned)((n + kEikSrc - 1) / kEikSrc);
    if (nb > INT32_MAX)
        return efail(KX_ESHAPE, "eikonal: grid too large");
    hipLaunchKernelGGL(eik_init_kernel, dim3((unsigned)nb, nsb), dim3(kEikSrc, kEikCells), 0, st, g,
                       slow, src, T);
    e = hipGetLastError();
    if (e != hipSuccess)
        return efail((int)e, "eikonal init: %s", hipGetErrorString(e));
    const int ndiag = (nx - 1) + (ny - 1) + (nz - 1) + 1;
    const int ndir = ndims == 3 ? 8 : 4;
    int rounds = 0, converged = 1;
    // first-order sweeps to convergence, then (order 2) second-order ones
    for (int phase = 1; phase <= order; ++phase) {
        for (int it = 0; it < max_iter; ++it) {
            ++rounds;
            e = hipMemsetAsync(flag, 0, sizeof(int32_t), st);
            if (e != hipSuccess)
                return efail((int)e, "eikonal: %s", hipGetErrorString(e));
            for (int q = 0; q < ndir; ++q) {
                const int dx = (q & 1) ? -1 : 1, dz = (q & 2) ? -1 : 1, dy = (q & 4) ? -1 : 1;
                for (int d = 0; d < ndiag; ++d) {
                    const int ixlo = std::max(0, d - (ny - 1) - (nz - 1));
                    const int ixhi = std::min(nx - 1, d);
                    const int nix = ixhi - ixlo + 1;
                    const int64_t npair = (int64_t)nix * ny;
                    const int64_t nbd = (npair + kEikCells - 1) / kEikCells;
                    hipLaunchKernelGGL(eik_sweep_kernel, dim3((unsigned)nbd, nsb),
                                       dim3(kEikSrc, kEikCells), 0,
                                       st, g, slow, src, T, d, dx, dy, dz, ixlo, nix, phase, flag);
                }
            }
            e = hipGetLastError();
            if (e != hipSuccess)
                return efail((int)e, "eikonal sweep: %s", hipGetErrorString(e));
            int32_t h = 0;
            e = hipMemcpyAsync(&h, flag, sizeof(int32_t), hipMemcpyDeviceToHost, st);
            if (e == hipSuccess)
                e = hipStreamSynchronize(st);
            if (e != hipSuccess)
                return efail((int)e, "eikonal: %s", hipGetErrorString(e));
            if (!h)
                break;
            if (it == max_iter - 1)
                converged = 0;  // values still changed in the last round
        }
    }
    if (iters) {
        iters[0] = rounds;
        iters[1] = converged;
    }
    return KX_OK;
}
