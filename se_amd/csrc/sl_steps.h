// sl_steps.h -- device code of the semi-Lagrangian steps (sl.hip): the mesh's
// lines, departure points, weights and sums, and the kernels of the first- and
// second-order step.  Orders above 8 are instantiated in a translation unit of
// their own (sl_high.hip): a process loads a unit's kernels at their first
// launch, and theirs are as large as all the others' together (first step of a
// process 13 ms without them, 16 with).
#pragma once
#include <cmath>
#include <cstring>

#include "glibc_pow.h"
#include "se_common.h"

namespace se_sl {

struct SLGeom {
    int N, nEls0, nEls1, nv0, nv1, per0, per1;
    int cubic;  // the advected field by bicubic Lagrange interpolation (Advector::Interpolate)
    double min0, min1, max0, max1, dx0, dx1;
    const double* xk;   // abscissae
    const double* D;    // derivative matrix
    const double* pnx;  // P_N(x_j)
    const double* pn;   // P_N monomial coefficients
    const double* X;    // field column coordinates
    const double* Y;    // field row coordinates
    const double* J00;
    const double* J10;
    const double* J11;
    const double* J01;
};

#define SE_NUMAPPROX(var, val) ((var) >= (val)-1.0e-12 && (var) <= (val) + 1.0e-12)

// One dimension of the mesh.  The departure-point kernels give every point a
// pair of neighbouring lanes, the even one for x and the odd one for y: all of
// a point's arithmetic but the sums over an element's nodes is separable, and
// of those each lane sums its own component of a velocity.  With one lane per
// node a mesh of 37 k nodes was one wave per SIMD walking a serial chain (powers,
// divisions, sums), and at 332 k nodes 167 registers were wanted.
struct Line {
    int dim, nEls, per, n0;  // n0: nodes from one element to the next, N or N nv0
    double min, max, dx, sc;  // sc = 2 / dx
};

template <int NN>
__device__ __forceinline__ Line line_of(const SLGeom& g, int dim) {
#pragma clang fp contract(off)
    Line l;
    l.dim = dim;
    l.nEls = dim ? g.nEls1 : g.nEls0;
    l.per = dim ? g.per1 : g.per0;
    l.n0 = (NN ? NN : g.N) * (dim ? g.nv0 : 1);
    l.min = dim ? g.min1 : g.min0;
    l.max = dim ? g.max1 : g.max0;
    l.dx = dim ? g.dx1 : g.dx0;
    l.sc = 2.0 / l.dx;
    return l;
}

// quad_perm of the doubles of a lane pair
template <int CTRL>
__device__ __forceinline__ double quad(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
constexpr int kEven = 0xA0, kOdd = 0xF5, kSwap = 0xB1;  // [0,0,2,2], [1,1,3,3], [1,0,3,2]

// Mesh::GetEl, src/base/Mesh.cpp:106-137, in one dimension
__device__ __forceinline__ int get_el(const Line& l, double c) {
#pragma clang fp contract(off)
    int t;
    double integer, frac;
    if (SE_NUMAPPROX(c - l.max, 0.0)) {
        t = l.nEls - 1;
    } else {
        double out = (c - l.min) / l.dx;
        frac = modf(out, &integer);
        t = (int)integer;
        if (t > 0 && SE_NUMAPPROX(frac, 0.0)) t--;
    }
    // A coordinate outside the domain (displacement beyond one period, or a
    // non-finite velocity) has no element in the reference either; clamp so
    // the gather stays inside the field arrays.
    return t < 0 ? 0 : (t >= l.nEls ? l.nEls - 1 : t);
}
__device__ __forceinline__ int get_el(const SLGeom& g, double cx, double cy) {
    return get_el(line_of<0>(g, 1), cy) * g.nEls0 + get_el(line_of<0>(g, 0), cx);
}

// Advector::PeriodicUpdate, src/base/Advector.cpp:122-134, in one dimension
__device__ __forceinline__ void wrap(const Line& l, double& c) {
#pragma clang fp contract(off)
    if (c < l.min) c = l.per ? l.max - l.min + c : l.min;
    if (c > l.max) c = l.per ? l.min - l.max + c : l.max;
}

// The kernels take the order as a template argument NN: the steps N = 2..12,
// the others N = 2..8 and, with NN = 0, the order of the geometry: the same
// operations either way, with fixed trip counts and arrays of N + 1 in registers
// when NN is known.  (In scratch memory two lanes' arrays cost more than they
// saved: 40 x 40 elements of order 9, first-order step, one lane 62 us, two 132,
// two with the order known 30; 60 x 60 of order 12 330, 819, 152.)
template <int NN> struct Ord {
    static constexpr int MAX = NN ? NN : 12;  // array bound
};
template <int NN>
__device__ __forceinline__ int order(const SLGeom& g) {
    return NN ? NN : g.N;
}

// Jacobi::EvalDeriv (Jacobi.cpp:58-66) of P_N; its powers of x share one log.
// Between two GLL points no special case of pow arises (but |x| below 2^-60 at
// odd orders): there the powers are free of branches and run side by side.
template <int NN>
__device__ __forceinline__ double pn_deriv(const SLGeom& g, double x) {
#pragma clang fp contract(off)
    double dp = 0.0;
    if (se_pow::pow_plain(x)) {
        double lo = 0.0, hi = 0.0;
        if (order<NN>(g) > 2) hi = se_pow::log_hi_lo(se_pow::bits(x) & 0x7fffffffffffffffULL, &lo);
        for (int i = order<NN>(g); i >= 1; i -= 2) dp += g.pn[i] * i * se_pow::pow_plain_at(x, hi, lo, i - 1);
    } else {
        const se_pow::PowBase b = se_pow::pow_base(x);
#pragma unroll 1
        for (int i = order<NN>(g); i >= 1; i -= 2) dp += g.pn[i] * i * se_pow::pow_int_at(b, i - 1);
    }
    return dp;
}

// a / b, correctly rounded, for operands whose quotient and steps are far from
// the limits of the exponent (or NaN): two Newton steps of the reciprocal, the
// quotient and its remainder's correction (Markstein) without the scaling
// around them.
__device__ __forceinline__ double div_plain(double a, double b) {
#pragma clang fp contract(off)
    double r = __builtin_amdgcn_rcp(b);
    r = fma(r, fma(-b, r, 1.0), r);
    r = fma(r, fma(-b, r, 1.0), r);
    const double q = a * r;
    return fma(fma(-b, q, a), r, q);
}

// 1-D GLL cardinal functions at local coordinate x in [-1, 1] (Legendre::IsRoot
// and the per-dimension factor of ShapeFuncsAtCoord, Legendre.cpp:145-169,
// 291-305).  At least 1e-8 from every GLL point, 1 - x^2 is 2e-8 or more and
// the divisor 1e-9 or more.
template <int NN>
__device__ __forceinline__ void cardinal(const SLGeom& g, double x, double (&L)[Ord<NN>::MAX + 1]) {
#pragma clang fp contract(off)
    const int N = order<NN>(g);
    int root = -1;
    for (int k = N; k >= 0; k--)
        if (fabs(x - g.xk[k]) < 1.0e-8) root = k;
    if (root >= 0) {
        for (int j = 0; j <= N; j++) L[j] = (j == root) ? 1.0 : 0.0;
        return;
    }
    const double dpx = pn_deriv<NN>(g, x);
    for (int j = 0; j <= N; j++)
        L[j] = -div_plain(1.0 - x * x, N * (N + 1) * g.pnx[j] * (x - g.xk[j])) * dpx;
}

// Mesh::GlobalToLocal (Mesh.cpp:163-177) in one dimension; n0: the first node
// of c's element along the dimension
__device__ __forceinline__ double local_of(const Line& l, double c, int& n0) {
#pragma clang fp contract(off)
    const int e = get_el(l, c);
    n0 = e * l.n0;
    double x = (c - l.min - e * l.dx) * l.sc - 1.0;
    if (x < -1.0) x = -1;
    if (x > +1.0) x = +1;
    return x;
}

// The element of a point whose coordinate in this lane's dimension is c
struct Place {
    double x;  // this dimension's local coordinate
    int node;  // the element's first node
};
template <int NN>
__device__ __forceinline__ Place place(const Line& l, double c) {
    Place p;
    int n0;
    p.x = local_of(l, c, n0);
    p.node = n0 + __builtin_amdgcn_mov_dpp(n0, kSwap, 0xf, 0xf, true);
    return p;
}

// A point's weights: a lane evaluates its own dimension's, the pair exchanges
template <int NN>
struct Weights {
    double x[Ord<NN>::MAX + 1], y[Ord<NN>::MAX + 1];
    // hides the weights from the compiler before a further sum, whose products
    // x y it would otherwise all keep from the one before
    __device__ __forceinline__ void fresh() {
#pragma unroll
        for (int j = 0; j <= NN; j++) asm volatile("" : "+v"(y[j]));
    }
};
template <int NN>
__device__ __forceinline__ void weights_at(const SLGeom& g, const Place& p, Weights<NN>& w) {
    double L[Ord<NN>::MAX + 1];
    cardinal<NN>(g, p.x, L);
    for (int j = 0; j <= order<NN>(g); j++) {
        w.x[j] = quad<kEven>(L[j]);
        w.y[j] = quad<kOdd>(L[j]);
    }
}

// Field::InterpGlobal (Field.cpp:57-76) of one component per lane of a field of
// nd components: a velocity's or a two-component field's own one (ND = 2), the
// only one (ND = 1, both lanes) or component comp (ND = 0).  The cache's
// lookups bound the sums on large meshes, so a lane reads 16 bytes at a time
// and the pair exchanges: of two components the nodes of its parity, of one
// every other two nodes.  The first AHEAD rows of the element's nodes are read
// before the weights are known, the others AHEAD rows before their use.
struct __attribute__((aligned(8))) Two {
    double a, b;
};
template <int NN, int ND>
struct Rows {
    static constexpr int AHEAD = NN > 6 ? 2 : 3, N1 = NN + 1;
    static constexpr int NR = ND == 2 ? (N1 + 1) / 2 : ND == 1 ? (N1 + 3) / 4 : (N1 + 1) / 2;  // 16-byte reads a row
    const double* p;
    int nd, pitch, dim;
    Two v[AHEAD][NR];

    __device__ __forceinline__ void read(int jj) {
        const double* r = p + jj * pitch;
#pragma unroll
        for (int k = 0; k < NR; k++) {
            Two& t = v[jj % AHEAD][k];
            if (ND == 2) {
                t = *(const Two*)(r + 4 * k + (2 * k < NN ? 2 * dim : 0));
            } else if (ND == 1) {
                const int i0 = 4 * k < NN ? 4 * k : NN - 1, i1 = 4 * k + 2 < NN ? 4 * k + 2 : NN - 1;
                t = *(const Two*)(r + (dim ? i1 : i0));
            } else {
                t.a = r[2 * k * nd];
                if (2 * k < NN) t.b = r[(2 * k + 1) * nd];
            }
        }
    }
    __device__ __forceinline__ double value(int jj, int ii) const {
        if (ND == 2) {  // lane 0 read the even nodes, lane 1 the odd ones
            const Two& t = v[jj % AHEAD][ii / 2];
            const double o = ii & 1 ? quad<kOdd>(t.a) : quad<kEven>(t.b);  // (with both lanes active)
            return ii & 1 ? (dim ? t.b : o) : (dim ? o : t.a);
        } else if (ND == 1) {
            const Two& t = v[jj % AHEAD][ii / 4];
            const int c = ii / 2 * 2, i0 = c < NN ? c : NN - 1;
            return (ii & 2) ? quad<kOdd>(ii > i0 ? t.b : t.a) : quad<kEven>(ii > i0 ? t.b : t.a);
        }
        const Two& t = v[jj % AHEAD][ii / 2];
        return ii & 1 ? t.b : t.a;
    }
    __device__ __forceinline__ Rows(const SLGeom& g, const Line& l, int node, const double* f, int nd_, int comp) {
        nd = nd_;
        dim = l.dim;
        pitch = g.nv0 * nd;
        p = f + (size_t)node * nd + (ND ? 0 : comp);
#pragma unroll
        for (int jj = 0; jj < AHEAD && jj <= NN; jj++) read(jj);
    }
    __device__ __forceinline__ double sum(const Weights<NN>& w) {
#pragma clang fp contract(off)
        double s = 0.0;
#pragma unroll
        for (int jj = 0; jj <= NN; jj++) {
#pragma unroll
            for (int ii = 0; ii <= NN; ii++) s += w.x[ii] * w.y[jj] * value(jj, ii);
            asm volatile("" : "+v"(s) : : "memory");  // the next rows' reads stay behind this row's sum
            if (jj + AHEAD <= NN) read(jj + AHEAD);
        }
        return s;
    }
};

// this lane's component of a velocity at the point whose coordinate in its
// dimension is c
template <int NN>
__device__ __forceinline__ double velocity_at(const SLGeom& g, const Line& l, double c, const double* __restrict__ vel,
                                              Weights<NN>& w) {
    const Place p = place<NN>(l, c);
    Rows<NN, 2> r(g, l, p.node, vel, 2, l.dim);
    weights_at<NN>(g, p, w);
    return r.sum(w);
}

// Field::InterpGlobal at any point, one thread per point; vals node-major with
// nd dofs
template <int NN, int ND>
__device__ __forceinline__ void interp_global(const SLGeom& g, const double* __restrict__ vals, int nd, double cx,
                                              double cy, double (&out)[ND]) {
#pragma clang fp contract(off)
    const int N = order<NN>(g);
    int nx, ny;
    const double lx = local_of(line_of<NN>(g, 0), cx, nx), ly = local_of(line_of<NN>(g, 1), cy, ny);
    double Lx[Ord<NN>::MAX + 1], Ly[Ord<NN>::MAX + 1];
    cardinal<NN>(g, lx, Lx);
    cardinal<NN>(g, ly, Ly);
    for (int d = 0; d < ND; d++) out[d] = 0.0;
    const int n0 = nx + ny;
#pragma unroll 1
    for (int jj = 0; jj <= N; jj++)
        for (int ii = 0; ii <= N; ii++) {
            double Ni = Lx[ii] * Ly[jj];
            const double* v = &vals[(size_t)(n0 + jj * g.nv0 + ii) * nd];
            for (int d = 0; d < ND; d++)
                if (d < nd) out[d] += Ni * v[d];
        }
}

// Advector::InterpLagrange, Advector.cpp:248-275
template <int ND>
__device__ __forceinline__ void interp_lagrange(double x, const double* c, double (&vals)[4][ND], double (&psi)[ND]) {
#pragma clang fp contract(off)
    for (int d = 0; d < ND; d++) psi[d] = 0.0;
    for (int node = 0; node < 4; node++) {
        double factor = 1.0;
        for (int o = 0; o < 4; o++)
            if (o != node) factor *= (x - c[o]) / (c[node] - c[o]);
        for (int d = 0; d < ND; d++) psi[d] += vals[node][d] * factor;
    }
}

// Advector::Interpolate (bicubic on the 4x4 node stencil, used when N < 3),
// Advector.cpp:278-337
template <int ND>
__device__ __forceinline__ void interp_bicubic(const SLGeom& g, const double* __restrict__ vals, int nd, double cx,
                                               double cy, double (&out)[ND]) {
#pragma clang fp contract(off)
    const int N = g.N;
    int el = get_el(g, cx, cy);
    int ex = el % g.nEls0, ey = el / g.nEls0;
    int node0 = N * ey * g.nv0 + N * ex;
    int x0 = node0 % g.nv0;
    int y0 = (node0 / g.nv0) % g.nv1;
    double ddx = g.dx0 / N, ddy = g.dx1 / N;
    if (cx <= g.X[x0 + 1]) x0--;
    if (cy <= g.Y[ey * N + 3 / (N + 1)]) y0--;  // row of entry 3 of the element's node list
    if (cx <= g.min0 + ddx) x0++;
    else if (cx >= g.max0 - ddx) x0--;
    if (cy <= g.min1 + ddy) y0++;
    else if (cy >= g.max1 - ddy) y0--;
    x0 = x0 < 0 ? 0 : (x0 > g.nv0 - 4 ? g.nv0 - 4 : x0);
    y0 = y0 < 0 ? 0 : (y0 > g.nv1 - 4 ? g.nv1 - 4 : y0);
    double px[4], py[4], pts[4][ND], rows[4][ND];
    for (int i = 0; i < 4; i++) px[i] = g.X[x0 + i];
    for (int j = 0; j < 4; j++) py[j] = g.Y[y0 + j];
    for (int j = 0; j < 4; j++) {
        for (int i = 0; i < 4; i++)
            for (int d = 0; d < ND; d++) pts[i][d] = d < nd ? vals[(size_t)(x0 + i + (y0 + j) * g.nv0) * nd + d] : 0.0;
        double r[ND];
        interp_lagrange<ND>(cx, px, pts, r);
        for (int d = 0; d < ND; d++) rows[j][d] = r[d];
    }
    interp_lagrange<ND>(cy, py, rows, out);
}

// The advected field's component of this lane -- and, of three, the last one
__device__ __forceinline__ int component(const Line& l, int nd) { return l.dim < nd ? l.dim : nd - 1; }
// the components at the point whose coordinate in this lane's dimension is c,
// bicubic
__device__ __forceinline__ void bicubic_at(const SLGeom& g, const Line& l, const double* __restrict__ q, int nd,
                                           double c, double& a, double& b) {
    const double o = quad<kSwap>(c);
    double v[3];
    interp_bicubic<3>(g, q, nd, l.dim ? o : c, l.dim ? c : o, v);
    a = l.dim && nd > 1 ? v[1] : v[0];
    b = v[2];
}
// the components by the weights of a place
template <int NN, int ND>
__device__ __forceinline__ void advected_at(const SLGeom& g, const Line& l, double c, const double* __restrict__ q,
                                            int nd, double& a, double& b) {
    Weights<NN> w;
    const Place p = place<NN>(l, c);
    Rows<NN, ND> r(g, l, p.node, q, nd, component(l, nd));
    weights_at<NN>(g, p, w);
    a = r.sum(w);
    b = 0.0;
    if (ND == 0 && nd == 3) {
        w.fresh();
        b = Rows<NN, 0>(g, l, p.node, q, nd, 2).sum(w);
    }
}
// Stores node v's value, with Field::PeriodicUpdate (Field.cpp:232-252): the
// first line's nodes of a periodic dimension also store their duplicates on the
// last line, whose own values go nowhere.  Against a launch of its own after each
// step, us, first and second order: 29 x 17 elements of order 5 8.1 / 14.7 -> 6.6 /
// 13.1, 96 x 96 of order 3 10.1 / 20.8 -> 8.3 / 19.1, periodic 64 x 64 of order 8 56.5 /
// 122 -> 53.7 / 120; 96 x 96 of order 6 43.5 / 88.6 -> 45.4 / 87.7.
__device__ __forceinline__ void put_advected(const SLGeom& g, const Line& l, int v, int nd, double a, double b,
                                             double* __restrict__ qsl) {
    const int J = v / g.nv0, I = v - J * g.nv0;
    if ((g.per0 && I == g.nv0 - 1) || (g.per1 && J == g.nv1 - 1)) return;
    auto put = [&](int at) {
        if (l.dim < nd) qsl[(size_t)at * nd + l.dim] = a;
        if (nd == 3 && l.dim == 0) qsl[(size_t)at * 3 + 2] = b;
    };
    const int x = g.per0 && I == 0 ? g.nv0 - 1 : 0, y = g.per1 && J == 0 ? (g.nv1 - 1) * g.nv0 : 0;
    put(v);
    if (x) put(v + x);
    if (y) put(v + y);
    if (x && y) put(v + x + y);
}

// Advector::FirstOrder + IntegrateRK2 (Advector.cpp:136-148,181-201).  Bound by
// latency: 29x17 order 5 22 -> 7.3 us, 32x32 order 6 29.5 -> 12 us with two lanes
// per node, branch-free powers and unscaled divisions.
template <int NN, int ND>
__global__ __launch_bounds__(256) void k_sl_first(SLGeom g, const double* __restrict__ q, int nd,
                                                   const double* __restrict__ vel, double dt, double* __restrict__ qsl,
                                                   int32_t* __restrict__ dep) {
#pragma clang fp contract(off)
    const int v = blockIdx.x * 128 + (threadIdx.x >> 1);
    if (v >= g.nv0 * g.nv1) return;
    const Line l = line_of<NN>(g, threadIdx.x & 1);
    const double o = l.dim ? g.Y[v / g.nv0] : g.X[v % g.nv0];
    Weights<NN> w;
    // velocity at the origin: the origin is a GLL node, so InterpGlobal
    // returns the nodal value exactly (IsRoot selects a Kronecker delta)
    double h = o - 0.5 * dt * velocity_at<NN>(g, l, o, vel, w);
    wrap(l, h);
    double c = o - dt * velocity_at<NN>(g, l, h, vel, w);
    wrap(l, c);
    double a, b;
    if (ND < 0) bicubic_at(g, l, q, nd, c, a, b);
    else advected_at<NN, ND>(g, l, c, q, nd, a, b);
    put_advected(g, l, v, nd, a, b, qsl);
    if (dep) {
        const int e = get_el(l, c);
        const int ey = __builtin_amdgcn_mov_dpp(e, kSwap, 0xf, 0xf, true);
        if (l.dim == 0) dep[v] = ey * g.nEls0 + e;
    }
}

// Advector::SecondOrder (Advector.cpp:203-246).  Four waves per SIMD (128
// VGPRs, no spills; the bicubic form takes 256, orders above 8 130 to 166).  32x32 order 6 54 -> 19 us;
// 96x96 order 6 135 -> 89 us: two thirds of it VALU issue (3300 instructions a
// wave), the rest the cache's lookups of the gathers (126 us while a lane read 8
// bytes at a time).
template <int NN, int ND>
__global__ __launch_bounds__(256, ND < 0 || NN > 8 ? 2 : 4) void k_sl_second(SLGeom g, const double* __restrict__ q, const double* __restrict__ qp,
                                                    int nd, const double* __restrict__ vel,
                                                    const double* __restrict__ vp1, const double* __restrict__ vph,
                                                    const double* __restrict__ vmh, double dt,
                                                    double* __restrict__ qsl) {
#pragma clang fp contract(off)
    const int v = blockIdx.x * 128 + (threadIdx.x >> 1);
    if (v >= g.nv0 * g.nv1) return;
    const Line l = line_of<NN>(g, threadIdx.x & 1);
    const double o = l.dim ? g.Y[v / g.nv0] : g.X[v % g.nv0];
    Weights<NN> w;
    double h = o - 0.5 * dt * velocity_at<NN>(g, l, o, vp1, w);
    wrap(l, h);
    double c = o - dt * velocity_at<NN>(g, l, h, vph, w);
    wrap(l, c);
    // the velocity and (GLL interpolation) the advected field at the first
    // point share one set of weights
    double a1, b1 = 0.0, a2, b2;
    if (ND < 0) {
        h = c - 0.5 * dt * velocity_at<NN>(g, l, c, vel, w);
        bicubic_at(g, l, q, nd, c, a1, b1);
    } else {
        const Place p = place<NN>(l, c);
        Rows<NN, 2> rv(g, l, p.node, vel, 2, l.dim);
        weights_at<NN>(g, p, w);
        h = c - 0.5 * dt * rv.sum(w);
        w.fresh();
        a1 = Rows<NN, ND>(g, l, p.node, q, nd, component(l, nd)).sum(w);
        if (ND == 0 && nd == 3) {
            w.fresh();
            b1 = Rows<NN, 0>(g, l, p.node, q, nd, 2).sum(w);
        }
    }
    wrap(l, h);
    c -= dt * velocity_at<NN>(g, l, h, vmh, w);
    wrap(l, c);
    if (ND < 0) bicubic_at(g, l, qp, nd, c, a2, b2);
    else advected_at<NN, ND>(g, l, c, qp, nd, a2, b2);
    put_advected(g, l, v, nd, 2.0 * a1 - 0.5 * a2, 2.0 * b1 - 0.5 * b2, qsl);
}

inline int pair_blocks(int n) { return n / 128 + (n % 128 != 0); }  // two lanes per node

// KERNEL<N, the advected components: 1, 2, else 0; -1: bicubic>
#define SE_SL_ADV(KERNEL, N, GRID, ...)                                                                   \
    if (g.cubic) hipLaunchKernelGGL((KERNEL<N, -1>), GRID, dim3(256), 0, __VA_ARGS__);                   \
    else if (nd == 1) hipLaunchKernelGGL((KERNEL<N, 1>), GRID, dim3(256), 0, __VA_ARGS__);               \
    else if (nd == 2) hipLaunchKernelGGL((KERNEL<N, 2>), GRID, dim3(256), 0, __VA_ARGS__);               \
    else hipLaunchKernelGGL((KERNEL<N, 0>), GRID, dim3(256), 0, __VA_ARGS__)

// the steps of the orders 9..12 (sl_high.hip)
void sl_first_high(int N, hipStream_t s, const SLGeom& g, const double* q, int nd, const double* vel, double dt,
                   double* qsl, int32_t* dep);
void sl_second_high(int N, hipStream_t s, const SLGeom& g, const double* q, const double* qp, int nd,
                    const double* vel, const double* vp1, const double* vph, const double* vmh, double dt,
                    double* qsl);

}  // namespace se_sl
