// sl.hip -- semi-Lagrangian advection (departure-point search + GLL
// interpolation), velocity from the stream function, CFL time step.
//
// Two lanes per field node, one for each dimension.  The coordinate arithmetic that decides the
// departure element (RK2 midpoint, wrap/clamp, GetEl's modf and its 1e-12
// edge rule, the local-coordinate map) follows the reference's operation order
// with FP contraction disabled.  P_N(x_j) is tabulated on the host with the
// reference's evaluation; P_N'(x) is evaluated on the device with the same
// monomial sum, its powers bit-identical to the C library's pow
// (glibc_pow.h), so interpolated values and departure elements agree with
// the reference's bit for bit.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <mutex>
#include <string>

#include "glibc_pow.h"
#include "se_common.h"

using namespace se;

namespace {

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
// last line, whose own values go nowhere (a launch of its own cost 4 us and an
// edge after each step).
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

// Advector::ExtrapolateVelocities (Advector.cpp:339-349)
__global__ void k_extrap(int n2, const double* __restrict__ vel, const double* __restrict__ velPrev,
                         double* __restrict__ vp1, double* __restrict__ vph, double* __restrict__ vmh) {
#pragma clang fp contract(off)
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n2) return;
    double a = vel[i], b = velPrev[i];
    vp1[i] = 2.0 * a - 1.0 * b;
    vph[i] = 1.5 * a - 0.5 * b;
    vmh[i] = 0.5 * a + 0.5 * b;
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

// Field::InterpGlobal (mode GLL) or Advector::Interpolate (mode BICUBIC) at
// arbitrary points, one thread per point; xy: npts x 2, out: npts x nd
template <int NN>
__global__ __launch_bounds__(256) void k_interp_points(SLGeom g, const double* __restrict__ vals, int nd, int npts,
                                                       const double* __restrict__ xy, int cubic,
                                                       double* __restrict__ out) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= npts) return;
    double v[3];
    if (cubic) interp_bicubic<3>(g, vals, nd, xy[2 * (size_t)p], xy[2 * (size_t)p + 1], v);
    else interp_global<NN, 3>(g, vals, nd, xy[2 * (size_t)p], xy[2 * (size_t)p + 1], v);
    for (int d = 0; d < nd; d++) out[(size_t)p * nd + d] = v[d];
}

// QuasiGeostrophicEqn::GenVel via Field::InterpDerivsGlobal and
// Mesh::ShapeFuncDerivsAtCoord (Mesh.cpp:252-285).  At a vertex both local
// coordinates are GLL roots, so the local derivative rows are columns of D
// and the Jacobian is the tabulated one of that GLL point.
template <int NN>
__global__ __launch_bounds__(256) void k_genvel(SLGeom g, const double* __restrict__ psi, double* __restrict__ vel) {
#pragma clang fp contract(off)
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= g.nv0 * g.nv1) return;
    const int N = order<NN>(g), n1 = N + 1;
    const double ox = g.X[v % g.nv0], oy = g.Y[v / g.nv0];
    int el = get_el(g, ox, oy);
    int ex = el % g.nEls0, ey = el / g.nEls0;
    double lx = (ox - g.min0 - ex * g.dx0) * (2.0 / g.dx0) - 1.0;
    double ly = (oy - g.min1 - ey * g.dx1) * (2.0 / g.dx1) - 1.0;
    if (lx < -1.0) lx = -1;
    if (lx > +1.0) lx = +1;
    if (ly < -1.0) ly = -1;
    if (ly > +1.0) ly = +1;
    int xi = -1, yi = -1;
    for (int k = 0; k <= N; k++)
        if (xi < 0 && fabs(lx - g.xk[k]) < 1.0e-8) xi = k;
    for (int k = 0; k <= N; k++)
        if (yi < 0 && fabs(ly - g.xk[k]) < 1.0e-8) yi = k;
    if (xi < 0 || yi < 0) {  // cannot happen at a vertex
        vel[2 * (size_t)v] = vel[2 * (size_t)v + 1] = __builtin_nan("");
        return;
    }
    double j00 = g.J00[ex * n1 + xi], j01 = g.J01[(ey * n1 + yi) * n1 + xi];
    double j10 = g.J10[(ex * n1 + xi) * n1 + yi], j11 = g.J11[ey * n1 + yi];
    double det = j00 * j11 - j01 * j10;
    double i00 = j11 / det, i11 = j00 / det, i01 = -j01 / det, i10 = -j10 / det;
    double g0 = 0.0, g1 = 0.0;
    const double* p = psi + (N * ey * g.nv0 + N * ex);
    // the element's nodes (jj, ii) in row-major order; only row yi and
    // column xi can carry a non-zero shape-function derivative, so the walk
    // visits those in the same order (the others were skipped anyway).
    // a0: GNx * Ny, a1: Nx * GNy
    auto node = [&](double a0, double a1, double pv) {
        if (a0 == 0.0 && a1 == 0.0) return;
        double t0 = 0.0;
        t0 += a0 * i00;
        t0 += a1 * i01;
        double t1 = 0.0;
        t1 += a0 * i10;
        t1 += a1 * i11;
        g0 += t0 * pv;
        g1 += t1 * pv;
    };
    if (NN) {
        // both lines of psi and of D before the first use (one node after the
        // other the loads' latency was most of the time: 96x96 order 6 16 ->
        // 12 us)
        double pr[NN + 1], pc[NN + 1], dr[NN + 1], dc[NN + 1];
#pragma unroll
        for (int k = 0; k <= NN; k++) {
            pr[k] = p[yi * g.nv0 + k];
            pc[k] = p[k * g.nv0 + xi];
            dr[k] = g.D[xi * n1 + k];
            dc[k] = g.D[yi * n1 + k];
        }
#pragma unroll
        for (int jj = 0; jj <= NN; jj++)
            if (jj < yi) node(0.0, dc[jj], pc[jj]);
        double dy = 0.0;  // D[yi][yi]
#pragma unroll
        for (int k = 0; k <= NN; k++)
            if (k == yi) dy = dc[k];
#pragma unroll
        for (int ii = 0; ii <= NN; ii++) node(dr[ii], ii == xi ? dy : 0.0, pr[ii]);
#pragma unroll
        for (int jj = 0; jj <= NN; jj++)
            if (jj > yi) node(0.0, dc[jj], pc[jj]);
    } else {
        for (int jj = 0; jj < yi; jj++) node(0.0, g.D[yi * n1 + jj], p[jj * g.nv0 + xi]);
        for (int ii = 0; ii <= N; ii++) node(g.D[xi * n1 + ii], ii == xi ? g.D[yi * n1 + yi] : 0.0, p[yi * g.nv0 + ii]);
        for (int jj = yi + 1; jj <= N; jj++) node(0.0, g.D[yi * n1 + jj], p[jj * g.nv0 + xi]);
    }
    vel[2 * (size_t)v] = -1.0 * g1;
    vel[2 * (size_t)v + 1] = +1.0 * g0;
}

__global__ void k_maxvel2(int nV, const double* __restrict__ vel, unsigned long long* __restrict__ out) {
    double m = 0.0;
    for (int v = blockIdx.x * blockDim.x + threadIdx.x; v < nV; v += gridDim.x * blockDim.x) {
        double a = vel[2 * (size_t)v], b = vel[2 * (size_t)v + 1];
        double s = a * a + b * b;
        if (s > m) m = s;
    }
    for (int off = 32; off >= 1; off >>= 1) {
        double o = __shfl_xor(m, off, 64);
        m = o > m ? o : m;
    }
    // non-negative doubles order like their bit patterns
    if ((threadIdx.x & 63) == 0) atomicMax(out, (unsigned long long)__double_as_longlong(m));
}

SLGeom sl_geom(const se_mesh* m) {
    SLGeom g;
    g.N = m->N;
    // Advector's cubicInterp: N < 3 unless the caller chose (Advector.cpp:33,60)
    g.cubic = m->sl_interp == SE_INTERP_BICUBIC || (m->sl_interp == SE_INTERP_DEFAULT && m->N < 3);
    g.nEls0 = m->nEls[0];
    g.nEls1 = m->nEls[1];
    g.nv0 = m->nVerts[0];
    g.nv1 = m->nVerts[1];
    g.per0 = m->periodic[0];
    g.per1 = m->periodic[1];
    g.min0 = m->min[0];
    g.min1 = m->min[1];
    g.max0 = m->max[0];
    g.max1 = m->max[1];
    g.dx0 = m->dx[0];
    g.dx1 = m->dx[1];
    const int n1 = m->N + 1;
    const double* b = m->d_basis.as<double>();
    g.xk = b;
    g.D = b + 2 * n1;
    g.pnx = b + 2 * n1 + n1 * n1;
    g.pn = b + 3 * n1 + n1 * n1;
    g.X = m->d_X.as<double>();
    g.Y = m->d_Y.as<double>();
    g.J00 = m->d_J00.as<double>();
    g.J10 = m->d_J10.as<double>();
    g.J11 = m->d_J11.as<double>();
    g.J01 = m->d_J01.as<double>();
    return g;
}

int blocks_for(int n) { return (n + 255) / 256; }
int pair_blocks(int n) { return n / 128 + (n % 128 != 0); }  // two lanes per node

// KERNEL<N> for the orders 2..8, KERNEL<0> (the order read from the
// geometry) for the others; 256 threads per workgroup
#define SE_SL_LAUNCH(KERNEL, N, GRID, ...)                                          \
    switch (N) {                                                                    \
        case 2: hipLaunchKernelGGL(KERNEL<2>, GRID, dim3(256), 0, __VA_ARGS__); break; \
        case 3: hipLaunchKernelGGL(KERNEL<3>, GRID, dim3(256), 0, __VA_ARGS__); break; \
        case 4: hipLaunchKernelGGL(KERNEL<4>, GRID, dim3(256), 0, __VA_ARGS__); break; \
        case 5: hipLaunchKernelGGL(KERNEL<5>, GRID, dim3(256), 0, __VA_ARGS__); break; \
        case 6: hipLaunchKernelGGL(KERNEL<6>, GRID, dim3(256), 0, __VA_ARGS__); break; \
        case 7: hipLaunchKernelGGL(KERNEL<7>, GRID, dim3(256), 0, __VA_ARGS__); break; \
        case 8: hipLaunchKernelGGL(KERNEL<8>, GRID, dim3(256), 0, __VA_ARGS__); break; \
        default: hipLaunchKernelGGL(KERNEL<0>, GRID, dim3(256), 0, __VA_ARGS__); break; \
    }

// KERNEL<N, the advected components: 1, 2, else 0; -1: bicubic> for the orders
// 2..12 (se_sl_advect_dev, sl_second_check)
#define SE_SL_ADV(KERNEL, N, GRID, ...)                                                                   \
    if (g.cubic) hipLaunchKernelGGL((KERNEL<N, -1>), GRID, dim3(256), 0, __VA_ARGS__);                   \
    else if (nd == 1) hipLaunchKernelGGL((KERNEL<N, 1>), GRID, dim3(256), 0, __VA_ARGS__);               \
    else if (nd == 2) hipLaunchKernelGGL((KERNEL<N, 2>), GRID, dim3(256), 0, __VA_ARGS__);               \
    else hipLaunchKernelGGL((KERNEL<N, 0>), GRID, dim3(256), 0, __VA_ARGS__)
#define SE_SL_LAUNCH_ADV(KERNEL, N, GRID, ...)                        \
    switch (N) {                                                      \
        case 2: SE_SL_ADV(KERNEL, 2, GRID, __VA_ARGS__); break;       \
        case 3: SE_SL_ADV(KERNEL, 3, GRID, __VA_ARGS__); break;       \
        case 4: SE_SL_ADV(KERNEL, 4, GRID, __VA_ARGS__); break;       \
        case 5: SE_SL_ADV(KERNEL, 5, GRID, __VA_ARGS__); break;       \
        case 6: SE_SL_ADV(KERNEL, 6, GRID, __VA_ARGS__); break;       \
        case 7: SE_SL_ADV(KERNEL, 7, GRID, __VA_ARGS__); break;       \
        case 8: SE_SL_ADV(KERNEL, 8, GRID, __VA_ARGS__); break;       \
        case 9: SE_SL_ADV(KERNEL, 9, GRID, __VA_ARGS__); break;       \
        case 10: SE_SL_ADV(KERNEL, 10, GRID, __VA_ARGS__); break;     \
        case 11: SE_SL_ADV(KERNEL, 11, GRID, __VA_ARGS__); break;     \
        default: SE_SL_ADV(KERNEL, 12, GRID, __VA_ARGS__); break;     \
    }

struct SLScratch {
    DevBuf a, b, c, d, e, f, g, h;
    ~SLScratch() {
        DevBuf* all[] = {&a, &b, &c, &d, &e, &f, &g, &h};
        for (DevBuf* p : all) p->release();
    }
};

}  // namespace

extern "C" int se_sl_advect_dev(se_mesh* m, const double* d_q, int nd, const double* d_vel, double dt, double* d_qsl,
                                int32_t* d_dep) {
    SE_CHECK(m && d_q && d_vel && d_qsl, SE_ERR_ARG, "se_sl_advect_dev: NULL argument");
    SE_CHECK(nd >= 1 && nd <= 3, SE_ERR_ARG, "se_sl_advect_dev: nDofs must be 1..3");
    SE_CHECK(m->N <= 12, SE_ERR_UNSUPPORTED, "se_sl_advect_dev: order above 12");
    SE_CHECK(m->N >= 3 || (m->nVerts[0] >= 4 && m->nVerts[1] >= 4), SE_ERR_UNSUPPORTED,
             "bicubic advection (N < 3) needs at least 4 nodes per direction");
    SLGeom g = sl_geom(m);
    hipStream_t s = m->ctx->stream;
    SE_SL_LAUNCH_ADV(k_sl_first, m->N, dim3(pair_blocks(m->nV)), s, g, d_q, nd, d_vel, dt, d_qsl, d_dep);
    SE_HIP(hipGetLastError());
    return SE_OK;
}

namespace {

int sl_second_check(const se_mesh* m, const void* d_q, const void* d_qp, int nd, const void* d_vel,
                    const void* d_velp, const void* d_qsl, const char* who) {
    SE_CHECK(m && d_q && d_qp && d_vel && d_velp && d_qsl, SE_ERR_ARG, std::string(who) + ": NULL argument");
    SE_CHECK(nd >= 1 && nd <= 3, SE_ERR_ARG, std::string(who) + ": nDofs must be 1..3");
    SE_CHECK(m->N <= 12, SE_ERR_UNSUPPORTED, std::string(who) + ": order above 12");
    SE_CHECK(m->N >= 3 || (m->nVerts[0] >= 4 && m->nVerts[1] >= 4), SE_ERR_UNSUPPORTED,
             "bicubic advection (N < 3) needs at least 4 nodes per direction");
    return SE_OK;
}

// the second-order step with the three extrapolated velocity fields in
// vp1 | vph | vmh (2 nV doubles each)
int sl_second(se_mesh* m, const double* d_q, const double* d_qp, int nd, const double* d_vel, const double* d_velp,
              double dt, double* d_qsl, double* vp1) {
    SLGeom g = sl_geom(m);
    hipStream_t s = m->ctx->stream;
    const size_t n2 = 2 * (size_t)m->nV;
    double* vph = vp1 + n2;
    double* vmh = vph + n2;
    hipLaunchKernelGGL(k_extrap, dim3(blocks_for((int)n2)), dim3(256), 0, s, (int)n2, d_vel, d_velp, vp1, vph, vmh);
    SE_SL_LAUNCH_ADV(k_sl_second, m->N, dim3(pair_blocks(m->nV)), s, g, d_q, d_qp, nd, d_vel, vp1, vph, vmh, dt, d_qsl);
    SE_HIP(hipGetLastError());
    return SE_OK;
}

// Scratch of the allocation-free second-order step: its three extrapolated
// velocity fields, 3 x 2 x SE_SL_NOALLOC_MAX_NODES doubles (24 MiB).  One
// copy per GPU, held until the process ends.  Host code never passes the
// array's name to a kernel (on the host it is only a stand-in for the device
// symbol): it passes the per-device address that hipGetSymbolAddress gives.
static __device__ __align__(256) double scratch[3 * 2 * (size_t)SE_SL_NOALLOC_MAX_NODES];

std::mutex g_scratch_mu;
std::map<int, double*> g_scratch_ptr;  // device -> address of that device's scratch

// this device's scratch address, looked up once per device with that device
// current (the caller's current device is restored afterwards)
int scratch_of(int device, double** out) {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    auto it = g_scratch_ptr.find(device);
    if (it == g_scratch_ptr.end()) {
        double* ptr = nullptr;
        int prev = 0;
        SE_HIP(hipGetDevice(&prev));
        SE_HIP(hipSetDevice(device));
        hipError_t e = hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch));
        SE_HIP(hipSetDevice(prev));
        SE_CHECK(e == hipSuccess, SE_ERR_HIP,
                 std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        SE_CHECK(ptr != nullptr, SE_ERR_HIP, "no device address for the SL scratch");
        it = g_scratch_ptr.emplace(device, ptr).first;
    }
    *out = it->second;
    return SE_OK;
}

}  // namespace

extern "C" int se_sl_advect2_dev_noalloc(se_mesh* m, const double* d_q, const double* d_qp, int nd,
                                         const double* d_vel, const double* d_velp, double dt, double* d_qsl) {
    int rc = sl_second_check(m, d_q, d_qp, nd, d_vel, d_velp, d_qsl, "se_sl_advect2_dev_noalloc");
    if (rc) return rc;
    SE_CHECK((size_t)m->nV <= (size_t)SE_SL_NOALLOC_MAX_NODES, SE_ERR_ARG,
             "se_sl_advect2_dev_noalloc: the mesh has " + std::to_string(m->nV) +
                 " field nodes, more than the fixed scratch holds (SE_SL_NOALLOC_MAX_NODES = " +
                 std::to_string(SE_SL_NOALLOC_MAX_NODES) + "); use se_sl_advect2_dev");
    double* sc = nullptr;
    rc = scratch_of(m->ctx->device, &sc);
    if (rc) return rc;
    return sl_second(m, d_q, d_qp, nd, d_vel, d_velp, dt, d_qsl, sc);
}

extern "C" int se_sl_advect2_dev(se_mesh* m, const double* d_q, const double* d_qp, int nd, const double* d_vel,
                                 const double* d_velp, double dt, double* d_qsl) {
    int rc = sl_second_check(m, d_q, d_qp, nd, d_vel, d_velp, d_qsl, "se_sl_advect2_dev");
    if (rc) return rc;
    size_t n2 = 2 * (size_t)m->nV;
    rc = m->d_sl.alloc(3 * n2 * sizeof(double));
    if (rc) return rc;
    return sl_second(m, d_q, d_qp, nd, d_vel, d_velp, dt, d_qsl, m->d_sl.as<double>());
}

extern "C" int se_genvel_dev(se_mesh* m, const double* d_psi, double* d_vel) {
    SE_CHECK(m && d_psi && d_vel, SE_ERR_ARG, "se_genvel_dev: NULL argument");
    SLGeom g = sl_geom(m);
    SE_SL_LAUNCH(k_genvel, m->N, dim3(blocks_for(m->nV)), m->ctx->stream, g, d_psi, d_vel);
    SE_HIP(hipGetLastError());
    return SE_OK;
}

extern "C" int se_calc_timestep_dev(se_mesh* m, const double* d_vel, double courant, double* dt) {
    SE_CHECK(m && d_vel && dt, SE_ERR_ARG, "se_calc_timestep_dev: NULL argument");
    int rc = m->d_red.alloc(sizeof(unsigned long long));
    if (rc) return rc;
    hipStream_t s = m->ctx->stream;
    SE_HIP(hipMemsetAsync(m->d_red.ptr, 0, sizeof(unsigned long long), s));
    int nb = std::min(blocks_for(m->nV), 1024);
    hipLaunchKernelGGL(k_maxvel2, dim3(nb), dim3(256), 0, s, m->nV, d_vel, m->d_red.as<unsigned long long>());
    unsigned long long bits = 0;
    SE_HIP(hipMemcpyAsync(&bits, m->d_red.ptr, sizeof(bits), hipMemcpyDeviceToHost, s));
    SE_HIP(hipStreamSynchronize(s));
    double maxVelSq;
    std::memcpy(&maxVelSq, &bits, sizeof(double));
    // Utils.cpp:23-40
    double minSep = (m->dx[0] < m->dx[1]) ? m->dx[0] : m->dx[1];
    *dt = courant * minSep / std::sqrt(maxVelSq);
    return SE_OK;
}

// ---- host-pointer wrappers ---------------------------------------------------
namespace {
int up(hipStream_t s, DevBuf& b, const void* h, size_t bytes) {
    int rc = b.alloc(std::max<size_t>(bytes, 8));
    if (rc) return rc;
    SE_HIP(hipMemcpyAsync(b.ptr, h, bytes, hipMemcpyHostToDevice, s));
    return SE_OK;
}
int down(hipStream_t s, void* h, const DevBuf& b, size_t bytes) {
    SE_HIP(hipMemcpyAsync(h, b.ptr, bytes, hipMemcpyDeviceToHost, s));
    SE_HIP(hipStreamSynchronize(s));
    return SE_OK;
}
}  // namespace

extern "C" int se_sl_advect(se_mesh* m, const double* q, int nd, const double* vel, double dt, double* qsl,
                            int32_t* dep) {
    SE_CHECK(m && q && vel && qsl, SE_ERR_ARG, "se_sl_advect: NULL argument");
    SE_CHECK(nd >= 1 && nd <= 3, SE_ERR_ARG, "se_sl_advect: nDofs must be 1..3");
    SE_HIP(hipSetDevice(m->ctx->device));
    hipStream_t s = m->ctx->stream;
    SLScratch b;
    size_t nV = m->nV;
    int rc = up(s, b.a, q, nV * nd * sizeof(double));
    if (!rc) rc = up(s, b.b, vel, nV * 2 * sizeof(double));
    if (!rc) rc = b.c.alloc(nV * nd * sizeof(double));
    if (!rc) rc = b.d.alloc(nV * sizeof(int32_t));
    if (!rc) rc = se_sl_advect_dev(m, b.a.as<double>(), nd, b.b.as<double>(), dt, b.c.as<double>(),
                                   dep ? b.d.as<int32_t>() : nullptr);
    if (!rc) rc = down(s, qsl, b.c, nV * nd * sizeof(double));
    if (!rc && dep) rc = down(s, dep, b.d, nV * sizeof(int32_t));
    return rc;
}

extern "C" int se_sl_advect2(se_mesh* m, const double* q, const double* qp, int nd, const double* vel,
                             const double* velp, double dt, double* qsl) {
    SE_CHECK(m && q && qp && vel && velp && qsl, SE_ERR_ARG, "se_sl_advect2: NULL argument");
    SE_CHECK(nd >= 1 && nd <= 3, SE_ERR_ARG, "se_sl_advect2: nDofs must be 1..3");
    SE_HIP(hipSetDevice(m->ctx->device));
    hipStream_t s = m->ctx->stream;
    SLScratch b;
    size_t nV = m->nV;
    int rc = up(s, b.a, q, nV * nd * sizeof(double));
    if (!rc) rc = up(s, b.b, qp, nV * nd * sizeof(double));
    if (!rc) rc = up(s, b.c, vel, nV * 2 * sizeof(double));
    if (!rc) rc = up(s, b.d, velp, nV * 2 * sizeof(double));
    if (!rc) rc = b.e.alloc(nV * nd * sizeof(double));
    if (!rc) rc = se_sl_advect2_dev(m, b.a.as<double>(), b.b.as<double>(), nd, b.c.as<double>(), b.d.as<double>(), dt,
                                    b.e.as<double>());
    if (!rc) rc = down(s, qsl, b.e, nV * nd * sizeof(double));
    return rc;
}

extern "C" int se_genvel(se_mesh* m, const double* psi, double* vel) {
    SE_CHECK(m && psi && vel, SE_ERR_ARG, "se_genvel: NULL argument");
    SE_HIP(hipSetDevice(m->ctx->device));
    hipStream_t s = m->ctx->stream;
    SLScratch b;
    size_t nV = m->nV;
    int rc = up(s, b.a, psi, nV * sizeof(double));
    if (!rc) rc = b.b.alloc(nV * 2 * sizeof(double));
    if (!rc) rc = se_genvel_dev(m, b.a.as<double>(), b.b.as<double>());
    if (!rc) rc = down(s, vel, b.b, nV * 2 * sizeof(double));
    return rc;
}

extern "C" int se_calc_timestep(se_mesh* m, const double* vel, double courant, double* dt) {
    SE_CHECK(m && vel && dt, SE_ERR_ARG, "se_calc_timestep: NULL argument");
    SE_HIP(hipSetDevice(m->ctx->device));
    hipStream_t s = m->ctx->stream;
    SLScratch b;
    int rc = up(s, b.a, vel, (size_t)m->nV * 2 * sizeof(double));
    if (!rc) rc = se_calc_timestep_dev(m, b.a.as<double>(), courant, dt);
    return rc;
}

extern "C" int se_mesh_set_sl_interp(se_mesh* m, int mode) {
    SE_CHECK(m, SE_ERR_ARG, "se_mesh_set_sl_interp: NULL argument");
    SE_CHECK(mode == SE_INTERP_DEFAULT || mode == SE_INTERP_GLL || mode == SE_INTERP_BICUBIC, SE_ERR_ARG,
             "se_mesh_set_sl_interp: mode must be SE_INTERP_DEFAULT, SE_INTERP_GLL or SE_INTERP_BICUBIC");
    const bool cubic = mode == SE_INTERP_BICUBIC || (mode == SE_INTERP_DEFAULT && m->N < 3);
    SE_CHECK(!cubic || (m->nVerts[0] >= 4 && m->nVerts[1] >= 4), SE_ERR_UNSUPPORTED,
             "bicubic interpolation needs at least 4 nodes per direction");
    m->sl_interp = mode;
    return SE_OK;
}

extern "C" int se_interp_points_dev(se_mesh* m, const double* d_vals, int nd, int npts, const double* d_xy, int mode,
                                    double* d_out) {
    SE_CHECK(m && (npts == 0 || (d_vals && d_xy && d_out)), SE_ERR_ARG, "se_interp_points_dev: NULL argument");
    SE_CHECK(nd >= 1 && nd <= 3 && npts >= 0, SE_ERR_ARG, "se_interp_points_dev: nDofs 1..3, npts >= 0");
    SE_CHECK(mode == SE_INTERP_DEFAULT || mode == SE_INTERP_GLL || mode == SE_INTERP_BICUBIC, SE_ERR_ARG,
             "se_interp_points_dev: bad mode");
    SE_CHECK(m->N <= 12, SE_ERR_UNSUPPORTED, "se_interp_points_dev: order above 12");
    const int cubic = mode == SE_INTERP_BICUBIC || (mode == SE_INTERP_DEFAULT && m->N < 3);
    SE_CHECK(!cubic || (m->nVerts[0] >= 4 && m->nVerts[1] >= 4), SE_ERR_UNSUPPORTED,
             "bicubic interpolation needs at least 4 nodes per direction");
    if (npts == 0) return SE_OK;
    SLGeom g = sl_geom(m);
    SE_SL_LAUNCH(k_interp_points, m->N, dim3(blocks_for(npts)), m->ctx->stream, g, d_vals, nd, npts, d_xy, cubic,
                 d_out);
    SE_HIP(hipGetLastError());
    return SE_OK;
}

extern "C" int se_interp_points(se_mesh* m, const double* vals, int nd, int npts, const double* xy, int mode,
                                double* out) {
    SE_CHECK(m && (npts == 0 || (vals && xy && out)), SE_ERR_ARG, "se_interp_points: NULL argument");
    SE_CHECK(nd >= 1 && nd <= 3 && npts >= 0, SE_ERR_ARG, "se_interp_points: nDofs 1..3, npts >= 0");
    if (npts == 0) return SE_OK;
    SE_HIP(hipSetDevice(m->ctx->device));
    hipStream_t s = m->ctx->stream;
    SLScratch b;
    const size_t nv = (size_t)m->nV * nd;
    int rc = up(s, b.a, vals, nv * sizeof(double));
    if (!rc) rc = up(s, b.b, xy, 2 * (size_t)npts * sizeof(double));
    if (!rc) rc = b.c.alloc((size_t)npts * nd * sizeof(double));
    if (!rc) rc = se_interp_points_dev(m, b.a.as<double>(), nd, npts, b.b.as<double>(), mode, b.c.as<double>());
    if (!rc) rc = down(s, out, b.c, (size_t)npts * nd * sizeof(double));
    return rc;
}
