// sl.hip -- semi-Lagrangian advection (departure-point search + GLL
// interpolation), velocity from the stream function, CFL time step.
//
// Two lanes per field node, one for each dimension (sl_steps.h).  The coordinate
// arithmetic that decides the departure element (RK2 midpoint, wrap/clamp,
// GetEl's modf and its 1e-12 edge rule, the local-coordinate map) follows the
// reference's operation order with FP contraction disabled.  P_N(x_j) is
// tabulated on the host with the reference's evaluation; P_N'(x) is evaluated on
// the device with the same monomial sum, its powers bit-identical to the C
// library's pow (glibc_pow.h), so interpolated values and departure elements
// agree with the reference's bit for bit.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <mutex>
#include <string>

#include "se_common.h"
#include "sl_steps.h"

using namespace se;
using namespace se_sl;

namespace {

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

// a step's kernel for the orders 2..12 (se_sl_advect_dev, sl_second_check):
// those above 8 by HIGH
#define SE_SL_LAUNCH_ADV(KERNEL, HIGH, N, S, ...)                                      \
    do {                                                                               \
        const dim3 grid(pair_blocks(g.nv0 * g.nv1));                                   \
        switch (N) {                                                                   \
            case 2: SE_SL_ADV(KERNEL, 2, grid, S, __VA_ARGS__); break;                 \
            case 3: SE_SL_ADV(KERNEL, 3, grid, S, __VA_ARGS__); break;                 \
            case 4: SE_SL_ADV(KERNEL, 4, grid, S, __VA_ARGS__); break;                 \
            case 5: SE_SL_ADV(KERNEL, 5, grid, S, __VA_ARGS__); break;                 \
            case 6: SE_SL_ADV(KERNEL, 6, grid, S, __VA_ARGS__); break;                 \
            case 7: SE_SL_ADV(KERNEL, 7, grid, S, __VA_ARGS__); break;                 \
            case 8: SE_SL_ADV(KERNEL, 8, grid, S, __VA_ARGS__); break;                 \
            default: HIGH(N, S, __VA_ARGS__); break;                                   \
        }                                                                              \
    } while (0)

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
    SE_SL_LAUNCH_ADV(k_sl_first, sl_first_high, m->N, s, g, d_q, nd, d_vel, dt, d_qsl, d_dep);
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
    SE_SL_LAUNCH_ADV(k_sl_second, sl_second_high, m->N, s, g, d_q, d_qp, nd, d_vel, vp1, vph, vmh, dt, d_qsl);
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
