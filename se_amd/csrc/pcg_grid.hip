// pcg_grid.hip -- the FP64 Jacobi-PCG of one operator as one launch.
//
// The reference's algorithm (KSPSolve with -ksp_type cg -pc_type jacobi,
// src/linsys/HelmholtzEqn.cpp:120-131) needs two global sums per iteration.
// As separate kernels (helm.hip) an iteration is three dependent launches of
// 5 to 19 us, whatever the size: 14 us at 1024 unknowns (p = 4), 20 us at
// 36 672 (p = 6), 36 us at 1 048 576 (p = 8).  Here every workgroup owns a tile
// of elements for the whole solve and the workgroups meet at grid-wide sums:
// 5.2, 8.3 and 18 us per iteration at those sizes, beside 15 to 40 us for the
// launch, the start and the check.
//   * p of the tile stays in LDS, r, and where they fit x and the inverse
//     diagonal, in registers.  A tile holds all nodes of its elements; a node
//     on an edge is held by every tile around it, with the same value.
//   * Each tile applies its own elements only, so no element is evaluated
//     twice; p.q is the sum of the tiles' own parts.  The parts of A p on the
//     tile's edges (one line a side) go through memory (ex) and every tile
//     sums the parts of its edge nodes in one common order.  (Evaluating the
//     neighbouring elements instead, with r of an element ring exchanged,
//     took 7.5 ms against 6.6 at 36 672 unknowns and 22 against 13.9 at
//     1 048 576: more elements, and rings an element wide.)
//   * A grid-wide sum is an all-to-all: each workgroup stores its partials to
//     slots of its own and every workgroup polls all slots, so a sum costs one
//     store and one load through the coherence point (1.6 us for 8
//     workgroups, 3.3 us for 256).  A slot holds a mark, a NaN no sum
//     produces, until its value arrives, so value and arrival are one 8-byte
//     word.  Three slot sets rotate: a workgroup that has passed sum s - 1
//     knows that all are done with set s - 2 = s + 1 (mod 3) and empties its
//     slots there.
//   * Everything another workgroup reads is written and read by relaxed
//     agent-scope atomics (write-through stores, loads past the XCD's L2); a
//     wave waits for its stores before its workgroup publishes a partial.
// The same totals in the same order reach every workgroup, so all take the
// same decisions and the result does not depend on timing.
//
// Bound by the latency of the two sums (4 to 8 us) and by VALU issue in the
// operator (2 us for 4 waves per CU, 6 us for 9).
//
// Waits are bounded: a workgroup whose partners do not arrive within `limit`
// (workgroups that are not resident together) gives up, all leave, and the
// caller runs the launch-per-phase solver instead.  The solves of a process
// share a device's CUs by turns (GridGate), so they cannot hold each other's
// workgroups out.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <condition_variable>
#include <cstdlib>
#include <mutex>

#include "apply_kernels.h"
#include "apply_lines.h"
#include "helm_kernels.h"
#include "se_common.h"
#include "se_op.h"

namespace se {

namespace {

typedef unsigned long long u64;
constexpr u64 kEmpty = ~0ull;       // a slot whose value has not arrived
constexpr int kSlots = 256;         // workgroups at most
constexpr int kSums = 4;            // values per grid-wide sum at most
constexpr double kWaitLimit = 0.1;  // seconds a workgroup waits for the others

// element at a 32-bit byte offset: a uniform base and one offset register
__device__ __forceinline__ const SE_GLOBAL double* at_byte(const double* p, unsigned off) {
    return (const SE_GLOBAL double*)((const SE_GLOBAL char*)p + off);
}
__device__ __forceinline__ SE_GLOBAL double* at_byte(double* p, unsigned off) {
    return (SE_GLOBAL double*)((SE_GLOBAL char*)p + off);
}
__device__ __forceinline__ void put_bits(double* p, unsigned off, u64 b) {
    __hip_atomic_store((SE_GLOBAL u64*)at_byte(p, off), b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 get_bits(double* p, unsigned off) {
    return __hip_atomic_load((SE_GLOBAL u64*)at_byte(p, off), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// sum over the first 16 lanes of a wave, to every lane
__device__ __forceinline__ double row_sum(double v) {
    v += dpp_shr(v, 1);
    v += dpp_shr(v, 2);
    v += dpp_shr(v, 4);
    v += dpp_shr(v, 8);
    return lane_value(v, 15);
}
// a value's bits: any NaN, but never the empty mark
__device__ __forceinline__ u64 value_bits(double v) {
    return v != v ? 0x7ff8000000000000ull : (u64)__double_as_longlong(v);
}

struct GridArgs {
    OpParams P;
    const double* f;      // right-hand side
    const double* dinv;   // inverse diagonal of sign*A
    double* x;            // result
    double* px;           // [G][NL T]: p over a failed true-residual check
    double* ex;           // [G][kEdge]: each tile's part of A p on its edges
    u64* slots;           // [3][kSums][kSlots]
    u64* next;            // the next solve's slots
    CgState* st;          // pinned host memory: the outcome; pad = 1: a wait ran out
    int tx, ty, tilesX, tilesY, G, n, null_space, maxit;
    double sgn, rtol;
    u64 limit;            // ticks of the constant 100 MHz clock
};

// nodes of a tile per thread (checked on the host)
constexpr int grid_cells(int N) { return N; }
constexpr int kEdge = 512;  // edge nodes of a tile at most

template <int N, int T>
__global__ __launch_bounds__(T) void k_pcg_grid(GridArgs g) {
    constexpr int N1 = N + 1, NP = N1 * N1, F = 4 * N1, QS = 2 * NP, NW = T / 64;
    constexpr int NL = grid_cells(N);
    // x in registers or LDS, the inverse diagonal in registers or read from
    // memory each time, the nodes' slots ready or formed from one word: what
    // the register file leaves beside the lines
    constexpr bool XREG = T == 256, DREG = T == 256 || N <= 6, PACK = DREG;
    extern __shared__ double lds[];
    __shared__ double s_red[2][kSums][NW], s_red2[2][kSums][4];
    __shared__ int s_give_up;

    const OpParams& P = g.P;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, wg = blockIdx.x;
    const int X = wg % g.tilesX, Y = wg / g.tilesX, ex0 = X * g.tx, ey0 = Y * g.ty;
    const int ncx = min(g.tx, P.nEls0 - ex0), ncy = min(g.ty, P.nEls1 - ey0), NE = ncx * ncy;
    const int W = ncx * N + 1, H = ncy * N + 1, BW = W | 1;
    const bool left = X > 0 || P.per0, right = X + 1 < g.tilesX || P.per0;
    const bool below = Y > 0 || P.per1, above = Y + 1 < g.tilesY || P.per1;

    double* s_u = lds;                       // the tile: p (or x in a check); node i = a BW + b
    double* s_o = s_u + NL * T;              // element outputs, FP32 exchange before; one zero
    const int zero = NE * NP;
    double* s_q = s_o + NE * NP + 1;         // A p on the tile's edges, all parts
    double* s_ex = s_q + kEdge;              // a single workgroup's ex
    double* s_cf = s_ex + (g.G == 1 ? kEdge : 0);
    double* s_rf = s_cf + ncx * F;
    float* s_cq = (float*)(s_rf + ncy * F);
    float* s_rq = s_cq + ncx * QS;
    double* s_x = (double*)(s_rq + ncy * QS);
    float* s_xf = (float*)s_o;
    float* s_ef = s_xf + NE * NP;

    for (int i = tid; i < ncx * F; i += T) s_cf[i] = gview(P.colTab)[(size_t)ex0 * F + i];
    for (int i = tid; i < ncy * F; i += T) s_rf[i] = gview(P.rowTab)[(size_t)ey0 * F + i];
    for (int i = tid; i < ncx * QS; i += T) s_cq[i] = gview(P.colQ)[(size_t)ex0 * QS + i];
    for (int i = tid; i < ncy * QS; i += T) s_rq[i] = gview(P.rowQ)[(size_t)ey0 * QS + i];
    if (tid == 0) s_give_up = 0, s_o[zero] = 0.0;
    if (tid < 3 * kSums)
        __hip_atomic_store((SE_GLOBAL u64*)g.next + tid * kSlots + wg, kEmpty, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);

    // where tile (tX, tY) keeps its part at its edge node (col, row) in its
    // run of ex: left edge, right edge, bottom, top
    auto edge_index = [&](int W_, int H_, int col, int row) {
        return col == 0 ? row : (col == W_ - 1 ? H_ + row : (row == 0 ? 2 * H_ + col : 2 * H_ + W_ + col));
    };
    // The s_o slots of node (col, row)'s up to four element outputs (bottom
    // left, bottom, left, own; the zero where there is no element): PACK, 16
    // bits each; else its own element's (virtual on a closing line) << 4 and
    // which of the four there are, below bit 20.
    auto node_slots = [&](int col, int row, unsigned& lo, unsigned& hi) {
        const int cq = col / N, lx = col - cq * N, rq = row / N, ly = row - rq * N;
        const bool cl = lx == 0 && cq > 0, co = cq < ncx, rl = ly == 0 && rq > 0, ro = rq < ncy;
        const int at = (rq * ncx + cq) * NP + ly * N1 + lx;
        lo = (at << 4) | (rl && cl ? 1 : 0) | (rl && co ? 2 : 0) | (ro && cl ? 4 : 0) | (ro && co ? 8 : 0);
        if (PACK) {
            const int m = lo;
            lo = (m & 1 ? at - (ncx + 1) * NP + N * N1 + N : zero) | (m & 2 ? at - ncx * NP + N * N1 : zero) << 16;
            hi = (m & 4 ? at - NP + N : zero) | (m & 8 ? at : zero) << 16;
        }
    };
    // sign times the sum of a node's element outputs
    auto node_sum = [&](unsigned lo, unsigned hi) {
        unsigned i0 = lo & 0xffff, i1 = lo >> 16, i2 = hi & 0xffff, i3 = hi >> 16;
        if (!PACK) {
            const int at = (lo >> 4) & 0xffff;
            i0 = lo & 1 ? at - (ncx + 1) * NP + N * N1 + N : zero;
            i1 = lo & 2 ? at - ncx * NP + N * N1 : zero;
            i2 = lo & 4 ? at - NP + N : zero;
            i3 = lo & 8 ? at : zero;
        }
        return g.sgn * (((s_o[i0] + s_o[i1]) + s_o[i2]) + s_o[i3]);
    };

    // ---- this thread's nodes of the tile ---------------------------------------
    // u: byte offset of the unknown, -1: none.  olo, ohi: node_slots; without
    // an unknown all zeros (q, r, p and x stay zero there).  edge: which nodes
    // other tiles hold too, and ei their edge indices (not
    // PACK: edge index + 1 from bit 20 of olo).
    int u[NL];
    unsigned olo[NL], ohi[PACK ? NL : 1], edge = 0, ei[PACK ? (NL + 1) / 2 : 1] = {};
    unsigned own = 0;  // this tile counts the node in the sums and writes x
    double r[NL], xr[XREG ? NL : 1], dr[DREG ? NL : 1];
#pragma unroll
    for (int k = 0; k < NL; k++) {
        const int i = tid + T * k, a = i / BW, b = i - a * BW;
        u[k] = -1, r[k] = 0.0;
        olo[k] = PACK ? zero | zero << 16 : 0;
        if (PACK) ohi[PACK ? k : 0] = zero | zero << 16;
        if (a < H && b < W) {
            const int I = unk_line(ex0 * N + b, P.nEls0 * N, P.per0, P.off0, P.nU0);
            const int J = unk_line(ey0 * N + a, P.nEls1 * N, P.per1, P.off1, P.nU1);
            if (I >= 0 && J >= 0) {
                u[k] = 8 * (J * P.nU0 + I);
                node_slots(b, a, olo[k], ohi[PACK ? k : 0]);
                const bool r_ = b == W - 1 && right, t_ = a == H - 1 && above;
                if (r_ || t_ || (b == 0 && left) || (a == 0 && below)) {
                    edge |= 1u << k;
                    const unsigned j = edge_index(W, H, b, a);
                    if (PACK) ei[PACK ? k / 2 : 0] |= j << (16 * (k & 1));
                    else olo[k] |= (j + 1) << 20;
                }
                if (!r_ && !t_) own |= 1u << k;
            }
        }
        if (XREG) xr[XREG ? k : 0] = 0.0;
        else s_x[i] = 0.0;
        if (DREG) dr[DREG ? k : 0] = u[k] >= 0 ? *at_byte(g.dinv, u[k]) : 0.0;
    }
    // ---- this thread's edge node -------------------------------------------------
    // elo, ehi: its node_slots; ep: the byte offsets in ex of the tiles' parts, in
    // an order all tiles share (the left tile's before the right's, the lower
    // tile's before the upper's), -1: none
    const int edge_nodes = 2 * H + 2 * W;
    unsigned elo = 0, ehi = 0;
    int ep[4] = {-1, -1, -1, -1};
    if (tid < edge_nodes) {
        const int col = tid < H ? 0 : (tid < 2 * H ? W - 1 : (tid < 2 * H + W ? tid - 2 * H : tid - 2 * H - W));
        const int row = tid < H ? tid : (tid < 2 * H ? tid - H : (tid < 2 * H + W ? 0 : H - 1));
        node_slots(col, row, elo, ehi);
        const bool l_ = col == 0 && left, r_ = col == W - 1 && right, b_ = row == 0 && below, t_ = row == H - 1 && above;
#pragma unroll
        for (int c = 0; c < 4; c++) {
            // bit 0: the copy at its tile's left edge; bit 1: at its bottom edge
            const bool zx = c & 1, zy = c & 2;
            int tX = X, tY = Y, cc = col, rr = row;
            bool have = true;
            if (l_ || r_) {
                if (l_ && !zx) tX = X > 0 ? X - 1 : g.tilesX - 1;
                if (r_ && zx) tX = X + 1 < g.tilesX ? X + 1 : 0;
                cc = zx ? 0 : min(g.tx, P.nEls0 - tX * g.tx) * N;
            } else if (zx) {
                have = false;
            }
            if (b_ || t_) {
                if (b_ && !zy) tY = Y > 0 ? Y - 1 : g.tilesY - 1;
                if (t_ && zy) tY = Y + 1 < g.tilesY ? Y + 1 : 0;
                rr = zy ? 0 : min(g.ty, P.nEls1 - tY * g.ty) * N;
            } else if (zy) {
                have = false;
            }
            const int W_ = min(g.tx, P.nEls0 - tX * g.tx) * N + 1, H_ = min(g.ty, P.nEls1 - tY * g.ty) * N + 1;
            if (have) ep[c] = 8 * ((tY * g.tilesX + tX) * kEdge + edge_index(W_, H_, cc, rr));
        }
    }
    int e = tid / N1, t = tid - e * N1, er = e / ncx, ec = e - er * ncx;
    const bool live = e < NE;

    int seq = 0;
    // the totals of v over all workgroups; false when a wait ran out
    auto grid_sum = [&](auto& v) -> bool {
        constexpr int K = sizeof(v) / sizeof(double);
        const int sp = seq & 1;
#pragma unroll
        for (int k = 0; k < K; k++) {
            const double s = wave_sum(v[k]);
            if (lane == 0) s_red[sp][k][wid] = s;
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's parts in ex have arrived
        __syncthreads();
        if (g.G == 1) {
#pragma unroll
            for (int k = 0; k < K; k++) v[k] = row_sum(lane < NW ? s_red[sp][k][lane] : 0.0);
            seq++;
            return true;
        }
        u64* cur = g.slots + (size_t)(seq % 3) * kSums * kSlots;
        if (wid == 0) {
#pragma unroll
            for (int k = 0; k < K; k++) {
                const double s = row_sum(lane < NW ? s_red[sp][k][lane] : 0.0);
                if (lane == k)
                    __hip_atomic_store((SE_GLOBAL u64*)cur + k * kSlots + wg, value_bits(s), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        u64 w[K];
#pragma unroll
        for (int k = 0; k < K; k++) w[k] = 0;
        if (tid < g.G) {
            const u64 t0 = wall_clock64();
            for (int spin = 0;; spin++) {
                bool all = true;
#pragma unroll
                for (int k = 0; k < K; k++)
                    w[k] = __hip_atomic_load((SE_GLOBAL u64*)cur + k * kSlots + tid, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                for (int k = 0; k < K; k++) all = all && w[k] != kEmpty;
                if (all) break;
                if (g.limit == 0 || ((spin & 63) == 63 && wall_clock64() - t0 > g.limit)) {
                    s_give_up = 1;
                    break;
                }
            }
        }
        if (tid < kSlots) {
#pragma unroll
            for (int k = 0; k < K; k++) {
                const double s = wave_sum(__longlong_as_double((long long)w[k]));
                if (lane == 0) s_red2[sp][k][wid] = s;
            }
        }
        __syncthreads();
        if (s_give_up) return false;
#pragma unroll
        for (int k = 0; k < K; k++)
            v[k] = ((s_red2[sp][k][0] + s_red2[sp][k][1]) + s_red2[sp][k][2]) + s_red2[sp][k][3];
        // all workgroups have passed sum seq - 1: its predecessor's set is free
        u64* nxt = g.slots + (size_t)((seq + 2) % 3) * kSums * kSlots;
        if (tid < kSums)
            __hip_atomic_store((SE_GLOBAL u64*)nxt + tid * kSlots + wg, kEmpty, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        seq++;
        return true;
    };
    // q = this tile's part of sign A s_u at the thread's nodes; its edge nodes'
    // parts go to ex (read after the next sum, and free again after the one
    // after that)
    double q[NL];
    auto apply = [&]() {
        double yx[N1], yy[N1], uxi[N1], uet[N1];
        if (live) line_gradients<N>(P, s_u, BW, er, ec, t, e, s_xf, s_ef, uxi, uet);
        __syncthreads();
        if (live)
            line_outputs<N>(P, s_u, BW, er, ec, t, e, s_xf, s_ef, s_cf + ec * F, s_rf + er * F, s_cq + ec * QS,
                            s_rq + er * QS, uxi, uet, yx, yy);
        __syncthreads();
        if (live) {
#pragma unroll
            for (int l = 0; l < N1; l++) s_o[e * NP + l * N1 + t] = yy[l];
        }
        __syncthreads();
        if (live) {
#pragma unroll
            for (int l = 0; l < N1; l++) yy[l] = s_o[e * NP + t * N1 + l];
#pragma unroll
            for (int l = 0; l < N1; l++) s_o[e * NP + t * N1 + l] = yy[l] + yx[l];
        }
        __syncthreads();
        if (tid < edge_nodes) {
            const double part = node_sum(elo, ehi);
            if (g.G == 1) s_ex[tid] = part;
            else put_bits(g.ex, 8 * (wg * kEdge + tid), (u64)__double_as_longlong(part));
        }
#pragma unroll
        for (int k = 0; k < NL; k++) q[k] = node_sum(olo[k], ohi[PACK ? k : 0]);
    };
    // after a sum: q of the edge nodes with all tiles' parts.  (Polling ex for
    // them beside the sum's slots, with no wait before its partials are
    // stored, measured slower, 17.3 against 13.6 ms at 128 x 128, p = 8: the
    // polls hold up the stores they wait for.)
    auto join_edges = [&]() {
        if (tid < edge_nodes) {
            double w[4];
#pragma unroll
            for (int c = 0; c < 4; c++) w[c] = 0.0;
            if (g.G == 1) {
#pragma unroll
                for (int c = 0; c < 4; c++)
                    if (ep[c] >= 0) w[c] = *(const double*)((const char*)s_ex + ep[c]);
            } else {
#pragma unroll
                for (int c = 0; c < 4; c++)
                    if (ep[c] >= 0) w[c] = __longlong_as_double((long long)get_bits(g.ex, ep[c]));
            }
            s_q[tid] = ((w[0] + w[1]) + w[2]) + w[3];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < NL; k++) {
            if (PACK) {
                if (edge & (1u << k)) q[k] = s_q[(ei[PACK ? k / 2 : 0] >> (16 * (k & 1))) & 0xffff];
            } else if (olo[k] >> 20) {
                q[k] = s_q[(olo[k] >> 20) - 1];
            }
        }
    };
    double d[NL], v[4];
    auto load_dinv = [&]() {
#pragma unroll
        for (int k = 0; k < NL; k++) {
            if (DREG) d[k] = dr[DREG ? k : 0];
            else d[k] = u[k] >= 0 ? *at_byte(g.dinv, u[k]) : 0.0;
        }
    };
    auto sums = [&]() {  // r.r, r.z, sum z, sum r of this thread's nodes
        v[0] = v[1] = v[2] = v[3] = 0.0;
#pragma unroll
        for (int k = 0; k < NL; k++) {
            const double rk = own & (1u << k) ? r[k] : 0.0, z = d[k] * rk;
            v[0] += rk * rk;
            v[1] += rk * z;
            v[2] += z;
            v[3] += rk;
        }
    };
    auto give_up = [&]() {
        if (tid == 0) g.st->pad = 1;
    };

    // ---- start: b = sgn f - mean, r = b, p = D^-1 r - mu --------------------------
    double mu_b = 0.0;
    if (g.null_space) {
        double w[1] = {0.0};
#pragma unroll
        for (int k = 0; k < NL; k++)
            if (own & (1u << k)) w[0] += g.sgn * *at_byte(g.f, u[k]);
        if (!grid_sum(w)) return give_up();
        mu_b = w[0] / g.n;
    }
    load_dinv();
#pragma unroll
    for (int k = 0; k < NL; k++) {
        if (u[k] >= 0) r[k] = g.sgn * *at_byte(g.f, u[k]) - mu_b;
        s_u[tid + T * k] = d[k] * r[k];  // (- mu below)
    }
    sums();
    if (!grid_sum(v)) return give_up();
    const double bb = v[0], tol2 = g.rtol * g.rtol * bb;
    double rr = bb, rho_prev = 0.0, tt = 0.0;
    double mu = g.null_space ? v[2] / g.n : 0.0;
    double rho = v[1] - mu * v[3];
    int iter = 0, guard = 0, status = CG_RUNNING;
    if (bb == 0.0) status = 0;
    else if (!(bb - bb == 0.0) || !(v[1] - v[1] == 0.0)) status = 3;
    if (status == 3 && bb - bb == 0.0) tt = bb;  // (x = 0: the residual is b)
    if (mu != 0.0 && status == CG_RUNNING) {
#pragma unroll
        for (int k = 0; k < NL; k++)
            if (u[k] >= 0) s_u[tid + T * k] -= mu;
    }
    __syncthreads();

    // One pass of the loop applies the operator to the tile: to p in an
    // iteration, to x when the residual is checked (the recursion has met the
    // target, or the solve stops without meeting it).
    bool check = false;
    while (status == CG_RUNNING || check) {
        // (keeps the addresses formed from these out of registers across the loop)
#pragma unroll
        for (int k = 0; k < NL; k++) asm volatile("" : "+v"(u[k]), "+v"(olo[k]), "+v"(ohi[PACK ? k : 0]));
        asm volatile("" : "+v"(e), "+v"(t), "+v"(er), "+v"(ec));
        apply();
        if (!check) {
            // ---- alpha, x, r -----------------------------------------------------
            load_dinv();
            double a[1] = {0.0};
#pragma unroll
            for (int k = 0; k < NL; k++) a[0] += s_u[tid + T * k] * q[k];
            if (!grid_sum(a)) return give_up();
            const double pq = a[0];
            if (!(pq > 0.0)) {
                status = (pq - pq == 0.0) ? 2 : 3;
                if (!grid_sum(a)) return give_up();  // (all are past this apply's parts)
            } else {
                const double alpha = rho / pq;
                rho_prev = rho;
                join_edges();
#pragma unroll
                for (int k = 0; k < NL; k++) {
                    r[k] -= alpha * q[k];
                    if (XREG) xr[XREG ? k : 0] += alpha * s_u[tid + T * k];
                    else s_x[tid + T * k] += alpha * s_u[tid + T * k];
                }
                sums();
                if (g.null_space) {
                    if (!grid_sum(v)) return give_up();
                } else {
                    double w[2] = {v[0], v[1]};
                    if (!grid_sum(w)) return give_up();
                    v[0] = w[0], v[1] = w[1];
                }
                rr = v[0];
                iter++;
                if (!(rr - rr == 0.0) || !(v[1] - v[1] == 0.0)) status = 3;
                else if (rr <= tol2) check = true;
                else if (iter >= g.maxit) status = 1;
            }
            if (check || status != CG_RUNNING) {
                // the tile takes x; p is kept in px
                check = true;
#pragma unroll
                for (int k = 0; k < NL; k++) {
                    const int i = tid + T * k;
                    *at_byte(g.px, 8 * (wg * NL * T + i)) = s_u[i];
                    s_u[i] = XREG ? xr[XREG ? k : 0] : s_x[i];
                }
                __syncthreads();
                continue;
            }
        } else {
            // ---- r = b - A x; ||r||^2 less its mean part ---------------------------
            check = false;
            double none[1] = {0.0};
            if (!grid_sum(none)) return give_up();
            join_edges();
            double a[2] = {0.0, 0.0};
#pragma unroll
            for (int k = 0; k < NL; k++) {
                if (u[k] >= 0) r[k] = (g.sgn * *at_byte(g.f, u[k]) - mu_b) - q[k];
                const double rk = own & (1u << k) ? r[k] : 0.0;
                a[0] += rk;
                a[1] += rk * rk;
            }
            if (!grid_sum(a)) return give_up();
            const double mt = g.null_space ? a[0] / g.n : 0.0;
            tt = g.null_space ? a[1] - a[0] * mt : a[1];
            if (status != CG_RUNNING) break;
            if (tt <= tol2) {
                status = 0;
                break;
            }
            if (iter >= g.maxit || ++guard > 1000) {
                status = 1;
                break;
            }
            // continue from the true residual with the old direction
#pragma unroll
            for (int k = 0; k < NL; k++) {
                if (u[k] >= 0) r[k] -= mt;
                s_u[tid + T * k] = *at_byte(g.px, 8 * (wg * NL * T + tid + T * k));
            }
            load_dinv();
            sums();
            if (!grid_sum(v)) return give_up();
            rr = v[0];
        }
        // ---- p = (D^-1 r - mu) + beta p ------------------------------------------
        mu = g.null_space ? v[2] / g.n : 0.0;
        const double rho_new = v[1] - mu * v[3];
        const double beta = rho_new / rho_prev;
        rho = rho_new;
#pragma unroll
        for (int k = 0; k < NL; k++)
            s_u[tid + T * k] = (d[k] * r[k] - (u[k] >= 0 ? mu : 0.0)) + beta * s_u[tid + T * k];
        __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < NL; k++)
        if (own & (1u << k)) *at_byte(g.x, u[k]) = XREG ? xr[XREG ? k : 0] : s_x[tid + T * k];
    if (wg == 0 && tid == 0) {
        g.st->bb = bb;
        g.st->rr = rr;
        g.st->tt = tt;
        g.st->iter = iter;
        g.st->status = status;
    }
}

// ---------------------------------------------------------------------------
// host
// ---------------------------------------------------------------------------
struct GridShape {
    int tx = 0, ty = 0, T = 0, G = 0;
    size_t lds = 0;
};

constexpr size_t kLdsMax = 156 * 1024;  // of the CU's 160 KB; the static arrays take the rest

size_t grid_lds(int N, int tx, int ty, int T, int G) {
    const int N1 = N + 1, NP = N1 * N1;
    size_t d = (size_t)N * T + (size_t)tx * ty * NP + 1 + kEdge + (G == 1 ? kEdge : 0);
    d += (size_t)(tx + ty) * (4 * N1 + NP);  // the FP32 tables: 2 NP floats each
    if (T != 256) d += (size_t)N * T;        // x
    return 8 * d;
}

// The tile: the cheapest of those whose line threads fill one pass, whose
// nodes fit the registers and LDS, and whose workgroups fit the chip.  An
// iteration costs two grid-wide sums (0.2 us in one workgroup, else 1.2 us and
// 0.26 per doubling of the workgroups) and the operator on the tile, by line
// length and waves per SIMD; the weights are fits to measured iterations, and
// the tiles they pick are within 2% of the best of those tried (at 32 x 32,
// p = 6: 2 x 16 elements 6.69 ms, 4 x 8 6.64, 4 x 4 6.89, 2 x 4 7.35, 8 x 8 8.76;
// at 8 x 8, p = 4: one workgroup 0.54 ms, two 0.59, four 0.60).  Elsewhere they
// are untried; what they pick beats the launches everywhere measured (ms, a
// solve): 60 x 60 p 8 46.6 -> 22.4, 100 x 100 p 2 / 3 / 4 / 5 / 7 8.3 -> 4.4 /
// 18.3 -> 10.5 / 28.8 -> 13.9 / 43.3 -> 21.2 / 72.1 -> 53.1, 150 x 2 p 6 45.6 -> 18.8,
// 30 x 30 p 4 with 4 iterations 0.28 -> 0.07.  The most a tile takes is 64 elements
// at p = 8, 72 at p = 7, 82 at p = 6: above 128 x 128 elements of p = 8 on 256 CUs
// no tiling fits and the solve is launches again (45 us an iteration at
// 128 x 132).
bool grid_shape(const se_mesh* m, int cu, GridShape& best) {
    const int N = m->N, N1 = N + 1;
    double cost = HUGE_VAL;
    auto consider = [&](int tx, int ty, int T) {
        const long tX = (m->nEls[0] + tx - 1) / tx, tY = (m->nEls[1] + ty - 1) / ty, G = tX * tY;
        if (tx * ty * N1 > T || G > std::min(cu, kSlots)) return;
        const long W = tx * N + 1, H = ty * N + 1;
        if ((W | 1) * H > (long)grid_cells(N) * T || 2 * (W + H) > std::min(T, kEdge)) return;
        const size_t lds = grid_lds(N, tx, ty, T, (int)G);
        if (lds > kLdsMax) return;
        const int waves = (tx * ty * N1 + 63) / 64, w = (waves + 3) / 4;
        const double sum = G == 1 ? 0.2 : 1.2 + 0.26 * std::log2((double)G);
        const double c = 2.0 * sum + N1 * N1 * (0.02 + 0.03 * w) + (T == 256 ? 0.0 : 0.3);
        if (c < cost) {
            cost = c;
            best.tx = tx, best.ty = ty, best.T = T, best.G = (int)G, best.lds = lds;
        }
    };
    for (int T : {256, 576})
        for (int tx = 1; tx <= m->nEls[0] && tx * N1 <= T; tx++)
            for (int ty = 1; ty <= m->nEls[1] && tx * ty * N1 <= T; ty++) consider(tx, ty, T);
    return cost < HUGE_VAL;
}

constexpr int kDevices = 64;

// The kernel may have kLdsMax of LDS and then fits a CU: set and asked once per
// kernel and device.
template <int N, int T>
bool grid_usable(int device) {
    static std::atomic<signed char> known[kDevices];  // 1: usable, -1: not
    signed char k = known[device].load();
    if (k == 0) {
        const void* f = reinterpret_cast<const void*>(k_pcg_grid<N, T>);
        int blocks = 0;
        const bool ok =
            hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsMax) == hipSuccess &&
            hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, f, T, kLdsMax) == hipSuccess && blocks >= 1;
        if (!ok) (void)hipGetLastError();
        k = ok ? 1 : -1;
        known[device].store(k);
    }
    return k > 0;
}

// SE_ERR_UNSUPPORTED: not launched
template <int N, int T>
int launch_grid(const GridArgs& a, const GridShape& sh, int device, hipStream_t s) {
    if (!grid_usable<N, T>(device)) return SE_ERR_UNSUPPORTED;
    hipLaunchKernelGGL((k_pcg_grid<N, T>), dim3(sh.G), dim3(T), sh.lds, s, a);
    return SE_OK;
}

template <int N>
int launch_grid_n(const GridArgs& a, const GridShape& sh, int device, hipStream_t s) {
    return sh.T == 256 ? launch_grid<N, 256>(a, sh, device, s) : launch_grid<N, 576>(a, sh, device, s);
}

// The CUs of a device that the solves in flight from this process may need.  A
// workgroup needs a CU at most, so the workgroups of a solve that was let in
// are all resident once other kernels have drained.  A solve waits its turn:
// going to the other solver where the device is taken would give it other
// round-off, and so a result that depends on what runs beside it.
struct GridGate {
    std::mutex mu;
    std::condition_variable cv;
    unsigned long long next = 0, serving = 0;  // tickets: solves enter in order of arrival
    int used = 0;
    void enter(int cus, int all) {
        std::unique_lock<std::mutex> lk(mu);
        const unsigned long long t = next++;
        cv.wait(lk, [&] { return t == serving && used + cus <= all; });
        serving++;
        used += cus;
        cv.notify_all();
    }
    void leave(int cus) {
        std::lock_guard<std::mutex> lk(mu);
        used -= cus;
        cv.notify_all();
    }
    // Waits that ran out in a row (another process on the device, masked CUs).
    // One may be a passing kernel's.  From the second on the next solves, 16 and
    // twice as many each time, are left to the other solver: a try costs the
    // whole wait, 0.1 s, ten times an ordinary solve.
    int strikes = 0, skip = 0;
    bool leaves_out() {
        std::lock_guard<std::mutex> lk(mu);
        return skip > 0 && skip--;
    }
    void ended(bool well) {
        std::lock_guard<std::mutex> lk(mu);
        strikes = well ? 0 : strikes + 1;
        if (strikes > 1) skip = 16 << std::min(strikes - 2, 16);
    }
};
GridGate g_gate[kDevices];
// a solve's stay, from before its launch until its kernel has ended; a lone
// workgroup waits for no other and needs none
struct GridStay {
    GridGate& gate;
    int cus;
    GridStay(GridGate& g, int n, int all) : gate(g), cus(n) {
        if (cus > 1) gate.enter(cus, all);
    }
    ~GridStay() {
        if (cus > 1) gate.leave(cus);
    }
};

}  // namespace

// The solve as one launch.  done = false: not of this form (too large for the
// chip's LDS and registers, an SVV term, a recorded history), or a wait ran
// out, now or in solves before it; f is whole then (d_x may hold part of a
// result: workgroups past the last sum have stored theirs) and the caller
// solves it launch by launch.
int pcg_grid(se_op* op, const double* d_f, double* d_x, const se_solve_opts& o, se_solve_info& info, bool& done) {
    done = false;
    se_mesh* m = op->mesh;
    se_ctx* c = m->ctx;
    if (o.history || op->svv_mN > 0 || m->n < 1 || c->device >= kDevices) return SE_OK;
    // the tile depends on the mesh and the device only: chosen once per operator
    int(&tile)[3] = op->grid_tile;
    GridShape sh;
    if (tile[2] == 0) {
        const bool fits = grid_shape(m, c->cu_count, sh);
        tile[0] = sh.tx, tile[1] = sh.ty, tile[2] = fits ? sh.T : -1;
    } else if (tile[2] > 0) {
        sh.tx = tile[0], sh.ty = tile[1], sh.T = tile[2];
        sh.G = ((m->nEls[0] + sh.tx - 1) / sh.tx) * ((m->nEls[1] + sh.ty - 1) / sh.ty);
        sh.lds = grid_lds(m->N, sh.tx, sh.ty, sh.T, sh.G);
    }
    if (tile[2] < 0) return SE_OK;
    GridGate& gate = g_gate[c->device];
    if (sh.G > 1 && gate.leaves_out()) return SE_OK;
    hipStream_t s = c->stream;
    // two regions of slots: a solve uses one and its workgroups empty theirs
    // in the other for the next solve
    constexpr size_t region = 3 * kSums * kSlots;
    // (memory too short for this form is enough for the other)
    if (op->grid_slots.alloc(2 * region * sizeof(u64)) != SE_OK ||
        op->grid_work.alloc(sizeof(double) * sh.G * ((size_t)kEdge + (size_t)grid_cells(m->N) * sh.T)) != SE_OK) {
        (void)hipGetLastError();
        return SE_OK;
    }
    if (op->grid_dirty) SE_HIP(hipMemsetAsync(op->grid_slots.ptr, 0xff, 2 * region * sizeof(u64), s));
    op->grid_dirty = true;  // until this solve has ended well
    CgState* hs = (CgState*)op->h_state;  // pinned: the kernel writes its outcome there
    *hs = CgState{};
    GridArgs a;
    a.P = op_params(op, (double)op->sign);
    a.f = d_f;
    a.dinv = op->dinv_s.as<double>();
    a.x = d_x == d_f ? op->x.as<double>() : d_x;  // f is read to the end
    if (a.x == d_f) return SE_OK;
    a.ex = op->grid_work.as<double>();
    a.px = a.ex + (size_t)sh.G * kEdge;
    a.slots = op->grid_slots.as<u64>() + (op->grid_turn ? region : 0);
    a.next = op->grid_slots.as<u64>() + (op->grid_turn ? 0 : region);
    a.st = hs;
    a.tx = sh.tx;
    a.ty = sh.ty;
    a.tilesX = (m->nEls[0] + sh.tx - 1) / sh.tx;
    a.tilesY = (m->nEls[1] + sh.ty - 1) / sh.ty;
    a.G = sh.G;
    a.n = m->n;
    a.null_space = o.null_space ? 1 : 0;
    a.maxit = std::max(o.maxit, 0);
    a.sgn = (double)op->sign;
    a.rtol = o.rtol;
    // SE_GRID_WAIT (seconds): another limit; 0: no wait at all
    const char* wait = getenv("SE_GRID_WAIT");
    a.limit = (u64)((wait ? atof(wait) : kWaitLimit) * 1e8);
    GridStay stay(gate, sh.G, c->cu_count);
    SE_HIP(hipEventRecord(c->ev0, s));
    int rc = SE_ERR_UNSUPPORTED;
    switch (m->N) {
        case 2: rc = launch_grid_n<2>(a, sh, c->device, s); break;
        case 3: rc = launch_grid_n<3>(a, sh, c->device, s); break;
        case 4: rc = launch_grid_n<4>(a, sh, c->device, s); break;
        case 5: rc = launch_grid_n<5>(a, sh, c->device, s); break;
        case 6: rc = launch_grid_n<6>(a, sh, c->device, s); break;
        case 7: rc = launch_grid_n<7>(a, sh, c->device, s); break;
        case 8: rc = launch_grid_n<8>(a, sh, c->device, s); break;
        default: break;
    }
    if (rc == SE_ERR_UNSUPPORTED) return SE_OK;
    SE_HIP(hipGetLastError());
    SE_HIP(hipEventRecord(c->ev1, s));
    SE_HIP(hipEventSynchronize(c->ev1));
    if (sh.G > 1) gate.ended(!hs->pad);
    if (hs->pad) {  // a wait ran out (the slots are cleared before the next use)
        c->grid_gave_up++;
        return SE_OK;
    }
    c->grid_solves++;
    op->grid_dirty = false;
    op->grid_turn ^= 1;
    if (a.x != d_x) {  // only now: a solve that gave up still needs f, which d_x is
        SE_HIP(hipMemcpyAsync(d_x, a.x, sizeof(double) * m->n, hipMemcpyDeviceToDevice, s));
        SE_HIP(hipEventRecord(c->ev1, s));
        SE_HIP(hipEventSynchronize(c->ev1));
    }
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, c->ev0, c->ev1);
    info.status = hs->status;
    info.iters = hs->iter;
    info.outer_iters = 1;
    info.true_rel_residual = hs->bb > 0.0 ? std::sqrt(std::max(hs->tt, 0.0) / hs->bb) : 0.0;
    info.seconds = ms * 1e-3;
    done = true;
    return SE_OK;
}

}  // namespace se
