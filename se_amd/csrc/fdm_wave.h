// fdm_wave.h -- device code of the wave form of the FDM transforms
// (wave_host.h): three kernels per application, FP64 throughout.
//   WAVE_X   rows of the residual -> x modes            (T1)
//   WAVE_Y   columns of T1: y modes, times 1/D, and back (T1, in place);
//            partials of r.z, a sum over modes
//   WAVE_XB  rows of T1 -> z (or p); with a null space, partials of sum z, sum r
//
// A workgroup takes R whole lines (8, or 4 of more than 64 elements) into LDS
// as U[slot][part][line] and transforms them there, so a line is read and
// written once per kernel and the two y transforms need no memory between
// them.  A forward transform is: fold the element's nodes into parts, then
// per kind of part (vertex, symmetric, antisymmetric) the E x E wave matrix
// over the slots -- a matrix product with all parts and lines of that kind as
// columns, on the FP64 matrix cores (v_mfma_f64_16x16x4f64; eight waves share
// the 16 x 16 output tiles, K = E runs through the LDS rows, the wave matrix
// is read in operand order from the cache) -- then per phase the N x N matrix,
// one (phase, pair of lines) per thread in registers.  The backward transform
// is the same backwards.
//
// Compared with dense eigenvector matrices (k_fdm_gemm) a line of E N
// unknowns takes E + N multiply-adds per unknown instead of E N, and the four
// passes over memory become three.  LDS rows are padded to 16 mod 32 doubles:
// the four rows an operand read touches then fall in different banks.
// T1 is kept in blocks of R lines, [block][mode][line], so that WAVE_Y reads
// and writes runs of R columns x R lines.
#pragma once
#include "apply_kernels.h"

namespace se {

typedef double wave_f64x4 __attribute__((ext_vector_type(4)));
typedef double wave_d2 __attribute__((ext_vector_type(2)));

// one 16 x 16 output tile of a block of a kind's waves (wave_host.h,
// Line::Block: even or odd about the line's middle)
struct WaveTile {
    int of;               // its operands in fwd or bwd
    int col, w, row;      // first column (part * R + line) and how many; first output row of the block
    int at, step;         // slots: LDS row at + step k
    int b0, cnt;          // phases: LDS row b0 + k modulo E; the block's output rows
};
// one direction of a member
struct WaveDim {
    const double *fwd, *bwd;  // wave matrices in MFMA operand order, per block [16-row tile][k step][64]
    const double* phi;        // [(part N + mode) E16 + phase]
    int n, ne, E, E16, logR, LD;  // unknowns, elements, slots, padded; lines per workgroup; LDS row length
    int off, vs;                  // node of the first unknown; vertex of slot 0
    int mirror;                   // the line is symmetric: slot s of parts mirrors to ne - 1 - s, of vertices to ne - s
    int kf, kb;                   // k steps forward, backward (even)
    int n0, n1;                   // mirrored slots of vertices, of parts
    const WaveTile *tf, *tb;      // output tiles forward (phases), backward (slots)
    int nf, nb;
};
struct WaveTask {
    WaveDim x, y;
    int N, nS;
    double* t1;                       // [y blocks of 1 << x.logR][x modes][1 << x.logR]
    const double *r, *b;              // the residual; the right-hand side (first direction)
    double *z, *p;                    // result; the CG's direction
    const double *lx, *ly, *ex, *ey;  // by mode: D = lx + ly + ex ey
    double dtol;                      // D below this: a null mode (1/D := 0)
    double* part_rz;                  // [y blocks]: r.z, as the sum of (mode of r)^2 / D
    double* part_zr;                  // [2][x blocks]: sum z, sum r (null space only)
    int null_space;
    const double* pv;                 // r.r partials of the CG (null outside one)
    const CgState* st;
    int nch;
};
enum { WAVE_X = 0, WAVE_Y = 1, WAVE_XB = 2 };
constexpr int kWaveT = 512;
constexpr int kWavePad = 8;  // cleared LDS rows before U

// lines per workgroup and LDS row length (host and device)
__host__ __device__ inline int wave_log_r(int E) { return E <= 64 ? 3 : 2; }
__host__ __device__ inline int wave_ld(int N, int logR) {
    const int w = N << logR;
    return w + (48 - w % 32) % 32;
}
// long lines: more output tiles than four a wave, and no room in LDS for the
// phases' N x N matrices beside U; kernels of their own
__host__ __device__ inline bool wave_long(int E) { return E > 128; }
__host__ __device__ inline size_t wave_lds(int N, int E, int E16, int LD) {
    return ((size_t)(kWavePad + E16) * LD + 16 + (wave_long(E) ? 0 : N * N * E16)) * sizeof(double);
}

// The thread, hidden from the compiler: each item derives its indices anew.
// Kept over the loop of items (of every order's N x N product) they spilled 14
// registers, and on the ensemble's short lines the scratch lines written back
// were more than the data (512 members 3060 -> 3000 us, 24 channels 227 -> 223).
__device__ __forceinline__ int wave_tid() {
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    return tid;
}

// U <- F U (FWD: slots -> phases, else phases -> slots): NQ output tiles of this
// wave, all K steps.  Operands of zero stand where a block has fewer rows than
// its tiles; the LDS rows they meet hold finite values (other blocks' or
// cleared rows).
constexpr int kWaveUN = 2;  // K steps a group of operands covers
template <int NA>
struct WaveTiles {
    WaveTile t[NA];
    double a[kWaveUN][NA];  // the first group of operands
};
template <int NQ, int NA, bool FWD>
__device__ __forceinline__ void wave_product(const WaveDim& d, const double* U, const WaveTiles<NA>& w,
                                             wave_f64x4 (&acc)[NA], int l) {
    const WaveTile(&t)[NA] = w.t;
    const int KS = FWD ? d.kf : d.kb;
    const SE_GLOBAL double* A = gview(FWD ? d.fwd : d.bwd) + l;
    const double* B = U + (l & 15);
    // the wave matrix's operands are loaded UN steps ahead
    constexpr int UN = kWaveUN;
    double a[2][UN][NQ];
    auto load_a = [&](int h, int ks) {
#pragma unroll
        for (int u = 0; u < UN; u++)
#pragma unroll
            for (int q = 0; q < NQ; q++) a[h][u][q] = A[t[q].of + (ks + u) * 64];
    };
    auto multiply = [&](int h, int ks) {
        double b[UN][NQ];
#pragma unroll
        for (int u = 0; u < UN; u++) {
            const int k = (ks + u) * 4 + (l >> 4);
#pragma unroll
            for (int q = 0; q < NQ; q++) {
                int r = FWD ? t[q].at + t[q].step * k : t[q].b0 + k;
                if (!FWD) r = r >= d.E ? r - d.E : r;
                b[u][q] = B[r * d.LD + t[q].col];
            }
        }
#pragma unroll
        for (int u = 0; u < UN; u++)
#pragma unroll
            for (int q = 0; q < NQ; q++)
                acc[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[h][u][q], b[u][q], acc[q], 0, 0, 0);
    };
#pragma unroll
    for (int u = 0; u < UN; u++)
#pragma unroll
        for (int q = 0; q < NQ; q++) a[0][u][q] = w.a[u][q];
    for (int ks = 0; ks < KS; ks += 2 * UN) {  // (KS is a multiple of UN)
        if (ks + UN < KS) load_a(1, ks + UN);
        multiply(0, ks);
        if (ks + UN >= KS) break;
        if (ks + 2 * UN < KS) load_a(0, ks + 2 * UN);
        multiply(1, ks + UN);
    }
}

// This wave's tiles of a product and the first of their operands, loaded well
// before the product (behind the lines' loads, the N x N matrices).
template <bool FWD, int NA>
__device__ __forceinline__ void wave_ahead(const WaveDim& d, WaveTiles<NA>& w) {
    const int l = wave_tid() & 63, wv = __builtin_amdgcn_readfirstlane(wave_tid() >> 6);
    const int nt = FWD ? d.nf : d.nb;
    typedef const __attribute__((address_space(4))) WaveTile ctile;  // (uniform: scalar loads)
    ctile* tab = (ctile*)(FWD ? d.tf : d.tb);
    const SE_GLOBAL double* A = gview(FWD ? d.fwd : d.bwd) + l;
#pragma unroll
    for (int q = 0; q < NA; q++) {
        ctile& c = tab[min(wv + 8 * q, nt - 1)];
        w.t[q] = WaveTile{c.of, c.col, c.w, c.row, c.at, c.step, c.b0, c.cnt};
#pragma unroll
        for (int u = 0; u < kWaveUN; u++) w.a[u][q] = A[w.t[q].of + u * 64];
    }
}

// the eight waves share the tiles; every wave is past its reads of U before
// the results go over it
template <bool FWD, int NA>
__device__ __forceinline__ void wave_matrix(double* U, const WaveDim& d, const WaveTiles<NA>& w) {
    constexpr bool LONG = NA > 4;
    const int l = wave_tid() & 63, wv = __builtin_amdgcn_readfirstlane(wave_tid() >> 6);
    const int nt = FWD ? d.nf : d.nb;
    const WaveTile(&t)[NA] = w.t;
    wave_f64x4 acc[NA];
#pragma unroll
    for (int q = 0; q < NA; q++) acc[q] = wave_f64x4{0.0, 0.0, 0.0, 0.0};
    const int mine = (nt - wv + 7) >> 3;
    // (a wave forms its own tiles only; 5 and 6 of the long lines' 7: at 256
    // elements of order 2 a product of 7 for 4 cost a fifth of a solve)
    switch (mine) {
        case 0: break;
        case 1: wave_product<1, NA, FWD>(d, U, w, acc, l); break;
        case 2: wave_product<2, NA, FWD>(d, U, w, acc, l); break;
        case 3: wave_product<3, NA, FWD>(d, U, w, acc, l); break;
        default:
            if constexpr (LONG) {
                if (mine == 4) wave_product<4, NA, FWD>(d, U, w, acc, l);
                else if (mine == 5) wave_product<5, NA, FWD>(d, U, w, acc, l);
                else if (mine == 6) wave_product<6, NA, FWD>(d, U, w, acc, l);
                else wave_product<NA, NA, FWD>(d, U, w, acc, l);
            } else {
                wave_product<NA, NA, FWD>(d, U, w, acc, l);
            }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NA; q++)
        if (q < mine && (l & 15) < t[q].w) {
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int i = t[q].row + (l >> 4) + 4 * v;
                int r = FWD ? t[q].b0 + i : t[q].at + t[q].step * i;
                if (FWD) r = r >= d.E ? r - d.E : r;
                if (i < t[q].cnt) U[r * d.LD + t[q].col + (l & 15)] = acc[q][v];
            }
        }
    __syncthreads();
}

// U's rows outside the phases, and the parts of a slot without an element:
// operands of zero meet them
__device__ __forceinline__ void wave_pad(const WaveDim& d, double* U, bool slots) {
    for (int k = wave_tid(); k < kWavePad * d.LD; k += kWaveT) U[k - kWavePad * d.LD] = 0.0;
    for (int k = d.E * d.LD + wave_tid(); k < d.E16 * d.LD; k += kWaveT) U[k] = 0.0;
    if (slots && d.ne < d.E)
        for (int k = (1 << d.logR) + wave_tid(); k < d.LD; k += kWaveT) U[(d.E - 1) * d.LD + k] = 0.0;
}

constexpr double kR2 = 0.70710678118654752440;

// Lines -> U with the folds: per element the vertex, the node pairs (i, N - i)
// as their symmetric and antisymmetric parts, the middle node; then the sums
// and differences of mirrored slots.  at(I): the address of unknown I of this
// thread's line; ok: the line exists.  Loads run B items a thread at once.
template <int B, typename AT>
__device__ __forceinline__ void wave_load(const WaveTask& t, const WaveDim& d, double* U, bool ok, AT&& at) {
    const int N = t.N, P1 = 1 + t.nS, mul = 65536 / P1 + 1;  // (exact below 2^16 / P1)
    const int cnt = (d.n0 * P1) << d.logR, r = wave_tid() & ((1 << d.logR) - 1);
    for (int k0 = wave_tid(); k0 < cnt; k0 += B * kWaveT) {
        double v[B][4];
        int s_[B], i_[B], m_[B];
#pragma unroll
        for (int j = 0; j < B; j++) {
            const int k = k0 + j * kWaveT, idx = k >> d.logR, s = (idx * mul) >> 16, i = idx - s * P1;
            const bool mid = 2 * i == N;
            int m = d.mirror ? d.ne - (i == 0 ? 0 : 1) - s : s;
            if (m >= d.E) m = 0;  // (the first vertex of a periodic line)
            const bool in = ok && k < cnt && (i == 0 || (s < d.n1 && s < d.ne));
            const int I = (i == 0 ? (s + d.vs) * N : s * N + i) - d.off, M = I + (m - s) * N;
            v[j][0] = v[j][1] = v[j][2] = v[j][3] = 0.0;
            if (in && I >= 0 && I < d.n) v[j][0] = *at(I);
            if (in && m != s && M >= 0 && M < d.n) v[j][2] = *at(M);
            if (in && i > 0 && !mid) {
                v[j][1] = *at(I + N - 2 * i);
                if (m != s) v[j][3] = *at(M + N - 2 * i);
            }
            s_[j] = k < cnt && (i == 0 || (s < d.n1 && s < d.ne)) ? s : -1;
            i_[j] = i;
            m_[j] = m;
        }
#pragma unroll
        for (int j = 0; j < B; j++) {
            if (s_[j] < 0) continue;
            const int i = i_[j], s = s_[j], m = m_[j], A = t.nS << d.logR;
            const bool pair = i > 0 && 2 * i != N;
            double* u = U + s * d.LD + (i << d.logR) + r;
            double* w = U + m * d.LD + (i << d.logR) + r;
            const double S0 = pair ? kR2 * (v[j][0] + v[j][1]) : v[j][0], A0 = kR2 * (v[j][0] - v[j][1]);
            const double S1 = pair ? kR2 * (v[j][2] + v[j][3]) : v[j][2], A1 = kR2 * (v[j][2] - v[j][3]);
            *u = S0 + S1;  // (S1 = A1 = 0 where the slot is its own mirror)
            if (pair) u[A] = A0 + A1;
            if (m != s) {
                *w = S0 - S1;
                if (pair) w[A] = A0 - A1;
            }
        }
    }
}
// U -> lines: out(I, value) of the unknowns of every pair of mirrored slots'
// pair of nodes.  TO_U: the node values go back to U instead (node i of slot s
// at part i, N - i at the antisymmetric part's place).
template <bool TO_U, typename OUT>
__device__ __forceinline__ void wave_unfold(const WaveTask& t, const WaveDim& d, double* U, bool ok, OUT&& out) {
    const int N = t.N, P1 = 1 + t.nS, mul = 65536 / P1 + 1;
    const int cnt = (d.n0 * P1) << d.logR, r = wave_tid() & ((1 << d.logR) - 1);
    if (!ok && !TO_U) return;
#pragma unroll 2
    for (int k = wave_tid(); k < cnt; k += kWaveT) {
        const int idx = k >> d.logR, s = (idx * mul) >> 16, i = idx - s * P1, A = t.nS << d.logR;
        const bool pair = i > 0 && 2 * i != N;
        if (i > 0 && (s >= d.n1 || s >= d.ne)) continue;
        int m = d.mirror ? d.ne - (i == 0 ? 0 : 1) - s : s;
        if (m >= d.E) m = 0;
        double* u = U + s * d.LD + (i << d.logR) + r;
        double* w = U + m * d.LD + (i << d.logR) + r;
        const double Sp = *u, Sm = m != s ? *w : 0.0, Ap = pair ? u[A] : 0.0, Am = pair && m != s ? w[A] : 0.0;
        const double S0 = Sp + Sm, S1 = Sp - Sm, A0 = Ap + Am, A1 = Ap - Am;
        const double x0 = pair ? kR2 * (S0 + A0) : S0, y0 = kR2 * (S0 - A0);
        const double x1 = pair ? kR2 * (S1 + A1) : S1, y1 = kR2 * (S1 - A1);
        if (TO_U) {
            *u = x0;
            if (pair) u[A] = y0;
            if (m != s) {
                *w = x1;
                if (pair) w[A] = y1;
            }
        } else {
            const int I = (i == 0 ? (s + d.vs) * N : s * N + i) - d.off, M = I + (m - s) * N;
            if (I >= 0 && I < d.n) out(I, x0);
            if (m != s && M >= 0 && M < d.n) out(M, x1);
            if (pair) {
                out(I + N - 2 * i, y0);
                if (m != s) out(M + N - 2 * i, y1);
            }
        }
    }
}

// the N x N matrices in place: parts -> modes (WAVE_X), modes -> parts
// (WAVE_XB), or parts -> modes, times 1/D, -> parts (WAVE_Y); one (phase, pair
// of lines) per thread.
template <int N, int MODE, bool LONG>
__device__ __forceinline__ double wave_modes(const WaveTask& t, const WaveDim& d, double* U, const double* Phi,
                                             int item) {
    double rz = 0.0;  // WAVE_Y: this thread's part of r.z
    const int R = 1 << d.logR, h = d.logR - 1;
    for (int k = wave_tid(); k < d.E << h; k += kWaveT) {
        const int r = 2 * (k & ((1 << h) - 1)), c = k >> h;
        double2* u = reinterpret_cast<double2*>(U + c * d.LD + r);
        auto f = [&](int p, int j) -> double {
            return !LONG ? Phi[(p * N + j) * d.E16 + c] : gview(d.phi)[(p * N + j) * d.E16 + c];
        };
        double2 m[N];
        if (MODE != WAVE_XB) {
#pragma unroll
            for (int j = 0; j < N; j++) m[j] = make_double2(0.0, 0.0);
#pragma unroll 2
            for (int p = 0; p < N; p++) {
                const double2 v = u[p * (R >> 1)];
#pragma unroll
                for (int j = 0; j < N; j++) {
                    const double w = f(p, j);
                    m[j].x += w * v.x;
                    m[j].y += w * v.y;
                }
            }
        } else {
#pragma unroll
            for (int j = 0; j < N; j++) m[j] = u[j * (R >> 1)];
        }
        if (MODE == WAVE_X) {
#pragma unroll
            for (int j = 0; j < N; j++) u[j * (R >> 1)] = m[j];
            continue;
        }
        if (MODE == WAVE_Y) {
            const int x = item * R + r;
            const double lx0 = gview(t.lx)[x], lx1 = gview(t.lx)[x + 1];
            const double ex0 = gview(t.ex)[x], ex1 = gview(t.ex)[x + 1];
#pragma unroll
            for (int j = 0; j < N; j++) {
                const double ly = gview(t.ly)[c * N + j], ey = gview(t.ey)[c * N + j];
                const double D0 = lx0 + ly + ex0 * ey, D1 = lx1 + ly + ex1 * ey;
                const double c0 = m[j].x, c1 = m[j].y;
                m[j].x = D0 > t.dtol ? c0 / D0 : 0.0;
                m[j].y = D1 > t.dtol ? c1 / D1 : 0.0;
                rz += c0 * m[j].x + c1 * m[j].y;
            }
        }
#pragma unroll 2
        for (int p = 0; p < N; p++) {
            double2 v = make_double2(0.0, 0.0);
#pragma unroll
            for (int j = 0; j < N; j++) {
                const double w = f(p, j);
                v.x += w * m[j].x;
                v.y += w * m[j].y;
            }
            u[p * (R >> 1)] = v;
        }
    }
    return rz;
}
template <int MODE, bool LONG>
__device__ __forceinline__ double wave_modes_n(const WaveTask& t, const WaveDim& d, double* U, const double* Phi,
                                             int item) {
#define SE_WAVE_MODES(NN) return wave_modes<NN, MODE, LONG>(t, d, U, Phi, item)
    switch (t.N) {
        case 2: SE_WAVE_MODES(2);
        case 3: SE_WAVE_MODES(3);
        case 4: SE_WAVE_MODES(4);
        case 5: SE_WAVE_MODES(5);
        case 6: SE_WAVE_MODES(6);
        case 7: SE_WAVE_MODES(7);
        default: SE_WAVE_MODES(8);
    }
#undef SE_WAVE_MODES
}

// Inside a CG iteration: as fdm_skip (fdm.hip), whose 256-thread sum it
// repeats to the bit (the direction kernel decides from that).
__device__ __forceinline__ bool wave_skip(const WaveTask& t) {
    __shared__ double s_part[4];
    if (!t.pv) return false;
    if (cg_stopped(t.st)) return true;
    double s = 0.0;
    if (threadIdx.x < 256) {
        for (int b = threadIdx.x; b < t.nch; b += 256) s += t.pv[b];
        s = wave_sum(s);
        if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = s;
    }
    __syncthreads();
    double rr = 0.0;
#pragma unroll
    for (int w = 0; w < 4; w++) rr += s_part[w];
    __syncthreads();
    return !(rr - rr == 0.0) || rr <= t.st->tol2;
}

// block `item` of T1 (contiguous: modes x R lines) from or to U
template <bool OUT>
__device__ __forceinline__ void wave_block(const WaveTask& t, const WaveDim& d, double* U, int item) {
    const int w = (t.N << d.logR) >> 1, cnt = d.E * w;  // 16-byte units of a phase, of the block
    const unsigned mul = (1u << 24) / w + 1;            // (exact: below 2^13 units, w at most 32)
    SE_GLOBAL wave_d2* T = (SE_GLOBAL wave_d2*)gview(t.t1) + (size_t)item * cnt;
#pragma unroll 4
    for (int k = wave_tid(); k < cnt; k += kWaveT) {
        const int c = (int)(((unsigned long long)k * mul) >> 24), j = k - c * w;
        wave_d2* u = (wave_d2*)(U + c * d.LD) + j;
        if (OUT) T[k] = *u;
        else *u = T[k];
    }
}

// one kernel's items (member, block of lines); item.x < 0: padding
template <int MODE, bool LONG>
__global__ __launch_bounds__(kWaveT, LONG ? 2 : 4) void k_fdm_wave(const WaveTask* __restrict__ tasks,
                                                        const int2* __restrict__ work, int nwork, int skip, int to_p) {
    extern __shared__ __attribute__((aligned(16))) double wave_u[];
    for (int w = blockIdx.x; w < nwork; w += gridDim.x) {
        const int2 it = work ? work[w] : make_int2(0, w);
        if (it.x < 0) continue;
        const WaveTask& t = tasks[it.x];
        if (skip && wave_skip(t)) continue;
        const WaveDim& d = MODE == WAVE_Y ? t.y : t.x;
        const int R = 1 << d.logR, lgx = t.x.logR, Rx = 1 << lgx, nMx = t.x.E * t.N;
        const int line = (it.y << d.logR) + (wave_tid() & (R - 1));  // this thread's line
        const bool ok = line < (MODE == WAVE_Y ? nMx : t.y.n);
        // unknown J of column `line` in T1
        auto in_t1 = [&](int J) { return (((size_t)(J >> lgx) * nMx + line) << lgx) + (J & (Rx - 1)); };
        double* U = wave_u + kWavePad * d.LD;
        double* Phi = U + d.E16 * d.LD + 16;
        WaveTiles<LONG ? 7 : 4> tiles;
        if (MODE == WAVE_XB) wave_ahead<false>(d, tiles);
        else wave_ahead<true>(d, tiles);
        __syncthreads();  // the previous item is done with U
        if (MODE == WAVE_X) {
            const SE_GLOBAL double* src = gview(to_p == 2 ? t.b : t.r) + (size_t)line * d.n;
            wave_load<3>(t, d, U, ok, [&](int I) { return src + I; });
        } else if (MODE == WAVE_Y) {
            const SE_GLOBAL double* T = gview(t.t1);
            wave_load<3>(t, d, U, ok, [&](int J) { return T + in_t1(J); });
        } else {
            wave_block<false>(t, d, U, it.y);
        }
        wave_pad(d, U, MODE != WAVE_XB);
        if (!LONG) {
            const SE_GLOBAL wave_d2* f = (const SE_GLOBAL wave_d2*)gview(d.phi);
#pragma unroll 4
            for (int k = wave_tid(); k < (t.N * t.N * d.E16) >> 1; k += kWaveT) ((wave_d2*)Phi)[k] = f[k];
        }
        __syncthreads();
        if (MODE != WAVE_XB) wave_matrix<true>(U, d, tiles);
        if (MODE == WAVE_Y) wave_ahead<false>(d, tiles);
        const double rz = wave_modes_n<MODE, LONG>(t, d, U, Phi, it.y);
        if (MODE == WAVE_Y) {
            const double v[1] = {rz};
            block_store_partials_at<1, kWaveT>(v, t.part_rz, it.y, (nMx + R - 1) >> d.logR);
        }
        __syncthreads();
        if (MODE == WAVE_X) {
            wave_block<true>(t, d, U, it.y);
            continue;
        }
        wave_matrix<false>(U, d, tiles);
        if (MODE == WAVE_Y) {
            SE_GLOBAL double* T = gview(t.t1);
            wave_unfold<false>(t, d, U, ok, [&](int J, double v) { T[in_t1(J)] = v; });
        } else {
            // whole runs of a line: the node values are unfolded in LDS first
            wave_unfold<true>(t, d, U, ok, [](int, double) {});
            __syncthreads();
            SE_GLOBAL double* Z = gview(to_p != 0 ? t.p : t.z) + (size_t)line * d.n;
            const int N = t.N, mul = 65536 / N + 1, r = wave_tid() & (R - 1);  // (nodes below 2^16 / N)
            auto node = [&](int I) {
                const int a = I + d.off, e = (a * mul) >> 16, i = a - e * N;
                const int p = i <= t.nS ? i : t.nS + N - i, s = i == 0 ? e - d.vs : e;
                return U[s * d.LD + (p << d.logR) + r];
            };
            if (!t.null_space) {
                if (ok) {
#pragma unroll 8
                    for (int I = wave_tid() >> d.logR; I < d.n; I += kWaveT >> d.logR) Z[I] = node(I);
                }
                continue;
            }
            const SE_GLOBAL double* Rs = gview(to_p == 2 ? t.b : t.r) + (size_t)line * d.n;
            double sz = 0.0, sr = 0.0;
#pragma unroll 4
            for (int I = wave_tid() >> d.logR; I < d.n; I += kWaveT >> d.logR)
                if (ok) {
                    const double v = node(I);
                    Z[I] = v;
                    sz += v;
                    sr += Rs[I];
                }
            const double pv[2] = {sz, sr};
            block_store_partials_at<2, kWaveT>(pv, t.part_zr, it.y, (t.y.n + R - 1) >> d.logR);
        }
    }
}

}  // namespace se
