// wave_host.h -- host side of the wave form of the fast diagonalisation: the
// eigenvectors of a line of equal elements as plane waves over the elements
// times small matrices, instead of one dense matrix.
//
// The 1-D operators of the separable form (fdm_host.h) repeat element by
// element on the reference's uniform meshes (Mesh::Mesh, src/base/Mesh.cpp:
// 17-84) up to a drift: the reference differentiates coordinates with a D whose
// rows sum to ~1e-13 (order 8), so an element's Jacobian differs from the mean by
// ~1e-11 in proportion to its distance from the origin.  The eigenvectors of the
// mean element are Bloch waves.  With an element's interior
// nodes i and N-i folded into a symmetric and an antisymmetric part, the
// amplitudes of a wave of phase theta per element,
//   vertices V cos(theta e),  symmetric parts S cos(theta (e + 1/2)),
//   antisymmetric parts -A sin(theta (e + 1/2))         (or sin, sin, cos),
// satisfy a real symmetric N x N eigenproblem in (V, S.., A..) per theta.  The
// phases that meet the line's ends are 2 pi k / ne (periodic), pi k / ne (two
// walls, or two natural ends) and pi (k + 1/2) / ne (one of each), so
//   V = (F_V + F_S + F_A, per part) * (N x N matrix per phase)
// and a transform of a line of ne N unknowns costs n (ne + N) multiply-adds
// instead of n^2: an N-fold less for long lines.  As an inverse of the operator
// they lack the drift, which dense eigenvectors have: ||A z - r|| / ||r|| of one
// application is 1.5 times the dense one's for white r (128 x 128 elements of
// order 8: 8.5e-11 against 5.7e-11) and some ten times for smooth r between
// walls (order 8: 4e-11 against 3e-12; little at orders up to 5).  What is left is
// high modes': the solutions are no further from the exact ones for it (128 x 128
// elements of order 8 1.9e-13 either way, the 512-member ensemble 1.1e-12 against
// 1.6e-12).
//
// Pure host C++ (no HIP types).
#pragma once

#include <cmath>
#include <cstddef>
#include <vector>

namespace se_wave {

constexpr int kMaxE = 256;  // element slots the device kernels take

struct Line {
    int ne = 0, N = 0, n = 0;      // elements, order, unknowns
    int E = 0, E16 = 0;            // element slots = phases, and padded to 16
    int nS = 0, nA = 0;            // symmetric / antisymmetric parts (1 + nS + nA = N)
    std::vector<double> F[3];      // [E16][E16] wave of phase c at slot s: F[s * E16 + c], of V, S, A
    // The waves of a line whose ends are alike are even or odd about its
    // middle.  Phases are numbered so that per kind of part the even ones and
    // the odd ones are runs (modulo E); slot s mirrors to mirror[kind] - s
    // (modulo E for the vertices of a periodic line).  Block 2 kind + odd takes
    // the sums (differences) of mirrored slots: slots 0 .. nk - 1, at LDS row k
    // (even) or top - k (odd), and the phases b0 .. b0 + np - 1 (modulo E).
    struct Block {
        int nk = 0, np = 0, b0 = 0, top = 0, s0 = 0;  // s0: first slot
    } blk[6];
    int mirror[3] = {-1, -1, -1};  // -1: no such symmetry (all in the even blocks)
    std::vector<double> phi;       // [(t N + j) E16 + c]: part t of mode j of phase c
    std::vector<double> lambda;    // [c N + j]
    int off = 0, vs = 0;           // node of the first unknown; vertex of slot 0
    std::vector<char> have;        // [c N + j]: a mode (else phi = 0 there)
};

// eigenvalues w and unit eigenvectors (columns of v) of the symmetric n x n
// matrix a by cyclic Jacobi rotations (Golub & Van Loan, Matrix Computations,
// section 8.5); a is destroyed
inline void jacobi_eig(int n, double (*a)[8], double* w, double (*v)[8]) {
    for (int i = 0; i < n; i++)
        for (int j = 0; j < n; j++) v[i][j] = i == j ? 1.0 : 0.0;
    for (int sweep = 0; sweep < 60; sweep++) {
        double off = 0.0, dia = 0.0;
        for (int i = 0; i < n; i++) {
            dia += a[i][i] * a[i][i];
            for (int j = i + 1; j < n; j++) off += a[i][j] * a[i][j];
        }
        if (off <= 1e-40 * dia) break;
        for (int p = 0; p < n; p++)
            for (int q = p + 1; q < n; q++) {
                if (a[p][q] == 0.0) continue;
                const double th = (a[q][q] - a[p][p]) / (2.0 * a[p][q]);
                const double t = (th >= 0.0 ? 1.0 : -1.0) / (std::fabs(th) + std::sqrt(th * th + 1.0));
                const double c = 1.0 / std::sqrt(t * t + 1.0), s = t * c;
                for (int k = 0; k < n; k++) {
                    const double x = a[k][p], y = a[k][q];
                    a[k][p] = c * x - s * y;
                    a[k][q] = s * x + c * y;
                }
                for (int k = 0; k < n; k++) {
                    const double x = a[p][k], y = a[q][k];
                    a[p][k] = c * x - s * y;
                    a[q][k] = s * x + c * y;
                    const double vx = v[k][p], vy = v[k][q];
                    v[k][p] = c * vx - s * vy;
                    v[k][q] = s * vx + c * vy;
                }
            }
    }
    for (int i = 0; i < n; i++) w[i] = a[i][i];
}

// cos / sin of pi num / den, the angle reduced exactly
inline double cos_pi(long num, long den) {
    num %= 2 * den;
    return (double)std::cos((long double)M_PIl * (long double)num / (long double)den);
}
inline double sin_pi(long num, long den) {
    num %= 2 * den;
    return (double)std::sin((long double)M_PIl * (long double)num / (long double)den);
}

// K: the element stiffness [N+1][N+1], s: the element's share of the diagonal
// S at its nodes (positive).  wall_lo, wall_hi: no unknown at that end (not
// periodic).  False if the line is longer than the kernels take.
inline bool wave_line(int ne, int N, bool per, bool wall_lo, bool wall_hi, const std::vector<double>& K,
                      const std::vector<double>& s, Line& L) {
    const bool natural = !per && !wall_lo && !wall_hi;
    L.ne = ne;
    L.N = N;
    L.E = natural ? ne + 1 : ne;
    if (L.E > kMaxE) return false;
    L.E16 = (L.E + 15) / 16 * 16;
    L.nS = N / 2;
    L.nA = N - 1 - L.nS;
    const int n1 = N + 1, E = L.E, P = L.E16, vs = !per && wall_lo && !wall_hi ? 1 : 0;
    // unknowns: nodes off .. of the line; vertex e at slot e - vs, the nodes
    // i, N - i of an element at its parts S_i, A_i
    const int off = wall_lo ? 1 : 0, last = ne * N - (per || wall_hi ? 1 : 0);
    L.n = last - off + 1;
    L.off = off;
    L.vs = vs;
    for (auto& f : L.F) f.assign((size_t)P * P, 0.0);
    L.phi.assign((size_t)N * N * P, 0.0);
    L.lambda.assign((size_t)E * N, 1.0);
    L.have.assign((size_t)E * N, 0);
    // element blocks in the folded basis; symmetrised against round-off
    auto sym = [&](int a, int b) {
        return 0.25 * (K[a * n1 + b] + K[b * n1 + a] + K[(N - a) * n1 + (N - b)] + K[(N - b) * n1 + (N - a)]);
    };
    auto wgt = [&](int i) { return 0.5 * (s[i] + s[N - i]); };
    const double r2 = std::sqrt(0.5);
    // part t (1 ..) of an element: coefficient of node i
    auto part = [&](int t, int i) {
        if (t <= L.nS) {
            if (2 * t == N) return i == t ? 1.0 : 0.0;
            return i == t || i == N - t ? r2 : 0.0;
        }
        const int j = t - L.nS;
        return i == j ? r2 : (i == N - j ? -r2 : 0.0);
    };
    std::vector<double> w(N);
    for (int t = 0; t < N; t++) w[t] = t == 0 ? 2.0 * wgt(0) : wgt(t <= L.nS ? t : t - L.nS);
    // the phases in their order, and the blocks
    std::vector<int> ord;
    if (per) {  // 0, cosines, [the phase pi,] sines
        const int h = (ne - 1) / 2, ny = ne % 2 == 0 ? 1 : 0;
        for (int c = 0; c < E; c += c == 0 ? 1 : 2) ord.push_back(c);
        for (int c = 2; c <= 2 * h; c += 2) ord.push_back(c);
        L.mirror[0] = ne;
        L.mirror[1] = L.mirror[2] = ne - 1;
        const int nev[3] = {1 + h + ny, 1 + h, 1 + h}, b0[3] = {0, 0, (1 + h + ny) % E};
        for (int k = 0; k < 3; k++) {
            const int ns = k == 0 ? ne / 2 + 1 : (ne + 1) / 2;
            L.blk[2 * k] = {ns, nev[k], b0[k], 0, 0};
            L.blk[2 * k + 1] = {ne - ns, E - nev[k], (b0[k] + nev[k]) % E, E - 1, k == 0 ? 1 : 0};
        }
    } else if (wall_lo && wall_hi) {  // odd k, 0, even k
        for (int c = 1; c < E; c += 2) ord.push_back(c);
        ord.push_back(0);
        for (int c = 2; c < E; c += 2) ord.push_back(c);
        const int o = E / 2, z = ne % 2;  // the symmetric parts' phase pi (number 0) is even for odd ne
        L.mirror[0] = ne;
        L.mirror[1] = L.mirror[2] = ne - 1;
        // (slot 0 holds no vertex: it mirrors to itself)
        L.blk[0] = {ne / 2 + 1, o, 0, 0, 0};
        L.blk[1] = {ne - ne / 2 - 1, E - o - 1, (o + 1) % E, E - 1, 1};
        L.blk[2] = {(ne + 1) / 2, o + z, 0, 0, 0};
        L.blk[3] = {ne / 2, E - o - z, (o + z) % E, E - 1, 0};
        L.blk[4] = {(ne + 1) / 2, E - o, o % E, 0, 0};
        L.blk[5] = {ne / 2, o, 0, E - 1, 0};
    } else if (natural) {  // even k, odd k
        for (int c = 0; c < E; c += 2) ord.push_back(c);
        for (int c = 1; c < E; c += 2) ord.push_back(c);
        const int ev = (E + 1) / 2;
        L.mirror[0] = ne;
        L.mirror[1] = L.mirror[2] = ne - 1;
        for (int k = 0; k < 3; k++) {
            const int m = k == 0 ? E : ne;  // slots
            L.blk[2 * k] = {(m + 1) / 2, k == 2 ? E - ev : ev, k == 2 ? ev % E : 0, 0, 0};
            L.blk[2 * k + 1] = {m / 2, k == 2 ? ev : E - ev, k == 2 ? 0 : ev % E, m - 1, 0};
        }
    } else {
        for (int c = 0; c < E; c++) ord.push_back(c);
        for (int k = 0; k < 3; k++) L.blk[2 * k] = {E, E, 0, 0, 0};
    }
    for (int at = 0; at < E; at++) {
        const int c = ord[at];
        // theta = pi num / den; cosine or sine family; which parts the waves have
        long num, den = ne;
        bool cosine, hV = true, hS = true, hA = true;
        double nrm = std::sqrt(2.0 / ne);
        bool mixed0 = false;  // a single phase that takes V, S of the cosines and A of the sines
        bool nyquist = false;
        if (per) {
            num = 2 * ((c + 1) / 2);
            cosine = c % 2 == 1;
            if (c == 0) {
                nrm = std::sqrt(1.0 / ne);
                mixed0 = true;
                cosine = true;
            } else if (num == ne) {
                nrm = std::sqrt(1.0 / ne);
                nyquist = true;
                cosine = true;
            }
        } else if (wall_lo && wall_hi) {
            num = c;
            cosine = false;
            if (c == 0) {  // the two phases 0 (A only) and pi (S only) share the slot
                hV = false;
                nrm = std::sqrt(1.0 / ne);
            }
        } else if (natural) {
            num = c;
            cosine = true;
            if (c == 0) hA = false, nrm = std::sqrt(1.0 / ne);
            if (c == ne) hS = false, nrm = std::sqrt(1.0 / ne);
        } else {
            num = 2 * c + 1;
            den = 2 * ne;
            cosine = wall_hi;
        }
        for (int e = 0; e < E; e++) {
            double fV, fS, fA;
            const long v = num * (e + vs), h = num * (2L * e + 1);  // theta e, theta (e + 1/2) over pi / den, pi / (2 den)
            if (mixed0) {
                fV = fS = fA = 1.0;
            } else if (nyquist) {
                fV = cos_pi(v, den);
                fS = sin_pi(h, 2 * den);
                fA = -sin_pi(h, 2 * den);
            } else if (!hV) {
                fV = 0.0;
                fS = (e % 2) ? -1.0 : 1.0;
                fA = 1.0;
            } else if (cosine) {
                fV = cos_pi(v, den);
                fS = cos_pi(h, 2 * den);
                fA = -sin_pi(h, 2 * den);
            } else {
                fV = sin_pi(v, den);
                fS = sin_pi(h, 2 * den);
                fA = cos_pi(h, 2 * den);
            }
            const bool el = e < ne;  // (natural ends: slot ne holds the last vertex only)
            const bool vx = !(wall_lo && wall_hi && e == 0);
            L.F[0][(size_t)e * P + at] = hV && vx ? nrm * fV : 0.0;
            L.F[1][(size_t)e * P + at] = hS && el ? nrm * fS : 0.0;
            L.F[2][(size_t)e * P + at] = hA && el ? nrm * fA : 0.0;
        }
        // the N x N eigenproblem of the parts this phase has
        int idx[8], m = 0;
        for (int t = 0; t < N; t++)
            if (t == 0 ? hV : (t <= L.nS ? hS : hA)) idx[m++] = t;
        const double ch = hV ? 2.0 * cos_pi(num, 2 * den) : 0.0, sh = hV ? -2.0 * sin_pi(num, 2 * den) : 0.0;
        double a[8][8], lam[8], v[8][8];
        for (int p = 0; p < m; p++)
            for (int q = 0; q < m; q++) {
                const int t = idx[p], u = idx[q];
                double h = 0.0;
                if (t == 0 && u == 0) {
                    h = 2.0 * sym(0, 0) + 2.0 * sym(0, N) * cos_pi(num, den);
                } else if (t == 0 || u == 0) {
                    const int o = t + u;  // the other part
                    for (int i = 1; i < N; i++) h += sym(0, i) * part(o, i);
                    h *= o <= L.nS ? ch : sh;
                } else if ((t <= L.nS) == (u <= L.nS)) {
                    for (int i = 1; i < N; i++)
                        for (int j = 1; j < N; j++) h += part(t, i) * sym(i, j) * part(u, j);
                }
                a[p][q] = h / std::sqrt(w[t] * w[u]);
            }
        jacobi_eig(m, a, lam, v);
        for (int j = 0; j < m; j++) {
            L.lambda[(size_t)at * N + j] = lam[j];
            L.have[(size_t)at * N + j] = 1;
            for (int p = 0; p < m; p++) L.phi[((size_t)idx[p] * N + j) * P + at] = v[p][j] / std::sqrt(w[idx[p]]);
        }
    }
    return true;
}

}  // namespace se_wave
