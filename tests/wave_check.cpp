// Host check of wave_host.h: for lines of every kind of end, with random
// element matrices, the waves are the generalised eigenvectors of the assembled
// line (V^T G V diagonal, V^T S V = I), every mode is there once, and each block
// holds its waves, even or odd about the line's middle.  Prints the worst
// error; exits 1 if it exceeds 1e-11.
#include <cstdio>
#include <cstdlib>

#include "wave_host.h"

int main() {
    double worst = 0.0;
    for (int N = 2; N <= 8; N++)
        for (int ne : {1, 2, 3, 4, 5, 8, 9, 16, 17})
            for (int ends = 0; ends < 5; ends++) {
                const bool per = ends == 0, lo = ends == 1 || ends == 2, hi = ends == 1 || ends == 3;
                const int n1 = N + 1;
                std::vector<double> A(n1 * n1), K(n1 * n1), s(n1);
                for (double& v : A) v = drand48();
                for (int i = 0; i < n1; i++)  // symmetric, and the same from either end
                    for (int j = 0; j < n1; j++)
                        K[i * n1 + j] = A[i * n1 + j] + A[j * n1 + i] + A[(N - i) * n1 + N - j] + A[(N - j) * n1 + N - i];
                for (int i = 0; i <= N / 2; i++) s[i] = s[N - i] = 0.5 + drand48();
                se_wave::Line L;
                if (!se_wave::wave_line(ne, N, per, lo, hi, K, s, L)) return 1;
                const int n = L.n;
                std::vector<double> G((size_t)n * n), S(n);
                auto unk = [&](int a) {
                    if (per) return a % (ne * N);
                    const int k = a - (lo ? 1 : 0);
                    return k >= 0 && k < n ? k : -1;
                };
                for (int e = 0; e < ne; e++)
                    for (int i = 0; i < n1; i++) {
                        const int a = unk(e * N + i);
                        if (a < 0) continue;
                        S[a] += s[i];
                        for (int j = 0; j < n1; j++) {
                            const int b = unk(e * N + j);
                            if (b >= 0) G[(size_t)a * n + b] += K[i * n1 + j];
                        }
                    }
                std::vector<std::vector<double>> V;
                std::vector<double> lam;
                const double r2 = std::sqrt(0.5);
                for (int c = 0; c < L.E; c++)
                    for (int j = 0; j < N; j++) {
                        if (!L.have[(size_t)c * N + j]) continue;
                        std::vector<double> v(n);
                        for (int k = 0; k < n; k++) {
                            const int a = k + L.off, i = a % N, slot = i == 0 ? a / N - L.vs : a / N;
                            auto part = [&](int t) {
                                return L.F[t == 0 ? 0 : (t <= L.nS ? 1 : 2)][(size_t)slot * L.E16 + c] *
                                       L.phi[((size_t)t * N + j) * L.E16 + c];
                            };
                            if (i == 0 || 2 * i == N) v[k] = part(i);
                            else if (i <= L.nS) v[k] = r2 * (part(i) + part(L.nS + i));
                            else v[k] = r2 * (part(N - i) - part(L.nS + N - i));
                        }
                        V.push_back(v);
                        lam.push_back(L.lambda[(size_t)c * N + j]);
                    }
                if ((int)V.size() != n) {
                    printf("N %d ne %d ends %d: %zu modes of %d\n", N, ne, ends, V.size(), n);
                    return 1;
                }
                double scale = 1e-300;
                for (double v : lam) scale = std::fmax(scale, std::fabs(v));
                for (int p = 0; p < n; p++) {
                    std::vector<double> gv(n, 0.0);
                    for (int a = 0; a < n; a++)
                        for (int b = 0; b < n; b++) gv[a] += G[(size_t)a * n + b] * V[p][b];
                    for (int q = 0; q < n; q++) {
                        double g = 0.0, o = 0.0;
                        for (int a = 0; a < n; a++) {
                            g += V[q][a] * gv[a];
                            o += V[q][a] * S[a] * V[p][a];
                        }
                        worst = std::fmax(worst, std::fabs(g - (p == q ? lam[p] : 0.0)) / scale);
                        worst = std::fmax(worst, std::fabs(o - (p == q ? 1.0 : 0.0)));
                    }
                }
                for (int kind = 0; kind < 3; kind++) {
                    std::vector<double> full((size_t)L.E * L.E, 0.0);
                    for (int odd = 0; odd < 2; odd++) {
                        const auto& b = L.blk[2 * kind + odd];
                        for (int q = 0; q < b.np; q++)
                            for (int k = 0; k < b.nk; k++) {
                                const int c = (b.b0 + q) % L.E, slot = b.s0 + k;
                                int m = L.mirror[kind] < 0 ? slot : L.mirror[kind] - slot;
                                if (m >= L.E) m = 0;
                                if (odd && m != b.top - k) return 1;
                                const double f = L.F[kind][(size_t)slot * L.E16 + c];
                                full[(size_t)slot * L.E + c] = f;
                                if (m != slot) full[(size_t)m * L.E + c] = odd ? -f : f;
                            }
                    }
                    for (int slot = 0; slot < L.E; slot++)
                        for (int c = 0; c < L.E; c++)
                            worst = std::fmax(worst, std::fabs(full[(size_t)slot * L.E + c] -
                                                               L.F[kind][(size_t)slot * L.E16 + c]));
                }
            }
    printf("worst %.3g\n", worst);
    return worst <= 1e-11 ? 0 : 1;
}
