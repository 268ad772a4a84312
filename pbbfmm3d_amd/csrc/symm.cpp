// symm.cpp -- reflection-adapted bases of an operator set (host, FP64).
//
// Every kernel that depends on |dx|, |dy|, |dz| only has K_{Rd} = R K_d R for
// the reflections R of the axes, so in a basis whose vectors are even or odd
// under each reflection the compressed operators satisfy E_{Rd} = D_R E_d D_R
// with D_R = diag(+-1).  The singular vectors of the precompute span such a
// basis but mix the parities within a degenerate cluster; sym_side finds it:
// columns C (n3 x rt, orthonormal, each of one parity class) and A = C^T U,
// with U ~ C A.  A cluster cut by the rank gives a few more columns than the
// rank, directions of singular values at the rounding level give fewer.
//
// The way back is A's pseudo-inverse, not A^T: the singular vectors of the
// precompute are orthonormal to 1e-14 at order 4 and 2e-13 at order 6 only, and
// the operators rebuilt with A^T carry that error (order 4 1.3e-14 of their
// norm, order 6 8.7e-14; with the pseudo-inverse 1.1e-15 and 7.0e-15, the
// rounding of the operators themselves).
#include <algorithm>
#include <cmath>

#include "host.hpp"

namespace pbb {

// X = Pi_p U diag(w): the part of parity class p (bits x 4, y 2, z 1; set =
// odd) of the weighted columns, n3 x r column-major
static void project_class(int n, int r, const double *U, const double *w, int p, std::vector<double> &X)
{
    const int n3 = n * n * n;
    X.resize((size_t)n3 * r);
    for (int c = 0; c < r; c++) {
        const double *u = U + (size_t)c * n3;
        double *x = &X[(size_t)c * n3];
        for (int a = 0; a < n; a++)
            for (int b = 0; b < n; b++)
                for (int d = 0; d < n; d++) {
                    double s = 0;
                    for (int R = 0; R < 8; R++) {
                        const int i = (R & 4) ? n - 1 - a : a, j = (R & 2) ? n - 1 - b : b, k = (R & 1) ? n - 1 - d : d;
                        const double v = u[(i * n + j) * n + k];
                        s += (__builtin_popcount(R & p) & 1) ? -v : v;
                    }
                    x[(a * n + b) * n + d] = 0.125 * s * w[c];
                }
    }
}

bool sym_side(int n, int r, const double *U, const double *w, double tau, int max_rt, SymSide &out)
{
    const int n3 = n * n * n;
    std::vector<std::vector<double>> cols[8];
    // the classes are independent: pivoted Gram-Schmidt (each column twice)
    // until what is left of the weighted columns is below the class's share
    parallel_for(8, [&](int64_t p) {
        std::vector<double> X, q(n3), t(r);
        project_class(n, r, U, w, (int)p, X);
        std::vector<double> one(1, 1.0), y;
        while ((int)cols[p].size() <= max_rt) {
            double tot = 0, best = -1;
            int j = 0;
            for (int c = 0; c < r; c++) {
                double s = 0;
                for (int i = 0; i < n3; i++) s += X[(size_t)c * n3 + i] * X[(size_t)c * n3 + i];
                tot += s;
                if (s > best) {
                    best = s;
                    j = c;
                }
            }
            if (!(tot > tau * tau / 8)) break;
            std::copy(X.begin() + (size_t)j * n3, X.begin() + (size_t)(j + 1) * n3, q.begin());
            for (int rep = 0; rep < 2; rep++)
                for (const auto &b : cols[p]) {
                    double s = 0;
                    for (int i = 0; i < n3; i++) s += b[i] * q[i];
                    for (int i = 0; i < n3; i++) q[i] -= s * b[i];
                }
            project_class(n, 1, q.data(), one.data(), (int)p, y);  // rounding of the other classes
            double s = 0;
            for (int i = 0; i < n3; i++) s += y[i] * y[i];
            s = 1.0 / std::sqrt(s);
            for (int i = 0; i < n3; i++) y[i] *= s;
            for (int c = 0; c < r; c++) {
                double d = 0;
                for (int i = 0; i < n3; i++) d += y[i] * X[(size_t)c * n3 + i];
                for (int i = 0; i < n3; i++) X[(size_t)c * n3 + i] -= d * y[i];
            }
            cols[p].push_back(y);
        }
    });
    out.rt = 0;
    for (int p = 0; p < 8; p++) {
        out.cnt[p] = (int)cols[p].size();
        out.rt += out.cnt[p];
    }
    if (out.rt == 0 || out.rt > max_rt) return false;
    out.A.assign((size_t)out.rt * r, 0.0);
    out.cls.clear();
    int at = 0;
    for (int p = 0; p < 8; p++)
        for (const auto &b : cols[p]) {
            for (int c = 0; c < r; c++) {
                double s = 0;
                for (int i = 0; i < n3; i++) s += b[i] * U[(size_t)c * n3 + i];
                out.A[at + (size_t)c * out.rt] = s;
            }
            out.cls.push_back(p);
            at++;
        }
    // X = (2 - A A^T) A: the singular values of A are 1 to the rounding of U,
    // or 0 (directions of U that no column holds): s (2 - s^2) is 1 / s there
    const int rt = out.rt;
    std::vector<double> G((size_t)rt * rt);
    out.X.assign((size_t)rt * r, 0.0);
    const double *A = out.A.data();
    parallel_for(rt, [&](int64_t j) {
        double *g = &G[(size_t)j * rt];
        for (int c = 0; c < r; c++) {
            const double *a = A + (size_t)c * rt;
            for (int i = 0; i < rt; i++) g[i] -= a[i] * a[j];
        }
        g[j] += 2.0;
    });
    parallel_for(r, [&](int64_t c) {
        double *x = &out.X[(size_t)c * rt];
        for (int j = 0; j < rt; j++) {
            const double a = A[j + (size_t)c * rt], *g = &G[(size_t)j * rt];
            for (int i = 0; i < rt; i++) x[i] += g[i] * a;
        }
    });
    return true;
}

// Solves T x = b (m x m, row-major, destroyed) by elimination with full
// pivoting; unknowns whose pivot vanishes stay 0.
static void solve_full_pivot(std::vector<double> &T, std::vector<double> &b, int m)
{
    std::vector<int> col(m);
    for (int i = 0; i < m; i++) col[i] = i;
    double first = 0;
    int rank = m;
    for (int k = 0; k < m; k++) {
        int pi = k, pj = k;
        for (int i = k; i < m; i++)
            for (int j = k; j < m; j++)
                if (std::fabs(T[(size_t)i * m + j]) > std::fabs(T[(size_t)pi * m + pj])) {
                    pi = i;
                    pj = j;
                }
        const double piv = std::fabs(T[(size_t)pi * m + pj]);
        if (k == 0) first = piv;
        if (!(piv > 1e-12 * first)) {
            rank = k;
            break;
        }
        for (int j = 0; j < m; j++) std::swap(T[(size_t)k * m + j], T[(size_t)pi * m + j]);
        std::swap(b[k], b[pi]);
        for (int i = 0; i < m; i++) std::swap(T[(size_t)i * m + k], T[(size_t)i * m + pj]);
        std::swap(col[k], col[pj]);
        for (int i = k + 1; i < m; i++) {
            const double f = T[(size_t)i * m + k] / T[(size_t)k * m + k];
            if (f == 0) continue;
            for (int j = k; j < m; j++) T[(size_t)i * m + j] -= f * T[(size_t)k * m + j];
            b[i] -= f * b[k];
        }
    }
    std::vector<double> x(m, 0.0);
    for (int k = rank - 1; k >= 0; k--) {
        double s = b[k];
        for (int j = k + 1; j < rank; j++) s -= T[(size_t)k * m + j] * x[col[j]];
        x[col[k]] = s / T[(size_t)k * m + k];
    }
    b.swap(x);
}

void sym_complete(const SymSide &f, const SymSide &s, int rf, int rs, double *M, int nblocks)
{
    // P = A X^T of each side: the identity but on the columns a cut cluster
    // added, of which the operators hold a projection only.  M holds
    // avg_R (D_R P D_R) K (D_R P' D_R); those rows and columns are undone.
    constexpr int DEF_MAX = 10;
    auto gram = [](const SymSide &q, int r, std::vector<double> &P, std::vector<int> &def) {
        P.assign((size_t)q.rt * q.rt, 0.0);
        for (int c = 0; c < r; c++)
            for (int j = 0; j < q.rt; j++) {
                const double v = q.X[j + (size_t)c * q.rt];
                for (int i = 0; i < q.rt; i++) P[i + (size_t)j * q.rt] += q.A[i + (size_t)c * q.rt] * v;
            }
        for (int i = 0; i < q.rt; i++) {
            const double d = P[i + (size_t)i * q.rt];
            if (std::fabs(d - 1.0) > 1e-9 && d > 1e-6) def.push_back(i);
        }
    };
    std::vector<double> P, Q;
    std::vector<int> df, ds;
    gram(f, rf, P, df);
    gram(s, rs, Q, ds);
    if (df.empty() && ds.empty()) return;
    std::vector<char> isf(f.rt, 0), iss(s.rt, 0);
    for (int i : df) isf[i] = 1;
    for (int j : ds) iss[j] = 1;
    const int nf = (int)df.size(), ns = (int)ds.size(), m = nf * ns;
    parallel_for(nblocks, [&](int64_t blk) {
        double *K = M + (size_t)blk * f.rt * s.rt;
        std::vector<double> b;
        if (m > 0 && nf <= DEF_MAX && ns <= DEF_MAX) {
            std::vector<double> T((size_t)m * m, 0.0);
            b.resize(m);
            for (int a = 0; a < nf; a++)
                for (int c = 0; c < ns; c++) {
                    const int i = df[a], j = ds[c];
                    b[a * ns + c] = K[i + (size_t)j * f.rt];
                    for (int a2 = 0; a2 < nf; a2++)
                        for (int c2 = 0; c2 < ns; c2++) {
                            const int k = df[a2], l = ds[c2];
                            if ((f.cls[i] ^ f.cls[k] ^ s.cls[l] ^ s.cls[j]) == 0)
                                T[(size_t)(a * ns + c) * m + a2 * ns + c2] =
                                    P[i + (size_t)k * f.rt] * Q[l + (size_t)j * s.rt];
                        }
                }
            solve_full_pivot(T, b, m);
        }
        for (int j = 0; j < s.rt; j++)
            for (int i = 0; i < f.rt; i++) {
                double &v = K[i + (size_t)j * f.rt];
                if (isf[i] && !iss[j]) v /= P[i + (size_t)i * f.rt];
                else if (!isf[i] && iss[j]) v /= Q[j + (size_t)j * s.rt];
            }
        if (!b.empty())
            for (int a = 0; a < nf; a++)
                for (int c = 0; c < ns; c++) K[df[a] + (size_t)ds[c] * f.rt] = b[a * ns + c];
    });
}

// The 56 orbits (|dx|, |dy|, |dz|), each at most 3 and not all at most 1: a
// component of 1 or 2 is reached with both signs from every box of an octant
// class, a component of 3 with the sign of the octant only.
void sym_orbits(SymOrbits &o)
{
    o = SymOrbits{};
    int slots = 0;
    for (int a = 0; a < 4; a++)
        for (int b = 0; b < 4; b++)
            for (int c = 0; c < 4; c++) {
                if (a < 2 && b < 2 && c < 2) continue;
                const int v[3] = {a, b, c};
                SymOrbit &w = o.orbit[o.n];
                for (int ax = 0; ax < 3; ax++) {
                    w.d[ax] = v[ax];
                    const int bit = 4 >> ax;
                    if (v[ax] == 0) w.zm |= bit;
                    else if (v[ax] < 3) w.pm |= bit;
                }
                w.slot = slots;
                for (int sig = 0; sig < 8; sig++)
                    if ((sig & ~w.pm) == 0) o.slot_orbit[slots] = o.n, o.slot_sign[slots++] = sig;
                o.n++;
            }
    o.nslots = slots;
}

}  // namespace pbb
