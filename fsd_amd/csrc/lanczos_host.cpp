// Host FP64 part of the Lanczos square roots of the Brownian sampler
// (Sqrt_multiply, Helper_Brownian.cu:476-583): t = T^(1/2) e_1 for the m x m
// symmetric tridiagonal Lanczos matrix T, through its eigendecomposition
// T = Q diag(lambda) Q^T by implicit QR steps with Wilkinson's shift on the two
// diagonals (Golub and Van Loan, Matrix Computations, 4th ed., section 8.3), in
// double precision.  40 us for m = 24; cyclic Jacobi rotations of the full matrix
// took 3.7 ms, since rounding kept them from their stopping rule.
#include "lanczos_host.h"

#include <cmath>
#include <vector>

// a (diagonal): the eigenvalues at the end; b (off-diagonal) is used up; row j of Qt
// (m x m): the eigenvector of a[j]
static void tridiag_eigen(int m, std::vector<double> &a, std::vector<double> &b, std::vector<double> &Qt)
{
    Qt.assign((size_t)m * m, 0.0);
    for (int i = 0; i < m; ++i) Qt[(size_t)i * m + i] = 1.0;
    auto negligible = [&](int k) {       // also where a NaN reached the matrix
        return !(std::fabs(b[k]) > 1.1e-16 * (std::fabs(a[k]) + std::fabs(a[k + 1])) && std::fabs(b[k]) > 1e-300);
    };
    int q = m - 1;                       // rows past q are done
    for (int it = 0; q > 0 && it < 60 * m; ++it) {
        if (negligible(q - 1)) { --q; continue; }
        int p = q - 1;                   // the unreduced block p .. q
        while (p > 0 && !negligible(p - 1)) --p;
        const double d = 0.5 * (a[q - 1] - a[q]), e = b[q - 1];
        const double mu = a[q] - e * (e / (d + std::copysign(std::sqrt(d * d + e * e), d)));
        double x = a[p] - mu, z = b[p];
        for (int k = p; k < q; ++k) {
            const double r = std::sqrt(x * x + z * z);
            const double c = r > 0.0 ? x / r : 1.0, s = r > 0.0 ? z / r : 0.0;
            if (k > p) b[k - 1] = r;
            const double ak = a[k], an = a[k + 1], bk = b[k];
            const double cs2 = 2.0 * c * s * bk;
            a[k] = c * c * ak + cs2 + s * s * an;
            a[k + 1] = s * s * ak - cs2 + c * c * an;
            b[k] = (c * c - s * s) * bk + c * s * (an - ak);
            if (k + 1 < q) {
                x = b[k];
                z = s * b[k + 1];
                b[k + 1] *= c;
            }
            double *u = &Qt[(size_t)k * m], *v = u + m;
            for (int i = 0; i < m; ++i) {
                const double ui = u[i], vi = v[i];
                u[i] = c * ui + s * vi;
                v[i] = c * vi - s * ui;
            }
        }
    }
}

double tridiag_sqrt_e1(int m, const double *alpha, const double *off, double *t)
{
    std::vector<double> A(alpha, alpha + m), b(off, off + (m - 1)), Qt;
    tridiag_eigen(m, A, b, Qt);
    double lmin = 1e300;
    std::vector<double> s(m);
    for (int j = 0; j < m; ++j) {
        lmin = std::fmin(lmin, A[j]);
        s[j] = std::sqrt(std::fmax(A[j], 0.0)) * Qt[(size_t)j * m];       // lambda_j^(1/2) (Q^T e_1)_j
    }
    for (int i = 0; i < m; ++i) {
        double acc = 0.0;
        for (int j = 0; j < m; ++j) acc += Qt[(size_t)j * m + i] * s[j];
        t[i] = acc;
    }
    return lmin;
}
