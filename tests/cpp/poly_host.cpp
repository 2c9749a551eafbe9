// A generated polynomial (gen/<POLY>.inc) on the host against the same polynomial in extended precision.
// argv: file of int32 {nvars, n, slots, rows, terms}, x[nvars][n], coefficients[slots], the rest of each
// row's coefficient rounded to double [rows], then int32 {slot, degree, factors[8]} per term of the rows.
// Prints, for the value and for every component of the gradient (in adapted coordinates): the error's mean
// and standard deviation over the n-mers.  The value of the energy-only code must be the same bits.
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <cmath>
#include <vector>

#define __device__
#define __forceinline__ inline
typedef const double* mbxg_cptr;
#define MBXG_NODE_FENCE(C, dep) (void)(dep)
template <int N>
inline void mbxg_opaque(const double*) {}
inline double __fma_rn(double a, double b, double c) { return std::fma(a, b, c); }

#include POLY_INC

#define CAT_(a, b) a##b
#define CAT(a, b) CAT_(a, b)

int main(int, char** argv) {
    FILE* f = fopen(argv[1], "rb");
    int32_t h[5];
    if (!f || fread(h, sizeof(h), 1, f) != 1) return 2;
    const int nv = h[0], n = h[1], slots = h[2], rows = h[3], terms = h[4];
    std::vector<double> x((size_t)nv * n), c(slots), rest(rows);
    std::vector<int32_t> t((size_t)10 * terms);
    if (fread(x.data(), 8, x.size(), f) != x.size() || fread(c.data(), 8, slots, f) != (size_t)slots ||
        fread(rest.data(), 8, rows, f) != (size_t)rows || fread(t.data(), 4, t.size(), f) != t.size())
        return 2;
    std::vector<double> sum(nv + 1), sq(nv + 1);
    for (int P = PARTS; P <= 8; P *= 8) {
        for (double& v : sum) v = 0.0;
        for (double& v : sq) v = 0.0;
        for (int i = 0; i < n; ++i) {
            std::vector<double> u(nv), g(nv, 0.0);
            for (int j = 0; j < nv; ++j) u[j] = x[(size_t)j * n + i];
            CAT(POLY, _sym)(u.data());
            double e[8 * 64], e2[8 * 64];
            for (int w = 0; w < P; ++w) {
                std::vector<double> gw(nv, 0.0);
                CAT(POLY, _parts)(w, P, c.data(), u.data(), gw.data(), e);
                for (int j = 0; j < nv; ++j) g[j] += gw[j];
#ifdef ENERGY_ONLY
                CAT(POLY, _e_parts)(w, P, c.data(), u.data(), e2);
#endif
            }
#ifdef ENERGY_ONLY
            for (int k = 0; k < 8; ++k)
                if (memcmp(e + 64 * k, e2 + 64 * k, 8)) return 3;
#endif
            const double E = ((e[0] + e[4 * 64]) + (e[2 * 64] + e[6 * 64])) + ((e[64] + e[5 * 64]) + (e[3 * 64] + e[7 * 64]));
            long double V = 0.0L;
            std::vector<long double> G(nv, 0.0L);
            for (int k = 0; k < terms; ++k) {
                const int32_t *q = &t[(size_t)10 * k], d = q[1];
                const long double b = (long double)c[q[0]] + rest[q[0]];
                long double p[9];  // b times the factors from the left
                p[0] = b;
                for (int m = 0; m < d; ++m) p[m + 1] = p[m] * u[q[2 + m]];
                V += p[d];
                long double r = 1.0L;
                for (int m = d - 1; m >= 0; --m) {
                    G[q[2 + m]] += p[m] * r;
                    r *= u[q[2 + m]];
                }
            }
            for (int j = 0; j <= nv; ++j) {
                const double err = (double)(j < nv ? g[j] - G[j] : E - V);
                sum[j] += err;
                sq[j] += err * err;
            }
        }
        for (int j = 0; j <= nv; ++j) {
            const double mean = sum[j] / n;
            printf("%d %d %.17g %.17g\n", P, j, mean, std::sqrt(std::fmax(sq[j] / n - mean * mean, 0.0)));
        }
    }
    return 0;
}
