// CPU check of the inference path's GELU (mpc_amd/csrc/gelu_poly.h and the form
// of fno_device.h's gelu_fast) against 64 bits: the polynomial in FP64 at its
// FP32 coefficients, then the whole function in FP32, by range of |x|, beside
// the erf form 0.5 x (1 + erf(x / sqrt 2)) with a correctly rounded erf.
// Errors are in units of |x| / 2, GELU's size near 0.  Prints the figures; exit
// 1 on failure.
#include "../../mpc_amd/csrc/gelu_poly.h"
#include <cmath>
#include <cstdio>

static float fast(float x) {
    const float a = std::fabs(x), e = (float)std::exp2((double)(-a * gelu_poly(a)));
    return std::fma(-std::fmin(0.5f * a, 64.f), e, std::fmax(x, 0.f));
}
static float erf_form(float x) { return 0.5f * x * (1.f + (float)std::erf((double)(x * 0.70710678118654752f))); }

int main() {
    double worst = 0, at = 0;
    for (int i = 1; i <= 400000; ++i) {
        const double a = 10.0 * i / 400000, d = std::fabs(std::exp2(-a * gelu_poly(a)) - std::erfc(a / std::sqrt(2.0)));
        if (d > worst) { worst = d; at = a; }
    }
    printf("polynomial: max %.2e at %.3f\n", worst, at);
    int bad = worst > 1e-9;
    const double edge[] = {0, 0.01, 0.1, 0.5, 1, 2, 4, 8, 16};
    for (int k = 0; k + 1 < 9; ++k)
        for (int sg = -1; sg <= 1; sg += 2) {
            double sf = 0, se = 0, mf = 0, me = 0;
            const int m = 100000;
            for (int i = 1; i <= m; ++i) {
                const float x = (float)(sg * (edge[k] + (edge[k + 1] - edge[k]) * i / m));
                const double ref = 0.5 * (double)x * std::erfc(-(double)x / std::sqrt(2.0)), s = std::fabs(x) / 2;
                const double f = std::fabs(fast(x) - ref) / s, e = std::fabs(erf_form(x) - ref) / s;
                sf += f * f;
                se += e * e;
                mf = std::fmax(mf, f);
                me = std::fmax(me, e);
            }
            sf = std::sqrt(sf / m);
            se = std::sqrt(se / m);
            printf("%c|x| %5.2f-%5.2f: rms %.2e (erf form %.2e), max %.2e (%.2e)\n", sg < 0 ? '-' : '+', edge[k],
                   edge[k + 1], sf, se, mf, me);
            if (sf > 1.01 * se) bad = 1;        /* an rms of 1e5 samples is itself known to 0.3% */
        }
    printf(bad ? "FAIL\n" : "OK\n");
    return bad;
}
