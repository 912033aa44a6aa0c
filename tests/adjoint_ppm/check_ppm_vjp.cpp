// Host check of the reverse of the limited parabola (para_vjp) against its
// Jacobian (para_jacobian): lam_l Jl + lam_r Jr on random, near-linear, spiked
// and tied stencils.  Exit status 0 when they agree.
#include <cmath>
#include <cstdio>
#include <random>
#include "hamr_adjoint.h"
using namespace hamr;
int main()
{
    std::mt19937_64 g(11);
    std::normal_distribution<double> nd(0., 1.);
    std::uniform_int_distribution<int> kind(0, 3);
    double worst = 0.;
    for (long it = 0; it < 1000000; it++) {
        double x[5];
        const int kk = kind(g);
        for (int k = 0; k < 5; k++) {
            if (kk == 0) x[k] = nd(g);
            else if (kk == 1) x[k] = k + 0.3 * nd(g);                   // near-linear
            else if (kk == 2) x[k] = (k == 2 ? 3. : 0.) + 0.1 * nd(g);  // spike
            else x[k] = std::floor(2 * nd(g));                          // ties
        }
        const double ll = nd(g), lr = (it & 7) ? nd(g) : 0.;
        double l, r, Jl[5], Jr[5], v[5] = {1., 2., 3., 4., 5.};
        para_jacobian(x, &l, &r, Jl, Jr);
        para_vjp(x, ll, lr, v);
        const double scale = std::fabs(ll) + std::fabs(lr) + 5.;  // the 1 .. 5 that v starts from
        for (int k = 0; k < 5; k++)
            worst = std::fmax(worst, std::fabs(v[k] - (k + 1.) - (ll * Jl[k] + lr * Jr[k])) / scale);
    }
    // partials are at most 3; a dozen roundings of 2^-53 relative to them
    printf("max |vjp - Jacobian| = %.3e of the weights over 1e6 stencils\n", worst);
    return worst < 3. * 12. * 0x1p-53 ? 0 : 2;
}
