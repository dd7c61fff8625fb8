// The block map's scale (block_map_params): reads lines "curve vol drift portfolio" (factors on the
// market that the first line gives: 51 forwards, 153 loadings) and prints the exponent and the
// largest scaled shock entry's and forward's binary exponents.
#include <stdio.h>

#include "hjm_mfma_plan.h"

using namespace hjm;

int main()
{
    double spot[kTenors], vols[3 * kTenors];
    for (double& x : spot)
        if (scanf("%lf", &x) != 1) return 2;
    for (double& x : vols)
        if (scanf("%lf", &x) != 1) return 2;
    double curve, vol, dr;
    int pf;
    while (scanf("%lf %lf %lf %d", &curve, &vol, &dr, &pf) == 4) {
        double f[kTenors], v[3 * kTenors], m[kTenors];
        for (int j = 0; j < kTenors; ++j) {
            f[j] = curve * spot[j];
            m[j] = dr;
            for (int k = 0; k < 3; ++k) v[k * kTenors + j] = vol * vols[k * kTenors + j];
        }
        const MfmaMap map = pf ? MfmaMap::kPortfolio : MfmaMap::kReference;
        const BlockMapParams p = block_map_params(f, m, v, 0.01, 0.5, 7, map);
        const std::vector<double> W = mfma_block_map_dense(m, v, 0.01, 0.5, map);
        double top = 0.0, high = 0.0;
        for (size_t i = 0; i < W.size(); ++i)
            if (i % kMfmaK >= 64) top = fmax(top, fabs(W[i]) * p.up);
        for (double x : f) high = fmax(high, fabs(x) * p.up);
        printf("%d %.17g %.17g\n", p.scale, top, high);
    }
}
