// The Morton grid's range (physkit_amd/csrc/pk_trim.hpp) on the host. Reads "S n": prints the
// sampled bodies of n; or "R m" and the m centroids of each axis: prints each axis' range.
#include "pk_trim.hpp"

#include <algorithm>
#include <cstdio>
#include <vector>

int main()
{
    char what;
    unsigned n;
    while (std::scanf(" %c %u", &what, &n) == 2)
    {
        if (what == 'S')
        {
            for (uint32_t t = 0; t < pk::kTrimSample; ++t) std::printf("%u ", pk::trim_sample(t, n));
            std::printf("\n");
            continue;
        }
        std::vector<double> v[3];
        double lo[3], hi[3], widest = 0.0;
        for (int k = 0; k < 3; ++k)
        {
            v[k].resize(n);
            for (double &x : v[k])
                if (std::scanf("%lf", &x) != 1) return 1;
            std::vector<double> s;
            for (uint32_t t = 0; t < std::min(n, pk::kTrimSample); ++t)
                s.push_back(v[k][n > pk::kTrimSample ? pk::trim_sample(t, n) : t]);
            std::sort(s.begin(), s.end());
            pk::trim_axis(s.data(), static_cast<int>(s.size()), lo[k], hi[k]);
            widest = std::max(widest, hi[k] - lo[k]);
        }
        for (int k = 0; k < 3; ++k)
        {
            double l, h;
            pk::trim_range(*std::min_element(v[k].begin(), v[k].end()), *std::max_element(v[k].begin(), v[k].end()), lo[k],
                           hi[k], widest, l, h);
            std::printf("%.17g %.17g ", l, h);
        }
        std::printf("\n");
    }
    return 0;
}
