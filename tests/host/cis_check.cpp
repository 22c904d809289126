// Host check of the polynomials of csrc/sarf_cis.hpp against libm in long double:
// prints the largest absolute error of each over a revolution.
#include "sarf_cis.hpp"

#include <algorithm>
#include <cmath>
#include <cstdio>

template <class F>
static double worst(double lo, double hi, int n, F cis) {
    double e = 0.0;
    for (int i = 0; i <= n; i++) {
        const double t = lo + (hi - lo) * i / n;
        const long double a = 6.283185307179586476925286766559L * (long double)t;
        long double c, s;
        cis(t, c, s);
        e = std::max({e, (double)fabsl(c - cosl(a)), (double)fabsl(s - sinl(a))});
    }
    return e;
}

int main() {
    printf("cis_rev64 %.3e\n", worst(-0.5, 0.5, 3000017, [](double t, long double &c, long double &s) {
               const double2 v = sarf::cis_rev64(t);
               c = v.x;
               s = v.y;
           }));
    printf("cis_rev %.3e\n", worst(0.0, 1.0, 1 << 21, [](double t, long double &c, long double &s) {
               const float2 v = sarf::cis_rev((float)t);
               c = v.x;
               s = v.y;
           }));
    return 0;
}
