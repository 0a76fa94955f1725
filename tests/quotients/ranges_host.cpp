// Host build of the gradient sums' range checks and of one summand both ways,
// for tests/test_gradient_ranges_cpu.py.  Test infrastructure: nothing in the
// library loads it.
#include <hip/hip_runtime.h>
#include "quot_dev.h"

using namespace phd;

// kind: 0 coordinate, 1 primitive, 2 area, 3 volume
extern "C" int rh_ok(int kind, double x)
{
    return kind == 0 ? coord_ok(x) : kind == 1 ? prim_ok(x) : kind == 2 ? area_ok(x) : vol_ok(x);
}

namespace {
template <class M>
double summand(const M& m, const double* v)
{
    // v: xi, xj, com, pi, pj, area, vol along one axis
    const double cfx = v[2] - 0.5 * (v[0] + v[1]), dr = v[0] - v[1];
    const double num = v[5] * ((v[4] - v[3]) * cfx - 0.5 * (v[4] + v[3]) * dr);
    return m.div(num, m.rcp(m.root(dr * dr) * v[6]));
}
} // namespace

// summand with the operators and with Shared; 0 where the distance is zero
extern "C" int rh_summand(const double* v, double* out)
{
    if (v[0] == v[1]) return 0;
    out[0] = summand(Ieee(), v);
    out[1] = summand(Shared(), v);
    return 1;
}
