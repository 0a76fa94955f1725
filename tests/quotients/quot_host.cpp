// Host build of the face functions under both arithmetics of quot_dev.h, for
// tests/test_quotients_cpu.py.  Test infrastructure: nothing in the library
// loads it.
#include <hip/hip_runtime.h>
#include <string.h>
#include "riemann_dev.h"
#include "states_dev.h"
#include "adjoint_dev.h"

using namespace phd;

namespace {

template <int D, int SOLVER, class M>
bool face(const double* ri, const double* rj, const double* com, double diff, const double* n,
          const double* fv, const Gas& g, double dt, int boost, int gizmo, M& m, double* F)
{
    constexpr int NF = D + 2, G0 = NF, C0 = NF + D * NF;
    double L[NF], R[NF];
    boost_copy<D>(ri, rj, fv, boost, L, R);
    spatial_states<D>(com, diff, ri + C0, rj + C0, ri, rj, ri + G0, rj + G0, gizmo, m, L, R);
    temporal_side<D>(ri, ri + G0, fv, boost, g.gamma, dt, m, L);
    temporal_side<D>(rj, rj + G0, fv, boost, g.gamma, dt, m, R);
    riemann_hll<D, SOLVER>(L, R, n, fv, g, boost, m, F);
    return m.ok;
}

template <int D, int SOLVER>
void faces(long nf, const double* ri, const double* rj, const double* com, const double* diff,
           const double* n, const double* fv, double gamma, double dt, int boost, int gizmo,
           unsigned char* ok, unsigned char* same)
{
    constexpr int NF = D + 2, W = NF + D * NF + D;
    const Gas g = make_gas(gamma);
    for (long f = 0; f < nf; f++) {
        double A[NF], B[NF];
        Ieee mi;
        Shared ms;
        ms.ok = g.shared;
        face<D, SOLVER>(ri + f * W, rj + f * W, com + f * D, diff[f], n + f * D, fv + f * D, g, dt,
                        boost, gizmo, mi, A);
        ok[f] = face<D, SOLVER>(ri + f * W, rj + f * W, com + f * D, diff[f], n + f * D, fv + f * D,
                                g, dt, boost, gizmo, ms, B);
        same[f] = memcmp(A, B, sizeof(A)) == 0;
    }
}

} // namespace

extern "C" void qh_faces(int dim, int hllc, long nf, const double* ri, const double* rj,
                         const double* com, const double* diff, const double* n, const double* fv,
                         double gamma, double dt, int boost, int gizmo, unsigned char* ok,
                         unsigned char* same)
{
    if (dim == 2 && hllc) faces<2, PHD_SOLVER_HLLC>(nf, ri, rj, com, diff, n, fv, gamma, dt, boost, gizmo, ok, same);
    else if (dim == 2) faces<2, PHD_SOLVER_HLL>(nf, ri, rj, com, diff, n, fv, gamma, dt, boost, gizmo, ok, same);
    else if (hllc) faces<3, PHD_SOLVER_HLLC>(nf, ri, rj, com, diff, n, fv, gamma, dt, boost, gizmo, ok, same);
    else faces<3, PHD_SOLVER_HLL>(nf, ri, rj, com, diff, n, fv, gamma, dt, boost, gizmo, ok, same);
}

namespace {

template <int D>
struct List {
    int n;
    const double *rows, *com, *area;
    double* lnb;
    int deg() const { return n; }
    bool valid(int e) const { return area[e] >= 0.0; }
    void row(int e, double* r) const { for (int q = 0; q < 8; q++) r[q] = rows[8 * e + q]; }
    void geo(int e, double* c, double& a) const
    {
        for (int k = 0; k < 3; k++) c[k] = com[3 * e + k];
        a = area[e];
    }
    void out(int e, const double* lam) const { for (int q = 0; q < D + 2; q++) lnb[(D + 2) * e + q] = lam[q]; }
};

template <int D>
void grad(int deg, const double* rows, const double* com, const double* area, const double* pv,
          const double* xi, const double* cx, double vol, const double* lgrad, int fast,
          double* lself, double* lnb)
{
    List<D> l{deg, rows, com, area, lnb};
    grad_cell_vjp<D>(l, pv, xi, cx, vol, lgrad, lself, fast != 0);
}

} // namespace

extern "C" void qh_grad_vjp(int dim, int deg, const double* rows, const double* com,
                            const double* area, const double* pv, const double* xi,
                            const double* cx, double vol, const double* lgrad, int fast,
                            double* lself, double* lnb)
{
    if (dim == 2) grad<2>(deg, rows, com, area, pv, xi, cx, vol, lgrad, fast, lself, lnb);
    else grad<3>(deg, rows, com, area, pv, xi, cx, vol, lgrad, fast, lself, lnb);
}

namespace {

// the same list with one field of its primitives
template <int D>
struct Field : List<D> {
    int q;
    void row(int e, double* r) const
    {
        for (int k = 0; k < D; k++) r[k] = this->rows[8 * e + k];
        r[D] = this->rows[8 * e + D + q];
    }
    void out(int e, const double* lam) const { this->lnb[(D + 2) * e + q] = lam[0]; }
};

template <int D>
void grad_fields(int deg, const double* rows, const double* com, const double* area,
                 const double* pv, const double* xi, const double* cx, double vol,
                 const double* lgrad, int fast, double* lself, double* lnb)
{
    for (int q = 0; q < D + 2; q++) {
        Field<D> l;
        static_cast<List<D>&>(l) = List<D>{deg, rows, com, area, lnb};
        l.q = q;
        grad_cell_vjp<D, Field<D>, 1>(l, pv + q, xi, cx, vol, lgrad + q * D, lself + q, fast != 0);
    }
}

} // namespace

extern "C" void qh_grad_vjp_fields(int dim, int deg, const double* rows, const double* com,
                                   const double* area, const double* pv, const double* xi,
                                   const double* cx, double vol, const double* lgrad, int fast,
                                   double* lself, double* lnb)
{
    if (dim == 2) grad_fields<2>(deg, rows, com, area, pv, xi, cx, vol, lgrad, fast, lself, lnb);
    else grad_fields<3>(deg, rows, com, area, pv, xi, cx, vol, lgrad, fast, lself, lnb);
}
