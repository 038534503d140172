// Host build of the pair kernels' coordinate grid, Coulomb factors and
// fused fixed-point rounding (tests/test_pair_math.py).
#include "fixed_point.h"
#include "nb_pair.h"

using namespace tmamd;

extern "C" {
double pc_wrap(double L, double x) { return BoxAxis(L).wrap(x); }
double pc_delta(double L, double xi, double xj) { return BoxAxis(L).delta(xi, xj); }
// the displacement as a tile in one frame around c forms it
double pc_frame_delta(double L, double xi, double xj, double c) {
    const BoxAxis a(L);
    return to_frame(a.wrap(xi), c, a.edge, a.inv) - to_frame(a.wrap(xj), c, a.edge, a.inv);
}
double pc_edge(double L) { return BoxAxis(L).edge; }
void pc_es(double d2, double beta, double *out) {
    const EsFactors e = es_factors<true>(d2, beta);
    out[0] = e.force;
    out[1] = e.pot;
    EsFactors n[2];
    const double both[2] = {d2, d2};
    es_factors_n<true, 2>(both, beta, n);
    out[2] = n[1].force;
    out[3] = n[1].pot;
}
uint64_t pc_product(double a, double b) { return product_to_fixed(a, b); }
void pc_product3(double s, double vmax, double x, double y, double z, uint64_t *out) {
    product3_to_fixed(s, fixed_small_factor(vmax), x, y, z, out[0], out[1], out[2]);
}
}
