// Host build of the collision form that FP64 storage runs (lb_amd/csrc/collide.hpp,
// Ops<true>), in double, for the CPU test suite.  Built with -ffp-contract=off.
#include <cstdint>

#include "collide.hpp"

using namespace lbm;

extern "C" {

// op: LBM_COLLISION_CUM2015, _CUM2017 or _COMBINED (that operator's 2017 branch).
void host_fp64_collide(int op, uint32_t compat, const double* fin, double rho, double ux, double uy, double uz,
                       double om, double* out)
{
    const Consts<double> K = make_consts<double>(compat);
    const Raw2<double> r = raw_moments(fin);
    const Cen2<double> c = Ops<true>::cen2(r, ux, uy, uz);
    if (op == LBM_COLLISION_CUM2015) Ops<true>::cum2015(K, c, r.m0, rho, ux, uy, uz, om, out);
    else if (op == LBM_COLLISION_CUM2017) cum2017_fused<CV_2017>(K, fin, c, r.m0, rho, ux, uy, uz, om, out);
    else cum2017_fused<CV_2017C>(K, fin, c, r.m0, rho, ux, uy, uz, om, out);
}

double host_fp64_omega_les(const double* fin, double rho, double ux, double uy, double uz, double tau, double cles)
{
    return Ops<true>::omega_les(Ops<true>::cen2(raw_moments(fin), ux, uy, uz), rho, tau, cles);
}

}  // extern "C"
