// The FP32 bulk's plastic return (plastic_flow_delta) built for the host, for tests/test_plastic_return.py:
// n cells at once.  k: pbg[7], pf[6], G; s: 6 stress differences (sxx syy szz sxy sxz syz), lam, gam per cell.
#include "../../tetemoko_amd/csrc/tmk_physics.hpp"

extern "C" void plastic_return(int ns, int n, const float* k, float dt, float* s)
{
    static tmk::DevParams P;
    for (int q = 0; q < 7; ++q) P.pbg[q] = k[q];
    for (int q = 0; q < 6; ++q) P.pf[q] = k[7 + q];
    P.fG = k[13];
    for (int c = 0; c < n; ++c) {
        float* u = s + 8 * c;
        if (ns == 2) tmk::plastic_flow_delta<float, 2, tmk::DevParams>(P, dt, u[0], u[1], u[2], u[3], u[4], u[5], u[6], u[7]);
        else tmk::plastic_flow_delta<float, 3, tmk::DevParams>(P, dt, u[0], u[1], u[2], u[3], u[4], u[5], u[6], u[7]);
    }
}
