// The device's rate-and-state fault solve (rs_solve, rs_newton) built for the host, for
// tests/test_fault_solve.py: n solves at once.
#include "../../tetemoko_amd/csrc/tmk_physics.hpp"

extern "C" void fault_solve(int reference, int n, double Zs, double V0, const double* phi, const double* psi,
                            const double* sn, const double* a, double* V, double* tau)
{
    static tmk::DevParams P;
    P.Zs = Zs;
    P.rs_V0 = V0;
    for (int k = 0; k < n; ++k)
        tau[k] = reference ? tmk::rs_newton(P, phi[k], psi[k], sn[k], a[k], V[k])
                           : tmk::rs_solve(P, phi[k], psi[k], sn[k], a[k], V[k]);
}
