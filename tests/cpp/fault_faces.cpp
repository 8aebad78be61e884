// The device's fault faces (rs_fault, sw_fault) built for the host, for tests/test_fault_faces.py: n faces.
// in: vx1 vx2 vy1 vy2 vz1 vz2 syy1 syy2 sxy1 sxy2 syz1 syz2 per face; out: vx vy vz syy sxy syz of both sides.
#include "../../tetemoko_amd/csrc/tmk_physics.hpp"

extern "C" void fault_faces(int sw, int n, double Zp, double Zs, double V0, double a, double b, double L, double tau0,
                            double state, const double* in, double* out)
{
    static tmk::DevParams P;
    P.Zp = Zp; P.Zs = Zs; P.iZp = 1.0 / Zp; P.iZs = 1.0 / Zs; P.rs_V0 = V0;
    P.dx = 1.0; P.fric_w0 = 1e40;
    tmk::FaultFace f{};
    f.s0 = state; f.tau0 = tau0; f.a = a; f.b = b; f.L = L;
    for (int k = 0; k < n; ++k) {
        const double* q = in + 12 * k;
        tmk::FaultIn w;
        tmk::FaultOut o;
        for (int s = 0; s < 2; ++s) {
            w.vx[s] = q[s]; w.vy[s] = q[2 + s]; w.vz[s] = q[4 + s];
            w.syy[s] = q[6 + s]; w.sxy[s] = q[8 + s]; w.syz[s] = q[10 + s];
        }
        if (sw) tmk::sw_fault(P, 0, f, state, w, o);
        else tmk::rs_fault(P, f, state, w, o);
        for (int s = 0; s < 2; ++s) {
            double* r = out + 12 * k + s;
            r[0] = o.vx[s]; r[2] = o.vy[s]; r[4] = o.vz[s]; r[6] = o.syy[s]; r[8] = o.sxy[s]; r[10] = o.syz[s];
        }
    }
}
