"""The collision on 16-bit deviations (collide_deviations) on the CPU against the
FP64 collision of the populations (collide<double>), both from the library's
header: random deviations of up to 0.3 about equilibria whose reference velocity
and whose own are up to 0.1 per axis, so that the reference state's moments (all
products of the velocity's distance from the reference) count, K15 and K17, with
and without a force.  Largest difference over the largest deviation: the FP32
collision of 27 values is worth about 10 roundings (6e-8 each) of them."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include "cumulant.hpp"
using namespace lbm3;

static double uniform(double a) { return a * (2.0 * std::rand() / RAND_MAX - 1.0); }

// equilibrium at rho = 1 + dRho and velocity u, a product over the axes, less the weight
static double feq(int q, double dRho, const double (&u)[3])
{
    const int c[3] = {cx(q), cy(q), cz(q)};
    double p = 1.0 + dRho;
    for (int a = 0; a < 3; ++a) p *= c[a] == 0 ? 1.0 - 1.5 * u[a] * u[a] : 1.0 + 3.0 * c[a] * u[a] + 3.0 * u[a] * u[a];
    return weight<double>(q) * (p - 1.0);
}

template <int MODE> static double worst(bool force, double limiter)
{
    const int dirs[9][3] = {{MMM, MMO, MMP}, {MOM, MOO, MOP}, {MPM, MPO, MPP}, {OMM, OMO, OMP}, {OOM, OOO, OOP},
                            {OPM, OPO, OPP}, {PMM, PMO, PMP}, {POM, POO, POP}, {PPM, PPO, PPP}};
    double err = 0.0;
    for (int trial = 0; trial < 20000; ++trial) {
        const double nu = 0.001 + 0.1 * std::rand() / RAND_MAX;
        double U[3], u[3], g[3];
        for (int a = 0; a < 3; ++a) {
            U[a] = (float)uniform(0.1);
            u[a] = uniform(0.1);
            g[a] = force ? (float)uniform(1e-3) : 0.0;
        }
        const double dRho = uniform(0.01), noise = trial % 3 == 0 ? 0.0 : uniform(0.1);
        float h[27];
        double f[27];
        for (int q = 0; q < 27; ++q) {
            h[q] = (float)((feq(q, dRho, u) - feq(q, 0.0, U)) / weight<double>(q) + noise * uniform(1.0));
            f[q] = weight<double>(q) * h[q] + feq(q, 0.0, U);
        }
        const Relax<float> Rf = make_relax<float>((float)nu, 1.f, (float)limiter, (float)g[0], (float)g[1], (float)g[2]);
        // next to a viscosity where a rate has a pole (nu = 0.0476 and others) it amplifies any rounding
        if (std::max({std::fabs(Rf.w3), std::fabs(Rf.w4), std::fabs(Rf.w5), std::fabs(Rf.A), std::fabs(Rf.B)}) > 3.f) continue;
        Relax<double> R = make_relax<double>(nu, 1.0, limiter, g[0], g[1], g[2]);
        // the same coefficients: their own rounding is not the collision's
        R.w1 = Rf.w1; R.w3 = Rf.w3; R.w4 = Rf.w4; R.w5 = Rf.w5; R.A = Rf.A; R.B = Rf.B; R.lambda = Rf.lambda;
        float s[9], d[9], k[9], out[27];
        for (int c = 0; c < 9; ++c) {
            const float m = h[dirs[c][0]], p = h[dirs[c][2]];
            s[c] = p + m;
            d[c] = p - m;
            k[c] = std::fma(4.f, h[dirs[c][1]], s[c]);
        }
        const float Uf[3] = {(float)U[0], (float)U[1], (float)U[2]};
        collide_deviations<MODE>(s, d, k, Uf, Rf, out);
        collide<double, MODE>(f, R);
        double scale = 0.0, e = 0.0;
        for (int q = 0; q < 27; ++q) {
            const double want = (f[q] - feq(q, 0.0, U)) / weight<double>(q);
            scale = std::max(scale, std::fabs(want));
            e = std::max(e, std::fabs(out[q] - want));
        }
        err = std::max(err, e / scale);
    }
    return err;
}

int main()
{
    std::srand(11);
    for (int force = 0; force < 2; ++force)
        std::printf("%.3e %.3e %.3e\n", worst<2>(force, 0.0), worst<1>(force, 0.1), worst<1>(force, 0.001));
    return 0;
}
"""


def _run(tmp_path, include):
    src = tmp_path / "deviations.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "deviations"
    subprocess.run(["g++", "-std=c++17", "-O2", "-mfma", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I", include, str(src),
                    "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    return [float(v) for v in out.split()]


def test_deviations_collide_as_the_populations_do(tmp_path):
    err = _run(tmp_path, os.path.join(ROOT, "lbm3_amd", "csrc"))
    print(err)
    assert len(err) == 6 and max(err) < 2e-6
