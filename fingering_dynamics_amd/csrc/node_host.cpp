// node_host.cpp - host (FP64) build of the per-node arithmetic in lbm_node.h.
//
// The GPU kernels instantiate lbm_node.h with T = float; this file
// instantiates the very same templates with T = double and exports them with
// a C ABI so the CPU test-suite can check the algebra the kernels run against
// the FP64 oracle without a GPU.  Not used by the solver itself.
#include "lbm_node.h"

namespace {
template <typename T = double>
fdn::Consts<T> consts_from(const double c[9]) {
    fdn::Consts<T> k;
    k.inv_tau_g = (T)c[0];
    k.eta_n = (T)c[1];
    k.M = (T)c[2];
    k.a = (T)c[3];
    k.kappa = (T)c[4];
    k.gamma = (T)c[5];
    k.psi_wall = (T)c[6];
    k.gx = (T)c[7];
    k.gy = (T)c[8];
    k.psi_visc = sizeof(T) == 4 ? (T)3e38 : (T)1e300;
    return k;
}

// Collides n nodes (f, g: [n][9]) whose psi is the sum of g; grad: [n][3],
// the stencil's dx, dy, lap.  With per_population, in the form
// f - (f - feq)/tau + F.
template <typename T>
void collide_nodes(int n, T* f, T* g, const T* grad, const double c[9], bool per_population) {
    const fdn::Consts<T> k = consts_from<T>(c);
    for (; n > 0; --n, f += 9, g += 9, grad += 3) {
        T psi = g[0];
        for (int i = 1; i < 9; ++i) psi += g[i];
        const fdn::Mom<T> m = fdn::moments(f, psi, grad[0], grad[1], grad[2], k);
        if (!per_population) {
            fdn::collide(f, g, m, k);
            continue;
        }
        T feq[9], geq[9];
        fdn::equilibria(m, k, feq, geq);
        for (int i = 0; i < 9; ++i) {
            const T ex = T(fdn::EX[i]), ey = T(fdn::EY[i]), eu = ex * m.ux + ey * m.uy;
            const T F = fdn::W9<T>::w(i) * (T(1) - T(0.5) * m.itau) *
                        ((T(3) * (ex - m.ux) + T(9) * eu * ex) * m.fx + (T(3) * (ey - m.uy) + T(9) * eu * ey) * m.fy);
            f[i] = f[i] - (f[i] - feq[i]) * m.itau + F;
            g[i] = g[i] - (g[i] - geq[i]) * k.inv_tau_g;
        }
    }
}
}  // namespace

extern "C" {

// 1 / tau_mix with the viscosity interpolation's |psi| bound (<= 0: none).
double fdn_inv_tau_mix_f64(double rho, double psi, const double c[9], double bound) {
    fdn::Consts<double> k = consts_from(c);
    if (bound > 0) k.psi_visc = bound;
    return fdn::inv_tau_mix(rho, psi, k);
}

// n[9] psi on the node and its neighbours (C E N W S NE NW SW SE) -> out[3] = dx, dy, lap
void fdn_stencil_f64(const double n[9], double out[3]) { fdn::stencil(n, out[0], out[1], out[2]); }

// Moments (rho, psi, mu, ux, uy, p, 1/tau_mix, Fx, Fy) from post-stream f.
void fdn_moments_f64(const double f[9], double psi, double dpx, double dpy, double lap, const double c[9],
                     double mom[9]) {
    const fdn::Mom<double> m = fdn::moments(f, psi, dpx, dpy, lap, consts_from(c));
    const double v[9] = {m.rho, m.psi, m.mu, m.ux, m.uy, m.p, m.itau, m.fx, m.fy};
    for (int i = 0; i < 9; ++i) mom[i] = v[i];
}

// feq, geq for given moments (same layout as fdn_moments_f64's output).
void fdn_equilibria_f64(const double mom[9], const double c[9], double feq[9], double geq[9]) {
    const fdn::Mom<double> m{mom[0], mom[1], mom[2], mom[3], mom[4], mom[5],
                             mom[6], mom[7], mom[8], mom[5] / 3.0, mom[2] / 3.0};
    fdn::equilibria(m, consts_from(c), feq, geq);
}

// In-place collision of f and g with the given moments.
void fdn_collide_f64(double f[9], double g[9], const double mom[9], const double c[9]) {
    const fdn::Mom<double> m{mom[0], mom[1], mom[2], mom[3], mom[4], mom[5],
                             mom[6], mom[7], mom[8], mom[5] / 3.0, mom[2] / 3.0};
    fdn::collide(f, g, m, consts_from(c));
}

// collide_nodes in single and double precision.
void fdn_collide_nodes_f32(int n, float* f, float* g, const float* grad, const double c[9], int per_population) {
    collide_nodes<float>(n, f, g, grad, c, per_population != 0);
}
void fdn_collide_nodes_f64(int n, double* f, double* g, const double* grad, const double c[9], int per_population) {
    collide_nodes<double>(n, f, g, grad, c, per_population != 0);
}

void fdn_inlet_f64(double f[9], double g[9], double u, double px, double py) {
    fdn::inlet_f(f, u, px, py);
    fdn::inlet_g(g);
}

void fdn_outlet_f64(double f[9], double g[9], double u, double px, double py, int pressure, double rho_out,
                    double c3) {
    fdn::outlet_f(f, u, px, py, pressure != 0, rho_out, c3);
    fdn::outlet_g(g);
}

void fdn_inlet_corner_f64(double f[9], double g[9], double rho_nb, int top) {
    if (top) {
        fdn::inlet_corner_top_f(f, rho_nb);
        fdn::inlet_corner_top_g(g);
    } else {
        fdn::inlet_corner_bottom_f(f, rho_nb);
        fdn::inlet_corner_bottom_g(g);
    }
}

double fdn_inlet_rho_f64(const double f[9], double u, double px) { return fdn::inlet_rho(f, u, px); }

}  // extern "C"
