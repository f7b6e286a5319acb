// lbm_node.h - per-node arithmetic of the two-phase free-energy D2Q9 step.
//
// Shared by the gfx950 kernels (T = float) and by a host build used in the
// CPU tests (T = double), so the algebra the GPU runs is checked against the
// FP64 oracle without a GPU.  Everything here is a pure function of its
// arguments.
//
// Reference formulas (lattice_boltzmann/fingering_periodic.py):
//   stencils      d_x psi, d_y psi, lap psi            :214-256
//   mu            a psi (1 - psi^2) - kappa lap psi    :141-149
//   velocity      (sum f e + mu grad psi / 2) / rho    :126-139
//   pressure      rho/3 + psi mu                       :123-124
//   tau_mix       3 * 2 nu1 nu2/(nu1(1-psi)+nu2(1+psi)) + 1/2, nu1 = Eta_n/rho,
//                 nu2 = M Eta_n/rho                    :201-208
//   equilibria    feq_i = w_i (A_i + rho Q_i), geq_i = w_i (B_i + psi Q_i),
//                 Q_i = 3 e.u + 4.5 (e.u)^2 - 1.5 u.u  :155-192
//   forcing       F_i = w_i (1 - 1/(2 tau_mix)) [(3(e-u) + 9 (e.u) e) . Force],
//                 Force = mu grad psi                  :194-199
//   collision     f* = f - (f - feq)/tau_mix + F,  g* = g - (g - geq)/tau   :258-264
//   Zou-He        inlet :268-302, outlet :305-324; walled corners
//                 lattice_boltzmann/fingering.py:334-364, :387-390
#pragma once

#if defined(__HIPCC__)
#define FD_HD __host__ __device__ __forceinline__
#else
#define FD_HD inline
#endif

namespace fdn {

// Reciprocal: the hardware approximation (v_rcp_f32, 1 ulp) in FP32 device
// code, an exact division elsewhere.
FD_HD float rcp(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rcpf(x);
#else
    return 1.0f / x;
#endif
}
FD_HD double rcp(double x) { return 1.0 / x; }

// x between -b and b (b > 0); one v_med3_f32 in FP32 device code.
FD_HD float clampv(float x, float b) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_fmed3f(x, -b, b);
#else
    return x < -b ? -b : (x > b ? b : x);
#endif
}
FD_HD double clampv(double x, double b) { return x < -b ? -b : (x > b ? b : x); }

// D2Q9 order of fingering_periodic.py:50-89.
constexpr int EX[9] = {0, 1, 0, -1, 0, 1, -1, -1, 1};
constexpr int EY[9] = {0, 0, 1, 0, -1, 1, 1, -1, -1};
constexpr int OPP[9] = {0, 3, 4, 1, 2, 7, 8, 5, 6};

template <typename T>
struct W9 {
    static constexpr T w0 = T(4) / T(9);
    static constexpr T w1 = T(1) / T(9);
    static constexpr T w5 = T(1) / T(36);
    static FD_HD T w(int i) { return i == 0 ? w0 : (i < 5 ? w1 : w5); }
};

template <typename T>
struct Consts {
    T inv_tau_g;   // 1/tau of the g equation
    T eta_n, M;    // viscosities
    T a, kappa, gamma;
    T psi_wall;
    T gx, gy;      // body force (0 in the reference)
    T psi_visc;    // |psi| bound of the viscosity interpolation (huge: none)
};

// psi on the node and its 8 neighbours in D2Q9 order:
// n[0]=C n[1]=E n[2]=N n[3]=W n[4]=S n[5]=NE n[6]=NW n[7]=SW n[8]=SE
template <typename T>
FD_HD void stencil(const T n[9], T& dx, T& dy, T& lap) {
    const T a = n[5] - n[7], b = n[8] - n[6];
    dx = (T(4) * (n[1] - n[3]) + (a + b)) * (T(1) / T(12));
    dy = (T(4) * (n[2] - n[4]) + (a - b)) * (T(1) / T(12));
    lap = (T(-20) * n[0] + T(4) * (n[2] + n[4] + n[1] + n[3]) + n[5] + n[6] + n[7] + n[8]) *
          (T(1) / T(6));
}

template <typename T>
FD_HD T chem_pot(T psi, T lap, const Consts<T>& c) {
    return c.a * psi * (T(1) - psi * psi) - c.kappa * lap;
}

template <typename T>
FD_HD T inv_tau_mix(T rho, T psi, const Consts<T>& c) {
    // 2 nu1 nu2 / (nu1 (1-psi) + nu2 (1+psi)) with nu1 = eta/rho, nu2 = M eta/rho
    // = 2 M eta / (rho ((1-psi) + M (1+psi))).  The denominator vanishes at
    // psi = -(1+M)/(M-1) (-1.14 for M = 15), which overshoots past -1 near
    // wetting solids reach; with c.psi_visc = 1 the interpolation uses psi
    // clamped to the pure phases.  With the default huge bound the clamp
    // leaves psi as it is.
    // 1/tau = y / (6 M eta + y/2) with y the denominator: one reciprocal, and
    // 0 at the pole.
    const T pv = clampv(psi, c.psi_visc);
    const T y = rho * (T(2) + (c.M - T(1)) * (T(1) + pv));
    return y * rcp(T(6) * c.M * c.eta_n + T(0.5) * y);
}

// tau_mix - 1/2 = 6 M eta / (rho ((1-psi) + M (1+psi))), with the same psi
// bound as inv_tau_mix: the health term of the watchdog.  BGK needs
// tau_mix > 1/2; a value <= 0 (or infinite) means psi has crossed the pole
// of the interpolation at psi = -(1+M)/(M-1) (fingering_periodic.py:201-208).
template <typename T>
FD_HD T tau_excess(T rho, T psi, const Consts<T>& c) {
    const T pv = psi < -c.psi_visc ? -c.psi_visc : (psi > c.psi_visc ? c.psi_visc : psi);
    return T(6) * c.M * c.eta_n * rcp(rho * ((T(1) - pv) + c.M * (T(1) + pv)));
}

// Moments the collision of one node uses.  p3 and mu3 are thirds of the
// pressure and of mu, each rounded once.
template <typename T>
struct Mom {
    T rho, psi, mu, ux, uy, p, itau, fx, fy, p3, mu3;
};

// p3 and mu3 of a pressure rho/3 + psi mu_p (mu_p is mu, or 0 where the
// pressure is evaluated before mu).
template <typename T>
FD_HD void thirds(Mom<T>& m, T mu_p) {
    m.mu3 = m.mu * (T(1) / T(3));
    const T e = m.psi * (mu_p * (T(1) / T(3)));
    m.p3 = m.rho * (T(1) / T(9)) + e;
}

// Moments from the node's post-stream populations (fingering_periodic.py:470-479).
template <typename T>
FD_HD Mom<T> moments(const T f[9], T psi, T dpx, T dpy, T lap, const Consts<T>& c) {
    Mom<T> m;
    m.rho = f[0] + f[1] + f[2] + f[3] + f[4] + f[5] + f[6] + f[7] + f[8];
    const T d57 = f[5] - f[7], d86 = f[8] - f[6];
    const T jx = (f[1] - f[3]) + (d57 + d86);
    const T jy = (f[2] - f[4]) + (d57 - d86);
    m.psi = psi;
    m.mu = chem_pot(psi, lap, c);
    m.fx = m.mu * dpx + c.gx;
    m.fy = m.mu * dpy + c.gy;
    const T ir = rcp(m.rho);
    m.ux = (jx + T(0.5) * m.fx) * ir;
    m.uy = (jy + T(0.5) * m.fy) * ir;
    m.p = m.rho * (T(1) / T(3)) + psi * m.mu;
    thirds(m, m.mu);
    m.itau = inv_tau_mix(m.rho, psi, c);
    return m;
}

template <typename T>
FD_HD void equilibria(const Mom<T>& m, const Consts<T>& c, T feq[9], T geq[9]) {
    const T usq = m.ux * m.ux + m.uy * m.uy;
    const T A = T(3) * m.p;
    const T B = T(3) * c.gamma * m.mu;
    // (x - 3 (1 - w0) y) / w0 with w0 = 4/9: (x - 5/3 y) * 9/4
    const T A0 = (m.rho - T(5) / T(3) * m.p) * T(2.25);
    const T B0 = (m.psi - T(5) / T(3) * c.gamma * m.mu) * T(2.25);
#pragma unroll
    for (int i = 0; i < 9; ++i) {
        const T eu = T(EX[i]) * m.ux + T(EY[i]) * m.uy;
        const T q = T(3) * eu + T(4.5) * eu * eu - T(1.5) * usq;
        const T w = W9<T>::w(i);
        feq[i] = w * ((i == 0 ? A0 : A) + m.rho * q);
        geq[i] = w * ((i == 0 ? B0 : B) + m.psi * q);
    }
}

// In-place BGK collision of both distributions with Guo forcing:
//   f*_i = (1 - s) f_i + s feq_i + F_i,  s = 1/tau_mix,  F_i = w_i (1 - s/2) [...]
//   g*_i = (1 - t) g_i + t geq_i,        t = 1/tau
// written over the direction pairs (i, opp(i)).  With the vectors
//   J = 3 w1 (s rho u + (1 - s/2) F),  K = J + 3 w1 (1 - s/2) F
// the part of s feq_i + F_i that is odd in e_i is (w_i/w1) e.J and the even
// part is (w_i/w1) (s w1 A_i - u.K/2 + 3/2 (e.u)(e.K)), so that px = ux Kx,
// py = uy Ky and the cross term ux Ky + uy Kx serve all nine directions; the
// same for g with H = 3 w1 t psi u in place of both.  The kernels spend most
// of their time issuing vector instructions; this form and the moments'
// shared differences and reciprocals take 74 fewer of them per node than
// equilibria formed for each pair (350 -> 276): 100 x 400 on tiles 8.0 ->
// 7.7 us per iteration, 2048 x 1024 45.7 -> 43.9, 24 domains of an ensemble
// 343 -> 325 per launch of three.
// Conservation.  A collision keeps the sums of f and of g if every rounded
// constant and product enters the rest population as it enters the others:
//   - 1 - s and s have to add up to 1: rest() rounds 1 - s and s is taken back
//     from it, which is exact (for 0 <= s <= 2).  For s < 1/2 (tau > 2) that
//     puts s on a grid of 2^-24, an error of at most 2^-25; what it multiplies
//     is f - feq, and with s in full at the price of an addition a population
//     no error below was smaller;
//   - the rest population's share of s p is 5 times that of direction 1: of the
//     same number (p3, a1).  With 5/3 p and 1/3 as constants of their own, one
//     rounded down and one up, density grew by 3e-8 s a collision.
// Errors in float over a droplet in shear (96 x 96; M = 1, 5, 20; tau 0.79,
// 1.5, 5) as parts of those of feq and geq formed for each pair, geometric
// means: one collision, f 0.94 at the interface and 0.98 elsewhere, g 0.95 and
// 0.86, sums of f 0.97 and of g 0.92; psi, rho, ux, uy after 50 to 8000
// iterations 0.36, 0.05, 0.63, 0.53.
// On the GPU, fields after 50 ... 100 iterations, relative to 64 bits (in
// parentheses that form, and this one with 5/3 and 1/3 as constants): 320 x 128
// 6e-7 (2.2e-6, 2.3e-6), 400 x 100 2.4e-7 (3.2e-6, 3.3e-6), 2048 x 1024 6.7e-7
// (2.6e-6, 1.8e-6), 24 domains 2.7e-7 (1.1e-6, 1.2e-6); the same time within
// 0.3 % (400 x 100: 0.8).
template <typename T>
FD_HD T rest(T s) {
    return T(1) - s;
}

template <typename T>
FD_HD void relax(T f[9], T om, T a0, T a1, T px, T py, T cross, T jx, T jy) {
    const T sp = px + py;
    const T s13 = (a1 + px) - T(0.5) * py, s24 = (a1 + py) - T(0.5) * px;
    const T q = T(0.25) * (a1 + sp);
    const T s57 = q + T(0.375) * cross, s68 = q - T(0.375) * cross;
    const T j57 = jx + jy, j68 = jy - jx;
    f[0] = om * f[0] + (a0 - T(2) * sp);
    f[1] = om * f[1] + (s13 + jx);
    f[3] = om * f[3] + (s13 - jx);
    f[2] = om * f[2] + (s24 + jy);
    f[4] = om * f[4] + (s24 - jy);
    f[5] = om * f[5] + (s57 + T(0.25) * j57);
    f[7] = om * f[7] + (s57 - T(0.25) * j57);
    f[6] = om * f[6] + (s68 + T(0.25) * j68);
    f[8] = om * f[8] + (s68 - T(0.25) * j68);
}

template <typename T>
FD_HD void collide(T f[9], T g[9], const Mom<T>& m, const Consts<T>& c) {
    {
        const T om = rest(m.itau), s = T(1) - om;
        const T s3 = s * (T(1) / T(3)), sr = s3 * m.rho;       // 3 w1 = 1/3
        const T f3 = T(1) / T(3) - T(0.5) * s3;                // 3 w1 (1 - s/2)
        const T jx = sr * m.ux + f3 * m.fx, jy = sr * m.uy + f3 * m.fy;
        const T kx = jx + f3 * m.fx, ky = jy + f3 * m.fy;
        // w1 A = p/3;  w0 A_0 = rho - 5/3 p
        relax(f, om, s * (m.rho - T(5) * m.p3), s * m.p3, m.ux * kx, m.uy * ky, m.ux * ky + m.uy * kx, jx, jy);
    }
    {
        const T om = rest(c.inv_tau_g), t = T(1) - om;
        const T t3 = t * (T(1) / T(3));
        const T a1 = t * (c.gamma * m.mu3), h = t3 * m.psi;
        const T hx = h * m.ux, hy = h * m.uy;
        // w1 B = gamma mu / 3;  w0 B_0 = psi - 5/3 gamma mu
        relax(g, om, t * m.psi - T(5) * a1, a1, m.ux * hx, m.uy * hy, T(2) * (m.ux * hy), hx, hy);
    }
}

// ---------------------------------------------------------------- Zou-He
// Inlet density from the known populations (fingering_periodic.py:276-277).
template <typename T>
FD_HD T inlet_rho(const T f[9], T u, T px) {
    return (f[0] + f[2] + f[4] + T(2) * (f[3] + f[6] + f[7]) - T(0.5) * px) * rcp(T(1) - u);
}

// Inlet, rows with the standard formulas (fingering_periodic.py:276-302).
template <typename T>
FD_HD void inlet_f(T f[9], T u, T px, T py) {
    const T r = inlet_rho(f, u, px);
    const T ur = u * r;
    f[1] = f[3] + (T(2) / T(3)) * ur - px * (T(1) / T(6));
    f[5] = f[7] - T(0.5) * (f[2] - f[4]) + ur * (T(1) / T(6)) - px * (T(1) / T(6)) - T(0.25) * py;
    f[8] = f[6] + T(0.5) * (f[2] - f[4]) + ur * (T(1) / T(6)) - px * (T(1) / T(6)) + T(0.25) * py;
}

template <typename T>
FD_HD void inlet_g(T g[9]) {
    // w_k psi_in / (w1 + w5 + w8): w1/(1/6) = 2/3, w5/(1/6) = 1/6
    const T s = T(1) - (g[0] + g[2] + g[3] + g[4] + g[6] + g[7]);
    g[1] = (T(2) / T(3)) * s;
    g[5] = (T(1) / T(6)) * s;
    g[8] = (T(1) / T(6)) * s;
}

// Walled inlet corner nodes (fingering.py:334-364); rho_nb is the inlet
// density of the adjacent row (row 1 for the bottom corner, row H-2 for the
// top corner).
template <typename T>
FD_HD void inlet_corner_bottom_f(T f[9], T rho_nb) {
    f[1] = f[3];
    f[2] = f[4];
    f[5] = f[7];
    f[6] = T(0.5) * (rho_nb - (f[0] + f[1] + f[2] + f[3] + f[4] + f[5] + f[7]));
    f[8] = f[6];
}

template <typename T>
FD_HD void inlet_corner_bottom_g(T g[9]) {
    // w6 (1 - sum) / (w6 + w8) = (1 - sum) / 2
    g[1] = g[3];
    g[2] = g[4];
    g[5] = g[7];
    g[6] = T(0.5) * (T(1) - (g[0] + g[1] + g[2] + g[3] + g[4] + g[5] + g[7]));
    g[8] = g[6];
}

template <typename T>
FD_HD void inlet_corner_top_f(T f[9], T rho_nb) {
    f[1] = f[3];
    f[4] = f[2];
    f[8] = f[6];
    f[5] = T(0.5) * (rho_nb - (f[0] + f[1] + f[2] + f[3] + f[4] + f[6] + f[8]));
    f[7] = f[5];
}

template <typename T>
FD_HD void inlet_corner_top_g(T g[9]) {
    g[1] = g[3];
    g[4] = g[2];
    g[8] = g[6];
    g[5] = T(0.5) * (T(1) - (g[0] + g[1] + g[2] + g[3] + g[4] + g[6] + g[8]));
    g[7] = g[5];
}

// Outlet (fingering_periodic.py:305-324).  Velocity outlet: u given, rho
// solved.  Pressure outlet (build-original): rho given, u solved from the
// same mass balance.  c3 is 2/3 (fingering_periodic.py:317) or 1.5
// (fingering.py:378).
template <typename T>
FD_HD void outlet_f(T f[9], T u, T px, T py, bool pressure, T rho_out, T c3) {
    const T known = f[0] + f[2] + f[4] + T(2) * (f[1] + f[5] + f[8]) + T(0.5) * px;
    T r;
    if (pressure) {
        r = rho_out;
        u = known * rcp(rho_out) - T(1);
    } else {
        r = known * rcp(T(1) + u);
    }
    const T ur = u * r;
    f[3] = f[1] - c3 * ur + px * (T(1) / T(6));
    f[6] = f[8] - T(0.5) * (f[2] - f[4]) - ur * (T(1) / T(6)) + T(0.25) * py + px * (T(1) / T(6));
    f[7] = f[5] + T(0.5) * (f[2] - f[4]) - ur * (T(1) / T(6)) - T(0.25) * py + px * (T(1) / T(6));
}

template <typename T>
FD_HD void outlet_g(T g[9]) {
    const T s = T(-1) - (g[0] + g[1] + g[2] + g[4] + g[5] + g[8]);
    g[3] = (T(2) / T(3)) * s;
    g[6] = (T(1) / T(6)) * s;
    g[7] = (T(1) / T(6)) * s;
}

}  // namespace fdn
