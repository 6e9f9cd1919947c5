// The EPL angular factor in FP64: Omega(psi) = sum_{k=0..10} C_k e^{i(2k+1) psi}
// with C_0 = 1, C_k = C_{k-1} (-f (2k - T)/(2k + T)), f = (1-q)/(1+q), T = 2-t
// (the tenth-order series of objects/epl.cl), and its psi derivative.
// Table nodes are taken in the diamond angle p of epl_table.h.
#pragma once

// C_k / C_{k-1}
__device__ inline double lensed_epl_ratio(double q, double t, int k)
{
    const double f = (1 - q) / (1 + q), T = 2 - t;
    return -f * (2 * k - T) / (2 * k + T);
}

// e P(z) and e Q(z), P(z) = sum C_k z^k and Q(z) = sum (2k+1) C_k z^k, for
// complex e and z (Horner's scheme): with e = e^{i psi} and z = e^{2 i psi}
// the first is Omega and i times the second its derivative
__device__ inline void lensed_epl_sum(const double* ratio, double ex, double ey, double zx, double zy, double& px,
                                      double& py, double& qx, double& qy)
{
    double c[11];
    c[0] = 1.0;
    for (int k = 1; k <= 10; ++k) c[k] = c[k - 1] * ratio[k - 1];
    double ax = c[10], ay = 0.0, bx = 21 * c[10], by = 0.0;
    for (int k = 9; k >= 0; --k) {
        const double an = c[k] + (zx * ax - zy * ay), bn = (2 * k + 1) * c[k] + (zx * bx - zy * by);
        ay = zy * ax + zx * ay;
        by = zy * bx + zx * by;
        ax = an;
        bx = bn;
    }
    px = ex * ax - ey * ay;
    py = ey * ax + ex * ay;
    qx = ex * bx - ey * by;
    qy = ey * bx + ex * by;
}

__device__ inline void lensed_epl_omega(double q, double t, double psi, double& ox, double& oy, double& dx,
                                        double& dy)
{
    double ratio[10], sn, cs, qx, qy;
    for (int k = 1; k <= 10; ++k) ratio[k - 1] = lensed_epl_ratio(q, t, k);
    sincos(psi, &sn, &cs);
    lensed_epl_sum(ratio, cs, sn, cs * cs - sn * sn, 2 * cs * sn, ox, oy, qx, qy);
    dx = -qy;
    dy = qx;
}

// The tabulated factor at diamond angle p = sin / (cos + sin) of psi in the
// first quadrant: W(p) = g(p)^h Omega(psi(p)) with g = p^2 + (1-p)^2
// (|u|^2 = (|u_x| + |u_y|)^2 g) and h = (1-t)/2, so that the deflection's
// |u|^(1-t) Omega is (|u_x| + |u_y|)^(1-t) W.  psi = atan2(p, 1-p), dpsi/dp
// = 1/g; the derivative is per unit of the interval coordinate f = p NT - i.
// No angle is formed: e^{i psi} = ((1-p) + i p) g^(-1/2), so a node takes one
// logarithm, one exponential and two real-coefficient sums instead of a
// power, an arctangent and eleven sines and cosines.
__device__ inline void lensed_epl_node(const double* ratio, double t, double p, double& wx, double& wy, double& dx,
                                       double& dy)
{
    const double c = 1 - p, g = p * p + c * c, h = 0.5 * (1 - t);
    const double s = exp((h - 0.5) * log(g));  // g^h / |(1-p) + i p|
    double qx, qy;
    lensed_epl_sum(ratio, s * c, s * p, (c * c - p * p) / g, 2 * c * p / g, wx, wy, qx, qy);
    const double lg = h * (4 * p - 2) / g;  // d log(g^h) / dp
    dx = (lg * wx - qy / g) / LENSED_EPL_NT;
    dy = (lg * wy + qx / g) / LENSED_EPL_NT;
}

// the node p = 1, where e^{i psi} = i and z = -1: two alternating sums
__device__ inline void lensed_epl_end(const double* ratio, double t, double& wx, double& wy, double& dx, double& dy)
{
    double c = 1.0, s = 1.0, m = 1.0;
    for (int k = 1; k <= 10; ++k) {
        c *= -ratio[k - 1];
        s += c;
        m += (2 * k + 1) * c;
    }
    wx = 0.0;
    wy = s;
    dx = -m / LENSED_EPL_NT;
    dy = (1 - t) * s / LENSED_EPL_NT;
}

__device__ inline void lensed_epl_node(double q, double t, double p, double& wx, double& wy, double& dx, double& dy)
{
    double ratio[10];
    for (int k = 1; k <= 10; ++k) ratio[k - 1] = lensed_epl_ratio(q, t, k);
    lensed_epl_node(ratio, t, p, wx, wy, dx, dy);
}

// cubic Hermite coefficients (a0, a1, a2, a3) of one interval from the
// values and f-derivatives at its ends
__device__ inline float4 lensed_hermite(double v0, double d0, double v1, double d1)
{
    return make_float4((float)v0, (float)d0, (float)(3 * (v1 - v0) - 2 * d0 - d1), (float)(2 * (v0 - v1) + d0 + d1));
}
