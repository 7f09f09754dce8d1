// Energy equation around the Stokes solve: the SUPG advection-diffusion
// operator of the implicit energy step, its Dirichlet data, the
// temperature-dependent viscosity and the advective time-step bound.
//
// SUPG operator (fe/wedge/operators/shell/unsteady_advection_diffusion_supg.hpp
// :19-49, :240-433; unsteady_advection_diffusion_supg_kerngen.hpp:1-60 for the
// collapsed form): per wedge and point q of the 6-point Felippa rule,
//   dst_i += w_q |det J_q| [ phi_i (m T(q) + dt u(q).grad T(q))
//                            + grad phi_i . (dt kappa grad T(q) + dt tau (u(q).grad T(q)) u(q)) ]
// with T(q), grad T(q) from the wedge's nodal values (boundary-layer values
// removed where the Dirichlet rows are treated), u(q) the interpolated
// velocity and tau the quadrature-weighted mean of supg_tau over the points
// (h = r_2 - r_1).  Boundary-layer rows keep their diagonal entry only; the
// diagonal mode keeps every row's diagonal entry; the lumped mass takes the
// row sums m sum_q w_q |det J_q| phi_i.
//
// Formulation used here.  The Jacobian at lateral point s and radius r is
// [e1, e2, p_s] diag(r, r, h/2) with e1, e2 the triangle's edges and p_s the
// point on it, so its inverse transpose has the columns M0_s / r, M1_s / r,
// M2 / (h/2) and |det J| = |det L| r^2 h/2, where M0_s = (e2 x p_s) / det L,
// M1_s = (p_s x e1) / det L, M2 = (e1 x e2) / det L are lateral data alone.
// With the contravariant velocity (u.M0_s / r, u.M1_s / r, u.M2 / (h/2)) and
// the Gram products M_i.M_j the bilinear form needs no physical gradients:
// the reference-space derivatives of T and of the test functions (three
// numbers per point each) carry everything.  tau depends on the velocity
// only; it comes from a kernel of its own (six square roots, hyperbolic
// tangents and divisions per wedge), once per energy step.
#include <algorithm>

#include "tng_internal.hpp"

namespace tng {

namespace {

__constant__ int kEW[2][6][3] = {{{0, 0, 0}, {1, 0, 0}, {0, 1, 0}, {0, 0, 1}, {1, 0, 1}, {0, 1, 1}},
                                 {{1, 1, 0}, {0, 1, 0}, {1, 0, 0}, {1, 1, 1}, {0, 1, 1}, {1, 0, 1}}};

__device__ double supg_tau_dev(double vel_norm, double kappa, double h, double pe_tol)
{
    const double kappa_virtual = fmax(kappa, 1e-8);
    const double eps_vel = 1e-12;
    if (vel_norm <= eps_vel) return 0.0;
    const double pe = vel_norm * h / (2.0 * kappa_virtual);
    if (pe <= pe_tol) return 0.0;
    const double tau_max = 10.0 * h / fmax(vel_norm, eps_vel);
    const double tau = (h / (2.0 * vel_norm)) * (1.0 / tanh(pe) - 1.0 / pe);
    return tau > tau_max ? tau_max : tau;
}

// Felippa rule: lateral point s has weight 2/3 at corner kPoint[s] and 1/6 at
// the two others, two radial Gauss points, all weights 1/6.
constexpr double kGauss = 0.5773502691896257;

struct SupgArgs {
    const double *src, *u0, *u1, *u2;
    const double *coords, *radii;
    const uint8_t *sd_cmb, *sd_surf;
    const double *tau;    // (cell, wedge), nullptr: no streamline term
    // (lateral cell, side, corner): its share of the treated boundary rows'
    // diagonal entries, read by the gather (bdiag) and written (bshare)
    const double *bdiag;
    double *bshare;
    double *partial;      // (lateral cell, corner, level)
    double *dst;
    double kappa, dt, mass;
    int treat_boundary, lumped, add;
    int bblocks;    // blocks of the cell kernel's grid that form bshare
    int nsd, nx, nr;
    int lr, lc;     // log2 of the radial and lateral cells per subdomain
    int plen, lseg; // entries per (lateral cell, corner), log2 of the cells per radial segment
    int64_t ncell;
};

// Lateral data of one triangle at the three lateral points.
struct SupgGeom {
    double m0[3][3], m1[3][3], g00[3], g01[3], g11[3], g02[3], g12[3];
    double m2[3], g22, det;
};

// The same at one point.
struct SupgPoint {
    double m0[3], m1[3], m2[3], g00, g01, g11, g02, g12, g22, det;
};

// Wedge w of lateral cell col at lateral point s.
__device__ __forceinline__ SupgPoint supg_point(const SupgArgs &a, int64_t col, int w, int s)
{
    const int nc = a.nx - 1;
    const int yc = (int)(col & (nc - 1)), xc = (int)((col >> a.lc) & (nc - 1)), sd = (int)(col >> (2 * a.lc));
    double P[3][3];
    for (int n = 0; n < 3; ++n) {
        const double *c = a.coords + 3 * (((int64_t)sd * a.nx + xc + kEW[w][n][0]) * a.nx + yc + kEW[w][n][1]);
        for (int d = 0; d < 3; ++d) P[n][d] = c[d];
    }
    const int ks = s == 0 ? 1 : (s == 1 ? 2 : 0);
    double e1[3], e2[3], p[3];
    for (int d = 0; d < 3; ++d) {
        e1[d] = P[1][d] - P[0][d];
        e2[d] = P[2][d] - P[0][d];
        const double pk = ks == 0 ? P[0][d] : (ks == 1 ? P[1][d] : P[2][d]);
        p[d] = (P[0][d] + P[1][d] + P[2][d]) * (1.0 / 6.0) + 0.5 * pk;
    }
    auto cross = [](const double *x, const double *y, double *o) {
        o[0] = x[1] * y[2] - x[2] * y[1];
        o[1] = x[2] * y[0] - x[0] * y[2];
        o[2] = x[0] * y[1] - x[1] * y[0];
    };
    auto dot = [](const double *x, const double *y) { return x[0] * y[0] + x[1] * y[1] + x[2] * y[2]; };
    SupgPoint g;
    cross(e1, e2, g.m2);
    cross(e2, p, g.m0);
    cross(p, e1, g.m1);
    const double det = dot(g.m2, p), id = 1.0 / det;
    for (int d = 0; d < 3; ++d) {
        g.m2[d] *= id;
        g.m0[d] *= id;
        g.m1[d] *= id;
    }
    g.g00 = dot(g.m0, g.m0);
    g.g01 = dot(g.m0, g.m1);
    g.g11 = dot(g.m1, g.m1);
    g.g02 = dot(g.m0, g.m2);
    g.g12 = dot(g.m1, g.m2);
    g.g22 = dot(g.m2, g.m2);
    g.det = fabs(det);
    return g;
}

// Fills entry (w, s) of the geometry of lateral cell col.
__device__ __forceinline__ void supg_geometry(const SupgArgs &a, int64_t col, int w, int s, SupgGeom &G)
{
    const SupgPoint g = supg_point(a, col, w, s);
    for (int d = 0; d < 3; ++d) {
        G.m0[s][d] = g.m0[d];
        G.m1[s][d] = g.m1[d];
        if (s == 0) G.m2[d] = g.m2[d];
    }
    G.g00[s] = g.g00;
    G.g01[s] = g.g01;
    G.g11[s] = g.g11;
    G.g02[s] = g.g02;
    G.g12[s] = g.g12;
    if (s == 0) {
        G.g22 = g.g22;
        G.det = g.det;
    }
}

// Diagonal entries of the six rows of one wedge, without the lumped mass.
__device__ __forceinline__ void supg_wedge_diag(const SupgArgs &a, const SupgGeom *geom, int gi, const double (&ub)[3][4],
                                                const double (&ut)[3][4], double r1, double r2, double tau,
                                                double (&db)[3], double (&dt_)[3])
{
    const double gr = 0.5 * (r2 - r1), igr = 1.0 / gr;
    const double mass = a.lumped ? 0.0 : a.mass;
#pragma unroll
    for (int k = 0; k < 3; ++k) db[k] = dt_[k] = 0.0;
#pragma unroll 1
    for (int z = 0; z < 2; ++z) {
        const double zeta = z == 0 ? -kGauss : kGauss;
        const double n0 = 0.5 * (1.0 - zeta), n1 = 0.5 * (1.0 + zeta);
        // the lateral data is read again for each z (an opaque index): kept
        // over the loop it costs 76 registers and with them the occupancy
        asm volatile("" : "+v"(gi));
        const SupgGeom &G = geom[gi];
        const double r = r1 + gr * (1.0 + zeta), ir = 1.0 / r, wz = G.det * r * r * gr * (1.0 / 6.0);
#pragma unroll
        for (int s = 0; s < 3; ++s) {
            const int ks = s == 0 ? 1 : (s == 1 ? 2 : 0);
            double u[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                const double z0 = n0 * ub[d][0] + n1 * ut[d][0], z1 = n0 * ub[d][1] + n1 * ut[d][1],
                             z2 = n0 * ub[d][2] + n1 * ut[d][2];
                u[d] = (z0 + z1 + z2) * (1.0 / 6.0) + 0.5 * (ks == 0 ? z0 : (ks == 1 ? z1 : z2));
            }
            const double al = (u[0] * G.m0[s][0] + u[1] * G.m0[s][1] + u[2] * G.m0[s][2]) * ir;
            const double be = (u[0] * G.m1[s][0] + u[1] * G.m1[s][1] + u[2] * G.m1[s][2]) * ir;
            const double ga = (u[0] * G.m2[0] + u[1] * G.m2[1] + u[2] * G.m2[2]) * igr;
            const double h00 = G.g00[s] * ir * ir, h01 = G.g01[s] * ir * ir, h11 = G.g11[s] * ir * ir,
                         h02 = G.g02[s] * ir * igr, h12 = G.g12[s] * ir * igr, h22 = G.g22 * igr * igr;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const double nl = k == ks ? 2.0 / 3.0 : 1.0 / 6.0;
                const double lx = k == 0 ? -1.0 : (k == 1 ? 1.0 : 0.0), ly = k == 0 ? -1.0 : (k == 2 ? 1.0 : 0.0);
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const double nr = t == 0 ? n0 : n1, dr = t == 0 ? -0.5 : 0.5;
                    const double fx = lx * nr, fy = ly * nr, fz = nl * dr, phi = nl * nr;
                    const double ug = fx * al + fy * be + fz * ga;
                    const double gg = fx * fx * h00 + fy * fy * h11 + fz * fz * h22 +
                                      2.0 * (fx * fy * h01 + fx * fz * h02 + fy * fz * h12);
                    const double v = wz * (mass * phi * phi + a.dt * (a.kappa * gg + ug * phi + tau * ug * ug));
                    if (t == 0) db[k] += v;
                    else dt_[k] += v;
                }
            }
        }
    }
}

// The wedge's action on the nodal values of its three corners, bottom (tb,
// ob) and top (tt, ot); zero_b / zero_t: the Dirichlet columns left out.
__device__ __forceinline__ void supg_wedge_apply(const SupgArgs &a, const SupgGeom *geom, int gi, const double (&Tb)[4],
                                                 const double (&Tt)[4], bool zero_b, bool zero_t,
                                                 const double (&ub)[3][4], const double (&ut)[3][4], double r1,
                                                 double r2, double tau, double (&ob)[3], double (&ot)[3])
{
    double tb[3], tt[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        tb[k] = zero_b ? 0.0 : Tb[k];
        tt[k] = zero_t ? 0.0 : Tt[k];
    }
    const double gr = 0.5 * (r2 - r1), igr = 1.0 / gr;
    const double mass = a.lumped ? 0.0 : a.mass, dk = a.dt * a.kappa, dtau = a.dt * tau;
    const double D[3] = {0.5 * (tt[0] - tb[0]), 0.5 * (tt[1] - tb[1]), 0.5 * (tt[2] - tb[2])};
    const double D6 = (D[0] + D[1] + D[2]) * (1.0 / 6.0);
#pragma unroll 1
    for (int z = 0; z < 2; ++z) {
        const double zeta = z == 0 ? -kGauss : kGauss;
        const double n0 = 0.5 * (1.0 - zeta), n1 = 0.5 * (1.0 + zeta);
        // the lateral data is read again for each z (an opaque index): kept
        // over the loop it costs 76 registers and with them the occupancy
        asm volatile("" : "+v"(gi));
        const SupgGeom &G = geom[gi];
        const double r = r1 + gr * (1.0 + zeta), ir = 1.0 / r, wz = G.det * r * r * gr * (1.0 / 6.0);
        double T[3], u[3][3], U6[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            T[k] = n0 * tb[k] + n1 * tt[k];
#pragma unroll
            for (int d = 0; d < 3; ++d) u[k][d] = n0 * ub[d][k] + n1 * ut[d][k];
        }
#pragma unroll
        for (int d = 0; d < 3; ++d) U6[d] = (u[0][d] + u[1][d] + u[2][d]) * (1.0 / 6.0);
        const double T6 = (T[0] + T[1] + T[2]) * (1.0 / 6.0);
        const double ax = T[1] - T[0], ay = T[2] - T[0];
        double L[3] = {0.0, 0.0, 0.0}, R[3] = {0.0, 0.0, 0.0}, S6 = 0.0, Z6 = 0.0, Fx = 0.0, Fy = 0.0;
#pragma unroll
        for (int s = 0; s < 3; ++s) {
            const int ks = s == 0 ? 1 : (s == 1 ? 2 : 0);
            const double q[3] = {U6[0] + 0.5 * u[ks][0], U6[1] + 0.5 * u[ks][1], U6[2] + 0.5 * u[ks][2]};
            const double al = (q[0] * G.m0[s][0] + q[1] * G.m0[s][1] + q[2] * G.m0[s][2]) * ir;
            const double be = (q[0] * G.m1[s][0] + q[1] * G.m1[s][1] + q[2] * G.m1[s][2]) * ir;
            const double ga = (q[0] * G.m2[0] + q[1] * G.m2[1] + q[2] * G.m2[2]) * igr;
            const double c = D6 + 0.5 * D[ks];
            const double ugT = al * ax + be * ay + ga * c;
            const double S = wz * (mass * (T6 + 0.5 * T[ks]) + a.dt * ugT);
            // diffusive flux in the dual basis: scaled derivatives, then the Gram products
            const double px = ax * ir, py = ay * ir, pz = c * igr, st = dtau * ugT;
            const double fx = wz * (dk * ir * (G.g00[s] * px + G.g01[s] * py + G.g02[s] * pz) + st * al);
            const double fy = wz * (dk * ir * (G.g01[s] * px + G.g11[s] * py + G.g12[s] * pz) + st * be);
            const double fz = wz * (dk * igr * (G.g02[s] * px + G.g12[s] * py + G.g22 * pz) + st * ga);
            Fx += fx;
            Fy += fy;
            S6 += S;
            Z6 += fz;
            L[ks] += 0.5 * S;
            R[ks] += 0.5 * fz;
        }
        S6 *= 1.0 / 6.0;
        Z6 *= 1.0 / 6.0;
        L[0] += S6 - (Fx + Fy);
        L[1] += S6 + Fx;
        L[2] += S6 + Fy;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const double rk = 0.5 * (Z6 + R[k]);
            ob[k] += n0 * L[k] - rk;
            ot[k] += n1 * L[k] + rk;
        }
    }
}

// Row sums of the wedge's mass (lumped mode): the same for the three corners.
__device__ __forceinline__ void supg_lumped_mass(const SupgArgs &a, const SupgGeom &G, double r1, double r2,
                                                 double &mb, double &mt)
{
    const double gr = 0.5 * (r2 - r1);
    mb = mt = 0.0;
    for (int z = 0; z < 2; ++z) {
        const double zeta = z == 0 ? -kGauss : kGauss;
        const double r = r1 + gr * (1.0 + zeta), wz = a.mass * G.det * r * r * gr * (1.0 / 6.0);
        mb += 0.5 * (1.0 - zeta) * wz;
        mt += 0.5 * (1.0 + zeta) * wz;
    }
}

struct SupgCell {
    int64_t col;  // lateral cell
    int rc, xc, yc, sd;
};

__device__ __forceinline__ SupgCell supg_cell_of(const SupgArgs &a, int64_t cell)
{
    const int nc = a.nx - 1;
    SupgCell c;
    c.rc = (int)(cell & ((1 << a.lr) - 1));
    c.col = cell >> a.lr;
    c.yc = (int)(c.col & (nc - 1));
    c.xc = (int)((c.col >> a.lc) & (nc - 1));
    c.sd = (int)(c.col >> (2 * a.lc));
    return c;
}

// One wedge of a lateral cell at one surface (thread = (cell, side, wedge)): the
// diagonal entries of its three corners there, summed over the cell's two
// wedges into its four corner columns.
__device__ __forceinline__ void supg_boundary(const SupgArgs &a, int64_t t)
{
    const int64_t ncol = a.ncell >> a.lr;
    if (t >= 4 * ncol) return;
    const int w = (int)(t & 1), side = (int)((t >> 1) & 1), nx = a.nx, nr = a.nr, nc = nx - 1;
    const int64_t col = t >> 2;
    const int yc = (int)(col & (nc - 1)), xc = (int)((col >> a.lc) & (nc - 1)), sd = (int)(col >> (2 * a.lc));
    if ((side == 0 ? a.sd_cmb[sd] : a.sd_surf[sd]) == 0) return;  // not read there
    const int rc = side == 0 ? 0 : nr - 2;
    const double r1 = a.radii[(int64_t)sd * nr + rc], r2 = a.radii[(int64_t)sd * nr + rc + 1];
    double ub[3][3], ut[3][3], out[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const int64_t i = (((int64_t)sd * nx + xc + kEW[w][j][0]) * nx + yc + kEW[w][j][1]) * nr + rc;
        ub[0][j] = a.u0[i];
        ub[1][j] = a.u1[i];
        ub[2][j] = a.u2[i];
        ut[0][j] = a.u0[i + 1];
        ut[1][j] = a.u1[i + 1];
        ut[2][j] = a.u2[i + 1];
    }
    const double tau = a.tau ? a.tau[2 * ((col << a.lr) + rc) + w] : 0.0;
    const double gr = 0.5 * (r2 - r1), igr = 1.0 / gr;
    // a real loop: unrolled, three points' geometry is live at once
#pragma unroll 1
    for (int s = 0; s < 3; ++s) {
        const int ks = s == 0 ? 1 : (s == 1 ? 2 : 0);
        const SupgPoint g = supg_point(a, col, w, s);
#pragma unroll
        for (int z = 0; z < 2; ++z) {
            const double zeta = z == 0 ? -kGauss : kGauss;
            const double n0 = 0.5 * (1.0 - zeta), n1 = 0.5 * (1.0 + zeta);
            const double r = r1 + gr * (1.0 + zeta), ir = 1.0 / r, wz = g.det * r * r * gr * (1.0 / 6.0);
            double u[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                const double z0 = n0 * ub[d][0] + n1 * ut[d][0], z1 = n0 * ub[d][1] + n1 * ut[d][1],
                             z2 = n0 * ub[d][2] + n1 * ut[d][2];
                u[d] = (z0 + z1 + z2) * (1.0 / 6.0) + 0.5 * (ks == 0 ? z0 : (ks == 1 ? z1 : z2));
            }
            const double al = (u[0] * g.m0[0] + u[1] * g.m0[1] + u[2] * g.m0[2]) * ir;
            const double be = (u[0] * g.m1[0] + u[1] * g.m1[1] + u[2] * g.m1[2]) * ir;
            const double ga = (u[0] * g.m2[0] + u[1] * g.m2[1] + u[2] * g.m2[2]) * igr;
            const double h00 = g.g00 * ir * ir, h01 = g.g01 * ir * ir, h11 = g.g11 * ir * ir, h02 = g.g02 * ir * igr,
                         h12 = g.g12 * ir * igr, h22 = g.g22 * igr * igr;
            const double nr_ = side == 0 ? n0 : n1, dr = side == 0 ? -0.5 : 0.5;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const double nl = k == ks ? 2.0 / 3.0 : 1.0 / 6.0;
                const double lx = k == 0 ? -1.0 : (k == 1 ? 1.0 : 0.0), ly = k == 0 ? -1.0 : (k == 2 ? 1.0 : 0.0);
                const double fx = lx * nr_, fy = ly * nr_, fz = nl * dr, phi = nl * nr_;
                const double ug = fx * al + fy * be + fz * ga;
                const double gg = fx * fx * h00 + fy * fy * h11 + fz * fz * h22 +
                                  2.0 * (fx * fy * h01 + fx * fz * h02 + fy * fz * h12);
                out[k] += wz * (a.mass * (a.lumped ? phi : phi * phi) + a.dt * (a.kappa * gg + ug * phi + tau * ug * ug));
            }
        }
    }
    // corner columns 00, 10, 01, 11: the first wedge's corners are 0, 1, 2, the
    // second's 3, 2, 1.  The wedges sit in neighbouring lanes.
    const double other = __shfl_xor(out[2], 1, 64);
    double *o = a.bshare + (col * 2 + side) * 4;
    o[w == 0 ? 0 : 3] = out[0];
    o[w == 0 ? 1 : 2] = out[1] + other;
}

// One thread per cell (lanes along r), its two wedges together: the eight
// nodes are loaded once, the lateral data of the block's columns is formed
// once per block in LDS.  A corner column's contributions to a node level (the
// cell above as its bottom, the cell below as its top) are summed through LDS,
// so a lateral cell writes four values per level instead of twelve per cell
// (84 MB against 250 MB at level 6), and the gather below reads four.  Bound
// by FP64 arithmetic at two waves per SIMD (221 VGPRs).  Level 6 (2.6 M
// cells): 167 us + 24 us for the gather, against 721 us + 140 us with the
// Jacobian inverse, tau and every row's diagonal formed at each of the six
// points of each wedge and twelve partials per cell; tau takes 257 us, once
// per step.  BND: the first blocks form the treated boundary rows' diagonal (an
// apply outside an energy step).  In the cells' waves every lane would wait for
// the boundary lanes; as a kernel of its own it cannot overlap, and one thread
// per node and side, which evaluates each wedge three times, took 24 us at level
// 4 and 250 us at level 7, 2 layers (a wedge once, in this launch: 1 and 35 us).
template <bool DIAG, bool BND> __global__ __launch_bounds__(256) void supg_cell_kernel(const SupgArgs a)
{
    extern __shared__ double smem[];
    const int tb_ = blockDim.x, ncr = 1 << a.lr;
    SupgGeom *geom = reinterpret_cast<SupgGeom *>(smem);
    if constexpr (BND)
        if ((int)blockIdx.x < a.bblocks) {
            supg_boundary(a, (int64_t)blockIdx.x * tb_ + threadIdx.x);
            return;
        }
    const int64_t cell0 = (int64_t)(blockIdx.x - (BND ? a.bblocks : 0)) * tb_, ncol = a.ncell >> a.lr;
    const int64_t col0 = cell0 >> a.lr;
    const int cols = tb_ > ncr ? tb_ >> a.lr : 1;
    double *tops = smem + cols * 2 * (sizeof(SupgGeom) / sizeof(double));  // (corner, thread)
    for (int t = threadIdx.x; t < cols * 6; t += tb_) {
        const int64_t col = min(col0 + t / 6, ncol - 1);
        supg_geometry(a, col, (t / 3) & 1, t % 3, geom[t / 3]);
    }
    __syncthreads();
    const int64_t cell = min(cell0 + (int64_t)threadIdx.x, a.ncell - 1);
    const bool live = cell0 + threadIdx.x < a.ncell;
    const SupgCell c = supg_cell_of(a, cell);
    const int nx = a.nx, nr = a.nr;
    const double r1 = a.radii[(int64_t)c.sd * nr + c.rc], r2 = a.radii[(int64_t)c.sd * nr + c.rc + 1];
    const bool zero_b = a.treat_boundary && c.rc == 0 && a.sd_cmb[c.sd];
    const bool zero_t = a.treat_boundary && c.rc == ncr - 1 && a.sd_surf[c.sd];
    // corners 00, 10, 01, 11
    double Tb[4], Tt[4], Ub[3][4], Ut[3][4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int64_t i = (((int64_t)c.sd * nx + c.xc + (k & 1)) * nx + c.yc + (k >> 1)) * nr + c.rc;
        Tb[k] = a.src[i];
        Tt[k] = a.src[i + 1];
        Ub[0][k] = a.u0[i];
        Ut[0][k] = a.u0[i + 1];
        Ub[1][k] = a.u1[i];
        Ut[1][k] = a.u1[i + 1];
        Ub[2][k] = a.u2[i];
        Ut[2][k] = a.u2[i + 1];
    }
    double ob[4] = {0, 0, 0, 0}, ot[4] = {0, 0, 0, 0};
    // A real loop over the two wedges: the corners of the second, (3, 2, 1),
    // are those of the first after the four are turned end for end, so one
    // body serves both and its registers are live once (unrolled, the compiler
    // keeps both wedges' lateral data and interpolants: 294 VGPRs, one wave
    // per SIMD).
#pragma unroll 1
    for (int w = 0; w < 2; ++w) {
        const SupgGeom &G = geom[2 * (c.col - col0) + w];
        const double tw = a.tau ? a.tau[2 * cell + w] : 0.0;
        double wb[3] = {0, 0, 0}, wt[3] = {0, 0, 0}, mb = 0.0, mt = 0.0;
        if constexpr (DIAG)
            supg_wedge_diag(a, geom, 2 * (int)(c.col - col0) + w, Ub, Ut, r1, r2, tw, wb, wt);
        else
            supg_wedge_apply(a, geom, 2 * (int)(c.col - col0) + w, Tb, Tt, zero_b, zero_t, Ub, Ut, r1, r2, tw, wb, wt);
        if (a.lumped) supg_lumped_mass(a, G, r1, r2, mb, mt);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            if constexpr (DIAG) {
                ob[k] += (wb[k] + mb) * Tb[k];
                ot[k] += (wt[k] + mt) * Tt[k];
            } else {
                ob[k] += wb[k] + mb * Tb[k];
                ot[k] += wt[k] + mt * Tt[k];
            }
        }
        auto turn = [](auto &v) {
            for (int k = 0; k < 2; ++k) {
                const double t = v[k];
                v[k] = v[3 - k];
                v[3 - k] = t;
            }
        };
        turn(Tb);
        turn(Tt);
        turn(ob);
        turn(ot);
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            turn(Ub[d]);
            turn(Ut[d]);
        }
    }
    // level rc of a corner column: this cell's bottom and the top of the cell
    // below; a segment's first cell has no cell below, its last one also
    // writes the level above
    const int seg = (1 << a.lseg) - 1;
    const bool first = (c.rc & seg) == 0, last = (c.rc & seg) == seg || c.rc == ncr - 1;
#pragma unroll
    for (int k = 0; k < 4; ++k) tops[k * tb_ + threadIdx.x] = ot[k];
    __syncthreads();
    if (!live) return;
    double *o = a.partial + c.col * 4 * a.plen + c.rc + (c.rc >> a.lseg);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        o[(int64_t)k * a.plen] = first ? ob[k] : ob[k] + tops[k * tb_ + threadIdx.x - 1];
        if (last) o[(int64_t)k * a.plen + 1] = ot[k];
    }
}

// Node values from the four lateral cells around a node; treated boundary
// rows are their diagonal entry times the value.
__global__ __launch_bounds__(256) void supg_gather_kernel(const SupgArgs a, const Index4 idx)
{
    const uint32_t n = (uint32_t)a.nsd * a.nx * a.nx * a.nr;
    const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= n) return;
    int sd, X, Y, l;
    idx.decode(gid, sd, X, Y, l);
    const int nc = a.nx - 1, ncr = a.nr - 1;
    const int seg = min(l, ncr - 1) >> a.lseg;
    const bool seam = l < ncr && l > 0 && (l & ((1 << a.lseg) - 1)) == 0;
    double v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int xc = X - (k & 1), yc = Y - (k >> 1);
        v[k] = 0.0;
        if (xc >= 0 && xc < nc && yc >= 0 && yc < nc) {
            const double *p = a.partial + ((((int64_t)sd * nc + xc) * nc + yc) * 4 + k) * a.plen + l + seg;
            v[k] = p[0];
            if (seam) v[k] += p[-1];
        }
    }
    double s = (v[0] + v[1]) + (v[2] + v[3]);
    if (a.bdiag && ((l == 0 && a.sd_cmb[sd]) || (l == ncr && a.sd_surf[sd]))) {
        double b[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int xc = X - (k & 1), yc = Y - (k >> 1);
            const bool in = xc >= 0 && xc < nc && yc >= 0 && yc < nc;
            b[k] = in ? a.bdiag[((((int64_t)sd * nc + xc) * nc + yc) * 2 + (l == 0 ? 0 : 1)) * 4 + k] : 0.0;
        }
        s = ((b[0] + b[1]) + (b[2] + b[3])) * a.src[gid];
    }
    a.dst[gid] = a.add ? a.dst[gid] + s : s;
}

// tau per wedge: one thread per cell, the velocity at the six points.
__global__ __launch_bounds__(256) void supg_tau_kernel(const SupgArgs a, double *tau)
{
    const int64_t cell = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (cell >= a.ncell) return;
    const SupgCell c = supg_cell_of(a, cell);
    const int nx = a.nx, nr = a.nr;
    const double h = a.radii[(int64_t)c.sd * nr + c.rc + 1] - a.radii[(int64_t)c.sd * nr + c.rc];
    double U[2][4][3];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int64_t i = (((int64_t)c.sd * nx + c.xc + (k & 1)) * nx + c.yc + (k >> 1)) * nr + c.rc;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            U[t][k][0] = a.u0[i + t];
            U[t][k][1] = a.u1[i + t];
            U[t][k][2] = a.u2[i + t];
        }
    }
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        constexpr int kC[2][3] = {{0, 1, 2}, {3, 2, 1}};
        double acc = 0.0;
#pragma unroll
        for (int z = 0; z < 2; ++z) {
            const double n0 = z == 0 ? 0.5 * (1.0 + kGauss) : 0.5 * (1.0 - kGauss), n1 = 1.0 - n0;
#pragma unroll
            for (int s = 0; s < 3; ++s) {
                const int ks = s == 0 ? 1 : (s == 1 ? 2 : 0);
                double vn = 0.0;
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    double u = 0.0;
#pragma unroll
                    for (int k = 0; k < 3; ++k)
                        u += (k == ks ? 2.0 / 3.0 : 1.0 / 6.0) * (n0 * U[0][kC[w][k]][d] + n1 * U[1][kC[w][k]][d]);
                    vn += u * u;
                }
                acc += supg_tau_dev(sqrt(vn), a.kappa, h, 1e-08);
            }
        }
        tau[2 * cell + w] = acc * (1.0 / 6.0);
    }
}

// The boundary rows alone (an energy step forms them once for all its applies).
__global__ __launch_bounds__(256) void supg_boundary_kernel(const SupgArgs a)
{
    supg_boundary(a, (int64_t)blockIdx.x * blockDim.x + threadIdx.x);
}

// g: the Dirichlet temperatures at the boundary nodes (CMB first), zero elsewhere
__global__ __launch_bounds__(256) void boundary_values_kernel(double *g, const uint8_t *bmask, double t_cmb,
                                                              double t_surf, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint8_t f = bmask[i], cmb = 2 | 4, surf = 2 | 8;
    g[i] = (f & cmb) == cmb ? t_cmb : ((f & surf) == surf ? t_surf : 0.0);
}

// b = src at the nodes carrying all bits of `flag`, b unchanged elsewhere
__global__ __launch_bounds__(256) void assign_masked_kernel(double *b, const double *src, const uint8_t *bmask,
                                                            uint8_t flag, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if ((bmask[i] & flag) == flag) b[i] = src[i];
}

// eta = rmu^(0.5 - T) (Frank-Kamenetskii, interpolators.hpp:219-244)
__global__ __launch_bounds__(256) void viscosity_fk_kernel(double *eta, const double *temp, double rmu, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    eta[i] = pow(rmu, 0.5 - temp[i]);
}

// per-block max of |u| over all copies; the last kernel combines
__global__ __launch_bounds__(256) void max_magnitude_kernel(const double *u0, const double *u1, const double *u2,
                                                            int64_t n, double *partials)
{
    __shared__ double red[4];
    double m = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        m = fmax(m, sqrt(u0[i] * u0[i] + u1[i] * u1[i] + u2[i] * u2[i]));
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) partials[blockIdx.x] = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
}

__global__ __launch_bounds__(256) void max_final_kernel(const double *partials, int nb, double *out)
{
    __shared__ double red[4];
    double m = 0.0;
    for (int b = threadIdx.x; b < nb; b += blockDim.x) m = fmax(m, partials[b]);
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) *out = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
}

unsigned grid1d(int64_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace

namespace {

int log2_of(int v)
{
    int l = 0;
    while ((1 << l) < v) ++l;
    TNG_REQUIRE((1 << l) == v, "SUPG: cells per subdomain must be a power of 2");
    return l;
}

// cells of one block of the cell kernel: a radial segment of up to 256 cells,
// or up to 64 whole columns (the lateral data of each sits in LDS)
int supg_block(int ncr) { return std::min(256, 64 * ncr); }

SupgArgs supg_args(const tng_operator &op)
{
    const tng_domain &m = *op.mesh;
    TNG_REQUIRE(op.vel && op.vel->mesh == &m && op.vel->ncomp == 3 && op.vel->dtype == TNG_F64,
                "SUPG: the velocity must be an FP64 vector on the operator's mesh");
    SupgArgs a{};
    a.u0 = (const double *)op.vel->comp(0);
    a.u1 = (const double *)op.vel->comp(1);
    a.u2 = (const double *)op.vel->comp(2);
    a.coords = m.d_coords.as<double>();
    a.radii = m.d_radii.as<double>();
    a.sd_cmb = m.d_sd_cmb.as<uint8_t>();
    a.sd_surf = m.d_sd_surf.as<uint8_t>();
    a.kappa = op.supg_kappa;
    a.dt = op.supg_dt;
    a.mass = op.supg_mass_scaling;
    a.treat_boundary = op.supg_treat_boundary ? 1 : 0;
    a.lumped = op.supg_lumped ? 1 : 0;
    a.nsd = m.nsd;
    a.nx = m.nx;
    a.nr = m.nr;
    a.lr = log2_of(m.nr - 1);
    a.lc = log2_of(m.nx - 1);
    a.lseg = std::min(a.lr, 8);
    a.plen = m.nr + ((1 << a.lr) >> a.lseg) - 1;
    a.ncell = (int64_t)m.nsd << (2 * a.lc + a.lr);
    TNG_REQUIRE(a.ncell < (int64_t)1 << 31, "SUPG: cells exceed 32-bit indexing");
    return a;
}

}  // namespace

void supg_tau(const tng_operator &op, double *tau, hipStream_t s)
{
    const SupgArgs a = supg_args(op);
    hipLaunchKernelGGL(supg_tau_kernel, dim3(grid1d(a.ncell)), dim3(256), 0, s, a, tau);
    TNG_HIP_CHECK(hipGetLastError());
}

void supg_boundary_diagonal(const tng_operator &op, const double *tau, double *bdiag, hipStream_t s)
{
    SupgArgs a = supg_args(op);
    a.tau = op.supg_enabled ? tau : nullptr;
    a.bshare = bdiag;
    hipLaunchKernelGGL(supg_boundary_kernel, dim3(grid1d(4 * (a.ncell >> a.lr))), dim3(256), 0, s, a);
    TNG_HIP_CHECK(hipGetLastError());
}

size_t supg_boundary_count(const tng_domain &m) { return (size_t)m.nsd * (m.nx - 1) * (m.nx - 1) * 8; }

size_t supg_tau_count(const tng_domain &m) { return (size_t)m.nsd * (m.nx - 1) * (m.nx - 1) * (m.nr - 1) * 2; }

void supg_apply(tng_operator &op, const tng_vector &src, tng_vector &dst, hipStream_t s)
{
    const tng_domain &m = *op.mesh;
    TNG_REQUIRE(src.dtype == TNG_F64 && m.nr >= 2, "SUPG: FP64 temperature");
    SupgArgs a = supg_args(op);
    // work space: corner partials, then (outside an energy step, which brings
    // its own) tau and the boundary diagonal of this apply's velocity
    const size_t npart = (size_t)(a.ncell >> a.lr) * 4 * a.plen, ntau = supg_tau_count(m), nb = supg_boundary_count(m);
    const bool own_tau = op.supg_enabled && !op.supg_step_tau;
    const bool treat = op.supg_treat_boundary && !op.diagonal;
    const bool own_bdiag = treat && !op.supg_step_bdiag;
    const size_t bytes = (npart + (own_tau ? ntau : 0) + (own_bdiag ? nb : 0)) * sizeof(double);
    if (op.scratch.bytes < bytes) op.scratch.alloc(bytes);
    a.src = (const double *)src.comp(0);
    a.dst = (double *)dst.comp(0);
    a.partial = op.scratch.as<double>();
    a.add = op.apply_mode == TNG_ADD ? 1 : 0;
    if (op.supg_enabled) {
        if (own_tau) supg_tau(op, a.partial + npart, s);
        a.tau = own_tau ? a.partial + npart : op.supg_step_tau;
    }
    const int tb = supg_block(1 << a.lr), cols = std::max(1, tb >> a.lr);
    const size_t lds = (size_t)cols * 2 * sizeof(SupgGeom) + (size_t)tb * 4 * sizeof(double);
    if (treat) {
        double *own = a.partial + npart + (own_tau ? ntau : 0);
        if (own_bdiag) {
            a.bshare = own;
            a.bblocks = (int)((4 * (a.ncell >> a.lr) + tb - 1) / tb);
        }
        a.bdiag = own_bdiag ? own : op.supg_step_bdiag;
    }
    const dim3 grid((unsigned)(a.bblocks + (a.ncell + tb - 1) / tb));
    if (op.diagonal) {
        a.treat_boundary = 0;  // every row keeps its own diagonal entry
        hipLaunchKernelGGL((supg_cell_kernel<true, false>), grid, dim3(tb), lds, s, a);
    } else if (a.bblocks > 0) {
        hipLaunchKernelGGL((supg_cell_kernel<false, true>), grid, dim3(tb), lds, s, a);
    } else {
        hipLaunchKernelGGL((supg_cell_kernel<false, false>), grid, dim3(tb), lds, s, a);
    }
    hipLaunchKernelGGL(supg_gather_kernel, dim3(grid1d(m.nalloc)), dim3(256), 0, s, a, Index4(m.nx, m.nr));
    TNG_HIP_CHECK(hipGetLastError());
    if (op.comm_mode == TNG_COMMUNICATE_ADDITIVELY) launch_halo_sum(m, dst, s);
}

void launch_boundary_values(tng_vector &g, double t_cmb, double t_surf, hipStream_t s)
{
    const tng_domain &m = *g.mesh;
    hipLaunchKernelGGL(boundary_values_kernel, dim3(grid1d(m.nalloc)), dim3(256), 0, s, (double *)g.comp(0),
                       m.d_bmask.as<uint8_t>(), t_cmb, t_surf, m.nalloc);
    TNG_HIP_CHECK(hipGetLastError());
}

void launch_assign_masked(tng_vector &b, const tng_vector &src, uint8_t flag, hipStream_t s)
{
    const tng_domain &m = *b.mesh;
    hipLaunchKernelGGL(assign_masked_kernel, dim3(grid1d(m.nalloc)), dim3(256), 0, s, (double *)b.comp(0),
                       (const double *)src.comp(0), m.d_bmask.as<uint8_t>(), flag, m.nalloc);
    TNG_HIP_CHECK(hipGetLastError());
}

void launch_viscosity_fk(tng_vector &eta, const tng_vector &temp, double rmu, hipStream_t s)
{
    const tng_domain &m = *eta.mesh;
    hipLaunchKernelGGL(viscosity_fk_kernel, dim3(grid1d(m.nalloc)), dim3(256), 0, s, (double *)eta.comp(0),
                       (const double *)temp.comp(0), rmu, m.nalloc);
    TNG_HIP_CHECK(hipGetLastError());
}

double max_vector_magnitude(const tng_vector &u, hipStream_t s)
{
    const tng_domain &m = *u.mesh;
    TNG_REQUIRE(u.ncomp == 3 && u.dtype == TNG_F64, "max |u|: FP64 velocity");
    tng_context &ctx = *m.ctx;
    const int nb = (int)std::min<int64_t>(1024, std::max<int64_t>(1, (m.nalloc + 255) / 256));
    double *part = ctx.red_partials.as<double>(), *out = ctx.red_result.as<double>() + 300;
    hipLaunchKernelGGL(max_magnitude_kernel, dim3(nb), dim3(256), 0, s, (const double *)u.comp(0),
                       (const double *)u.comp(1), (const double *)u.comp(2), m.nalloc, part);
    hipLaunchKernelGGL(max_final_kernel, dim3(1), dim3(256), 0, s, (const double *)part, nb, out);
    TNG_HIP_CHECK(hipGetLastError());
    double v = 0.0;
    TNG_HIP_CHECK(hipMemcpyAsync(&v, out, sizeof(double), hipMemcpyDeviceToHost, s));
    TNG_HIP_CHECK(hipStreamSynchronize(s));
    return v;
}

}  // namespace tng
