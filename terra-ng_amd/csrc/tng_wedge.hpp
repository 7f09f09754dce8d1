// Geometry of a wedge for the kernels that form local matrices (device code).
#pragma once

#include "tng_internal.hpp"

namespace tng {

namespace {

// wedge node n = lateral corner n % 3 (kWN offsets), radial n / 3
__constant__ int kWN[2][3][2] = {{{0, 0}, {1, 0}, {0, 1}}, {{1, 1}, {0, 1}, {1, 0}}};

// Geometry of one wedge at the centroid: |det J| k_eval and the six physical
// gradients (wedge node order: bottom corners 0..2, top corners 3..5).
__device__ __forceinline__ void wedge_gradients(const double *coords, const double *radii, const double *k, int nx, int nr, int sd,
                                int xc, int yc, int rc, int w, double g[6][3], double *jkw)
{
    double p[3][3];
    for (int c = 0; c < 3; ++c) {
        const double *q = coords + 3 * (((int64_t)sd * nx + xc + kWN[w][c][0]) * nx + yc + kWN[w][c][1]);
        p[c][0] = q[0]; p[c][1] = q[1]; p[c][2] = q[2];
    }
    const double r0 = radii[(int64_t)sd * nr + rc], r1 = radii[(int64_t)sd * nr + rc + 1];
    const double rmid = 0.5 * (r0 + r1), h = 0.5 * (r1 - r0);
    double J[3][3];
    for (int i = 0; i < 3; ++i) {
        J[i][0] = rmid * (p[1][i] - p[0][i]);
        J[i][1] = rmid * (p[2][i] - p[0][i]);
        J[i][2] = h * ((p[0][i] + p[1][i] + p[2][i]) * (1.0 / 3.0));
    }
    const double det = J[0][0] * (J[1][1] * J[2][2] - J[1][2] * J[2][1]) -
                       J[0][1] * (J[1][0] * J[2][2] - J[1][2] * J[2][0]) +
                       J[0][2] * (J[1][0] * J[2][1] - J[1][1] * J[2][0]);
    const double id = 1.0 / det;
    // (J^{-T})_{ab} = cof(J)_{ab} / det
    double iT[3][3];
    iT[0][0] = id * (J[1][1] * J[2][2] - J[1][2] * J[2][1]);
    iT[0][1] = id * (J[1][2] * J[2][0] - J[1][0] * J[2][2]);
    iT[0][2] = id * (J[1][0] * J[2][1] - J[1][1] * J[2][0]);
    iT[1][0] = id * (J[0][2] * J[2][1] - J[0][1] * J[2][2]);
    iT[1][1] = id * (J[0][0] * J[2][2] - J[0][2] * J[2][0]);
    iT[1][2] = id * (J[0][1] * J[2][0] - J[0][0] * J[2][1]);
    iT[2][0] = id * (J[0][1] * J[1][2] - J[0][2] * J[1][1]);
    iT[2][1] = id * (J[0][2] * J[1][0] - J[0][0] * J[1][2]);
    iT[2][2] = id * (J[0][0] * J[1][1] - J[0][1] * J[1][0]);
    // reference gradients at (1/3, 1/3, 0)
    const double dxi[3] = {-0.5, 0.5, 0.0}, deta[3] = {-0.5, 0.0, 0.5};
    double ks = 0.0;
    for (int n = 0; n < 6; ++n) {
        const int c = n % 3, e = n / 3;
        const double dz = e == 0 ? -1.0 / 6.0 : 1.0 / 6.0;
        for (int a = 0; a < 3; ++a) g[n][a] = iT[a][0] * dxi[c] + iT[a][1] * deta[c] + iT[a][2] * dz;
        ks += k[(((int64_t)sd * nx + xc + kWN[w][c][0]) * nx + yc + kWN[w][c][1]) * nr + rc + e];
    }
    *jkw = (ks * (1.0 / 6.0)) * fabs(det);
}

}  // namespace

}  // namespace tng
