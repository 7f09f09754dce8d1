// Coefficient gradient of the viscous operator, the element kernel of the
// viscosity adjoint:  g_i = d(lam^T A(k) u) / d log k_i.
//
// A is linear in the wedge coefficient k_w = mean of the six nodal k, so
//   g_i = (k_i / 6) sum_{wedges w of copy i} Phi_w,   Phi_w = lam_w^T A_w(k=1) u_w,
// summed afterwards over the copies of each node.  With one-point quadrature
// Phi_w = |det J| [2 eps(lam_t) : eps(u_t) - 2/3 div lam_t div u_t] on the
// boundary-modified trial and test values (Dirichlet: boundary values removed;
// free slip: tangential projection), plus the wedge's share of the boundary
// rows: Dirichlet  lam_b . diag_b u_b,  diag_b[d] = |det J| (|g_b|^2 + g_b[d]^2/3);
// free slip  (n.lam_b)(n.u_b) |det J| (|g_b|^2 + (g_b.n)^2/3).
// Two passes, no atomics: Phi per wedge (and the boundary rows' share) into
// scratch, then a per-node gather.
#include "tng_internal.hpp"

namespace tng {

namespace {

// Blocks of one XCD take neighbouring items (their node columns meet in its L2).
__device__ __forceinline__ uint32_t xcd_block(uint32_t b, uint32_t nb)
{
    const uint32_t x = b & 7, i = b >> 3, q = nb >> 3, r = nb & 7;
    return x * q + min(x, r) + i;
}

struct PhiArgs {
    const double *u[3], *l[3];
    const double *coords, *radii, *latgeom;
    const uint8_t *sd_cmb, *sd_surf;
    double2 *phi;  // (nsd, nc, nc, ncr), the two wedges of a cell side by side
    double *bphi;  // (2, nsd, nc, nc, 2): the boundary rows' share of the first and last radial cell
    int bblocks;   // blocks of the boundary rows
    int nsd, nx, nr, bc_cmb, bc_surf;
    int rows, nchunk;  // cell rows a thread sweeps, threads per cell column line
    FastDiv dr, dchunk, dcol;
};

// i / f.d where n (the number of items) may exceed 32 bits
__device__ __forceinline__ uint32_t div_any(const FastDiv &f, int64_t i, int64_t n)
{
    return n <= 0x7fffffff ? f.div((uint32_t)i) : (uint32_t)(i / f.d);
}

// The boundary rows' share, one thread per wedge of a boundary cell.  Apart
// from the sweep, whose waves hold a boundary lane each and would all wait for
// it (164 us for the whole gradient at level 6 with them in the sweep, 115 with a
// launch of its own, 111 so); these blocks come first in the sweep's grid.
__device__ void phi_boundary(const PhiArgs &a, int64_t block)
{
    const int nx = a.nx, nr = a.nr, nc = nx - 1, ncr = nr - 1;
    const int64_t n = (int64_t)a.nsd * nc * nc * 4;
    const int64_t gid = block * blockDim.x + threadIdx.x;
    if (gid >= n) return;
    const int w = (int)(gid & 1), layer = (int)((gid >> 1) & 1);
    const int64_t cell = gid >> 2;
    const uint32_t t = a.dcol.div((uint32_t)cell);
    const int yc = (int)((uint32_t)cell - t * nc);
    const int sd = (int)a.dcol.div(t);
    const int xc = (int)(t - (uint32_t)sd * nc);
    const int cbc = (layer == 0 ? a.sd_cmb[sd] : a.sd_surf[sd]) == 0 ? TNG_NEUMANN : (layer == 0 ? a.bc_cmb : a.bc_surf);
    double *out = a.bphi + ((int64_t)layer * (n >> 2) + cell) * 2 + w;
    if (cbc == TNG_NEUMANN) {
        *out = 0.0;
        return;
    }
    const int rc = layer == 0 ? 0 : ncr - 1;
    const double r0 = a.radii[(int64_t)sd * nr + rc], r1 = a.radii[(int64_t)sd * nr + rc + 1];
    const double rmid = 0.5 * (r0 + r1), h = 0.5 * (r1 - r0), vol = rmid * rmid * h;
    const double s = 0.5 / rmid, dz = 1.0 / (6.0 * h), sdz = layer == 0 ? -dz : dz;
    double g[10], uu[3][3], ll[3][3], nn[3][3];
#pragma unroll
    for (int v = 0; v < 10; ++v) g[v] = a.latgeom[cell * 20 + 10 * w + v];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const int dx = c == 1 ? 1 - w : w, dy = c == 2 ? 1 - w : w;
        const int64_t col = ((int64_t)sd * nx + xc + dx) * nx + yc + dy;
        const int64_t i = col * nr + rc + layer;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            uu[c][d] = a.u[d][i];
            ll[c][d] = a.l[d][i];
            nn[c][d] = a.coords[3 * col + d];
        }
    }
    double bt = 0.0;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const double xi = c == 0 ? -1.0 : (c == 1 ? 1.0 : 0.0), eta = c == 0 ? -1.0 : (c == 2 ? 1.0 : 0.0);
        double gj[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) gj[d] = s * (xi * g[d] + eta * g[3 + d]) + sdz * g[6 + d];
        const double gg = gj[0] * gj[0] + gj[1] * gj[1] + gj[2] * gj[2];
        if (cbc == TNG_DIRICHLET) {
#pragma unroll
            for (int d = 0; d < 3; ++d) bt += ll[c][d] * (gg + gj[d] * gj[d] * (1.0 / 3.0)) * uu[c][d];
        } else {
            const double *m = nn[c];
            const double un = m[0] * uu[c][0] + m[1] * uu[c][1] + m[2] * uu[c][2];
            const double ln = m[0] * ll[c][0] + m[1] * ll[c][1] + m[2] * ll[c][2];
            const double gn = gj[0] * m[0] + gj[1] * m[1] + gj[2] * m[2];
            bt += ln * un * (gg + gn * gn * (1.0 / 3.0));
        }
    }
    *out = (g[9] * vol) * bt;
}

// One radial cell of the column (xc, y) per thread, swept over `rows` values of
// y.  A wedge sees a field only through S = bottom + top and D = top - bottom of
// its three node columns,
//   grad = [ (S_1 - S_0) (x) G_0 + (S_2 - S_0) (x) G_1 ] / (2 r_mid) + sum_k D_k (x) G_2 / (6h),
// 27 products a wedge instead of the 108 of six node gradients; S and D of the
// row shared by two cells stay in registers, so that each cell reads two node
// columns.  The lateral geometry and normals are scalars where a wave stays in one
// column (radial cells a multiple of 64): 129 VGPRs, three waves per SIMD, against
// 198.  Bound by the latency of a row's loads (two more registers for a fourth
// wave spill, loads one row ahead gain nothing).  Level 6, 64 layers, both
// kernels and the halo sum: 172 us with six node gradients per wedge and 64-bit
// index divisions, 104 us as swept with vector geometry, 91 us so.
template <bool UNIFORM> __global__ __launch_bounds__(256) void phi_kernel(const PhiArgs a)
{
    const int nx = a.nx, nr = a.nr, nc = nx - 1, ncr = nr - 1;
    const int64_t n = (int64_t)a.nsd * nc * a.nchunk * ncr;
    if (blockIdx.x < (unsigned)a.bblocks) {
        phi_boundary(a, blockIdx.x);
        return;
    }
    const int64_t gid = (int64_t)xcd_block(blockIdx.x - a.bblocks, gridDim.x - a.bblocks) * blockDim.x + threadIdx.x;
    if (gid >= n) return;
    uint32_t t = div_any(a.dr, gid, n);
    const int rc = (int)(gid - (int64_t)t * ncr);
    const uint32_t t2 = a.dchunk.div(t);
    const int chunk = (int)(t - t2 * a.nchunk);
    const int sd = (int)a.dcol.div(t2);
    const int xc = (int)(t2 - (uint32_t)sd * nc);
    // the node column line (sd, xc) at y = 0, and the cells', as the index that the
    // lateral tables are read with
    int64_t col0 = ((int64_t)sd * nx + xc) * nx, cell0 = ((int64_t)sd * nc + xc) * nc;
    int y0 = chunk * a.rows;
    using CD = const double __attribute__((address_space(4)));
    if constexpr (UNIFORM) {
        col0 = __builtin_amdgcn_readfirstlane((int)col0);
        cell0 = __builtin_amdgcn_readfirstlane((int)cell0);
        y0 = __builtin_amdgcn_readfirstlane(y0);
    }
    int layer = -1, cbc = TNG_NEUMANN;
    if (rc == 0 && a.sd_cmb[sd] != 0) { layer = 0; cbc = a.bc_cmb; }
    else if (rc + 1 == nr - 1 && a.sd_surf[sd] != 0) { layer = 1; cbc = a.bc_surf; }
    const bool any_fs = a.bc_cmb == TNG_FREESLIP || a.bc_surf == TNG_FREESLIP;
    const bool any_dir = a.bc_cmb == TNG_DIRICHLET || a.bc_surf == TNG_DIRICHLET;
    const double f_lo = layer == 0 && cbc == TNG_FREESLIP ? 1.0 : 0.0, f_hi = layer == 1 && cbc == TNG_FREESLIP ? 1.0 : 0.0;
    const bool dir_lo = layer == 0 && cbc == TNG_DIRICHLET, dir_hi = layer == 1 && cbc == TNG_DIRICHLET;
    const double r0 = a.radii[(int64_t)sd * nr + rc], r1 = a.radii[(int64_t)sd * nr + rc + 1];
    const double rmid = 0.5 * (r0 + r1), h = 0.5 * (r1 - r0), vol = rmid * rmid * h;
    const double s = 0.5 / rmid, dz = 1.0 / (6.0 * h);
    const int y1 = min(y0 + a.rows, nc);

    // S and D of both fields on a node column, boundary values modified
    auto node = [&](int X, int Y, double (&S)[6], double (&D)[6]) {
        const int64_t col = col0 + X * nx + Y;
        const int64_t i = col * nr + rc;
        double lo[6], hi[6];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            lo[d] = a.u[d][i];
            hi[d] = a.u[d][i + 1];
            lo[3 + d] = a.l[d][i];
            hi[3 + d] = a.l[d][i + 1];
        }
        if (any_fs) {
            // the lanes' factors are 0 or 1; the column's normal is loaded by all
            double n0, n1, n2;
            if constexpr (UNIFORM) {
                CD *c = reinterpret_cast<CD *>(reinterpret_cast<uintptr_t>(a.coords + 3 * col));
                n0 = c[0]; n1 = c[1]; n2 = c[2];
            } else {
                n0 = a.coords[3 * col]; n1 = a.coords[3 * col + 1]; n2 = a.coords[3 * col + 2];
            }
#pragma unroll
            for (int f = 0; f < 6; f += 3) {
                const double dl = f_lo * (n0 * lo[f] + n1 * lo[f + 1] + n2 * lo[f + 2]);
                const double dh = f_hi * (n0 * hi[f] + n1 * hi[f + 1] + n2 * hi[f + 2]);
                lo[f] -= dl * n0; lo[f + 1] -= dl * n1; lo[f + 2] -= dl * n2;
                hi[f] -= dh * n0; hi[f + 1] -= dh * n1; hi[f + 2] -= dh * n2;
            }
        }
        if (any_dir) {
#pragma unroll
            for (int d = 0; d < 6; ++d) {
                lo[d] = dir_lo ? 0.0 : lo[d];
                hi[d] = dir_hi ? 0.0 : hi[d];
            }
        }
#pragma unroll
        for (int d = 0; d < 6; ++d) {
            S[d] = lo[d] + hi[d];
            D[d] = hi[d] - lo[d];
        }
    };

    double S[2][2][6], D[2][2][6];  // [x - xc][y - yc]
    node(0, y0, S[0][0], D[0][0]);
    node(1, y0, S[1][0], D[1][0]);
    for (int yc = y0; yc < y1; ++yc) {
        double G[20];
        const int64_t cell = cell0 + yc;
        if constexpr (UNIFORM) {
            CD *gp = reinterpret_cast<CD *>(reinterpret_cast<uintptr_t>(a.latgeom + cell * 20));
#pragma unroll
            for (int v = 0; v < 20; ++v) G[v] = gp[v];
        } else {
            const double2 *gp = reinterpret_cast<const double2 *>(a.latgeom + cell * 20);
#pragma unroll
            for (int v = 0; v < 10; ++v) {
                const double2 g2 = gp[v];
                G[2 * v] = g2.x;
                G[2 * v + 1] = g2.y;
            }
        }
        node(0, yc + 1, S[0][1], D[0][1]);
        node(1, yc + 1, S[1][1], D[1][1]);
        double res[2];
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            // wedge 0: (0,0), (1,0), (0,1); wedge 1: (1,1), (0,1), (1,0)
            const double *g = G + 10 * w;
            const double(&S0)[6] = S[w][w], (&S1)[6] = S[1 - w][w], (&S2)[6] = S[w][1 - w];
            const double(&D0)[6] = D[w][w], (&D1)[6] = D[1 - w][w], (&D2)[6] = D[w][1 - w];
            double M[6][3];
#pragma unroll
            for (int p = 0; p < 6; ++p) {
                const double e1 = s * (S1[p] - S0[p]), e2 = s * (S2[p] - S0[p]), e3 = dz * (D0[p] + D1[p] + D2[p]);
#pragma unroll
                for (int q = 0; q < 3; ++q) M[p][q] = e1 * g[q] + e2 * g[3 + q] + e3 * g[6 + q];
            }
            double dc = 0.0;
#pragma unroll
            for (int p = 0; p < 3; ++p)
#pragma unroll
                for (int q = 0; q < 3; ++q) dc += M[3 + p][q] * (M[p][q] + M[q][p]);
            const double divu = M[0][0] + M[1][1] + M[2][2], divl = M[3][0] + M[4][1] + M[5][2];
            res[w] = (g[9] * vol) * (dc - (2.0 / 3.0) * divl * divu);
        }
        a.phi[cell * ncr + rc] = make_double2(res[0], res[1]);
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int d = 0; d < 6; ++d) {
                S[x][0][d] = S[x][1][d];
                D[x][0][d] = D[x][1][d];
            }
    }
}

// The six wedges on each radial side of a node: loads independent of each
// other, masked where the cell does not exist.
__global__ __launch_bounds__(256) void phi_gather_kernel(const double2 *phi, const double2 *bphi, const double *k, double *g,
                                                         int nsd, int nx, int nr, const FastDiv dr, const FastDiv dx)
{
    const int64_t n = (int64_t)nsd * nx * nx * nr;
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= n) return;
    const uint32_t col = div_any(dr, gid, n);
    const int l = (int)(gid - (int64_t)col * nr);
    const uint32_t t = dx.div(col);
    const int Y = (int)(col - t * nx);
    const int sd = (int)dx.div(t);
    const int X = (int)(t - (uint32_t)sd * nx);
    const int nc = nx - 1, ncr = nr - 1;
    double2 v[2][2][2];  // [xc - X + 1][yc - Y + 1][rc - l + 1]
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int xc = X - 1 + (i >> 2), yc = Y - 1 + ((i >> 1) & 1), rc = l - 1 + (i & 1);
        const bool in = (unsigned)xc < (unsigned)nc && (unsigned)yc < (unsigned)nc && (unsigned)rc < (unsigned)ncr;
        const int64_t cell = (((int64_t)sd * nc + xc) * nc + yc) * ncr + rc;
        const double2 q = phi[in ? cell : 0];
        v[i >> 2][(i >> 1) & 1][i & 1] = in ? q : make_double2(0.0, 0.0);
    }
    double s = 0.0;
    s += v[0][0][0].y; s += v[0][0][1].y;
    s += v[0][1][0].x; s += v[0][1][1].x;
    s += v[0][1][0].y; s += v[0][1][1].y;
    s += v[1][0][0].x; s += v[1][0][1].x;
    s += v[1][0][0].y; s += v[1][0][1].y;
    s += v[1][1][0].x; s += v[1][1][1].x;
    if (bphi) {
        const int64_t nlat = (int64_t)nsd * nc * nc;
#pragma unroll
        for (int layer = 0; layer < 2; ++layer) {
            if (!(layer == 0 ? l <= 1 : l >= nr - 2)) continue;
            double2 b[2][2];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int xc = X - 1 + (i >> 1), yc = Y - 1 + (i & 1);
                const bool in = (unsigned)xc < (unsigned)nc && (unsigned)yc < (unsigned)nc;
                const double2 q = bphi[in ? layer * nlat + ((int64_t)sd * nc + xc) * nc + yc : 0];
                b[i >> 1][i & 1] = in ? q : make_double2(0.0, 0.0);
            }
            s += b[0][0].y + b[0][1].x + b[0][1].y + b[1][0].x + b[1][0].y + b[1][1].x;
        }
    }
    g[gid] = s * k[gid] * (1.0 / 6.0);
}

}  // namespace

void epsdivdiv_log_k_gradient(tng_operator &op, const tng_vector &lam, const tng_vector &u, tng_vector &g,
                              hipStream_t s)
{
    const tng_domain &m = *op.mesh;
    TNG_REQUIRE(op.kind == OP_EPSDIVDIV, "coefficient gradient of the viscous operator only");
    TNG_REQUIRE(op.k->dtype == TNG_F64 && lam.dtype == TNG_F64 && u.dtype == TNG_F64 && g.dtype == TNG_F64,
                "coefficient gradient: FP64 operator and vectors");
    TNG_REQUIRE(lam.mesh == &m && u.mesh == &m && g.mesh == &m && lam.ncomp == 3 && u.ncomp == 3 && g.ncomp == 1,
                "coefficient gradient: lam, u (velocity) and g (scalar) on the operator's mesh");
    TNG_REQUIRE(m.nr >= 3, "coefficient gradient: at least two radial layers");
    const int64_t ncell = (int64_t)m.nsd * (m.nx - 1) * (m.nx - 1) * (m.nr - 1);
    // Phi per wedge, then the boundary rows' share of the first and last radial cells
    const size_t bytes = ((size_t)ncell * 2 + (size_t)m.nsd * (m.nx - 1) * (m.nx - 1) * 4) * sizeof(double);
    if (op.scratch.bytes < bytes) op.scratch.alloc(bytes);
    PhiArgs a{};
    for (int d = 0; d < 3; ++d) {
        a.u[d] = (const double *)u.comp(d);
        a.l[d] = (const double *)lam.comp(d);
    }
    a.coords = m.d_coords.as<double>(); a.radii = m.d_radii.as<double>(); a.latgeom = m.d_latgeom.as<double>();
    a.sd_cmb = m.d_sd_cmb.as<uint8_t>(); a.sd_surf = m.d_sd_surf.as<uint8_t>();
    a.phi = op.scratch.as<double2>();
    a.nsd = m.nsd; a.nx = m.nx; a.nr = m.nr; a.bc_cmb = op.bc_cmb; a.bc_surf = op.bc_surf;
    const int nc = m.nx - 1, ncr = m.nr - 1;
    const int64_t line = (int64_t)m.nsd * nc * ncr;
    // rows per thread: 8 (16: 93 us against 91) unless that leaves few waves
    a.rows = 8;
    while (a.rows > 1 && line * ((nc + a.rows - 1) / a.rows) < (int64_t)4096 * 64) a.rows /= 2;
    a.nchunk = (nc + a.rows - 1) / a.rows;
    a.dr = FastDiv((uint32_t)ncr); a.dchunk = FastDiv((uint32_t)a.nchunk); a.dcol = FastDiv((uint32_t)nc);
    const int64_t nthr = line * a.nchunk;
    const bool bnd = op.bc_cmb != TNG_NEUMANN || op.bc_surf != TNG_NEUMANN;
    a.bphi = op.scratch.as<double>() + ncell * 2;
    a.bblocks = bnd ? (int)(((int64_t)m.nsd * nc * nc * 4 + 255) / 256) : 0;
    const dim3 grid((unsigned)(a.bblocks + (nthr + 255) / 256));
    // whole waves in one column: its lateral geometry as scalars
    if (ncr % 64 == 0) hipLaunchKernelGGL(phi_kernel<true>, grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL(phi_kernel<false>, grid, dim3(256), 0, s, a);
    TNG_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(phi_gather_kernel, dim3((unsigned)((m.nalloc + 255) / 256)), dim3(256), 0, s,
                       op.scratch.as<double2>(), bnd ? reinterpret_cast<const double2 *>(a.bphi) : nullptr,
                       (const double *)op.k->comp(0), (double *)g.comp(0), m.nsd, m.nx, m.nr, FastDiv((uint32_t)m.nr), FastDiv((uint32_t)m.nx));
    TNG_HIP_CHECK(hipGetLastError());
    launch_halo_sum(m, g, s);
}

}  // namespace tng
