// Direct solve on the coarsest multigrid level (an option beside the
// reference's PCG, linalg/solvers/pcg.hpp): the level's operator, boundary
// rows and fs/fs penalty included, as a dense matrix over the unique node
// components, inverted once per viscosity update by Gauss-Jordan on the GPU
// (no pivoting: the operator is symmetric positive definite), and applied
// per V-cycle as one matrix-vector product.
//
//   unique numbering: uid[copy] = unique node of a node copy; rep[node] = one
//   copy of it.  Unknown 3 u + c is component c of unique node u.
#include <cfloat>
#include <cmath>
#include <string>
#include <vector>

#include "tng_coarse.hpp"
#include "tng_wedge.hpp"

namespace tng {

namespace {

// x = e_(node, comp) on every copy of the node
__global__ __launch_bounds__(256) void unit_vector_kernel(double *x0, double *x1, double *x2, const int32_t *uid,
                                                          int64_t ncopies, int node, int comp)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ncopies) return;
    const bool on = uid[i] == node;
    x0[i] = on && comp == 0 ? 1.0 : 0.0;
    x1[i] = on && comp == 1 ? 1.0 : 0.0;
    x2[i] = on && comp == 2 ? 1.0 : 0.0;
}

// column `col` of the row-major n x n matrix from an applied unit vector
__global__ __launch_bounds__(256) void column_kernel(const double *y0, const double *y1, const double *y2,
                                                     const int32_t *rep, int nu, double *M, int n, int col)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n) return;
    const int u = r / 3, c = r - 3 * u;
    const double *y = c == 0 ? y0 : (c == 1 ? y1 : y2);
    M[(int64_t)r * n + col] = y[rep[u]];
}

// Gauss-Jordan step k, part 1: row k and column k before the step
__global__ __launch_bounds__(256) void gj_copy_kernel(const double *M, int n, int k, double *rowk, double *colk)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    rowk[i] = M[(int64_t)k * n + i];
    colk[i] = M[(int64_t)i * n + k];
}

// part 2: every entry from the saved row and column (in place):
//   (k, k) -> 1 / p, (k, j) -> a_kj / p, (i, k) -> -a_ik / p,
//   (i, j) -> a_ij - a_ik a_kj / p
__global__ __launch_bounds__(256) void gj_update_kernel(double *M, int n, int k, const double *rowk,
                                                        const double *colk)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (int64_t)n * n) return;
    const int i = (int)(e / n), j = (int)(e - (int64_t)i * n);
    const double p = rowk[k];
    double v;
    if (i == k && j == k) v = 1.0 / p;
    else if (i == k) v = rowk[j] / p;
    else if (j == k) v = -colk[i] / p;
    else v = M[e] - colk[i] * (rowk[j] / p);
    M[e] = v;
}

// U = M Z and V = M^T W (n x 3 each, row-major), one thread per row
__global__ __launch_bounds__(256) void proj_vectors_kernel(const double *M, int n, const double *Z, const double *W,
                                                           double *U, double *V)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double u[3] = {0.0, 0.0, 0.0}, v[3] = {0.0, 0.0, 0.0};
    for (int j = 0; j < n; ++j) {
        const double mij = M[(int64_t)i * n + j], mji = M[(int64_t)j * n + i];
        for (int k = 0; k < 3; ++k) {
            u[k] = fma(mij, Z[3 * j + k], u[k]);
            v[k] = fma(mji, W[3 * j + k], v[k]);
        }
    }
    for (int k = 0; k < 3; ++k) {
        U[3 * i + k] = u[k];
        V[3 * i + k] = v[k];
    }
}

struct Proj3 {
    double C[9];  // W^T M Z
};

// M <- P M P with P = I - Z W^T:  M - Z V^T - U W^T + Z C W^T
__global__ __launch_bounds__(256) void proj_update_kernel(double *M, int n, const double *Z, const double *W,
                                                          const double *U, const double *V, const Proj3 c)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (int64_t)n * n) return;
    const int i = (int)(e / n), j = (int)(e - (int64_t)i * n);
    double s = M[e];
    for (int k = 0; k < 3; ++k) s -= Z[3 * i + k] * V[3 * j + k] + U[3 * i + k] * W[3 * j + k];
    for (int k = 0; k < 3; ++k)
        for (int l = 0; l < 3; ++l) s += Z[3 * i + k] * c.C[3 * k + l] * W[3 * j + l];
    M[e] = s;
}

__global__ __launch_bounds__(256) void diag_kernel(const double *M, int n, double *d)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) d[i] = M[(int64_t)i * n + i];
}

template <typename T>
__global__ __launch_bounds__(256) void gather_kernel(const T *r0, const T *r1, const T *r2, const int32_t *rep, int nu,
                                                     double *b)
{
    const int u = blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= nu) return;
    const int64_t i = rep[u];
    b[3 * u] = (double)r0[i];
    b[3 * u + 1] = (double)r1[i];
    b[3 * u + 2] = (double)r2[i];
}

// x = M b, one wave per row, lanes over the columns in a fixed order
__global__ __launch_bounds__(256) void gemv_kernel(const double *M, const double *b, double *x, int n)
{
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= n) return;
    const double *m = M + (int64_t)row * n;
    double s = 0.0;
    for (int j = lane; j < n; j += 64) s = fma(m[j], b[j], s);
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (lane == 0) x[row] = s;
}

template <typename T>
__global__ __launch_bounds__(256) void scatter_kernel(T *e0, T *e1, T *e2, const int32_t *uid, int64_t ncopies,
                                                      const double *x)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ncopies) return;
    const int u = uid[i];
    e0[i] = (T)x[3 * u];
    e1[i] = (T)x[3 * u + 1];
    e2[i] = (T)x[3 * u + 2];
}

unsigned blocks(int64_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace

namespace {

// uid[copy] = unique node of a node copy, rep[node] = its first copy
void number_nodes(const tng_domain &m, std::vector<int32_t> &uid, std::vector<int32_t> &rep)
{
    const int64_t nc = m.nalloc;
    std::vector<int32_t> hidx((size_t)m.halo_maxc * m.halo_n);
    uid.resize(nc);
    rep.clear();
    if (!hidx.empty())
        TNG_HIP_CHECK(hipMemcpy(hidx.data(), m.d_halo_idx.p, hidx.size() * sizeof(int32_t), hipMemcpyDeviceToHost));
    for (int64_t i = 0; i < nc; ++i) uid[i] = (int32_t)i;
    // every copy of a shared node points at the group's first copy
    for (int64_t t = 0; t < m.halo_n; ++t) {
        const int32_t first = hidx[t];
        for (int j = 1; j < m.halo_maxc; ++j) {
            const int32_t c = hidx[(size_t)j * m.halo_n + t];
            if (c >= 0) uid[c] = first;
        }
    }
    std::vector<int32_t> compact(nc, -1);
    for (int64_t i = 0; i < nc; ++i)
        if (uid[i] == i) {
            compact[i] = (int32_t)rep.size();
            rep.push_back((int32_t)i);
        }
    for (int64_t i = 0; i < nc; ++i) uid[i] = compact[uid[i]];
}

void upload(DevBuf &b, const void *src, size_t bytes)
{
    b.alloc(bytes);
    TNG_HIP_CHECK(hipMemcpy(b.p, src, bytes, hipMemcpyHostToDevice));
}

}  // namespace

void CoarseDirect::numbering(const tng_domain &m)
{
    std::vector<int32_t> uid, rep;
    number_nodes(m, uid, rep);
    nu = (int)rep.size();
    n = 3 * nu;
    TNG_REQUIRE(n <= kMaxUnknowns, "direct coarse solve: the coarsest level has " + std::to_string(n) +
                                       " unknowns, more than " + std::to_string(kMaxUnknowns));
    ncopies = m.nalloc;
    upload(d_uid, uid.data(), uid.size() * sizeof(int32_t));
    upload(d_rep, rep.data(), rep.size() * sizeof(int32_t));
    d_M.alloc((size_t)n * n * sizeof(double));
    d_row.alloc(n * sizeof(double));
    d_col.alloc(n * sizeof(double));
    d_b.alloc(n * sizeof(double));
    d_x.alloc(n * sizeof(double));
}

void CoarseDirect::build(tng_operator &A, tng_vector &x, tng_vector &y, bool fp32_levels, hipStream_t s)
{
    TNG_REQUIRE(x.dtype == TNG_F64 && y.dtype == TNG_F64 && x.ncomp == 3 && y.ncomp == 3,
                "direct coarse solve: FP64 work vectors required");
    if (!d_uid.p) numbering(*A.mesh);
    double *M = d_M.as<double>();
    const int32_t *uid = d_uid.as<int32_t>(), *rep = d_rep.as<int32_t>();
    for (int col = 0; col < n; ++col) {
        hipLaunchKernelGGL(unit_vector_kernel, dim3(blocks(ncopies)), dim3(256), 0, s, (double *)x.comp(0),
                           (double *)x.comp(1), (double *)x.comp(2), uid, ncopies, col / 3, col % 3);
        op_apply(A, x, y);
        hipLaunchKernelGGL(column_kernel, dim3(blocks(n)), dim3(256), 0, s, (const double *)y.comp(0),
                           (const double *)y.comp(1), (const double *)y.comp(2), rep, nu, M, n, col);
    }
    for (int k = 0; k < n; ++k) {
        hipLaunchKernelGGL(gj_copy_kernel, dim3(blocks(n)), dim3(256), 0, s, (const double *)M, n, k,
                           d_row.as<double>(), d_col.as<double>());
        hipLaunchKernelGGL(gj_update_kernel, dim3(blocks((int64_t)n * n)), dim3(256), 0, s, M, n, k,
                           (const double *)d_row.p, (const double *)d_col.p);
    }
    TNG_HIP_CHECK(hipGetLastError());
    // the inverse of a symmetric positive definite matrix has a positive,
    // finite diagonal; a vanishing pivot leaves non-finite entries
    hipLaunchKernelGGL(diag_kernel, dim3(blocks(n)), dim3(256), 0, s, (const double *)M, n, d_b.as<double>());
    std::vector<double> diag(n);
    TNG_HIP_CHECK(hipMemcpyAsync(diag.data(), d_b.p, n * sizeof(double), hipMemcpyDeviceToHost, s));
    TNG_HIP_CHECK(hipStreamSynchronize(s));
    for (int i = 0; i < n; ++i)
        TNG_REQUIRE(std::isfinite(diag[i]) && diag[i] > 0.0,
                    "direct coarse solve: the coarsest operator is not positive definite");
    if (A.penalty_active && fp32_levels) project_rotations(*A.mesh, s);
    ready = true;
}

// With the fs/fs penalty the three rigid rotations are near-null modes whose
// inverse gain is 1 / eps.  FP32 levels do not resolve the eps-sized
// penalty, so the rotational part of their restricted residual is rounding
// noise that an exact inverse would amplify: there the coarse correction is
// taken in the rotations' Euclidean complement, M <- P M P with
// P = I - Z (Z^T Z)^{-1} Z^T (Z: the rotations e_k x x at the unique nodes),
// and the rotations are left to the fine levels and the Krylov method.
void CoarseDirect::project_rotations(const tng_domain &m, hipStream_t s)
{
    std::vector<int32_t> rep(nu);
    TNG_HIP_CHECK(hipMemcpy(rep.data(), d_rep.p, nu * sizeof(int32_t), hipMemcpyDeviceToHost));
    std::vector<double> Z((size_t)n * 3), W((size_t)n * 3);
    for (int u = 0; u < nu; ++u) {
        const int64_t i = rep[u], lcol = i / m.nr;
        const int l = (int)(i - lcol * m.nr);
        const int64_t sd = lcol / ((int64_t)m.nx * m.nx);
        const double r = m.radii[sd * m.nr + l];
        const double x[3] = {m.coords[3 * lcol] * r, m.coords[3 * lcol + 1] * r, m.coords[3 * lcol + 2] * r};
        for (int k = 0; k < 3; ++k) {
            // e_k x x, component c at row 3 u + c
            const double e[3] = {k == 0 ? 1.0 : 0.0, k == 1 ? 1.0 : 0.0, k == 2 ? 1.0 : 0.0};
            const double z[3] = {e[1] * x[2] - e[2] * x[1], e[2] * x[0] - e[0] * x[2], e[0] * x[1] - e[1] * x[0]};
            for (int c = 0; c < 3; ++c) Z[(size_t)(3 * u + c) * 3 + k] = z[c];
        }
    }
    // W = Z (Z^T Z)^{-1}
    double G[9] = {0}, Gi[9];
    for (int r = 0; r < n; ++r)
        for (int a = 0; a < 3; ++a)
            for (int b = 0; b < 3; ++b) G[3 * a + b] += Z[(size_t)r * 3 + a] * Z[(size_t)r * 3 + b];
    const double det = G[0] * (G[4] * G[8] - G[5] * G[7]) - G[1] * (G[3] * G[8] - G[5] * G[6]) +
                       G[2] * (G[3] * G[7] - G[4] * G[6]);
    TNG_REQUIRE(std::isfinite(det) && det > 0.0, "direct coarse solve: degenerate rotation fields");
    Gi[0] = (G[4] * G[8] - G[5] * G[7]) / det;
    Gi[1] = (G[2] * G[7] - G[1] * G[8]) / det;
    Gi[2] = (G[1] * G[5] - G[2] * G[4]) / det;
    Gi[3] = (G[5] * G[6] - G[3] * G[8]) / det;
    Gi[4] = (G[0] * G[8] - G[2] * G[6]) / det;
    Gi[5] = (G[2] * G[3] - G[0] * G[5]) / det;
    Gi[6] = (G[3] * G[7] - G[4] * G[6]) / det;
    Gi[7] = (G[1] * G[6] - G[0] * G[7]) / det;
    Gi[8] = (G[0] * G[4] - G[1] * G[3]) / det;
    for (int r = 0; r < n; ++r)
        for (int a = 0; a < 3; ++a) {
            double v = 0.0;
            for (int b = 0; b < 3; ++b) v += Z[(size_t)r * 3 + b] * Gi[3 * b + a];
            W[(size_t)r * 3 + a] = v;
        }
    DevBuf dZ, dW, dU, dV;
    dZ.alloc(Z.size() * sizeof(double));
    dW.alloc(W.size() * sizeof(double));
    dU.alloc(Z.size() * sizeof(double));
    dV.alloc(Z.size() * sizeof(double));
    TNG_HIP_CHECK(hipMemcpyAsync(dZ.p, Z.data(), Z.size() * sizeof(double), hipMemcpyHostToDevice, s));
    TNG_HIP_CHECK(hipMemcpyAsync(dW.p, W.data(), W.size() * sizeof(double), hipMemcpyHostToDevice, s));
    double *M = d_M.as<double>();
    hipLaunchKernelGGL(proj_vectors_kernel, dim3(blocks(n)), dim3(256), 0, s, (const double *)M, n,
                       (const double *)dZ.p, (const double *)dW.p, dU.as<double>(), dV.as<double>());
    std::vector<double> U((size_t)n * 3);
    TNG_HIP_CHECK(hipMemcpyAsync(U.data(), dU.p, U.size() * sizeof(double), hipMemcpyDeviceToHost, s));
    TNG_HIP_CHECK(hipStreamSynchronize(s));
    Proj3 c{};
    for (int a = 0; a < 3; ++a)
        for (int b = 0; b < 3; ++b) {
            double v = 0.0;
            for (int r = 0; r < n; ++r) v += W[(size_t)r * 3 + a] * U[(size_t)r * 3 + b];
            c.C[3 * a + b] = v;
        }
    hipLaunchKernelGGL(proj_update_kernel, dim3(blocks((int64_t)n * n)), dim3(256), 0, s, M, n, (const double *)dZ.p,
                       (const double *)dW.p, (const double *)dU.p, (const double *)dV.p, c);
    TNG_HIP_CHECK(hipGetLastError());
    TNG_HIP_CHECK(hipStreamSynchronize(s));
}

void CoarseDirect::solve(tng_vector &e0, const tng_vector &r0, hipStream_t s)
{
    TNG_REQUIRE(ready, "direct coarse solve: not built");
    const int32_t *uid = d_uid.as<int32_t>(), *rep = d_rep.as<int32_t>();
    double *b = d_b.as<double>(), *x = d_x.as<double>();
    if (r0.dtype == TNG_F64)
        hipLaunchKernelGGL(gather_kernel<double>, dim3(blocks(nu)), dim3(256), 0, s, (const double *)r0.comp(0),
                           (const double *)r0.comp(1), (const double *)r0.comp(2), rep, nu, b);
    else
        hipLaunchKernelGGL(gather_kernel<float>, dim3(blocks(nu)), dim3(256), 0, s, (const float *)r0.comp(0),
                           (const float *)r0.comp(1), (const float *)r0.comp(2), rep, nu, b);
    hipLaunchKernelGGL(gemv_kernel, dim3((n + 3) / 4), dim3(256), 0, s, (const double *)d_M.p, (const double *)b, x, n);
    if (e0.dtype == TNG_F64)
        hipLaunchKernelGGL(scatter_kernel<double>, dim3(blocks(ncopies)), dim3(256), 0, s, (double *)e0.comp(0),
                           (double *)e0.comp(1), (double *)e0.comp(2), uid, ncopies, (const double *)x);
    else
        hipLaunchKernelGGL(scatter_kernel<float>, dim3(blocks(ncopies)), dim3(256), 0, s, (float *)e0.comp(0),
                           (float *)e0.comp(1), (float *)e0.comp(2), uid, ncopies, (const double *)x);
    TNG_HIP_CHECK(hipGetLastError());
}

// ----------------------------------------------------------------------------
// PCG on the assembled coarsest operator.  A coarsest level has a few hundred
// to a few thousand nodes: its PCG is bound by launches and by the chain of
// loads in each kernel, not by bandwidth.  Assembled over the unique nodes the
// halo sum and the boundary handling are in the matrix (1.2 MB at level 2
// against 3.3 MB of wedge matrices, most of which five blocks of gathering
// threads read per apply), and each of an iteration's two reductions ends in
// the next kernel, where every block sums the partials itself.  Level 2 (810
// nodes), Galerkin operator: 8.8 us of kernel time per iteration (5.2 + 3.6; 9.0
// with the gaps, 0.45 ms for 50), 71 us with the
// stored-matrix apply, halo sum and five vector kernels.  Used up to 8192
// nodes (lateral level 3), where the matrix kernel's 10 MB still come from
// cache; above, and with the rotation penalty (a rank-3 term over all nodes),
// the general PCG on the operator's own apply runs.
// ----------------------------------------------------------------------------
namespace {

// The wedge (dxc, dyc, w, rc) around a node copy (X, Y, l), q = 0 .. 11, as the
// lateral cell offsets, the wedge, the radial cell offset and the node's
// lateral corner in it.
__host__ __device__ __forceinline__ void wedge_around(int q, int &dx, int &dy, int &w, int &dr, int &corner)
{
    // lateral triangles around a node: cell offsets, wedge, corner
    constexpr int8_t kT[6][4] = {{0, 0, 0, 0}, {-1, 0, 1, 2}, {-1, 0, 0, 1}, {-1, -1, 1, 0}, {0, -1, 0, 2}, {0, -1, 1, 1}};
    const int t = q >> 1;
    dr = (q & 1) - 1;
    dx = kT[t][0];
    dy = kT[t][1];
    w = kT[t][2];
    corner = kT[t][3];
}

struct CpcgArgs {
    const double *lmat;      // stored wedge matrices, or nullptr: formed from the coefficient
    const double *k, *radii;
    const int32_t *rep, *copy_begin, *copy_list;
    const uint8_t *slot;
    const double *coords;
    const uint8_t *sd_cmb, *sd_surf;
    double *A;  // (node, entry 9, slot)
    const int32_t *col;
    int nu, nx, nr, bc_cmb, bc_surf;
};

// Entry (d1, d2) of the blocks of node i's row of a wedge matrix:
// k |det J| [ (g_i . g_j) d_{d1,d2} + g_i[d2] g_j[d1] - 2/3 g_i[d1] g_j[d2] ].
__device__ __forceinline__ void cpcg_row(const double (&g)[6][3], double jkw, int i, int d1, int d2, double (&m)[6])
{
    auto pick = [](const double *v, int d) { return d == 0 ? v[0] : (d == 1 ? v[1] : v[2]); };
    double gi[3] = {g[0][0], g[0][1], g[0][2]};
#pragma unroll
    for (int n = 1; n < 6; ++n)
#pragma unroll
        for (int c = 0; c < 3; ++c) gi[c] = n == i ? g[n][c] : gi[c];
    const double gi1 = pick(gi, d1), gi2 = pick(gi, d2);
#pragma unroll
    for (int j = 0; j < 6; ++j) {
        const double gg = gi[0] * g[j][0] + gi[1] * g[j][1] + gi[2] * g[j][2];
        m[j] = jkw * ((d1 == d2 ? gg : 0.0) + gi2 * pick(g[j], d1) - (2.0 / 3.0) * gi1 * pick(g[j], d2));
    }
}

// Sum of the wedge matrices' 3 x 3 blocks into the row's slots: four threads per
// (node, entry), each with a quarter of the wedges around the node, sum that
// entry of every slot in LDS.  Without stored matrices the blocks come from the
// coefficient as they are needed.  Bound by the chain of loads and divisions per
// wedge.
__global__ __launch_bounds__(64) void cpcg_assemble_kernel(const CpcgArgs a)
{
    const int t = (blockIdx.x * blockDim.x + threadIdx.x) >> 2, part = threadIdx.x & 3;
    const bool live = t < a.nu * 9;
    const int u = live ? t / 9 : 0, e = t - 9 * u, d1 = e / 3, d2 = e - 3 * d1;
    constexpr int W = CoarsePcg::kWidth;
    __shared__ double rows[64][W + 1];
    double *row = rows[threadIdx.x];
    for (int s = 0; s < W; ++s) row[s] = 0.0;
    const int nx = a.nx, nr = a.nr, nc = nx - 1, ncr = nr - 1;
    for (int j = a.copy_begin[u]; live && j < a.copy_begin[u + 1]; ++j) {
        const int i = a.copy_list[j];
        const int l = i % nr, c = i / nr, Y = c % nx, X = (c / nx) % nx, sd = c / (nx * nx);
        for (int q = part; q < 12; q += 4) {
            int dx, dy, w, dr, corner;
            wedge_around(q, dx, dy, w, dr, corner);
            const int xc = X + dx, yc = Y + dy, rc = l + dr;
            if (xc < 0 || xc >= nc || yc < 0 || yc >= nc || rc < 0 || rc >= ncr) continue;
            const int node = corner + (dr == 0 ? 0 : 3);
            double m[6];
            if (a.lmat) {
                const double *l = a.lmat + (((((int64_t)sd * nc + xc) * nc + yc) * ncr + rc) * 2 + w) * 324 +
                                  (node + 6 * d1) * 18 + 6 * d2;
                for (int k = 0; k < 6; ++k) m[k] = l[k];
            } else {
                double g[6][3], jkw;
                wedge_gradients(a.coords, a.radii, a.k, nx, nr, sd, xc, yc, rc, w, g, &jkw);
                cpcg_row(g, jkw, node, d1, d2, m);
            }
            const uint8_t *sl = a.slot + (int64_t)i * CoarsePcg::kMaxSlots + 6 * q;
            for (int k = 0; k < 6; ++k) row[sl[k]] += m[k];
        }
    }
    __syncthreads();
    if (!live) return;
    const double(*r)[W + 1] = rows + (threadIdx.x & ~3);
    double *out = a.A + ((int64_t)u * 9 + e) * W;
    for (int s = part; s < W; s += 4) out[s] = (r[0][s] + r[1][s]) + (r[2][s] + r[3][s]);
}

// kind of a node: 0 interior or Neumann, else its boundary condition; n its unit normal
__device__ __forceinline__ int cpcg_node_bc(const CpcgArgs &a, int u, double n[3])
{
    const int i = a.rep[u], nx = a.nx, nr = a.nr, l = i % nr, c = i / nr, sd = c / (nx * nx);
    const int bc = l == 0 && a.sd_cmb[sd] ? a.bc_cmb : (l == nr - 1 && a.sd_surf[sd] ? a.bc_surf : TNG_NEUMANN);
    const double *q = a.coords + 3 * (int64_t)c;
    const double mag = sqrt(q[0] * q[0] + q[1] * q[1] + q[2] * q[2]);
    for (int d = 0; d < 3; ++d) n[d] = q[d] / mag;
    return bc;
}

// Boundary rows and columns, per block: Dirichlet rows keep their diagonal
// entries, Dirichlet columns vanish; free slip projects the normal component
// out on both sides and keeps the normal-normal entry of the diagonal block.
__global__ __launch_bounds__(64) void cpcg_boundary_kernel(const CpcgArgs a)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    constexpr int W = CoarsePcg::kWidth;
    if (t >= a.nu * W) return;
    const int u = t / W, s = t - W * u, v = a.col[t];
    if (v < 0) return;
    double nu_[3], nv[3], B[3][3];
    const int bu = cpcg_node_bc(a, u, nu_), bv = cpcg_node_bc(a, v, nv);
    double *row = a.A + (int64_t)u * 9 * W + s;
    for (int e = 0; e < 9; ++e) B[e / 3][e % 3] = row[e * W];
    if (bu == TNG_DIRICHLET || bv == TNG_DIRICHLET) {
        for (int e = 0; e < 9; ++e) row[e * W] = u == v && bu == TNG_DIRICHLET && e % 4 == 0 ? B[e / 3][e / 3] : 0.0;
        return;
    }
    if (bu != TNG_FREESLIP && bv != TNG_FREESLIP) return;
    double ann = 0.0;
    if (u == v)
        for (int e = 0; e < 9; ++e) ann += nu_[e / 3] * B[e / 3][e % 3] * nu_[e % 3];
    if (bv == TNG_FREESLIP)
        for (int i = 0; i < 3; ++i) {
            const double d = B[i][0] * nv[0] + B[i][1] * nv[1] + B[i][2] * nv[2];
            for (int j = 0; j < 3; ++j) B[i][j] -= d * nv[j];
        }
    if (bu == TNG_FREESLIP)
        for (int j = 0; j < 3; ++j) {
            const double d = nu_[0] * B[0][j] + nu_[1] * B[1][j] + nu_[2] * B[2][j];
            for (int i = 0; i < 3; ++i) B[i][j] -= d * nu_[i];
        }
    for (int e = 0; e < 9; ++e) row[e * W] = B[e / 3][e % 3] + (u == v ? ann * nu_[e / 3] * nu_[e % 3] : 0.0);
}

// state: iteration count, the launch that ended the solve (0 while it runs),
// first residual norm, total iterations, then r.r in two slots used in turn
enum { CS_ITERS = 0, CS_DONE, CS_INIT, CS_TOTAL, CS_RR, CS_N = CS_RR + 2 };
constexpr int kCpcgNodes = 16;    // nodes per block of the matrix kernel: 16 lanes each
constexpr int kCpcgMaxParts = 1024;

__device__ __forceinline__ double block_sum256(double v, double *red)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    const double s = (red[0] + red[1]) + (red[2] + red[3]);
    __syncthreads();
    return s;
}
__device__ __forceinline__ double parts_sum(const double *p, int n, double *red)
{
    double v = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) v += p[i];
    return block_sum256(v, red);
}

// Launch numbers within a solve: 2 it for the matrix kernel of iteration it,
// 2 it + 1 for the update kernel.  The block that ends the solve records the
// number while other blocks of the launch may still be reading it: only an
// earlier launch's number ends a block here, so that all threads of a block,
// whichever value they saw, reach the block sums and take the decision there.
__device__ __forceinline__ bool cpcg_ended_before(const double *st, int launch)
{
    const double done = st[CS_DONE];
    return done != 0.0 && done < (double)launch;
}

// r = b, p = 0, x = 0; partials of r.r
template <typename T>
__global__ __launch_bounds__(256) void cpcg_begin_kernel(const Comp3<const T> b, const int32_t *rep, int nu, double *x,
                                                         double *r, double *p, double *parts, double *st)
{
    __shared__ double red[4];
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    double v = 0.0;
    if (t < 3 * nu) {
        const int u = t / 3, c = t - 3 * u;
        v = (double)(c == 0 ? b.p[0] : (c == 1 ? b.p[1] : b.p[2]))[rep[u]];
        r[t] = v;
        p[t] = 0.0;
        x[t] = 0.0;
    }
    const double s = block_sum256(v * v, red);
    if (threadIdx.x == 0) parts[blockIdx.x] = s;
    if (t == 0) {
        st[CS_ITERS] = 0.0;
        st[CS_DONE] = 0.0;
    }
}

// First kernel of iteration it (1, 2, ...): ends the iteration before (r.r, the
// stopping test, beta), forms the direction p = r + beta p_old of the row's own
// and neighbour nodes as it reads them, and A p with the partials of p.(A p).
// Every block combines the partials in one fixed order, so all take the same
// decision; block 0 records it.  16 lanes per row, lane j the slots j, j + 16.
__global__ __launch_bounds__(256) void cpcg_matrix_kernel(const double *A, const int32_t *col, int nu, const double *r,
                                                          const double *p_old, double *p, double *ap, const double *rparts,
                                                          int nrp, double *pparts, double *st, int it, double rtol,
                                                          double atol)
{
    __shared__ double red[4];
    if (cpcg_ended_before(st, 2 * it)) return;
    constexpr int W = CoarsePcg::kWidth;
    const int u = blockIdx.x * kCpcgNodes + (threadIdx.x >> 4), lane = threadIdx.x & 15;
    int v[2];
    double B[2][9];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int s = lane + 16 * k;
        v[k] = u < nu && s < W ? col[u * W + s] : -1;
#pragma unroll
        for (int e = 0; e < 9; ++e) B[k][e] = v[k] >= 0 ? A[((int64_t)u * 9 + e) * W + s] : 0.0;
    }
    const double rr = parts_sum(rparts, nrp, red);
    double beta = 0.0;
    if (it == 1) {
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            const double init = sqrt(rr);
            st[CS_INIT] = init;
            st[CS_RR + 1] = rr;
            if (init < atol) st[CS_DONE] = 2 * it;
        }
        if (sqrt(rr) < atol) return;
    } else {
        const double rr_old = st[CS_RR + ((it - 1) & 1)], res = sqrt(rr);
        const bool stop = res / st[CS_INIT] <= rtol || res < atol || fabs(rr_old) < DBL_MIN;
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            st[CS_RR + (it & 1)] = rr;
            st[CS_ITERS] = it - 1;
            if (stop) {
                st[CS_DONE] = 2 * it;
                st[CS_TOTAL] += it - 1;
            }
        }
        if (stop) return;
        beta = rr / rr_old;
    }
    double y[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < 2; ++k)
        if (v[k] >= 0) {
            double q[3];
#pragma unroll
            for (int c = 0; c < 3; ++c) q[c] = fma(beta, p_old[3 * v[k] + c], r[3 * v[k] + c]);
#pragma unroll
            for (int c = 0; c < 3; ++c) y[c] += B[k][3 * c] * q[0] + B[k][3 * c + 1] * q[1] + B[k][3 * c + 2] * q[2];
        }
    double d = 0.0;
#pragma unroll
    for (int c = 0; c < 3; ++c)
        for (int o = 8; o > 0; o >>= 1) y[c] += __shfl_xor(y[c], o, 16);
    if (u < nu && lane < 3) {
        const double yc = lane == 0 ? y[0] : (lane == 1 ? y[1] : y[2]);
        const double pc = fma(beta, p_old[3 * u + lane], r[3 * u + lane]);
        p[3 * u + lane] = pc;
        ap[3 * u + lane] = yc;
        d = pc * yc;
    }
    const double s = block_sum256(d, red);
    if (threadIdx.x == 0) pparts[blockIdx.x] = s;
}

// Second kernel: alpha, x += alpha p, r -= alpha A p, partials of r.r; the last
// one allowed counts itself (no later kernel runs the test).
__global__ __launch_bounds__(256) void cpcg_update_kernel(int n, double *x, double *r, const double *p, const double *ap,
                                                          const double *pparts, int npp, double *rparts, double *st,
                                                          int it, int max_it)
{
    __shared__ double red[4];
    if (cpcg_ended_before(st, 2 * it + 1)) return;
    const double pap = parts_sum(pparts, npp, red);
    const bool stop = fabs(pap) < DBL_MIN;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t == 0 && (stop || it == max_it)) {
        st[CS_ITERS] = it;
        st[CS_TOTAL] += it;
        if (stop) st[CS_DONE] = 2 * it + 1;
    }
    if (stop) return;
    const double alpha = st[CS_RR + (it & 1)] / pap;
    double rn = 0.0;
    if (t < n) {
        x[t] = fma(alpha, p[t], x[t]);
        rn = fma(-alpha, ap[t], r[t]);
        r[t] = rn;
    }
    const double s = block_sum256(rn * rn, red);
    if (threadIdx.x == 0) rparts[blockIdx.x] = s;
}

}  // namespace

bool CoarsePcg::accepts(const tng_operator &A)
{
    const tng_domain &m = *A.mesh;
    return !A.penalty_active && m.nr >= 3 && m.num_owned <= kMaxNodes;
}

void CoarsePcg::numbering(const tng_domain &m)
{
    std::vector<int32_t> uid, rep;
    number_nodes(m, uid, rep);
    nu = (int)rep.size();
    ncopies = m.nalloc;
    const int nx = m.nx, nr = m.nr, nc = nx - 1, ncr = nr - 1;
    std::vector<int32_t> begin(nu + 1, 0), list(ncopies), col((size_t)nu * kWidth, -1);
    for (int64_t i = 0; i < ncopies; ++i) begin[uid[i] + 1]++;
    for (int u = 0; u < nu; ++u) begin[u + 1] += begin[u];
    std::vector<int32_t> at(begin.begin(), begin.end() - 1);
    for (int64_t i = 0; i < ncopies; ++i) list[at[uid[i]]++] = (int32_t)i;
    std::vector<uint8_t> slot((size_t)ncopies * kMaxSlots, 0);
    static const int WN[2][3][2] = {{{0, 0}, {1, 0}, {0, 1}}, {{1, 1}, {0, 1}, {1, 0}}};
    for (int64_t i = 0; i < ncopies; ++i) {
        const int u = uid[i], l = (int)(i % nr), c = (int)(i / nr), Y = c % nx, X = (c / nx) % nx, sd = c / (nx * nx);
        int32_t *row = &col[(size_t)u * kWidth];
        for (int q = 0; q < 12; ++q) {
            int dx, dy, w, dr, corner;
            wedge_around(q, dx, dy, w, dr, corner);
            const int xc = X + dx, yc = Y + dy, rc = l + dr;
            if (xc < 0 || xc >= nc || yc < 0 || yc >= nc || rc < 0 || rc >= ncr) continue;
            TNG_REQUIRE(xc + WN[w][corner][0] == X && yc + WN[w][corner][1] == Y, "coarse PCG: wedge table");
            for (int k = 0; k < 6; ++k) {
                const int32_t v = uid[m.lin(sd, xc + WN[w][k % 3][0], yc + WN[w][k % 3][1], rc + k / 3)];
                int s = 0;
                while (s < kWidth && row[s] >= 0 && row[s] != v) ++s;
                TNG_REQUIRE(s < kWidth, "coarse PCG: a node with more neighbours than a row holds");
                row[s] = v;
                slot[(size_t)i * kMaxSlots + 6 * q + k] = (uint8_t)s;
            }
        }
    }
    upload(d_uid, uid.data(), uid.size() * sizeof(int32_t));
    upload(d_rep, rep.data(), rep.size() * sizeof(int32_t));
    upload(d_copy_begin, begin.data(), begin.size() * sizeof(int32_t));
    upload(d_copy_list, list.data(), list.size() * sizeof(int32_t));
    upload(d_slot, slot.data(), slot.size());
    upload(d_col, col.data(), col.size() * sizeof(int32_t));
    d_A.alloc((size_t)nu * 9 * kWidth * sizeof(double));
    // x, r, A p, two directions, two sets of partials, the state
    const std::vector<double> zero(CS_N, 0.0);
    d_vec.alloc(((size_t)5 * 3 * nu + 2 * kCpcgMaxParts) * sizeof(double));
    upload(d_state, zero.data(), zero.size() * sizeof(double));
}

void CoarsePcg::build(tng_operator &A, hipStream_t s)
{
    const tng_domain &m = *A.mesh;
    if (!d_uid.p) numbering(m);
    TNG_REQUIRE(A.stored ? A.lmat_dtype == TNG_F64 : A.k && A.k->dtype == TNG_F64,
                "coarse PCG: FP64 matrices or an FP64 coefficient required");
    CpcgArgs a{};
    a.lmat = A.stored ? A.d_lmat.as<double>() : nullptr;
    a.k = A.k ? (const double *)A.k->comp(0) : nullptr;
    a.radii = m.d_radii.as<double>();
    a.rep = d_rep.as<int32_t>();
    a.copy_begin = d_copy_begin.as<int32_t>();
    a.copy_list = d_copy_list.as<int32_t>();
    a.slot = d_slot.as<uint8_t>();
    a.col = d_col.as<int32_t>();
    a.coords = m.d_coords.as<double>();
    a.sd_cmb = m.d_sd_cmb.as<uint8_t>();
    a.sd_surf = m.d_sd_surf.as<uint8_t>();
    a.A = d_A.as<double>();
    a.nu = nu; a.nx = m.nx; a.nr = m.nr; a.bc_cmb = A.bc_cmb; a.bc_surf = A.bc_surf;
    hipLaunchKernelGGL(cpcg_assemble_kernel, dim3((nu * 36 + 63) / 64), dim3(64), 0, s, a);
    hipLaunchKernelGGL(cpcg_boundary_kernel, dim3((nu * kWidth + 63) / 64), dim3(64), 0, s, a);
    TNG_HIP_CHECK(hipGetLastError());
    ready = true;
}

void CoarsePcg::solve(tng_vector &e0, const tng_vector &r0, int max_it, double rtol, double atol, hipStream_t s)
{
    TNG_REQUIRE(ready, "coarse PCG: not built");
    // the host looks for an early end this often; until then the launches of a
    // finished solve return at once
    constexpr int kCheckEvery = 25;
    const int n = 3 * nu, gu = (n + 255) / 256, gm = (nu + kCpcgNodes - 1) / kCpcgNodes;
    double *x = d_vec.as<double>(), *r = x + n, *ap = r + n, *p[2] = {ap + n, ap + 2 * n};
    double *rparts = ap + 3 * n, *pparts = rparts + kCpcgMaxParts, *st = d_state.as<double>();
    TNG_REQUIRE(gm <= kCpcgMaxParts && gu <= kCpcgMaxParts, "coarse PCG: too many blocks");
    const int32_t *uid = d_uid.as<int32_t>(), *rep = d_rep.as<int32_t>();
    auto begin = [&](auto tag) {
        using T = decltype(tag);
        hipLaunchKernelGGL(cpcg_begin_kernel<T>, dim3(gu), dim3(256), 0, s,
                           Comp3<const T>{{(const T *)r0.comp(0), (const T *)r0.comp(1), (const T *)r0.comp(2)}}, rep, nu,
                           x, r, p[0], rparts, st);
    };
    if (r0.dtype == TNG_F64) begin(double());
    else begin(float());
    for (int it = 1; it <= max_it; ++it) {
        hipLaunchKernelGGL(cpcg_matrix_kernel, dim3(gm), dim3(256), 0, s, d_A.as<double>(), d_col.as<int32_t>(), nu, r,
                           p[(it - 1) & 1], p[it & 1], ap, rparts, gu, pparts, st, it, rtol, atol);
        hipLaunchKernelGGL(cpcg_update_kernel, dim3(gu), dim3(256), 0, s, n, x, r, p[it & 1], ap, pparts, gm, rparts, st,
                           it, max_it);
        if (it % kCheckEvery == 0 && it < max_it) {
            double done = 0.0;
            TNG_HIP_CHECK(hipMemcpyAsync(&done, st + CS_DONE, sizeof(double), hipMemcpyDeviceToHost, s));
            TNG_HIP_CHECK(hipStreamSynchronize(s));
            if (done != 0.0) break;
        }
    }
    auto scatter = [&](auto tag) {
        using T = decltype(tag);
        hipLaunchKernelGGL(scatter_kernel<T>, dim3(blocks(ncopies)), dim3(256), 0, s, (T *)e0.comp(0), (T *)e0.comp(1),
                           (T *)e0.comp(2), uid, ncopies, (const double *)x);
    };
    if (e0.dtype == TNG_F64) scatter(double());
    else scatter(float());
    TNG_HIP_CHECK(hipGetLastError());
}

long CoarsePcg::take_iterations(hipStream_t s)
{
    if (!d_state.p) return 0;
    double total = 0.0;
    const double zero = 0.0;
    double *slot = d_state.as<double>() + CS_TOTAL;
    TNG_HIP_CHECK(hipMemcpyAsync(&total, slot, sizeof(double), hipMemcpyDeviceToHost, s));
    TNG_HIP_CHECK(hipMemcpyAsync(slot, &zero, sizeof(double), hipMemcpyHostToDevice, s));
    TNG_HIP_CHECK(hipStreamSynchronize(s));
    return (long)total;
}

}  // namespace tng
