// EpsilonDivDiv apply for meshes of 4 to 32 radial layers that do not fill the
// chip (fan_pays; the small multigrid levels), halo sum and Chebyshev sub-step
// included: one launch for what the sweeping apply, the halo sum and the
// vector update do in three (the discretisation and its references are those
// of kernels_epsdivdiv.hip).  Sub-step of the smoother, FP32 no-slip: level 3
// 20.8 -> 6.6 us, level 4 22 -> 7.3 us, level 5 31.7 -> 20.4 us; FP64: level 3
// 19 -> 8.6 us, level 4 20 -> 11.5 us.  Apply with halo sum alone, level 4 FP64:
// 13.5 -> 7.6 us.
//
// What bounds these sizes is not arithmetic or bandwidth but launches and the
// chain inside one: a sweep over a row of cells is a serial loop of loads,
// exchange and barrier, 8 to 33 steps long, with few workgroups to hide it.
// Here a group of R lanes (one radial cell each) owns one lateral node copy and
// evaluates the fan of the up to six triangles around it in its subdomain, all
// loads independent.  A triangle is evaluated once per corner (three times in
// all), which pays while the chip is not full; only the centre's contribution
// is formed (tau . grad lambda_centre), so an evaluation is about 70 instead of
// 88 operations.  The copies of a shared node are laid out in one block (the
// task table of the mesh): their partial results meet in LDS, where every copy
// takes the sum in ascending copy order and finishes its own entry.
#include "tng_internal.hpp"

namespace tng {

namespace {

template <typename T> struct FanArgs {
    const T *src[3];
    T *dst[3];  // A x; with the sub-step: x + d
    const T *k, *latgeom, *coords, *btab;
    const double *radii;  // FP64
    const uint8_t *sd_cmb, *sd_surf;
    const int32_t *task_col, *task_grp;  // (block, slot): lateral column or -1; first | count << 8 of its copies
    int nx, bc_cmb, bc_surf, add, sum;
    FastDiv div_x;
    // Chebyshev sub-step: d = az (b - A x) invd [+ ad d]
    const T *b[3], *invd[3];
    T *d[3];
    T az, ad;
    int read_d;
    const T *layer;  // FP32: q and cv of each layer, formed in FP64 with the mesh
};

enum { FAN_APPLY = 0, FAN_CHEB = 1 };

// Lane i receives lane i - 1 of the wave (0 enters at lane 0).
__device__ __forceinline__ double shr1(double v)
{
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x138, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x138, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ float shr1(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x138, 0xf, 0xf, true));
}

// One node column at the two levels of a lane's cell, boundary values removed:
// sums and differences of top and bottom.
template <typename T> struct FanCol {
    T su[3], du[3], kk;
};

template <typename T> struct FanBc {
    T z_lo, f_lo, z_hi, f_hi;  // Dirichlet factor, free-slip projection at the lane's bottom and top
};

// Node values of one column at the two levels of a lane's cell.
template <typename T> struct FanRaw {
    T lo[3], hi[3], k0, k1;
};

template <typename T>
__device__ __forceinline__ void fan_load(const FanArgs<T> &a, uint32_t col, int nr, int l, FanRaw<T> &o)
{
    const uint32_t i = col * (uint32_t)nr + l;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        o.lo[c] = a.src[c][i];
        o.hi[c] = a.src[c][i + 1];
    }
    o.k0 = a.k[i];
    o.k1 = a.k[i + 1];
}

// BCM: bit 0 free slip, bit 1 Dirichlet present in the operator
template <typename T, int BCM>
__device__ __forceinline__ FanCol<T> fan_column(const FanArgs<T> &a, uint32_t col, const FanRaw<T> &r, const FanBc<T> &bc)
{
#pragma clang fp contract(off)
    T lo[3], hi[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        lo[c] = r.lo[c];
        hi[c] = r.hi[c];
    }
    FanCol<T> o;
    o.kk = r.k0 + r.k1;
    if constexpr ((BCM & 1) != 0) {
        const T n0 = a.coords[3 * col], n1 = a.coords[3 * col + 1], n2 = a.coords[3 * col + 2];
        const T dl = bc.f_lo * fma(n2, lo[2], fma(n1, lo[1], n0 * lo[0]));
        const T dh = bc.f_hi * fma(n2, hi[2], fma(n1, hi[1], n0 * hi[0]));
        lo[0] = fma(-dl, n0, lo[0]);
        lo[1] = fma(-dl, n1, lo[1]);
        lo[2] = fma(-dl, n2, lo[2]);
        hi[0] = fma(-dh, n0, hi[0]);
        hi[1] = fma(-dh, n1, hi[1]);
        hi[2] = fma(-dh, n2, hi[2]);
    }
    if constexpr ((BCM & 2) != 0) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            lo[c] *= bc.z_lo;
            hi[c] *= bc.z_hi;
        }
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        o.su[c] = lo[c] + hi[c];
        o.du[c] = hi[c] - lo[c];
    }
    return o;
}

// One triangle with corners (centre, A, B): its contribution to the centre's
// column, L (bottom and top alike) and C (minus at the bottom, plus at the top,
// without the factor q).  Ma, Mb: gradients of A's and B's barycentric
// coordinates, Mc the centre's.  The trial gradient goes without its factor
// hs = 1 / (2 r_mid), which f = hs^2 k |det J| carries.
template <typename T>
__device__ __forceinline__ void fan_triangle(const FanCol<T> &P, const FanCol<T> &A, const FanCol<T> &B, const T Ma[3],
                                             const T Mb[3], const T Mc[3], const T M2[3], T detl, T q, T cv, T L[3],
                                             T C[3])
{
#pragma clang fp contract(off)
    T G[3][3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const T e1 = A.su[d] - P.su[d], e2 = B.su[d] - P.su[d], D = q * (P.du[d] + A.du[d] + B.du[d]);
#pragma unroll
        for (int e = 0; e < 3; ++e) G[d][e] = fma(e1, Ma[e], fma(e2, Mb[e], D * M2[e]));
    }
    const T f = cv * (P.kk + A.kk + B.kk) * detl, f2 = T(2) * f;
    const T fd = T(-2.0 / 3.0) * f * (G[0][0] + G[1][1] + G[2][2]);
    const T t00 = fma(f2, G[0][0], fd), t11 = fma(f2, G[1][1], fd), t22 = fma(f2, G[2][2], fd);
    const T t01 = f * (G[0][1] + G[1][0]), t02 = f * (G[0][2] + G[2][0]), t12 = f * (G[1][2] + G[2][1]);
    auto add = [&](T *o, const T *g) {
        o[0] = fma(t00, g[0], fma(t01, g[1], fma(t02, g[2], o[0])));
        o[1] = fma(t01, g[0], fma(t11, g[1], fma(t12, g[2], o[1])));
        o[2] = fma(t02, g[0], fma(t12, g[1], fma(t22, g[2], o[2])));
    };
    add(L, Mc);
    add(C, M2);
}

// Two groups of R lanes per node copy, three triangles each: half the chain of
// a group that takes all six (levels 3 and 4: 8.6 and 8.4 us per FP32 sub-step
// with one group, 6.6 and 7.4 with two).  At level 5, where the chip is full,
// one group was the faster by a tenth (18.5 against 20.9 us); 32 layers take two
// like the rest, for one layout of table, block and epilogue.
template <int R> constexpr int kFanBlock = R == 32 ? 512 : 256;
template <int R> constexpr int kFanCap = kFanBlock<R> / (2 * R);  // node copies per block, at least 8

template <typename T, int R, int BCM, int MODE>
__global__ __launch_bounds__(kFanBlock<R>) void fan_kernel(const FanArgs<T> a)
{
#pragma clang fp contract(off)
    constexpr int CAP = kFanCap<R>, nr = R + 1;
    __shared__ T part[CAP][3][nr];
    const int slot = threadIdx.x / (2 * R), half = (threadIdx.x / R) & 1, rl = threadIdx.x % R;
    // consecutive logical blocks (neighbouring columns) on one XCD
    uint32_t blk;
    {
        const uint32_t nb = gridDim.x, x = blockIdx.x & 7, i = blockIdx.x >> 3, q = nb >> 3, r = nb & 7;
        blk = x * q + min(x, r) + i;
    }
    const int32_t tc = a.task_col[blk * CAP + slot];
    const int grp = a.task_grp[blk * CAP + slot];
    const bool on = tc >= 0;
    const uint32_t col = on ? (uint32_t)tc : 0u;
    const int nx = a.nx, nc = nx - 1;
    const uint32_t t = a.div_x.div(col), sd = a.div_x.div(t);
    const int Y = (int)(col - t * (uint32_t)nx), X = (int)(t - sd * (uint32_t)nx);
    const bool has_cmb = a.sd_cmb[sd] != 0, has_surf = a.sd_surf[sd] != 0;
    const int bc_lo = rl == 0 && has_cmb ? a.bc_cmb : TNG_NEUMANN;
    const int bc_hi = rl == R - 1 && has_surf ? a.bc_surf : TNG_NEUMANN;
    FanBc<T> bc;
    bc.z_lo = bc_lo == TNG_DIRICHLET ? T(0) : T(1);
    bc.f_lo = bc_lo == TNG_FREESLIP ? T(1) : T(0);
    bc.z_hi = bc_hi == TNG_DIRICHLET ? T(0) : T(1);
    bc.f_hi = bc_hi == TNG_FREESLIP ? T(1) : T(0);

    // Ring: neighbour n at kNb[n], triangle n between neighbours n and n + 1 in
    // lateral cell kTri[n] (offsets, wedge), with the centre as corner kTri[n][3]
    // of that wedge.  The ring is point-symmetric: neighbour n + 3 lies opposite,
    // triangle n + 3 in the opposite cell's other wedge with the same corner, so
    // the second half is the first with the signs turned.
    constexpr int kNb[4][2] = {{1, 0}, {0, 1}, {-1, 1}, {-1, 0}};
    constexpr int kTri[3][4] = {{0, 0, 0, 0}, {-1, 0, 1, 2}, {-1, 0, 0, 1}};
    const int sgn = half ? -1 : 1;
    // a column outside the subdomain belongs to no triangle here: the centre is read instead
    auto neighbour = [&](int n) {
        const int dx = sgn * kNb[n][0], dy = sgn * kNb[n][1], x = X + dx, y = Y + dy;
        const bool in = x >= 0 && x < nx && y >= 0 && y < nx;
        return in ? (uint32_t)((int)col + dx * nx + dy) : col;
    };
    FanRaw<T> rp, rn[4];
    fan_load(a, col, nr, rl, rp);
#pragma unroll
    for (int n = 0; n < 4; ++n) fan_load(a, neighbour(n), nr, rl, rn[n]);
    T q, cv;
    if constexpr (sizeof(T) == 8) {
        const double r0 = a.radii[sd * nr + rl], r1 = a.radii[sd * nr + rl + 1];
        const double rmid = 0.5 * (r0 + r1), h = 0.5 * (r1 - r0), hs = 0.5 / rmid;
        q = (1.0 / (6.0 * h)) / hs;
        cv = hs * hs * rmid * rmid * h * (1.0 / 6.0);
    } else {
        const T *y = a.layer + 2 * (sd * R + rl);
        q = y[0];
        cv = y[1];
    }
    T L[3] = {T(0), T(0), T(0)}, C[3] = {T(0), T(0), T(0)};
    const FanCol<T> P = fan_column<T, BCM>(a, col, rp, bc);
    FanCol<T> prev = fan_column<T, BCM>(a, neighbour(0), rn[0], bc);
#pragma unroll
    for (int n = 0; n < 3; ++n) {
        const int xc = X + (half ? -1 - kTri[n][0] : kTri[n][0]), yc = Y + (half ? -1 - kTri[n][1] : kTri[n][1]);
        const bool in = xc >= 0 && xc < nc && yc >= 0 && yc < nc;
        const int xq = min(max(xc, 0), nc - 1), yq = min(max(yc, 0), nc - 1);
        const T *g = a.latgeom + ((((int64_t)sd * nc + xq) * nc + yq) * 2 + (kTri[n][2] ^ half)) * 10;
        const FanCol<T> next = fan_column<T, BCM>(a, neighbour(n + 1), rn[n + 1], bc);
        // gradients of the wedge's barycentric coordinates: corner 1 M0, corner 2 M1, corner 0 -(M0 + M1)
        T m[3][3], M2[3];
#pragma unroll
        for (int e = 0; e < 3; ++e) {
            m[1][e] = g[e];
            m[2][e] = g[3 + e];
            m[0][e] = -(g[e] + g[3 + e]);
            M2[e] = g[6 + e];
        }
        constexpr int rot[3][3] = {{0, 1, 2}, {1, 2, 0}, {2, 0, 1}};
        const int *ro = rot[kTri[n][3]];
        fan_triangle<T>(P, prev, next, m[ro[1]], m[ro[2]], m[ro[0]], M2, in ? g[9] : T(0), q, cv, L, C);
        prev = next;
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        L[c] += __shfl_xor(L[c], R, 64);
        C[c] += __shfl_xor(C[c], R, 64);
    }
    // level rl: this cell's bottom and the top of the cell below; the last
    // lane also holds the top level
    T val[2][3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const T qc = q * C[c], top = L[c] + qc;
        const T up = shr1(top);
        val[0][c] = (L[c] - qc) + (rl > 0 ? up : T(0));
        val[1][c] = top;
    }
    const uint32_t base = col * (uint32_t)nr + rl;
    const bool last = rl == R - 1;
    if constexpr (BCM != 0) {
        // boundary rows of this copy
        auto row = [&](T (&v)[3], int bcv, int side, uint32_t i) {
            const T *bt = a.btab + (col * 2 + side) * 3;
            const T u0 = a.src[0][i], u1 = a.src[1][i], u2 = a.src[2][i];
            if ((BCM & 2) != 0 && bcv == TNG_DIRICHLET) {
                v[0] = bt[0] * u0;
                v[1] = bt[1] * u1;
                v[2] = bt[2] * u2;
            } else if constexpr ((BCM & 1) != 0) {
                const T n0 = a.coords[3 * col], n1 = a.coords[3 * col + 1], n2 = a.coords[3 * col + 2];
                const T dv = fma(n2, v[2], fma(n1, v[1], n0 * v[0]));
                const T un = bt[0] * fma(n2, u2, fma(n1, u1, n0 * u0));
                v[0] = fma(un, n0, fma(-dv, n0, v[0]));
                v[1] = fma(un, n1, fma(-dv, n1, v[1]));
                v[2] = fma(un, n2, fma(-dv, n2, v[2]));
            }
        };
        if (bc_lo != TNG_NEUMANN) row(val[0], bc_lo, 0, base);
        if (bc_hi != TNG_NEUMANN) row(val[1], bc_hi, 1, base + 1);
    }
    // from here the first half owns level rl, the second the top level (its last lane)
    T v[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) v[c] = half ? val[1][c] : val[0][c];
    const uint32_t at = base + half;
    const bool owner = on && (half == 0 || last);
    if (MODE == FAN_APPLY && a.add && owner) {
#pragma unroll
        for (int c = 0; c < 3; ++c) v[c] += a.dst[c][at];
    }
    // sum over the copies of a shared node, ascending
    const int cnt = grp >> 8, first_slot = grp & 255;
    if (a.sum) {
        if (cnt > 1 && owner) {
#pragma unroll
            for (int c = 0; c < 3; ++c) part[slot][c][rl + half] = v[c];
        }
        __syncthreads();
        if (cnt > 1 && owner) {
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                T s = T(0);
                for (int j = 0; j < cnt; ++j) s += part[first_slot + j][c][rl + half];
                v[c] = s;
            }
        }
    }
    if (!owner) return;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        if constexpr (MODE == FAN_APPLY) {
            a.dst[c][at] = v[c];
        } else {
            // the rounding of the separate update kernel
            const T r = a.b[c][at] - v[c];
            const T z = r * a.invd[c][at];
            T s = a.az * z;
            if (a.read_d) s = fma(a.ad, a.d[c][at], s);
            a.d[c][at] = s;
            a.dst[c][at] = a.src[c][at] + s;
        }
    }
}

template <typename T> FanArgs<T> fan_args(const tng_operator &op, const tng_vector &src, const tng_vector &dst)
{
    const tng_domain &m = *op.mesh;
    FanArgs<T> a{};
    for (int c = 0; c < 3; ++c) {
        a.src[c] = (const T *)src.comp(c);
        a.dst[c] = (T *)dst.comp(c);
    }
    constexpr bool f64 = sizeof(T) == 8;
    a.k = (const T *)op.k->comp(0);
    a.radii = m.d_radii.as<double>();
    if constexpr (!f64) a.layer = m.d_layer_f.as<float>();
    a.latgeom = (const T *)(f64 ? m.d_latgeom.p : m.d_latgeom_f.p);
    a.coords = (const T *)(f64 ? m.d_coords.p : m.d_coords_f.p);
    a.btab = op.d_btab.as<T>();
    a.sd_cmb = m.d_sd_cmb.as<uint8_t>();
    a.sd_surf = m.d_sd_surf.as<uint8_t>();
    a.task_col = m.d_fan_col.as<int32_t>();
    a.task_grp = m.d_fan_grp.as<int32_t>();
    a.nx = m.nx;
    a.bc_cmb = op.bc_cmb;
    a.bc_surf = op.bc_surf;
    a.div_x = FastDiv((uint32_t)m.nx);
    return a;
}

template <typename T, int R, int MODE> void fan_launch_bc(const FanArgs<T> &a, int blocks, hipStream_t s)
{
    const int bcm = (a.bc_cmb == TNG_FREESLIP || a.bc_surf == TNG_FREESLIP ? 1 : 0) |
                    (a.bc_cmb == TNG_DIRICHLET || a.bc_surf == TNG_DIRICHLET ? 2 : 0);
    switch (bcm) {
    case 0: hipLaunchKernelGGL((fan_kernel<T, R, 0, MODE>), dim3(blocks), dim3(kFanBlock<R>), 0, s, a); break;
    case 1: hipLaunchKernelGGL((fan_kernel<T, R, 1, MODE>), dim3(blocks), dim3(kFanBlock<R>), 0, s, a); break;
    case 2: hipLaunchKernelGGL((fan_kernel<T, R, 2, MODE>), dim3(blocks), dim3(kFanBlock<R>), 0, s, a); break;
    default: hipLaunchKernelGGL((fan_kernel<T, R, 3, MODE>), dim3(blocks), dim3(kFanBlock<R>), 0, s, a); break;
    }
    TNG_HIP_CHECK(hipGetLastError());
}

template <typename T, int MODE> void fan_launch(const tng_domain &m, const FanArgs<T> &a, hipStream_t s)
{
    if constexpr (sizeof(T) == 4)
        if (m.nr - 1 == 32) return fan_launch_bc<T, 32, MODE>(a, m.fan_blocks, s);
    switch (m.nr - 1) {
    case 4: fan_launch_bc<T, 4, MODE>(a, m.fan_blocks, s); break;
    case 8: fan_launch_bc<T, 8, MODE>(a, m.fan_blocks, s); break;
    default: fan_launch_bc<T, 16, MODE>(a, m.fan_blocks, s); break;
    }
}

}  // namespace

// The fan evaluates a triangle three times, the sweep (with its halo sum) once
// but as a serial loop over the rows of a strip, whose lanes may reach past
// narrow subdomains.  Measured at lateral levels 2 to 10, diamonds whole and
// split up to 16 x 16 (fan against sweep, no-slip):
//   lanes F <= 2^20, one filling of the chip: the fan always (FP64 level 4, 16
//     layers 7.6 against 13.9 us, level 6, 8 layers 30 against 35; FP32 level 5,
//     32 layers 14.7 against 23.3);
//   more: against the sweep's lanes times steps S.  FP64 from S = 2 F on
//     (level 7, 8 layers: S / F = 0.76 105 against 79 us, 2.2 121 against 150;
//     level 6, 16 layers: 0.77 56 against 43, 1.08 62 against 51, 2.3 70 against
//     86); 4 layers, where the sweep fills its strips badly, up to 2^23
//     (level 8 256 against 306, level 9 with free slip 1193 against 1081);
//   FP32, 4 layers: always (level 9 412 against 839 us).  Up to 2^21 lanes, 8
//     layers without free slip at any size, from S = 0.75 F on, with the free-slip
//     projections of every column it reads from S = F on (level 6, 16 layers: 0.77
//     21.5 against 24.3, free slip 26.2 against 25.9, 1.04 22.6 against 29.7 and
//     27.1 against 31.3; level 7, 8 layers: 0.76 43.8 against 50.2, free slip 54.3
//     against 53.2); else from S = 2 F on (level 6, 32 layers: 0.64 47.7
//     against 34.6; level 7, 16 layers: 0.63 81 against 57).
// Sub-steps of the smoother divide the same way: with the update kernel that
// the fan spares, V-cycles on level 6, 8 layers gain 1.46 (FP32) and 1.03 (FP64),
// level 6, 16 layers with free slip lose 0.94 and 0.75.  FP64 at 32 layers
// always takes the sweep: 174 to 216 registers leave two waves per SIMD, and 21,780
// groups of three triangles take 44 us at level 5 against 28 us.
bool fan_pays(const tng_domain &m, bool f32, bool free_slip)
{
    const int cells = m.nr - 1;
    if (m.rad_sdr != 0 || cells < 4 || cells > (f32 ? 32 : 16)) return false;
    const double fan = 2.0 * cells * (double)m.nlat;
    if (fan <= 1 << 20) return true;
    // workgroups of eight waves take 512 / cells - 1 new columns of one subdomain
    const int columns = 512 / cells - 1, strips = (m.nx + columns - 1) / columns;
    const double sweep = 512.0 * m.nsd * strips * (m.nx + 2.5);
    if (cells == 4 && (f32 || fan <= 1 << 23)) return true;
    if (f32 && (fan <= 1 << 21 || (cells == 8 && !free_slip))) return sweep >= (free_slip ? 1.0 : 0.75) * fan;
    return sweep >= 2.0 * fan;
}

bool fan_applies(const tng_operator &op)
{
    if (op.mesh->fan_blocks == 0 || op.stored || op.diagonal || op.penalty_active) return false;
    return fan_pays(*op.mesh, op.k->dtype == TNG_F32, op.bc_cmb == TNG_FREESLIP || op.bc_surf == TNG_FREESLIP);
}

void fan_apply(tng_operator &op, const tng_vector &src, tng_vector &dst, hipStream_t s)
{
    auto run = [&](auto tag) {
        using T = decltype(tag);
        FanArgs<T> a = fan_args<T>(op, src, dst);
        a.add = op.apply_mode == TNG_ADD ? 1 : 0;
        a.sum = op.comm_mode == TNG_COMMUNICATE_ADDITIVELY ? 1 : 0;
        fan_launch<T, FAN_APPLY>(*op.mesh, a, s);
    };
    if (src.dtype == TNG_F64) run(double());
    else run(float());
}

void fan_apply_cheb(tng_operator &op, const tng_vector &x, tng_vector &x_out, tng_vector &d, const tng_vector &b,
                    const tng_vector &invd, double az, double ad, bool read_d, hipStream_t s)
{
    auto run = [&](auto tag) {
        using T = decltype(tag);
        FanArgs<T> a = fan_args<T>(op, x, x_out);
        a.sum = 1;
        for (int c = 0; c < 3; ++c) {
            a.b[c] = (const T *)b.comp(c);
            a.invd[c] = (const T *)invd.comp(c);
            a.d[c] = (T *)d.comp(c);
        }
        a.az = (T)az;
        a.ad = (T)ad;
        a.read_d = read_d ? 1 : 0;
        fan_launch<T, FAN_CHEB>(*op.mesh, a, s);
    };
    if (x.dtype == TNG_F64) run(double());
    else run(float());
}

}  // namespace tng
