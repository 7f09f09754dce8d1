"""Kernel variants at the sizes where their decompositions change: against
the oracle at 1e-12 (FP64: sums of at most a few hundred products of one
sign-free magnitude, 1e-16 each)."""
import ctypes
import time

import numpy as np
import pytest

import oracle as O
import tng
from conftest import consistent, rel_err

pytestmark = pytest.mark.gpu

D, F, N = tng.DIRICHLET, tng.FREESLIP, tng.NEUMANN


def field(om, ncomp, seed, scale=1.0):
    r = np.random.default_rng(seed)
    return consistent(om, scale * r.uniform(-1, 1, ((ncomp,) if ncomp > 1 else ()) + om.shape))


def vec(dom, data, dtype=tng.F64):
    return (tng.VectorQ1Vec if data.ndim == 5 else tng.VectorQ1Scalar)(dom, dtype).upload(data)


def microseconds(dom, fn, n=20):
    best = 1e9
    for _ in range(5):
        dom.ctx.synchronize()
        t = time.perf_counter()
        for _ in range(n):
            fn()
        dom.ctx.synchronize()
        best = min(best, (time.perf_counter() - t) / n)
    return 1e6 * best


# columns per block of the SUPG cell kernel: 64 (2 and 4 cells), 32, one, and
# radial segments of 256 cells whose seam levels two blocks share (512 layers)
@pytest.mark.parametrize("L,Lr,ls,rs", [(2, 1, 0, 0), (3, 2, 1, 0), (2, 3, 0, 0), (2, 8, 0, 0), (1, 9, 0, 0), (1, 9, 0, 1)])
@pytest.mark.parametrize("flags", [dict(), dict(lumped_mass=True), dict(diagonal=True, treat_boundary=False)])
def test_supg_block_shapes(L, Lr, ls, rs, flags, gpu_ctx):
    dom = tng.DistributedDomain.create_uniform(L, Lr, 0.55, 1.0, ls, rs)
    om = O.Mesh(L, Lr, 0.55, 1.0, ls, rs)
    vel, T = field(om, 3, 1, 50.0), field(om, 1, 2)
    op = tng.UnsteadyAdvectionDiffusionSUPG(dom, vec(dom, vel), 0.01, 0.02, **flags)
    out = vec(dom, T)
    op.apply(vec(dom, T), out)
    ref = O.supg_apply(om, vel, T, kappa=0.01, dt=0.02, treat_boundary=flags.get("treat_boundary", True),
                       diagonal=flags.get("diagonal", False), lumped=flags.get("lumped_mass", False))
    assert rel_err(out.download(), ref) < 1e-12


# the treated boundary rows must not cost more than a little beside the apply: the untreated diagonal mode has the same
# kernels without them
@pytest.mark.parametrize("L,Lr", [(4, 4), (6, 2), (5, 5)])
def test_supg_boundary_rows_cost_little(L, Lr, gpu_ctx):
    dom = tng.DistributedDomain.create_uniform(L, Lr, 0.55, 1.0)
    v, t, out = tng.VectorQ1Vec(dom), tng.VectorQ1Scalar(dom), tng.VectorQ1Scalar(dom)
    v.fill(1.0)
    t.fill(1.0)
    ops = [tng.UnsteadyAdvectionDiffusionSUPG(dom, v, 0.01, 0.02, **kw)
           for kw in ({}, dict(diagonal=True, treat_boundary=False))]
    treated, diagonal = (microseconds(dom, lambda op=op: op.apply(t, out)) for op in ops)
    assert treated < 1.3 * diagonal


def test_supg_reads_the_velocity_at_every_apply(gpu_ctx):
    """tau and the boundary rows follow a velocity changed in place between two applies of one operator."""
    dom, om = tng.DistributedDomain.create_uniform(3, 3, 0.55, 1.0), O.Mesh(3)
    T, v = field(om, 1, 2), vec(dom, field(om, 3, 1, 50.0))
    op = tng.UnsteadyAdvectionDiffusionSUPG(dom, v, 0.01, 0.02)
    out = vec(dom, T)
    op.apply(vec(dom, T), out)
    vel = field(om, 3, 3, 5.0)
    v.upload(vel)
    op.apply(vec(dom, T), out)
    assert rel_err(out.download(), O.supg_apply(om, vel, T, kappa=0.01, dt=0.02)) < 1e-12


# rows at every kind of node: subdomain edges and corners, single cells between surfaces, 128 layers
@pytest.mark.parametrize("L,Lr,ls,rs", [(1, 1, 0, 0), (2, 3, 1, 1), (3, 2, 0, 0), (2, 7, 0, 0)])
def test_mass_matches_oracle(L, Lr, ls, rs, gpu_ctx):
    dom = tng.DistributedDomain.create_uniform(L, Lr, 0.55, 1.0, ls, rs)
    om = O.Mesh(L, Lr, 0.55, 1.0, ls, rs)
    x, u = field(om, 1, 4), field(om, 3, 5)
    out = vec(dom, x)
    tng.mass_apply(vec(dom, x), out)
    assert rel_err(out.download(), O.scalar_mass(om, x)) < 1e-12
    for dtype, tol in ((tng.F64, 1e-12), (tng.F32, 2e-6)):  # FP32: inputs and tables rounded to 6e-8, sums of 63 terms
        out = vec(dom, u, dtype)
        tng.VectorMass(dom).apply(vec(dom, u, dtype), out)
        assert rel_err(out.download(), O.vector_mass(om, u)) < tol


# the assembled coarse PCG: run to convergence it is the direct solve (relative residual 1e-13 times a condition
# number of some 1e4), whatever the boundary rows, split diamonds, or Galerkin / re-discretised coarsest operator
@pytest.mark.parametrize("bcs", [(D, D), (F, D), (D, F), (tng.NEUMANN, D)])
@pytest.mark.parametrize("gca,sdr,dtype", [(0, 0, tng.F64), (1, 1, tng.F64), (1, 0, tng.F32)])
def test_assembled_coarse_pcg_solves_the_coarse_system(bcs, gca, sdr, dtype, gpu_ctx):
    om = O.Mesh(3, 3, 0.55, 1.0, sdr, 0)
    eta, b = np.exp(0.5 * field(om, 1, 11)), field(om, 3, 12)
    out = []
    for kw in (dict(coarse_solver=1), dict(coarse_solver=0, coarse_max_iterations=4000, coarse_relative_tolerance=1e-13)):
        S = tng.StokesSolver(2, 3, 0.55, 1.0, bcs, tng.StokesParams.defaults(gca=gca, viscous_pc_dtype=dtype, **kw),
                             lateral_sdr=sdr)
        dv = S.domain_velocity
        S.set_viscosity(vec(dv, eta))
        x = tng.VectorQ1Vec(dv)
        S.precondition_velocity(x, vec(dv, b))
        out.append(x.download())
    assert rel_err(out[1], out[0]) < (1e-8 if dtype == tng.F64 else 1e-6)


# a new viscosity assembles that operator; with the rotation penalty, whose coarse PCG is not assembled, it does not
def test_assembled_coarse_operator_costs_little_per_viscosity(gpu_ctx):
    times = []
    for bcs in ((D, F), (F, F)):
        S = tng.StokesSolver(2, 3, 0.55, 1.0, bcs, tng.StokesParams.defaults(krylov_restart=2))
        eta = tng.VectorQ1Scalar(S.domain_velocity)
        eta.fill(1.0)
        times.append(microseconds(S.domain_velocity, lambda: S.set_viscosity(eta)))
    assert times[0] < 2 * times[1]


# launches after the end of a coarse solve change nothing, wherever in the host's look at the end (every 25) it falls:
# ended by the tolerance within the first 25 iterations, and by a zero right-hand side, for which p.(A p) is zero
@pytest.mark.parametrize("dtype", [tng.F64, tng.F32])
def test_coarse_pcg_keeps_its_result_after_the_end(dtype, gpu_ctx):
    om = O.Mesh(3, 3)
    eta, b = np.exp(0.5 * field(om, 1, 13)), field(om, 3, 14)
    out, zero = [], []
    for max_it in (24, 25, 26, 400):
        S = tng.StokesSolver(2, 3, 0.55, 1.0, (D, D), tng.StokesParams.defaults(
            viscous_pc_dtype=dtype, coarse_max_iterations=max_it, coarse_relative_tolerance=1e-2,
            coarse_absolute_tolerance=0.0))
        dv = S.domain_velocity
        S.set_viscosity(vec(dv, eta))
        for rhs, res in ((b, out), (0 * b, zero)):
            x = tng.VectorQ1Vec(dv)
            S.precondition_velocity(x, vec(dv, rhs))
            res.append(x.download())
    assert np.any(out[0]) and all(np.array_equal(o, out[0]) for o in out)
    assert all(not np.any(z) for z in zero)


# the fan kernel: every lane-group size (4 to 32 layers; 32 in FP32 only, FP64 takes the sweep there), shared nodes of
# two to five copies inside and across diamonds, every boundary mix, Add mode and skipped communication
@pytest.mark.parametrize("L,Lr,ls", [(2, 2, 1), (3, 3, 2), (3, 4, 1), (4, 5, 0), (1, 3, 0), (5, 2, 2)])
@pytest.mark.parametrize("bcs", [(D, D), (F, D), (D, F), (tng.NEUMANN, F), (tng.NEUMANN, tng.NEUMANN)])
def test_fan_apply_matches_oracle(L, Lr, ls, bcs, gpu_ctx):
    dom = tng.DistributedDomain.create_uniform(L, Lr, 0.55, 1.0, ls, 0)
    om = O.Mesh(L, Lr, 0.55, 1.0, ls, 0)
    k, u, base = np.exp(0.5 * field(om, 1, 21)), field(om, 3, 22), field(om, 3, 23)
    # FP32: eight rounded factors (up to 6e-8, 2e-8 on average) and sums of random terms; radii kept in FP32 would cost
    # 6e-8 radius / thickness, 2e-6 at 32 layers
    for dtype, tol in ((tng.F64, 1e-12), (tng.F32, 5e-7)):
        kv, uv = vec(dom, k, dtype), vec(dom, u, dtype)
        op = tng.EpsilonDivDivKerngen(dom, kv, bcs)
        out = vec(dom, base, dtype)
        op.apply(uv, out)
        assert rel_err(out.download(), om.epsdivdiv(k, u, *bcs)) < tol
        for mode in ((tng.ADD, tng.SKIP_COMMUNICATION), (tng.ADD, tng.COMMUNICATE_ADDITIVELY),
                     (tng.REPLACE, tng.SKIP_COMMUNICATION)):
            op.set_operator_apply_and_communication_modes(*mode)
            out = vec(dom, base, dtype)
            op.apply(uv, out)
            ref = om.epsdivdiv(k, u, *bcs, apply_mode=mode[0], comm=mode[1], dst=base)
            assert rel_err(out.download(), ref) < tol


# wide meshes of few layers: the fan kernel's triple evaluation must not be taken there.  The rotation penalty of free
# slip on both surfaces always takes the sweep, and does strictly more than an apply without it
@pytest.mark.parametrize("L,Lr,dtype", [(7, 4, tng.F64), (7, 3, tng.F64), (7, 5, tng.F32), (7, 4, tng.F32)])
def test_wide_meshes_take_no_longer_than_with_the_penalty(L, Lr, dtype, gpu_ctx):
    dom = tng.DistributedDomain.create_uniform(L, Lr, 0.55, 1.0)
    k, u, out = tng.VectorQ1Scalar(dom, dtype), tng.VectorQ1Vec(dom, dtype), tng.VectorQ1Vec(dom, dtype)
    k.fill(1.0)
    u.fill(1.0)
    ops = [tng.EpsilonDivDivKerngen(dom, k, bcs) for bcs in ((D, F), (F, F))]
    ops[1].set_penalty_epsilon(1.0)
    plain, penalised = (microseconds(dom, lambda op=op: op.apply(u, out)) for op in ops)
    assert plain < penalised


# both sides of the line, and meshes whose narrow subdomains move it
@pytest.mark.parametrize("L,Lr,ls", [(6, 4, 0), (6, 4, 3), (7, 2, 0), (6, 5, 0)])
def test_fan_and_sweep_on_wide_meshes_match_oracle(L, Lr, ls, gpu_ctx):
    dom, om = tng.DistributedDomain.create_uniform(L, Lr, 0.55, 1.0, ls, 0), O.Mesh(L, Lr, 0.55, 1.0, ls, 0)
    k, u = np.exp(0.5 * field(om, 1, 36)), field(om, 3, 37)
    ref = om.epsdivdiv(k, u, D, F)
    for dtype, tol in ((tng.F64, 1e-12), (tng.F32, 1e-6)):  # FP32: operands and tables rounded to 6e-8, sums of 36 terms
        out = tng.VectorQ1Vec(dom, dtype)
        tng.EpsilonDivDivKerngen(dom, vec(dom, k, dtype), (D, F)).apply(vec(dom, u, dtype), out)
        assert rel_err(out.download(), ref) < tol


# copies that differ (a vector that no exchange has made consistent): each copy's cells read their own subdomain's values
def test_fan_apply_reads_each_subdomains_own_copies(gpu_ctx):
    dom, om = tng.DistributedDomain.create_uniform(3, 3, 0.55, 1.0, 1, 0), O.Mesh(3, 3, 0.55, 1.0, 1, 0)
    k = np.exp(0.5 * field(om, 1, 24))
    u = np.random.default_rng(25).uniform(-1, 1, (3,) + om.shape)
    for bcs in ((D, F), (F, D)):
        out = vec(dom, u)
        tng.EpsilonDivDivKerngen(dom, vec(dom, k), bcs).apply(vec(dom, u), out)
        assert rel_err(out.download(), om.epsdivdiv(k, u, *bcs)) < 1e-12


@pytest.mark.parametrize("dtype", [tng.F64, tng.F32])
@pytest.mark.parametrize("bcs,sdr", [((D, D), 0), ((D, F), 1)])
def test_fan_chebyshev_has_the_bits_of_the_separate_kernels(dtype, bcs, sdr, gpu_ctx):
    om = O.Mesh(5, 5, 0.55, 1.0, sdr, 0)
    eta, b = np.exp(0.5 * field(om, 1, 26)), field(om, 3, 27)
    out = []
    for fuse in (0, 1):
        with tng.default_context().tuning(cheb_fuse=fuse):
            S = tng.StokesSolver(2, 5, 0.55, 1.0, bcs, tng.StokesParams.defaults(
                viscous_pc_dtype=dtype, viscous_pc_chebyshev_order=3, coarse_solver=1), lateral_sdr=sdr)
        S.set_viscosity(vec(S.domain_velocity, eta))
        x = tng.VectorQ1Vec(S.domain_velocity)
        for _ in range(2):  # from zero, then from a start vector
            S.precondition_velocity(x, vec(S.domain_velocity, b))
        out.append(x.download())
    assert np.array_equal(out[0], out[1])


# B and its transpose are adjoint: the one-pass divergence with chunks of 2, 4 and 8 coarse rows and the three kernels of
# small FP64 meshes, at 64 layers per subdomain (random entries: a wrong one moves the product by 1e-7 or more of the
# norms' product, rounding by a few 1e-16)
@pytest.mark.parametrize("L,Lr,rs", [(4, 6, 0), (5, 6, 0), (7, 6, 0), (7, 7, 1)])
def test_divergence_is_the_adjoint_of_the_gradient(L, Lr, rs, gpu_ctx):
    fine, coarse = (tng.DistributedDomain.create_uniform(L - i, Lr - i, 0.55, 1.0, 0, rs) for i in range(2))

    def noise(dom, k):  # the same on all copies of a node
        s = (dom.coords() @ (1e3 * np.random.default_rng(k).uniform(1, 2, 3)))[..., None]
        return np.sin(s + 1e4 * dom.radii()[:, None, None, :])

    u = tng.VectorQ1Vec(fine).upload(np.stack([noise(fine, k) for k in range(3)]))
    p = tng.VectorQ1Scalar(coarse).upload(noise(coarse, 3))
    bu, btp = tng.VectorQ1Scalar(coarse), tng.VectorQ1Vec(fine)
    tng.DivergenceKerngen(fine, coarse, (D, F)).apply(u, bu)
    tng.GradientKerngen(fine, coarse, (D, F)).apply(p, btp)
    assert abs(tng.dot(bu, p) - tng.dot(u, btp)) < 1e-13 * tng.norm_2(bu) * tng.norm_2(p)


# the one-pass divergence's serial rows on small FP64 meshes: FP32, which takes it at every size, is the yardstick
def test_small_divergence_takes_no_longer_in_fp64(gpu_ctx):
    fine, coarse = (tng.DistributedDomain.create_uniform(3 - i, 6 - i, 0.55, 1.0) for i in range(2))
    times = []
    for dtype in (tng.F64, tng.F32):
        u, out = tng.VectorQ1Vec(fine, dtype), tng.VectorQ1Scalar(coarse, dtype)
        u.fill(1.0)
        op = tng.DivergenceKerngen(fine, coarse, (D, F))
        times.append(microseconds(fine, lambda: op.apply(u, out)))
    assert times[0] < 1.08 * times[1]  # 0.94; 1.12 with one pass


# spare vectors of the fused sub-step only where a level takes it: none with the rotation penalty below 64 layers
def test_no_spare_vectors_where_no_sub_step_is_fused(gpu_ctx):
    def free_memory():
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert tng.load_library().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    used = []
    for fuse in (0, 1):
        free = free_memory()
        with tng.default_context().tuning(cheb_fuse=fuse):
            S = tng.StokesSolver(2, 5, 0.55, 1.0, (F, F), tng.StokesParams.defaults(krylov_restart=2))
        used.append(free - free_memory())
        S.close()
    assert used[1] - used[0] < 4 << 20  # one vector of the finest level is 8.6 MB


# FP32 at 128 layers, two cells per lane: strips of eight columns within one subdomain and across several, every
# boundary mix and the penalty, both apply modes, copies that differ
@pytest.mark.parametrize("L,ls,rs", [(1, 0, 0), (2, 1, 0), (3, 0, 1)])
@pytest.mark.parametrize("bcs", [(D, D), (F, F), (N, N), (F, D), (D, F), (N, F)])
@pytest.mark.parametrize("chunks", [0, 1])  # 1: the kernel with four waves and the boundary mix at run time
def test_fp32_pairs_of_cells_match_oracle(L, ls, rs, bcs, chunks, gpu_ctx):
    dom, om = tng.DistributedDomain.create_uniform(L, 7 + rs, 0.55, 1.0, ls, rs), O.Mesh(L, 7 + rs, 0.55, 1.0, ls, rs)
    k, base = np.exp(0.5 * field(om, 1, 28)), field(om, 3, 29)
    u = np.random.default_rng(30).uniform(-1, 1, (3,) + om.shape)
    op = tng.EpsilonDivDivKerngen(dom, vec(dom, k, tng.F32), bcs)
    op.set_penalty_epsilon(1.0)
    for mode in ((tng.REPLACE, tng.COMMUNICATE_ADDITIVELY), (tng.ADD, tng.SKIP_COMMUNICATION)):
        op.set_operator_apply_and_communication_modes(*mode)
        out = vec(dom, base, tng.F32)
        with dom.ctx.tuning(apply_radial_chunks=chunks):
            op.apply(vec(dom, u, tng.F32), out)
        ref = om.epsdivdiv(k, u, *bcs, path="fast", penalty_eps=1.0, apply_mode=mode[0], comm=mode[1], dst=base)
        # eight rounded factors (up to 6e-8, 2e-8 on average) and sums of random terms; radii kept in FP32 would cost 6e-8
        # radius / thickness, 1e-5
        assert rel_err(out.download(), ref) < 5e-7


# chunks (the fused step below 2048 columns), parts and pairs of cells form the same products per level
@pytest.mark.parametrize("L", [3, 4])
def test_fp32_shapes_at_128_layers_have_the_same_bits(L, gpu_ctx):
    om = O.Mesh(L, 7)
    eta, b = np.exp(0.5 * field(om, 1, 39)), field(om, 3, 40)
    out = []
    for fuse, split in ((0, 0), (1, 0), (1, 1)):
        with tng.default_context().tuning(cheb_fuse=fuse, apply_radial_split=split):
            S = tng.StokesSolver(1, L, 0.55, 1.0, (D, F), tng.StokesParams.defaults(
                viscous_pc_dtype=tng.F32, viscous_pc_chebyshev_order=3, coarse_solver=1), radial_extra_levels=7 - L)
            S.set_viscosity(vec(S.domain_velocity, eta))
            x = tng.VectorQ1Vec(S.domain_velocity)
            for _ in range(2):
                S.precondition_velocity(x, vec(S.domain_velocity, b))
            out.append(x.download())
    assert all(np.array_equal(out[0], o) for o in out)


@pytest.mark.parametrize("bcs", [(D, D), (F, F), (D, F)])
def test_fp32_pairs_fused_have_the_bits_of_the_separate_kernels(bcs, gpu_ctx):
    om = O.Mesh(4, 7, 0.55, 1.0, 0, 0)
    eta, b = np.exp(0.5 * field(om, 1, 31)), field(om, 3, 32)
    out = []
    for fuse in (0, 1):
        with tng.default_context().tuning(cheb_fuse=fuse):
            S = tng.StokesSolver(1, 4, 0.55, 1.0, bcs, tng.StokesParams.defaults(
                viscous_pc_dtype=tng.F32, viscous_pc_chebyshev_order=3, coarse_solver=1), radial_extra_levels=3)
        S.set_viscosity(vec(S.domain_velocity, eta))
        x = tng.VectorQ1Vec(S.domain_velocity)
        for _ in range(2):
            S.precondition_velocity(x, vec(S.domain_velocity, b))
        out.append(x.download())
    assert np.array_equal(out[0], out[1])


# the same on split diamonds, and on a level that the last cache does not hold (the step's vectors pass by the caches)
@pytest.mark.parametrize("L,extra,ls", [(4, 3, 1), (6, 1, 0)])
def test_fp32_pairs_fused_split_and_streamed(L, extra, ls, gpu_ctx):
    out, rng = [], np.random.default_rng(38)
    for fuse in (0, 1):
        with tng.default_context().tuning(cheb_fuse=fuse):
            S = tng.StokesSolver(L - 1, L, 0.55, 1.0, (D, F), tng.StokesParams.defaults(
                viscous_pc_dtype=tng.F32, viscous_pc_chebyshev_order=3, coarse_max_iterations=1, krylov_restart=2),
                radial_extra_levels=extra, lateral_sdr=ls)
        dv = S.domain_velocity
        if not out:  # the same values on every copy of a node
            s = dv.coords() @ (1e3 * rng.uniform(1, 2, (3, 4)))
            noise = np.sin(np.moveaxis(s, -1, 0)[..., None] + 1e4 * dv.radii()[:, None, None, :])
        S.set_viscosity(vec(dv, np.exp(0.5 * noise[3])))
        x, b = tng.VectorQ1Vec(dv), vec(dv, noise[:3])
        for _ in range(2):
            S.precondition_velocity(x, b)
        out.append(x.download())
    assert np.any(out[0]) and np.array_equal(out[0], out[1])


# a level that the last cache holds: the fused step is worth it only if it does not stream past that cache
def test_fp32_pairs_fused_pay_on_a_cached_level(gpu_ctx):
    times = []
    for fuse in (0, 1):
        with tng.default_context().tuning(cheb_fuse=fuse):
            S = tng.StokesSolver(4, 5, 0.55, 1.0, (D, F), tng.StokesParams.defaults(
                viscous_pc_dtype=tng.F32, viscous_pc_chebyshev_order=6, coarse_max_iterations=1, krylov_restart=2),
                radial_extra_levels=2)
        x, b = tng.VectorQ1Vec(S.domain_velocity), tng.VectorQ1Vec(S.domain_velocity)
        b.fill(1.0)
        times.append(microseconds(S.domain_velocity, lambda: S.precondition_velocity(x, b)))
    assert times[1] < 0.96 * times[0]


# the adjoint's wedge products: two layers (cells that meet at one node level), one and several rows per thread,
# waves in one column (64 and 128 layers) and in several, radial subdomains without a boundary
@pytest.mark.parametrize("L,Lr,ls,rs", [(1, 1, 0, 0), (2, 3, 1, 0), (2, 6, 0, 0), (1, 7, 0, 0), (3, 8, 0, 2), (5, 5, 0, 0),
                                        (6, 6, 0, 0)])
@pytest.mark.parametrize("bcs", [(N, N), (D, F), (F, D)])
def test_adjoint_sweep_matches_oracle(L, Lr, ls, rs, bcs, gpu_ctx):
    dom, om = tng.DistributedDomain.create_uniform(L, Lr, 0.55, 1.0, ls, rs), O.Mesh(L, Lr, 0.55, 1.0, ls, rs)
    k, lam, u = np.exp(field(om, 1, 33)), field(om, 3, 34), field(om, 3, 35)
    g = vec(dom, k)
    tng.EpsilonDivDivKerngen(dom, vec(dom, k), bcs).log_coefficient_gradient(vec(dom, lam), vec(dom, u), g)
    assert rel_err(g.download(), om.log_k_gradient(k, lam, u, *bcs)) < 1e-12
