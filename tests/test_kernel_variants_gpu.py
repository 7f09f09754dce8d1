"""Kernel variants at the sizes where their decompositions change: against
the oracle at 1e-12 (FP64: sums of at most a few hundred products of one
sign-free magnitude, 1e-16 each)."""
import numpy as np
import pytest

import oracle as O
import tng
from conftest import consistent, rel_err

pytestmark = pytest.mark.gpu

D, F = tng.DIRICHLET, tng.FREESLIP


def field(om, ncomp, seed, scale=1.0):
    r = np.random.default_rng(seed)
    return consistent(om, scale * r.uniform(-1, 1, ((ncomp,) if ncomp > 1 else ()) + om.shape))


def vec(dom, data, dtype=tng.F64):
    return (tng.VectorQ1Vec if data.ndim == 5 else tng.VectorQ1Scalar)(dom, dtype).upload(data)


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
