"""Caller-given star matrices and flux solvers (edge_el_create_raw) on the
kernels that read them: the element-batched kernels of one run and the MFMA
kernels that exchange projections, separate and fused, at every order against
the FP64 oracle.  (Geometry-built solvers of the same selectors run the
kernels over the matrices' non-zeros.)"""
import numpy as np
import pytest

import oracle as orc
from edge_amd import mesh as M
from edge_amd import setups as S
from edge_amd.mesh import FA_FREE_SURFACE, FA_OUTFLOW, FA_PERIODIC
from edge_amd.solver import KERNEL_EC64, KERNEL_MFMA, PATH_FUSED, PATH_PROJECTIONS, ElasticSolver

pytestmark = pytest.mark.gpu
TOL = {32: 1e-5, 64: 1e-12}  # against the FP64 oracle, as every path of the precision


def rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.linalg.norm((a - b).ravel()) / np.linalg.norm(b.ravel()))


@pytest.mark.parametrize("order", [2, 3, 4, 5])
@pytest.mark.parametrize("precision,runs,kernel", [(32, 1, KERNEL_EC64), (64, 1, KERNEL_EC64), (32, 16, KERNEL_MFMA)])
def test_raw_kernels_match_oracle(gpu, precision, runs, kernel, order):
    """Local, neighbour, three steps in one call, then (16 runs) the fused
    launch step by step; 162 elements fill neither a tile of 16 elements nor
    the last workgroup."""
    import torch
    m = M.box(3, bc=(FA_FREE_SURFACE, FA_OUTFLOW, FA_PERIODIC), jitter=0.1, seed=order)
    rho, lam, mu = S.random_materials(m.n_el, seed=order)
    star, fs, _ = orc.setup_mesh(m, rho, lam, mu)
    dt, tol = S.dt_cfl(m, rho, lam, mu, order), TOL[precision]
    s = ElasticSolver(m, order, runs, precision, star=star, fs=fs, kernel=kernel)
    assert s.kernel_info()[0] == kernel and s.kernel_info()[1] & PATH_PROJECTIONS
    mo = orc.MeshOracle(m, order, runs, star=star, fs=fs)
    real = torch.float64 if precision == 64 else torch.float32
    d = np.random.default_rng(order).normal(size=(m.n_el, 9, S.n_modes(order), runs))
    gd = torch.tensor(d, dtype=real, device="cuda").contiguous()
    d = gd.double().cpu().numpy()
    t, gt = np.zeros_like(d), torch.zeros_like(gd)

    def same():
        assert rel(gd.cpu().numpy(), d) <= tol
        assert rel(gt.cpu().numpy(), t) <= tol

    mo.local(d, t, dt)
    s.local(gd, gt, dt)
    same()
    mo.neigh(d, t)
    s.neigh(gd, gt)
    same()
    mo.step(d, t, dt, 3)
    s.step(gd, gt, dt, 3)
    same()
    if s.kernel_info()[1] & PATH_FUSED:
        s.local(gd, gt, dt)
        s.neigh_local(gd, gt, dt)
        s.neigh(gd, gt)
        mo.step(d, t, dt, 2)
        same()
    else:
        assert runs == 1
    s.close()
