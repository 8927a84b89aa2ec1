"""Rounding of the FP32 elastic kernels: the error of four steps of smooth
waves against the FP64 oracle is no larger than that of the MFMA kernels that
the same solvers ran on before the sparse kernels (measured on this problem)."""
import numpy as np
import pytest

import oracle as orc
from edge_amd import mesh as M
from edge_amd import setups as S
from edge_amd.solver import ElasticSolver

pytestmark = pytest.mark.gpu
# error of the MFMA kernels, (order, runs) -> relative L2; one run: the element-batched ones
MFMA_ERROR = {(2, 1): 1.492e-7, (2, 16): 1.600e-7, (3, 1): 1.963e-7, (3, 16): 2.069e-7,
              (4, 1): 2.780e-7, (4, 16): 2.797e-7, (5, 1): 3.828e-7, (5, 16): 3.786e-7}


def error(order, runs, seed=11, steps=4):
    """(FP32 solver against the FP64 oracle, from the same FP32 DOFs)"""
    import torch
    m = M.box((5, 5, 4), jitter=0.1, seed=seed)
    rho, lam, mu = S.random_materials(m.n_el, seed=seed)
    dt = S.dt_cfl(m, rho, lam, mu, order)
    rng = np.random.default_rng(seed)
    d = np.stack([S.project(m, order, S.PlaneWave(2.5, 25.0, 12.5, 2 * np.pi * rng.permutation([1, 2, -1])))[..., 0]
                  for _ in range(runs)], axis=-1)
    gd = torch.from_numpy(d.astype(np.float32)).cuda().contiguous()
    d = gd.double().cpu().numpy()
    s = ElasticSolver(m, order, runs, 32, rho, lam, mu)
    s.step(gd, torch.zeros_like(gd), dt, steps)
    got = gd.double().cpu().numpy()
    s.close()
    orc.MeshOracle(m, order, runs, rho=rho, lam=lam, mu=mu).step(d, np.zeros_like(d), dt, steps)
    return float(np.linalg.norm(got - d) / np.linalg.norm(d))


@pytest.mark.parametrize("order,runs", [(o, r) for o in (2, 3, 4, 5) for r in (1, 16)])
def test_error_is_that_of_the_mfma_kernels(gpu, order, runs):
    assert error(order, runs) <= MFMA_ERROR[order, runs]
