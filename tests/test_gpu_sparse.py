"""The kernels over the matrices' non-zeros (kernels_sparse_impl.hpp),
64 (element, run) columns per workgroup, against the FP64 oracle: every order
and run count on meshes whose last tile is partly filled, element ranges that
start inside a tile, free-surface, outflow and periodic faces in every
orientation; meshes that only the flux solvers describe, which take the other
kernels; steps that overlap on streams, and graphs."""
import numpy as np
import pytest

import oracle as orc
from edge_amd import mesh as M
from edge_amd import setups as S
from edge_amd._lib import EdgeError
from edge_amd.mesh import FA_FREE_SURFACE, FA_OUTFLOW, FA_PERIODIC
from edge_amd.solver import KERNEL_EC64, KERNEL_GENERIC, KERNEL_MFMA, PATH_PROJECTIONS, ElasticSolver

pytestmark = pytest.mark.gpu
TOL = {32: 1e-5, 64: 1e-12}  # against the FP64 oracle, as every path of the precision
NP = {32: np.float32, 64: np.float64}


def rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.linalg.norm((a - b).ravel()) / np.linalg.norm(b.ravel()))


def _problem(runs, order, precision=32, n=(3, 4, 3), seed=5):
    import torch
    m = M.box(n, bc=(FA_FREE_SURFACE, FA_OUTFLOW, FA_PERIODIC), jitter=0.1, seed=seed)
    rho, lam, mu = S.random_materials(m.n_el, seed=seed)
    d0 = np.random.default_rng(order).normal(size=(m.n_el, 9, S.n_modes(order), runs)).astype(NP[precision])
    dev = torch.from_numpy(d0).cuda()
    return m, (rho, lam, mu), S.dt_cfl(m, rho, lam, mu, order), d0.astype(np.float64), dev


@pytest.mark.parametrize("runs", [1, 8, 16])
@pytest.mark.parametrize("order", [2, 3, 4, 5])
@pytest.mark.parametrize("precision", [32, 64])
def test_steps_match_oracle(gpu, precision, order, runs):
    """162 elements (2 tiles of 64 and 34, 20 of 8 and 2, 40 of 4 and 2): local,
    neighbour, then three steps in one call."""
    import torch
    m, mat, dt, d, gd = _problem(runs, order, precision, n=(3, 3, 3))
    if (precision, order, runs) == (64, 5, 16):  # no kernel that reads tInt fits
        with pytest.raises(EdgeError, match="no kernel"):
            ElasticSolver(m, order, runs, precision, *mat)
        return
    tol = TOL[precision]
    s = ElasticSolver(m, order, runs, precision, *mat)
    assert s.kernel_info()[0] == (2 if (precision, runs) == (32, 16) else 5)
    mo = orc.MeshOracle(m, order, runs, rho=mat[0], lam=mat[1], mu=mat[2])
    t, gt = np.zeros_like(d), torch.zeros_like(gd)
    mo.local(d, t, dt)
    s.local(gd, gt, dt)
    assert rel(gt.cpu().numpy(), t) <= tol
    assert rel(gd.cpu().numpy(), d) <= tol
    mo.neigh(d, t)
    s.neigh(gd, gt)
    assert rel(gd.cpu().numpy(), d) <= tol
    mo.step(d, t, dt, 3)
    s.step(gd, gt, dt, 3)
    assert rel(gt.cpu().numpy(), t) <= tol
    assert rel(gd.cpu().numpy(), d) <= tol
    s.close()


@pytest.mark.parametrize("runs", [1, 8, 16])
@pytest.mark.parametrize("precision", [32, 64])
def test_ranges_equal_whole(gpu, precision, runs):
    """Element ranges that start and end inside a tile (and inside a block of
    the constants) write their elements only, and the same values as one call."""
    import torch
    order = 4
    m, mat, dt, _, gd = _problem(runs, order, precision)
    s = ElasticSolver(m, order, runs, precision, *mat)
    cuts = [0, 1, 62, 67, 130, 131, 215, m.n_el]
    a, ta = gd.clone(), torch.zeros_like(gd)
    s.local(a, ta, dt)
    local = a.clone()
    s.neigh(a, ta)
    b, tb = gd.clone(), torch.zeros_like(gd)
    for lo, hi in zip(cuts[:-1], cuts[1:]):
        before, tbefore = b.clone(), tb.clone()
        s.local(b, tb, dt, first=lo, n=hi - lo)
        assert torch.equal(b[:lo], before[:lo]) and torch.equal(b[hi:], before[hi:])
        assert torch.equal(tb[:lo], tbefore[:lo]) and torch.equal(tb[hi:], tbefore[hi:])
    assert torch.equal(local, b) and torch.equal(ta, tb)
    for lo, hi in zip(cuts[:-1], cuts[1:]):
        before = b.clone()
        s.neigh(b, tb, first=lo, n=hi - lo)
        assert torch.equal(b[:lo], before[:lo]) and torch.equal(b[hi:], before[hi:])
    assert torch.equal(a, b)
    s.close()


@pytest.mark.parametrize("swap", [False, True])
@pytest.mark.parametrize("runs", [1, 8, 16])
def test_neighbours_that_do_not_pair(gpu, runs, swap):
    """One face's neighbour replaced by another element: the projections no
    longer have one receiver each, so a kernel runs that reads tInt.  Two faces'
    neighbours swapped: they have, but the faces' two elements are not each
    other's neighbours, so the kernels run that read the flux solvers."""
    import torch
    order = 3
    m, mat, dt, d, gd = _problem(runs, order)
    inner = np.argwhere((m.fa_el[m.el_fa] >= 0).all(axis=2) & (m.fa_type[m.el_fa] == 0))
    (el, fa), (e2, f2) = inner[5], inner[90]
    if swap:
        for a in (m.el_fa_el, m.f_id, m.v_id):
            a[el, fa], a[e2, f2] = a[e2, f2], a[el, fa]
    else:
        m.el_fa_el[el, fa] = (m.el_fa_el[el, fa] + 7) % m.n_el
    s = ElasticSolver(m, order, runs, 32, *mat)
    kernel, flags = s.kernel_info()
    assert kernel == {1: KERNEL_EC64 if swap else KERNEL_GENERIC, 8: KERNEL_GENERIC, 16: KERNEL_MFMA}[runs]
    assert bool(flags & PATH_PROJECTIONS) == (swap and runs != 8)
    mo = orc.MeshOracle(m, order, runs, rho=mat[0], lam=mat[1], mu=mat[2])
    t, gt = np.zeros_like(d), torch.zeros_like(gd)
    mo.step(d, t, dt, 2)
    s.step(gd, gt, dt, 2)
    assert rel(gd.cpu().numpy(), d) <= TOL[32]
    s.close()


@pytest.mark.parametrize("form", ["skew frame", "long normal", "free surface inside"])
@pytest.mark.parametrize("precision,runs", [(32, 1), (32, 8), (32, 16), (64, 1), (64, 8)])
def test_general_forms_of_a_face(gpu, precision, runs, form):
    """Faces that only their flux solvers describe: tangents or a normal off
    the orthonormal frame, a free surface that two elements share."""
    import torch
    order = 3
    m, mat, dt, d, gd = _problem(runs, order, precision)
    f = np.argwhere((m.fa_el >= 0).all(axis=1) & (m.fa_type == 0))[17, 0]
    if form == "skew frame":
        m.tangents[f, 0] += 0.1 * m.tangents[f, 1]
    elif form == "long normal":
        m.normals[f] *= 1 + (1e-9 if precision == 64 else 1e-5)  # (just past the bound)
    else:
        m.fa_type[f] = FA_FREE_SURFACE
    s = ElasticSolver(m, order, runs, precision, *mat)
    if runs == 8:
        assert s.kernel_info()[0] == KERNEL_GENERIC
    mo = orc.MeshOracle(m, order, runs, rho=mat[0], lam=mat[1], mu=mat[2])
    t, gt = np.zeros_like(d), torch.zeros_like(gd)
    mo.step(d, t, dt, 2)
    s.step(gd, gt, dt, 2)
    assert rel(gd.cpu().numpy(), d) <= TOL[precision]
    s.close()


@pytest.mark.parametrize("precision,runs", [(32, 8), (64, 8), (64, 16)])
def test_neighbour_step_reads_tint(gpu, precision, runs):
    """Solvers whose general kernels read tInt: a separate neighbour step takes
    what it is handed, changed since the local step, in another array, after a
    multi-step call or without any local step."""
    import torch
    order, tol = 3, TOL[precision]
    m, mat, dt, d, gd = _problem(runs, order, precision)
    s = ElasticSolver(m, order, runs, precision, *mat)
    assert s.kernel_info() == (5, 1)
    mo = orc.MeshOracle(m, order, runs, rho=mat[0], lam=mat[1], mu=mat[2])
    t, gt = np.zeros_like(d), torch.zeros_like(gd)
    t2 = (np.random.default_rng(8).normal(size=d.shape) * dt).astype(NP[precision])
    mo.neigh(d, t2.astype(np.float64))
    s.neigh(gd, torch.from_numpy(t2).cuda())
    assert rel(gd.cpu().numpy(), d) <= tol
    mo.local(d, t, dt)
    s.local(gd, gt, dt)
    gt *= 0.5
    mo.neigh(d, 0.5 * t)
    s.neigh(gd, gt)
    assert rel(gd.cpu().numpy(), d) <= tol
    mo.step(d, t, dt, 2)
    s.step(gd, gt, dt, 2)
    mo.neigh(d, t)
    s.neigh(gd, gt)
    assert rel(gd.cpu().numpy(), d) <= tol
    s.close()


@pytest.mark.parametrize("precision", [32, 64])
def test_one_run_after_and_under_capture(gpu, precision):
    """One run: multi-step calls captured by the caller before the second
    projection buffer exists (they go launch by launch), replayed between eager
    work; and a neighbour step after a multi-step call, eager and as a graph."""
    import torch
    order, tol = 4, TOL[precision]
    m, mat, dt, d, gd = _problem(1, order, precision)
    s = ElasticSolver(m, order, 1, precision, *mat)
    mo = orc.MeshOracle(m, order, 1, rho=mat[0], lam=mat[1], mu=mat[2])
    t, gt = np.zeros_like(d), torch.zeros_like(gd)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        s.step(gd, gt, dt, 2, stream=torch.cuda.current_stream())
    for _ in range(3):
        g.replay()
        torch.cuda.synchronize()
        mo.step(d, t, dt, 2)
        assert rel(gd.cpu().numpy(), d) <= tol
    for n, graph in ((2, False), (3, False), (3, True), (2, True)):
        s.step(gd, gt, dt, n, graph=graph)
        mo.step(d, t, dt, n)
        s.neigh(gd, gt)
        mo.neigh(d, t)
        assert rel(gd.cpu().numpy(), d) <= tol
    s.close()


@pytest.mark.parametrize("precision,runs", [(32, 8), (64, 16)])
def test_overlapping_steps_on_two_streams(gpu, precision, runs):
    """Solvers whose neighbour step reads tInt: steps of independent arrays
    that overlap on two streams, eager, as the solver's own graph, and captured
    by the caller and replayed beside eager ones, give the bits of steps one
    after the other (captured by the caller: with the neighbour kernel that
    reads tInt, so to rounding)."""
    import torch
    order, n, tol = 4, 3, TOL[precision]
    m, mat, dt, _, gd = _problem(runs, order, precision, n=(9, 8, 10))
    s = ElasticSolver(m, order, runs, precision, *mat)
    start = [gd, torch.flip(gd, dims=[0]) * 0.5]
    want = []
    for x in start:
        x = x.clone()
        t = torch.zeros_like(x)
        s.step(x, t, dt, 1)
        for _ in range(3):
            s.step(x, t, dt, n)
        want.append(x)
    streams = [torch.cuda.Stream() for _ in start]
    torch.cuda.synchronize()
    for graph in (False, True):  # (the first array's steps of one call as the solver's graph)
        got, tint = [x.clone() for x in start], [torch.zeros_like(x) for x in start]
        torch.cuda.synchronize()
        for k in (1, n, n, n):
            s.step(got[0], tint[0], dt, k, graph=graph and k == n, stream=streams[0])
            s.step(got[1], tint[1], dt, k, stream=streams[1])
        torch.cuda.synchronize()
        for x, w in zip(got, want):
            assert torch.equal(x, w)
    x, t = start[0].clone(), torch.zeros_like(gd)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=streams[0]):
        s.step(x, t, dt, n, stream=torch.cuda.current_stream())
    x.copy_(start[0])
    y, ty = start[1].clone(), torch.zeros_like(gd)
    torch.cuda.synchronize()
    s.step(x, t, dt, 1, stream=streams[0])
    s.step(y, ty, dt, 1, stream=streams[1])
    for _ in range(3):
        with torch.cuda.stream(streams[0]):
            g.replay()
        s.step(y, ty, dt, n, stream=streams[1])
    torch.cuda.synchronize()
    assert rel(x.cpu().numpy(), want[0].cpu().numpy()) <= tol
    assert torch.equal(y, want[1])
    s.close()


@pytest.mark.parametrize("precision,runs", [(32, 1), (64, 1), (32, 8)])
def test_repeated_graph_calls(gpu, precision, runs):
    """Calls that ask for a graph: launched, captured when the call repeats,
    replayed, with eager and other calls between, each against the oracle."""
    import torch
    order, tol = 4, TOL[precision]
    m, mat, dt, d, gd = _problem(runs, order, precision)
    s = ElasticSolver(m, order, runs, precision, *mat)
    mo = orc.MeshOracle(m, order, runs, rho=mat[0], lam=mat[1], mu=mat[2])
    t, gt = np.zeros_like(d), torch.zeros_like(gd)
    for n, graph in ((2, True), (2, True), (2, True), (3, True), (3, False), (2, True), (1, True), (1, True), (2, True)):
        mo.step(d, t, dt, n)
        s.step(gd, gt, dt, n, graph=graph)
        assert rel(gd.cpu().numpy(), d) <= tol
        assert rel(gt.cpu().numpy(), t) <= tol
    s.close()


@pytest.mark.parametrize("precision,runs,order", [(32, 8, 4), (64, 8, 3), (64, 16, 4)])
def test_fault_of_several_runs(gpu, precision, runs, order):
    """A fault between the fused launches of solvers of several runs on kernel 5
    (their tInt is written in every step for the fault's elements only), and
    between separate steps, against the coupled oracle."""
    import torch
    from edge_amd import fault as FL
    from test_gpu_fault import _problem as fault_problem
    m, rho, lam, mu, frame, glob, st0 = fault_problem(order, runs)
    dt, tol = S.dt_cfl(m, rho, lam, mu, order), TOL[precision]
    s = ElasticSolver(m, order, runs, precision, rho, lam, mu)
    assert s.kernel_info()[0] == KERNEL_EC64
    f = FL.Fault(s, m, rho, lam, mu, frame, glob, st0)
    fo = orc.FaultOracle(m, order, runs, rho, lam, mu, frame, glob, st0)
    d = 0.01 * np.random.default_rng(5).normal(size=(m.n_el, 9, S.n_modes(order), runs))
    gd = torch.tensor(d.astype(NP[precision]), device="cuda").contiguous()
    d = gd.double().cpu().numpy()
    t, gt = np.zeros_like(d), torch.zeros_like(gd)
    for n in (3, 1, 2):
        fo.step(d, t, dt, n)
        s.step(gd, gt, dt, n)
        assert rel(gd.cpu().numpy(), d) <= tol
        assert rel(gt.cpu().numpy(), t) <= tol
    fo.step(d, t, dt, 1)
    s.local(gd, gt, dt)
    f.apply(gd, gt, dt)
    s.neigh(gd, gt)
    assert rel(gd.cpu().numpy(), d) <= tol
    f.close()
    s.close()
