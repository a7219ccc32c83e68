"""Solver kernels whose launch shape depends on the size: the Gram-Schmidt dots and
updates (row remainders of their 1024- and 128-row tiles, one to several vectors to
a wave), and the sweeps and products with several waves to a chunk of rows (systems
of few chunks) against the plain ones (large systems, tests at full size).

Solves reach the relative residual they are asked for, evaluated by the oracle; the
one-sweep SGS and the product are within 1e-13 and 1e-12 of the oracle's largest
entry (sums of 27 terms of one row; the mixed-precision system applies SGS in FP64
to its FP32-assembled matrix here)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import nalu_amd as na  # noqa: E402
from nalu_amd.problems import heat_problem  # noqa: E402

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def dev(a, dtype=torch.float64):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=dtype, device=DEV)


# 64, 125, 1331, 2197, 9261 rows: below one wave's rows, one partial and several 1024-row chunks
@pytest.mark.parametrize("n", [3, 4, 10, 12, 20])
@pytest.mark.parametrize("method,precision", [("gmres", "fp64"), ("fgmres", "mixed"), ("cg", "fp64")])
def test_solve_sizes(oracle, n, method, precision):
    print("case: %s %s heat %d^3" % (method, precision, n), flush=True)
    P = heat_problem(n, seed=77)
    mesh = na.Mesh(P["coords"], P["conn"])
    ls = na.LinearSystem(1, na.SolverConfig(method, "sgs", tolerance=1e-10, kspace=12, max_iterations=800,
                                            precision=precision))
    ls.buildElemToNodeGraph(mesh)
    ls.finalizeLinearSystem()
    T, k = dev(P["T"]), dev(P["k"])
    ls.zeroSystem()
    na.assemble_scalar_diff(ls, mesh, T, k)
    if method != "cg":
        ls.applyDirichletBCs(dev(P["bc_nodes"], torch.int32), T, dev(P["bc_values"]))
    ls.loadComplete()
    rp, ci, v, r = ls.csr()
    N = r.shape[0]
    if method == "cg":  # symmetric: the pure-Neumann operator with a zero-mean rhs
        rng = np.random.default_rng(n)
        r = rng.normal(size=N)
        r -= r.mean()
    # the product and one SGS application against the oracle
    rng = np.random.default_rng(5)
    x = rng.normal(size=N)
    y, z = dev(np.zeros(N)), dev(np.zeros(N))
    ls.precond_setup()
    ls.precond_apply(dev(x), z)
    cp, cr = ls.coloring()
    zo = oracle.mcsgs_apply(rp, ci, v, cp, cr, x)
    assert np.abs(z.cpu().numpy() - zo).max() <= 1e-13 * np.abs(zo).max()
    perm = ls.permutation()
    yp = dev(np.zeros(N))
    ls.spmv_permuted(dev(x[perm]), yp)
    yo = oracle.spmv(rp, ci, v, x)
    assert np.abs(yp.cpu().numpy() - yo[perm]).max() <= 1e-12 * np.abs(yo).max()
    sol = dev(np.zeros(N))
    st, it, rel = ls.solve_rhs(dev(r), sol)
    res = np.linalg.norm(r - oracle.spmv(rp, ci, v, sol.cpu().numpy())) / np.linalg.norm(r)
    print("  iterations %d, relative residual %.2e (reported %.2e)" % (it, res, rel), flush=True)
    assert st == 0 and res <= 1e-10 * 1.01


def test_gmres_iterations_match_the_oracle(oracle):
    """Iteration counts of the FP64 GMRES over several restart cycles (the next
    column's product is enqueued before the current one's norm is read; the cycle
    ends, the last column and the converged column must not count it)."""
    P = heat_problem(10, seed=5)
    mesh = na.Mesh(P["coords"], P["conn"])
    for kspace, maxit in ((5, 500), (12, 500), (50, 500), (7, 9), (50, 1)):
        ls = na.LinearSystem(1, na.SolverConfig("gmres", "sgs", tolerance=1e-9, kspace=kspace, max_iterations=maxit))
        ls.buildElemToNodeGraph(mesh)
        ls.finalizeLinearSystem()
        T = dev(P["T"])
        ls.zeroSystem()
        na.assemble_scalar_diff(ls, mesh, T, dev(P["k"]))
        ls.applyDirichletBCs(dev(P["bc_nodes"], torch.int32), T, dev(P["bc_values"]))
        ls.loadComplete()
        rp, ci, v, r = ls.csr()
        cp, cr = ls.coloring()
        x = dev(np.zeros_like(r))
        st, it, rel = ls.solve_rhs(dev(r), x)
        xo, ito, _ = oracle.gmres(rp, ci, v, r, kspace=kspace, maxit=maxit, tol=1e-9, precond="mcsgs", color_ptr=cp,
                                  color_rows=cr)
        print("  kspace %d maxit %d: %d iterations, oracle %d" % (kspace, maxit, it, ito), flush=True)
        assert abs(it - ito) <= 1 and it <= maxit and (st == 0) == (rel <= 1e-9)
