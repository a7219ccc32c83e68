"""GPU test of the AMG set-up's sparse products and MIS-2 rounds at the sizes where
they change course: one partial block, row counts that leave one, and rows short and
wide of the 32 lanes, with every neighbour strong and with weak entries dropped.

Aggregates are integer work and equal the oracle's.  Each Galerkin entry is a sum of
products in FP64 in any order: the difference from another order is at most
2 k eps (|R| |A| |P|) with k the number of terms, taken from the patterns.
"""
import numpy as np
import pytest
import scipy.sparse as sp

torch = pytest.importorskip("torch")

import nalu_amd as na  # noqa: E402
from nalu_amd.problems import lowmach_problem  # noqa: E402
from oracle import amg as M  # noqa: E402

pytestmark = pytest.mark.gpu


def level(ls, l, which="A"):
    rp, ci, v, n, m = ls.amg_level_csr(l, which)
    return sp.csr_matrix((v, ci, rp), shape=(n, m))


def ones(A):
    B = A.copy()
    B.data = np.ones_like(B.data)
    return B


@pytest.mark.parametrize("n,drop_tol", [(3, 0.0), (13, 0.0), (13, 0.02), (24, 0.0), (24, 0.02)])
def test_products_and_rounds(n, drop_tol):
    print("case: amg products n=%d drop_tol=%g" % (n, drop_tol), flush=True)
    P = lowmach_problem(n, rho_sigma=0.3, seed=5)
    mesh = na.Mesh(P["coords"], P["conn"])
    ls = na.LinearSystem(1, na.SolverConfig("cg", "muelu", tolerance=1e-8))
    ls.set_muelu_params(na.MueLuParams(max_coarse_size=8, cheb_degree=2, drop_tol=drop_tol))
    ls.buildElemToNodeGraph(mesh)
    ls.finalizeLinearSystem()
    ls.zeroSystem()
    dev = lambda k: torch.as_tensor(np.ascontiguousarray(P[k]), dtype=torch.float64, device="cuda:0")  # noqa: E731
    na.assemble_continuity(ls, mesh, dev("rho"), dev("p"), dev("u"), dev("gpdx"), tau=1.0)
    ls.loadComplete()
    ls.removeRhsMean()
    ls.precond_setup()
    eps = np.finfo(np.float64).eps
    L = len(ls.amg_info()["rows"])
    assert L >= 2
    for l in range(L - 1):
        A, Pl = level(ls, l), level(ls, l, "P")
        if A.shape[0] <= 4000:
            agg, nc, _ = M.aggregate(A, drop_tol)
            assert np.array_equal(ls.amg_aggregates(l), agg)
        AP = (ones(A) @ ones(Pl)).tocsr()
        print("  level %d rows %d widest A %d, P %d, AP %d, avg AP %.1f" %
              (l, A.shape[0], np.diff(A.indptr).max(), np.diff(Pl.indptr).max(), np.diff(AP.indptr).max(),
               AP.nnz / A.shape[0]), flush=True)
        ref = (Pl.T @ (A @ Pl)).tocsr()
        mag = (abs(Pl).T @ (abs(A) @ abs(Pl))).tocsr()
        terms = (ones(Pl).T @ AP).max()
        D = abs(level(ls, l + 1) - ref)
        excess = (D - 2.0 * terms * eps * mag).tocsr()
        assert excess.nnz == 0 or excess.data.max() <= 0.0
