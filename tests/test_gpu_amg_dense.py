"""The dense coarse operator of the V-cycle (the cycle below a small level
as one matrix product) against the oracle's level-by-level V-cycle: every
smoother, several levels below the dense one, row counts on both sides of
the product's four-row blocks and not multiples of its padding.

Tolerances: FP64 1e-12 relative (n sums of rounding 1.1e-16 each, n < 1e4);
FP32 1e-5 relative, the FP32 V-cycle's own bound (test_gpu_poisson.py)."""
import numpy as np
import pytest
import scipy.sparse as sp

from nodals_amd import p1
from oracle import h8_oracle as O

pytestmark = pytest.mark.gpu

CASES = [
    # cube, system options, oracle smoother
    (10, "smoother=mcgs sweeps=1 order=symmetric terminal=16", dict(kind="mcgs")),
    (9, "smoother=mcgs sweeps=2 order=backward terminal=16",
     dict(kind="mcgs", mcgs_fine_sweeps=2, mcgs_coarse_sweeps=2, mcgs_order="backward")),
    (17, "smoother=jacobi sweeps=1 omega=0.7 terminal=16", dict(kind="jacobi")),
    (13, "smoother=jacobi sweeps=3 omega=0.7 terminal=16",
     dict(kind="jacobi", jacobi_fine_sweeps=3, jacobi_coarse_sweeps=3)),
    (16, "smoother=l1jacobi sweeps=1 omega=0.7 terminal=16", dict(kind="l1jacobi")),
    (15, "smoother=cheb2 power_its=8 terminal=16", dict(kind="cheb2")),
    # a dense level of more than 4096 rows (four rows a block)
    (23, "smoother=cheb2 cheb_degree=6 power_its=8 hierarchy=cf terminal=200", dict(kind="cheb2", cheb_degree=6)),
]


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("fp32", 1e-5)])
@pytest.mark.parametrize("n,options,smoother", CASES)
def test_dense_coarse_cycle_matches_levels(n, options, smoother, precision, tol):
    from nodals_amd._lib import System

    row, col, val = p1.kuhn_p1_laplacian(n)
    A = sp.csr_matrix((val, col, row))
    S = System(row, col, val, f"precision={precision} {options}")
    print(f"\n[gpu] dense coarse cycle, {n}^3, {options}, {precision}, level rows {S.level_rows}", flush=True)
    vc = O.VCycle(S.hierarchy(), O.Smoother(**smoother))
    vc.set_fine(A, A.diagonal())
    r = p1.poisson_rhs(A.shape[0], seed=3)
    z, zo = S.precond(r), vc.apply(r)
    err = float(np.linalg.norm(z - zo) / np.linalg.norm(zo))
    print(f"[gpu]   relative difference {err:.2e}", flush=True)
    assert err < tol
    S.close()
