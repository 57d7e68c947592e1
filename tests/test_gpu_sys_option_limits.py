"""Smoother counts and orders at and beyond the ends of their ranges through the
explicit-system options: a Jacobi or Chebyshev smoother makes at least one
step, a multicolour one without passes (a count below one, an order that is
not one of the three) leaves the cycle its coarse corrections alone.  Checked
on a hierarchy whose coarse levels are one dense product and on one with an
explicit coarse level, after a pass on other data (nothing is left over from
it), against the oracle's level-by-level V-cycle.

Tolerance: 1e-12 relative, FP64 sums in another order."""
import numpy as np
import pytest
import scipy.sparse as sp

from oracle import h8_oracle as O

pytestmark = pytest.mark.gpu

NO_PASS = dict(kind="mcgs", mcgs_fine_sweeps=0, mcgs_coarse_sweeps=0)
CASES = [
    ("smoother=mcgs sweeps=0", NO_PASS),
    ("smoother=mcgs sweeps=-3 order=forward", NO_PASS),
    ("smoother=mcgs sweeps=2 order=upwards", NO_PASS),
    ("smoother=jacobi sweeps=0 omega=0.7", dict(kind="jacobi")),
    ("smoother=l1jacobi sweeps=-2 omega=0.7", dict(kind="l1jacobi")),
    ("smoother=cheb2 cheb_degree=-1 power_its=8", dict(kind="cheb2", cheb_degree=-1)),
]


def weighted_laplacian(n, seed=5):
    """7-point Laplacian of an n^3 grid with random weights and a mass term."""
    i = np.arange(n ** 3).reshape(n, n, n)
    a = np.concatenate([i[1:].ravel(), i[:, 1:].ravel(), i[:, :, 1:].ravel()])
    b = np.concatenate([i[:-1].ravel(), i[:, :-1].ravel(), i[:, :, :-1].ravel()])
    w = -1.0 - np.random.default_rng(seed).random(a.size)
    U = sp.coo_matrix((np.r_[w, w], (np.r_[a, b], np.r_[b, a])), shape=(n ** 3, n ** 3)).tocsr()
    A = (U + sp.diags(0.01 - np.asarray(U.sum(axis=1)).ravel())).tocsr()
    A.sort_indices()
    return A


@pytest.mark.parametrize("n,hierarchy", [(11, "terminal=16"), (33, "hierarchy=cf terminal=500")])
@pytest.mark.parametrize("options,smoother", CASES)
def test_counts_and_orders_out_of_range(options, smoother, n, hierarchy):
    from nodals_amd._lib import System

    A = weighted_laplacian(n)
    print(f"\n[gpu] {options} {hierarchy}, {n}^3", flush=True)
    S = System(A.indptr.astype(np.int64), A.indices.astype(np.int32), A.data,
               f"precision=fp64 {options} {hierarchy}")
    if n == 33:
        assert S.level_rows[0] > 9000  # above the dense product's largest level
    vc = O.VCycle(S.hierarchy(), O.Smoother(**smoother))
    vc.set_fine(A, A.diagonal())
    rng = np.random.default_rng(3)
    S.precond(1e3 * rng.standard_normal(A.shape[0]))
    r = rng.standard_normal(A.shape[0])
    z, zo = S.precond(r), vc.apply(r)
    assert np.linalg.norm(z - zo) <= 1e-12 * np.linalg.norm(zo)
    S.close()
