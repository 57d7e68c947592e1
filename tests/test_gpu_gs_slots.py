"""Multicolour Gauss-Seidel on tiled slots (k_gs_colour) at the edges of its
layout, against the oracle's V-cycle: hub rows of several hundred entries
(more than 64 lanes hold at eight slots each), leaf rows of one entry, colours
of one row and of row counts that leave a tile partly filled, halves with no
entries (the first and the last colour), every order and one to three
sweeps.

Tolerances: FP64 1e-12, FP32 1e-5, BF16-finest 3e-2 relative, as for the
V-cycle in test_gpu_poisson.py."""
import numpy as np
import pytest
import scipy.sparse as sp

from oracle import h8_oracle as O


def hub_system(n=1203, hubs=3, seed=4):
    """SPD: a path with `hubs` rows coupled to most of the others."""
    rng = np.random.default_rng(seed)
    i = np.arange(n - 1)
    r, c, v = [i], [i + 1], [-1.0 - rng.random(n - 1)]
    for h in range(hubs):
        j = np.flatnonzero(rng.random(n) < (0.6, 0.45, 0.02)[h % 3])
        j = j[np.abs(j - h * 17) > 1]
        r.append(np.full(j.size, h * 17))
        c.append(j)
        v.append(-0.01 - 0.02 * rng.random(j.size))
    r, c, v = (np.concatenate(x) for x in (r, c, v))
    U = sp.coo_matrix((v, (r, c)), shape=(n, n)).tocsr()
    U = U + U.T
    A = (U + sp.diags(1.0 + np.asarray(abs(U).sum(axis=1)).ravel())).tocsr()
    A.sort_indices()
    return A


@pytest.mark.gpu
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("fp32", 1e-5), ("bf16", 3e-2)])
@pytest.mark.parametrize("order,sweeps", [("symmetric", 1), ("symmetric", 2), ("forward", 1), ("forward", 3),
                                          ("backward", 1), ("backward", 2)])
def test_slots_match_oracle(order, sweeps, precision, tol):
    from nodals_amd._lib import System

    A = hub_system()
    S = System(A.indptr.astype(np.int64), A.indices.astype(np.int32), A.data,
               f"precision={precision} smoother=mcgs sweeps={sweeps} order={order} terminal=100")
    vc = O.VCycle(S.hierarchy(), O.Smoother(kind="mcgs", mcgs_fine_sweeps=sweeps, mcgs_coarse_sweeps=sweeps,
                                            mcgs_order=order))
    vc.set_fine(A, A.diagonal())
    r = np.random.default_rng(2).standard_normal(A.shape[0])
    z, zo = S.precond(r), vc.apply(r)
    err = float(np.linalg.norm(z - zo) / np.linalg.norm(zo))
    print(f"\n[gpu] slots, {order} x {sweeps}, {precision}: relative difference {err:.2e}", flush=True)
    assert err < tol
    S.close()


@pytest.mark.gpu
@pytest.mark.parametrize("order,sweeps", [("symmetric", 2), ("forward", 2), ("backward", 1)])
def test_split_colours_match_oracle(order, sweeps):
    """Hub rows of thousands of entries: their colours are cut into classes by
    width, which also gives the layout a row list of its own."""
    from nodals_amd._lib import System
    from tests.test_gs_layout import hub_system as hubs

    A = hubs(12001, 2)
    S = System(A.indptr.astype(np.int64), A.indices.astype(np.int32), A.data,
               f"precision=fp64 smoother=mcgs sweeps={sweeps} order={order} terminal=100")
    widest, slots = int(np.diff(A.indptr).max()), S.get("gs_slots", 3, np.int64)
    assert slots.max() < 1000 * widest  # the padded colours would take some 6,000 rows x 4,800 entries
    vc = O.VCycle(S.hierarchy(), O.Smoother(kind="mcgs", mcgs_fine_sweeps=sweeps, mcgs_coarse_sweeps=sweeps,
                                            mcgs_order=order))
    vc.set_fine(A, A.diagonal())
    r = np.random.default_rng(2).standard_normal(A.shape[0])
    z, zo = S.precond(r), vc.apply(r)
    err = float(np.linalg.norm(z - zo) / np.linalg.norm(zo))
    print(f"\n[gpu] split colours, {order} x {sweeps}: levels {S.level_rows}, relative difference {err:.2e}", flush=True)
    assert err < 1e-12
    S.close()


@pytest.mark.gpu
@pytest.mark.parametrize("precision,tol", [("fp32", 1e-5), ("bf16", 3e-2)])
@pytest.mark.parametrize("order", ["symmetric", "forward"])
def test_tiny_diagonals(order, precision, tol):
    """Rows whose diagonal is below the reciprocal of the largest FP32 number:
    the quotient by it is finite, a product with its reciprocal is not."""
    from nodals_amd._lib import System
    from tests.test_gpu_sys_option_limits import weighted_laplacian

    A, tiny, m = weighted_laplacian(9), 2.0 ** -130, 40
    n = A.shape[0]
    rng = np.random.default_rng(0)
    link = sp.coo_matrix((np.full(m, -tiny / 2), (np.arange(m), rng.choice(n, m, replace=False))), shape=(m, n))
    B = sp.bmat([[A, link.T], [link, sp.diags([tiny] * m)]]).tocsr()
    B.sort_indices()
    S = System(B.indptr.astype(np.int64), B.indices.astype(np.int32), B.data,
               f"precision={precision} smoother=mcgs sweeps=1 order={order} terminal=100")
    vc = O.VCycle(S.hierarchy(), O.Smoother(kind="mcgs", mcgs_order=order))
    vc.set_fine(B, B.diagonal())
    r = np.concatenate([rng.standard_normal(n), tiny * rng.integers(-8, 9, m) / 4.0])
    z, zo = S.precond(r), vc.apply(r)
    print(f"\n[gpu] tiny diagonals, {order}, {precision}", flush=True)
    for part in (slice(0, n), slice(n, n + m)):
        assert np.linalg.norm(z[part] - zo[part]) <= tol * np.linalg.norm(zo[part])
    S.close()
