"""Storage of the multicolour Gauss-Seidel slots (csrc/host/gs_layout.hpp, no
GPU): linear in the entries, also where a colour holds a few rows of thousands
of entries beside thousands of short ones."""
import numpy as np
import scipy.sparse as sp

from nodals_amd import p1
from nodals_amd._lib import System


def hub_system(n, hubs, share=0.4, seed=4):
    """SPD: a path with `hubs` rows coupled to a share of the others."""
    rng = np.random.default_rng(seed)
    i = np.arange(n - 1)
    r, c, v = [i], [i + 1], [-1.0 - rng.random(n - 1)]
    for h in range(hubs):
        j = np.flatnonzero(rng.random(n) < share)
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


def slots(A, **kw):
    S = System(A.indptr.astype(np.int64), A.indices.astype(np.int32), A.data, "terminal=100", device=False)
    s = S.get("gs_slots", 3, np.int64)
    S.close()
    return s


def test_hub_rows_keep_storage_linear():
    for n, hubs in ((4000, 1), (30000, 2)):
        A = hub_system(n, hubs)
        # at most four slots an entry and row, and 2^16 a colour
        assert np.all(slots(A) <= 4 * (A.nnz + n) + 8 * 65536), (n, hubs)


def test_mesh_operator_storage():
    row, col, val = p1.kuhn_p1_laplacian(23)
    A = sp.csr_matrix((val, col, row))
    lower, upper, both = slots(A)
    off = A.nnz - A.shape[0]
    assert lower < 1.7 * off / 2 and upper < 1.7 * off / 2 and both < 1.3 * off
