"""Storage of the multicolour Gauss-Seidel slots (csrc/host/gs_layout.hpp, no
GPU): linear in the entries, also where a colour holds a few rows of thousands
of entries beside thousands of short ones."""
import resource
import subprocess
import sys
from pathlib import Path

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


LIMITED = """
import resource, sys
import numpy as np
from nodals_amd._lib import System
from tests.test_gs_layout import hub_system
A = hub_system(12001, 2)
S = System(A.indptr.astype(np.int64), A.indices.astype(np.int32), A.data, "terminal=100", device=False)
used = int(open("/proc/self/statm").read().split()[0]) * resource.getpagesize()
resource.setrlimit(resource.RLIMIT_AS, (used + int(sys.argv[1]), resource.RLIM_INFINITY))
try:
    print(*S.get("gs_slots", 3, np.int64))
except Exception as e:
    print(type(e).__name__, e)
"""


def test_layout_without_room_for_threads():
    """The workers' stacks (8 MB each) do not fit the address space: their
    colours are laid out by the caller; without room for the layout either,
    the call ends with an error, never the process."""
    root = Path(__file__).resolve().parents[1]
    out = []
    for room in (7 << 20, 1 << 18):
        r = subprocess.run([sys.executable, "-c", LIMITED, str(room)], cwd=root, capture_output=True, text=True,
                           timeout=120, preexec_fn=lambda: resource.setrlimit(resource.RLIMIT_STACK, (8 << 20, 8 << 20)))
        assert r.returncode == 0, r.stderr[-500:]
        out.append(r.stdout.strip())
    assert out[0] == " ".join(map(str, slots(hub_system(12001, 2))))
    assert out[1] == out[0] or out[1].startswith(("NodalsError", "MemoryError"))
