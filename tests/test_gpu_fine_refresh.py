"""Fine Schur refresh at cell counts that leave the last block of sixteen rows
partly empty and with rows both shorter and longer than one pass of a row's
lanes (80 nonzeros), for the value types and row-sum options, against the
oracle.

Tolerance: 1e-12 relative, float64 sums of at most 24 products per entry in
another order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "core,ring,nslab,args",
    [(2, 1, 2, []), (3, 1, 5, ["--amg-precision", "fp32"]), (3, 2, 7, ["--amg-smoother", "l1jacobi"]),
     (3, 2, 7, ["--amg-precision", "bf16", "--amg-smoother", "l1jacobi"])])
def test_refresh_matches_oracle(tmp_path, core, ring, nslab, args):
    from nodals_amd import _lib, meshgen
    from oracle import h8_oracle as O

    d = str(meshgen.write_pipe_case(tmp_path / "pipe", core=core, ring=ring, nslab=nslab))
    print(f"\n[gpu] refresh core={core} ring={ring} nslab={nslab} {args}", flush=True)
    h = _lib.H8(["--mesh", d, "--max-outer", "10", "--verbose", "0", *args])
    case = O.case_from_product(h)
    rng = np.random.default_rng(core * 100 + nslab)
    for x in range(3):
        h.set(f"u{x}", 0.3 * rng.standard_normal(case.nv))
    h.set("p", rng.standard_normal(case.nc))
    for alpha in (0.5, 0.8):  # the second call: new weights over the first's
        h.assemble(alpha)
        h.pressure_refresh()
        A, diag = O.fine_refresh(case, h.get("rau", case.nv))
        val = h.get("fine_val", A.nnz)
        assert np.linalg.norm(val - A.data) <= 1e-12 * np.linalg.norm(A.data)
        scale = np.abs(A).max(axis=1).toarray().ravel()  # row by row: no short row hides behind a long one
        err = np.maximum.reduceat(np.abs(val - A.data), A.indptr[:-1])
        assert np.all(err <= 1e-12 * scale)
        assert np.allclose(h.get("fine_diag", case.nc), diag, rtol=1e-12, atol=0)
    h.close()
