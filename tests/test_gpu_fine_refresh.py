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


def doubled_cell_case(directory, core=4, ring=2, nslab=6):
    """A pipe with one inner cell doubled: its copy shares all four vertices and
    two faces with it, so their nonzero has six terms where a conforming
    neighbour has at most four.  The faces that lose their partner become
    outlet faces."""
    from nodals_amd import meshgen

    pts, tets = meshgen.straight_pipe(core, ring, nslab)
    ends = (0.0, pts[:, 2].max())

    def classify(fc, n):
        return np.where(np.abs(fc[:, 2] - ends[0]) < 1e-8, 1, np.where(np.abs(fc[:, 2] - ends[1]) < 1e-8, 2, 0))

    m = meshgen.tets_to_polymesh(pts, tets, classify, ["patch_0_0", "patch_2_0", "patch_1_0"])
    faces, owner, neighbour = m.faces.tolist(), m.owner.tolist(), m.neighbour.tolist()
    ni, nc = len(neighbour), m.n_cells
    outer = {v for f in faces[ni:] for v in f}
    of = {}
    for f in range(ni):
        of.setdefault(owner[f], []).append(f)
        of.setdefault(neighbour[f], []).append(f)
    cell = next(c for c in sorted(of) if len(of[c]) == 4 and not any(v in outer for f in of[c] for v in faces[f]))
    for k, f in enumerate(of[cell]):
        out = faces[f] if owner[f] == cell else faces[f][::-1]
        if k < 2:  # now between the cell and its copy
            faces.append(out[::-1])
            owner.append(neighbour[f] if owner[f] == cell else owner[f])
            faces[f], owner[f], neighbour[f] = out, cell, nc
        else:
            faces.append(list(out))
            owner.append(nc)
    name, start, count = m.patches[-1]
    m.patches[-1] = (name, start, count + 4)
    m.faces, m.owner, m.neighbour = np.array(faces), np.array(owner), np.array(neighbour)
    return str(meshgen.write_polymesh(directory, m)), cell, nc


@pytest.mark.parametrize("args", [[], ["--amg-precision", "fp32", "--amg-smoother", "l1jacobi"]])
def test_refresh_of_unpacked_terms(tmp_path, args):
    """A nonzero of more terms than a word holds goes through the term list."""
    from nodals_amd import _lib
    from oracle import h8_oracle as O

    d, cell, copy = doubled_cell_case(tmp_path / "doubled")
    h = _lib.H8(["--mesh", d, "--max-outer", "10", "--verbose", "0", *args])
    case = O.case_from_product(h)
    shared = set(case.cell_ref[cell]) & set(case.cell_ref[copy])
    assert len([g for g in shared if g >= 0]) == 6
    print(f"\n[gpu] refresh of a doubled cell {args}", flush=True)
    rng = np.random.default_rng(8)
    for x in range(3):
        h.set(f"u{x}", 0.3 * rng.standard_normal(case.nv))
    h.assemble(0.5)
    h.pressure_refresh()
    A, diag = O.fine_refresh(case, h.get("rau", case.nv))
    val = h.get("fine_val", A.nnz)
    scale = np.abs(A).max(axis=1).toarray().ravel()
    assert np.all(np.maximum.reduceat(np.abs(val - A.data), A.indptr[:-1]) <= 1e-12 * scale)
    k = A.indptr[cell] + np.flatnonzero(A.indices[A.indptr[cell]:A.indptr[cell + 1]] == copy)
    assert abs(val[k] - A.data[k]) <= 1e-12 * abs(A.data[k])
    h.close()
