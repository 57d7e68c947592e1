"""Smoothers of several steps: odd and even step counts (the steps alternate
between two buffers), one step on one side only, and the value types, on a
mesh whose cell count is not a multiple of a block, against the oracle's
V-cycle.

Tolerances: 1e-12 relative for FP64 values (other summation order); FP32 and
BF16 hierarchies round values and vectors to 24 and 8 bits, so they are held
against the FP64 V-cycle to 1e-5 and 5e-2."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    ("jacobi", dict(jacobi_fine_sweeps=2, jacobi_coarse_sweeps=1), "fp64"),
    ("jacobi", dict(jacobi_fine_sweeps=1, jacobi_coarse_sweeps=3), "fp64"),
    ("l1jacobi", dict(jacobi_fine_sweeps=3, jacobi_coarse_sweeps=2), "fp64"),
    ("jacobi", dict(jacobi_fine_sweeps=4, jacobi_coarse_sweeps=4), "fp32"),
    ("cheb2", dict(cheb_degree=1), "fp64"),
    ("cheb2", dict(cheb_degree=2), "bf16"),
    ("cheb2", dict(cheb_degree=3), "fp32"),
]
FLAGS = {"jacobi_fine_sweeps": "--amg-jacobi-fine-sweeps", "jacobi_coarse_sweeps": "--amg-jacobi-coarse-sweeps",
         "cheb_degree": "--amg-cheb-degree"}


@pytest.mark.parametrize("kind,kw,precision", CASES)
def test_step_smoothers(tmp_path, kind, kw, precision):
    from nodals_amd import _lib, meshgen
    from oracle import h8_oracle as O

    d = str(meshgen.write_pipe_case(tmp_path / "pipe", core=3, ring=2, nslab=7))
    print(f"\n[gpu] smoother {kind} {kw} {precision}", flush=True)
    args = [x for k, v in kw.items() for x in (FLAGS[k], str(v))]
    h = _lib.H8(["--mesh", d, "--max-outer", "10", "--verbose", "0", "--amg-smoother", kind, "--amg-precision",
                 precision, *args])
    case = O.case_from_product(h)
    rng = np.random.default_rng(4)
    for x in range(3):
        h.set(f"u{x}", 0.3 * rng.standard_normal(case.nv))
    h.assemble(0.5)
    h.pressure_refresh()
    A, diag = O.fine_refresh(case, h.get("rau", case.nv))
    vc = O.VCycle(case.hier, O.Smoother(kind=kind, **kw))
    vc.set_fine(A, diag)
    tol = {"fp64": 1e-12, "fp32": 1e-5, "bf16": 5e-2}[precision]
    for rep in range(3):  # replays of the captured cycle on new right-hand sides
        r = rng.standard_normal(case.nc)
        z = vc.apply(r)
        assert np.linalg.norm(h.precond(r) - z) <= tol * np.linalg.norm(z)
    h.close()


@pytest.mark.parametrize("options,smoother", [
    ("smoother=cheb2 cheb_degree=2 power_its=8", dict(kind="cheb2", cheb_degree=2)),
    ("smoother=jacobi sweeps=3 omega=0.7", dict(kind="jacobi", jacobi_fine_sweeps=3, jacobi_coarse_sweeps=3))])
def test_steps_on_explicit_coarse_levels(options, smoother):
    """A hierarchy whose first coarse level is too large for the dense product."""
    import scipy.sparse as sp
    from nodals_amd import p1
    from nodals_amd._lib import System
    from oracle import h8_oracle as O

    row, col, val = p1.kuhn_p1_laplacian(36)
    A = sp.csr_matrix((val, col, row))
    S = System(row, col, val, f"precision=fp64 hierarchy=cf terminal=500 {options}")
    print(f"\n[gpu] steps on coarse levels, {options}, level rows {S.level_rows}", flush=True)
    assert S.level_rows[0] > 9000  # the first coarse level; the largest dense one has 9,000 rows
    vc = O.VCycle(S.hierarchy(), O.Smoother(**smoother))
    vc.set_fine(A, A.diagonal())
    r = p1.poisson_rhs(A.shape[0], seed=3)
    z = vc.apply(r)
    assert np.linalg.norm(S.precond(r) - z) <= 1e-12 * np.linalg.norm(z)
