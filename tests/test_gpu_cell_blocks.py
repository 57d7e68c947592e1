"""Cell-block kernels at cell counts that do not fill their wavefronts and
blocks (630 cells: not a multiple of four or eight): the k-omega volume terms,
the mixing-length and SUPG blocks, and the wall path's deviatoric tensors
through the assembled 3x3 block operator, against the oracles with the
product's own pointwise SST state (nodals_sst_local) as the provider.

Tolerances: 1e-10 of the largest entry for the volume terms (device
transcendentals on both sides, other summation orders), 1e-11 relative for
the assembled operator, 1e-9 for the ten-iteration trajectory, as in
test_gpu_sst_volume.py, test_gpu_wall.py and test_gpu_rans.py."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def odd_pipe(tmp_path_factory):
    from nodals_amd import meshgen

    return str(meshgen.write_pipe_case(tmp_path_factory.mktemp("odd") / "pipe", core=3, ring=1, nslab=5))


@pytest.mark.parametrize("equation", [0, 1])
def test_sst_volume_odd_cells(odd_pipe, equation):
    from nodals_amd import _lib
    from oracle import h8_oracle as O
    from oracle import sst_oracle as S

    h = _lib.H8(["--mesh", odd_pipe, "--max-outer", "10", "--verbose", "0"])
    case = O.case_from_product(h, with_hierarchy=False)
    assert case.nc % 8 == 6
    rng = np.random.default_rng(20 + equation)
    nv, nf = case.nv, h.info["nfixed"]
    U = rng.standard_normal((3, nv)) * 0.5
    for d in range(3):
        h.set(f"u{d}", U[d])
    k = 10.0 ** rng.uniform(-4, -1, nv + nf)
    w = 10.0 ** rng.uniform(0, 3, nv + nf)
    mat, rhs = h.sst_volume(equation, k[:nv], k[nv:], w[:nv], w[nv:])
    pipe = h.get("pipe", 5)
    mo, ro, _ = S.volume_terms(_lib, case.cell_ref, case.cell_invJ, case.cell_det,
                               h.get("cell_xy", case.nc * 8).reshape(case.nc, 4, 2), U, case.fixed_value, k[:nv],
                               k[nv:], w[:nv], w[nv:], float(pipe[3]), float(pipe[0]), equation)
    print(f"\n[gpu] volume terms {np.abs(mat - mo).max() / np.abs(mo).max():.1e} "
          f"{np.abs(rhs - ro).max() / np.abs(ro).max():.1e}", flush=True)
    assert np.abs(mat - mo).max() <= 1e-10 * np.abs(mo).max()
    assert np.abs(rhs - ro).max() <= 1e-10 * np.abs(ro).max()
    h.close()


@pytest.mark.parametrize("mixing,supg", [(True, False), (False, True), (True, True)])
def test_rans_blocks_odd_cells(odd_pipe, mixing, supg):
    from nodals_amd._lib import H8
    from oracle import h8_oracle as O
    from oracle import rans_oracle as R

    extra = (["--mixing-length", "1", "--mixlen-scale", "0.7"] if mixing else []) + (
        ["--supg", "1", "--supg-tau-scale", "0.1", "--supg-magic", "4.0"] if supg else [])
    h = H8(["--mesh", odd_pipe, "--max-outer", "10", "--amg-smoother", "jacobi", "--pressure-solver", "pcg", "--p-max",
            "200", "--re", "200", "--verbose", "0", *extra])
    h.run()
    case = O.case_from_product(h)
    pts, cx, cy, radius = R.product_geometry(h)
    nu = float(h.get("pipe", 5)[0])
    blocks = R.extra_blocks_fn(case, pts, nu, (0.7, radius, cx, cy) if mixing else None,
                               (0.1, 4.0) if supg else None)
    ref = O.simple(case, p_solver="pcg", p_max=200, smoother=O.Smoother(kind="jacobi"), max_outer=10,
                   extra_blocks=blocks)
    err = max(np.linalg.norm(h.get(f"u{d}", case.nv) - ref["U"][d]) / np.linalg.norm(ref["U"][d]) for d in range(3))
    print(f"\n[gpu] rans blocks mixing={mixing} supg={supg}: {err:.1e}", flush=True)
    assert err < 1e-9
    h.close()


def test_wall_operator_odd_cells(tmp_path):
    from nodals_amd import _lib, meshgen
    from oracle import h8_oracle as O
    from oracle import turb_oracle as TO
    from oracle import wall_oracle as WO

    mesh = str(meshgen.write_helix_case(tmp_path / "helix", core=3, ring=2, nslab=25))
    h = _lib.H8(["--mesh", mesh, "--max-outer", "10", "--duct", "1", "--wall-model", "spalding", "--re", "5000",
                 "--alpha-u", "0.7", "--alpha-p", "0.3", "--amg-hierarchy", "cf", "--cf-interp", "exti",
                 "--amg-smoother", "mcgs", "--pressure-solver", "pcg", "--p-rtol", "1e-3", "--p-max", "600", "--verbose",
                 "0"])
    h.turb_init([])
    h.wall_init([])
    case = O.case_from_product(h)
    assert case.nc % 8 != 0
    m = TO.mesh_from_product(h)
    st = TO.Step(m, case, h.get("pipe_geometry", 12), TO.Params(active_points=1), _lib,
                 wall_distance=h.get("wall_distance", m.nvert))
    wp = WO.WallPath(case, st, _lib)
    rng = np.random.default_rng(3)
    U = h.get("wall_u0", 3 * case.nv).reshape(case.nv, 3).T + 0.05 * rng.standard_normal((3, case.nv))
    p = 0.1 * rng.standard_normal(case.nc)
    for d in range(3):
        h.set(f"u{d}", U[d])
    h.set("p", p)
    st.k = st.k * (1.0 + 0.2 * rng.random(m.ns))
    st.w = st.w * (1.0 + 0.2 * rng.random(m.ns))
    h.set("k", st.k)
    h.set("omega", st.w)
    h.wall_assemble()
    nf = wp.W.nf
    A = wp.assemble(U, p, fit=h.get("wall_fit", 3 * nf).reshape(nf, 3))
    r = np.repeat(np.arange(case.nv), np.diff(case.mom_row))
    K = np.empty((case.nnz, 9))
    for i in range(3):
        for j in range(3):
            K[:, 3 * i + j] = np.asarray(A["K"][3 * r + i, 3 * case.mom_col + j]).ravel()
    Kg = h.get("wall_K", 9 * case.nnz).reshape(case.nnz, 9)
    rel = lambda a, b: float(np.linalg.norm(a - b) / np.linalg.norm(b))  # noqa: E731
    errs = [rel(Kg, K), rel(h.get("wall_rhs", 3 * case.nv), A["b"])]
    print(f"\n[gpu] wall operator, {case.nc} cells: K {errs[0]:.1e} rhs {errs[1]:.1e}", flush=True)
    assert max(errs) < 1e-11
    h.wall_momentum()
    Un = wp.momentum(A)
    e = max(rel(h.get(f"u{d}", case.nv), Un[d]) for d in range(3))
    print(f"[gpu]   after the block sweeps: {e:.1e}", flush=True)
    assert e < 1e-11
    h.close()
