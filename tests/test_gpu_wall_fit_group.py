"""The omega wall fit of the k-omega step for every number of active points
(one thread a point below three, eight lanes a point from three on) against
the oracle's step with the product's one-thread pointwise fit
(nodals_wall_fit_tangential) as its provider.

The fit of two or more points can end in a golden-section search of
resolution 1e-5 whose branches rounding decides, so targets agree to 3e-5 there
(the bound of test_gpu_turb.py) and to 1e-9 for one point and in the median."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class Pointwise:
    """refbind.RefSst's calls on the product's pointwise entries."""

    def __init__(self):
        from nodals_amd import _lib

        self.sst_local = _lib.sst_local
        self._lib = _lib

    def fit_values(self, U, y, nu, count):
        n = U.shape[0]
        samples = np.zeros((n, 5, 3))
        samples[:, :, 0] = U
        nrm, pic = np.tile([0.0, 0.0, 1.0], (n, 1)), np.tile([1.0, 0.0, 0.0], (n, 1))
        out, valid = self._lib.wall_fit_tangential(samples, y, nrm, pic, nu, count)
        return out[:, 1:3], valid

    def of_auto(self, inp, shared):
        return self._lib.wall_omega_target(inp, shared)


@pytest.mark.parametrize("points", [1, 2, 3, 4, 5])
def test_wall_targets(mesh_dir, points):
    from nodals_amd._lib import H8
    from oracle import h8_oracle as H
    from oracle import turb_oracle as T

    h = H8(["--mesh", mesh_dir["small"], "--run-mode", "fixed10", "--max-outer", "10", "--verbose", "0"])
    h.run()
    U = np.stack([h.get(f"u{d}", h.info["nv"]) for d in range(3)])
    h.turb_init(["--sst-wall-active-points", str(points)])
    st = T.Step(T.mesh_from_product(h), H.case_from_product(h, with_hierarchy=False), h.get("pipe_geometry", 12),
                T.Params(active_points=points), Pointwise())
    r = h.turb_step()
    st.step(U)
    assert r["wall_invalid"] == 0
    _, want, _, _, _ = st.wall_data(H.cell_values(st.case, U))
    got = h.get("turb_wall_target", want.size)
    e = np.abs(got - want) / want
    print(f"\n[gpu] {points} points: targets max {e.max():.1e} median {np.median(e):.1e}, "
          f"above 1e-9 at {int((e > 1e-9).sum())} of {e.size}", flush=True)
    assert np.median(e) < 1e-9 and e.max() < (1e-9 if points == 1 else 3e-5)
    h.close()
