"""The face tiles' shared-reciprocal flux against the IEEE forms of the split kernels, on states whose
quotients and roots leave its range: same residuals and states bit for bit, same error reports."""
import numpy as np
import pytest

from helpers import channel_case

pytestmark = pytest.mark.gpu


def patch(q, rho=None, mx=None, my=None, E=None):
    for c in (40, 41, 42, 43, 200):   # neighbours in a strip, and one cell alone
        for k, v in enumerate((rho, mx, my, E)):
            if v is not None:
                q[c, k] = v


STATES = {"at_rest": lambda q: q.__setitem__((slice(None), slice(1, 3)), 0.0),
          "no_density": lambda q: patch(q, rho=0.0), "subnormal_density": lambda q: patch(q, rho=1e-310),
          "negative_density": lambda q: patch(q, rho=-1.0), "huge_density": lambda q: patch(q, rho=1e200),
          "no_pressure": lambda q: patch(q, mx=0.0, my=0.0, E=0.0),
          "small_pressure": lambda q: patch(q, mx=0.0, my=0.0, E=1e-250),
          "negative_pressure": lambda q: patch(q, E=-1.0), "infinite_energy": lambda q: patch(q, E=np.inf),
          "nan": lambda q: patch(q, E=np.nan), "faint_flow": lambda q: patch(q, mx=1e-200, my=-1e-200)}


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("viscous", [False, True])
@pytest.mark.parametrize("flux", ["roeFlux", "rusanovFlux"])
@pytest.mark.parametrize("state", sorted(STATES))
def test_states_beyond_the_range_take_the_ieee_forms(state, flux, viscous, order, precision):
    from ebbcfd_amd import Solver, build_mesh
    raw, cfg = channel_case(32, 8, walls="viscidWall" if viscous else "inviscidWall", flux=flux, viscosity=viscous,
                            order=order)
    mesh = build_mesh(raw)
    got = []
    for path in ("faceTiles", "split"):
        cfg["extensions"] = {"stagePath": path, "precision": precision}
        s = Solver(mesh, cfg)
        q = s.q.copy()
        STATES[state](q)
        out = []
        for call in (lambda: s.ufvm_solver(), lambda: s.step(1e-4)):
            s.q = q
            try:
                out.append(call())
            except Exception as e:
                out.append(str(e))
            out.append(s.q)
        got.append(out)
    for a, b in zip(*got):
        if isinstance(a, str) or isinstance(b, str):
            assert a == b
        else:
            for x, y in zip(a, b) if isinstance(a, tuple) else [(a, b)]:
                assert np.array_equal(x, y, equal_nan=True)
