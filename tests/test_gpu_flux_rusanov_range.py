"""The face tiles' Rusanov flux where the terms that it leaves out are not finite (an enthalpy beyond the
type's range times a zero): the split kernels report the edge, and so do the face tiles."""
import numpy as np
import pytest

from helpers import channel_case

pytestmark = pytest.mark.gpu


def everywhere(rho, E):
    def fill(q):
        q[:, 0], q[:, 1], q[:, 2], q[:, 3] = rho, 0.0, 0.0, E
    return fill


def one_cell(rho, E):
    """a light cell away from the boundary, in ordinary gas"""
    def fill(q):
        q[201] = rho, 0.0, 0.0, E
    return fill


# gas at rest.  Energy / density: 4e38 in FP32 and 5e308 / 3.5 and more in FP64, whose enthalpies are infinite
# while pressure over mean density is not; and values that are large and finite
STATES = {"fp32_everywhere": ("mixed", everywhere(1e-18, 4e20), True), "fp32_one_cell": ("mixed", one_cell(1e-37, 40.0), True),
          "fp64_one_cell": ("fp64", one_cell(1e-290, 5e18), True), "fp32_finite": ("mixed", everywhere(1e-18, 4e18), False),
          "fp32_one_finite": ("mixed", one_cell(1e-30, 40.0), False),
          "fp64_one_finite": ("fp64", one_cell(1e-280, 5e18), False)}


@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("state", sorted(STATES))
def test_an_enthalpy_out_of_range_is_reported(state, order):
    from ebbcfd_amd import Solver, build_mesh
    precision, fill, fails = STATES[state]
    raw, cfg = channel_case(32, 8, flux="rusanovFlux", order=order)
    for bc in cfg["boudaryConditions"]:
        bc["type"] = "inviscidWall"
    mesh = build_mesh(raw)
    got = []
    for path in ("faceTiles", "split"):
        cfg["extensions"] = {"stagePath": path, "precision": precision}
        s = Solver(mesh, cfg)
        q = s.q.copy()
        fill(q)
        out = []
        for call in (lambda: s.ufvm_solver(), lambda: s.step(1e-40)):
            s.q = q
            try:
                out.append(call())
            except Exception as e:
                out.append(str(e))
        got.append(out)
    if order == 1:   # (the second order's reconstructions differ from cell to cell)
        assert [isinstance(x, str) and "interior edge" in x for x in got[1]] == [fails, fails]
    for a, b in zip(*got):
        if isinstance(a, str) or isinstance(b, str):
            assert a == b
        else:
            for x, y in zip(a, b):
                assert np.array_equal(x, y, equal_nan=True)
