"""The face tiles against the IEEE forms of the split kernels at the limits of each precision's type: densities
whose reciprocal is subnormal, and momenta, pressures and densities whose quotients' corrections are.  The
same residuals and states bit for bit, the same error reports."""
import numpy as np
import pytest

from helpers import channel_case

pytestmark = pytest.mark.gpu


def gas(rho, vel, p, spread=0.1):
    """every cell near one state, so that gradients and jumps stay representable too"""
    def fill(q, rng):
        n = len(q)
        r = rho * rng.uniform(1 - spread, 1 + spread, n)
        u, v = (vel * rng.uniform(0.5, 1.5, n) for _ in range(2))
        q[:, 0], q[:, 1], q[:, 2] = r, r * u, r * v
        q[:, 3] = p * rng.uniform(1 - spread, 1 + spread, n) / 0.4 + 0.5 * r * (u * u + v * v)
    return fill


def quiet(vel):
    """no jumps in density and pressure, so that the mass flux is the faint velocity's"""
    return gas(1.1, vel, 1.0, 0.0)


STATES = {"mixed": {"dense_2^126": gas(1.0e38, 1e-10, 4e18), "dense_2^127": gas(2.5e38, 1e-10, 4e18),
                    "faint_1e-33": gas(1.1, 1e-33, 1.0), "faint_1e-36": gas(1.1, 1e-36, 1.0), "faint_1e-40": gas(1.1, 1e-40, 1.0),
                    "quiet_1e-33": quiet(1e-33), "quiet_1e-36": quiet(1e-36), "quiet_1e-37": quiet(1e-37), "quiet_1e-38": quiet(1e-38),
                    "low_1e-30": gas(1.1, 0.0, 1e-30), "low_1e-38": gas(1.1, 0.0, 1e-38), "thin_1e-30": gas(1e-30, 0.3, 1e-30),
                    "thin_1e-36": gas(1e-36, 0.3, 1e-36), "thin_1e-38": gas(2e-38, 0.3, 2e-38)},
          "fp64": {"dense_1e307": gas(4e307, 1e-280, 1e60), "dense_1e308": gas(1.6e308, 1e-280, 1e60),
                   "faint_1e-270": gas(1.1, 1e-270, 1.0), "faint_1e-289": gas(1.1, 1e-289, 1.0),
                   "quiet_1e-270": quiet(1e-270), "quiet_1e-289": quiet(1e-289),
                   "low_1e-295": gas(1.1, 0.0, 1e-295), "low_1e-306": gas(1.1, 0.0, 1e-306),
                   "thin_1e-295": gas(1e-295, 0.3, 1e-295), "thin_1e-306": gas(2e-306, 0.3, 2e-306)}}
CASES = [(p, s) for p in sorted(STATES) for s in sorted(STATES[p])]


@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("viscous", [False, True])
@pytest.mark.parametrize("flux", ["roeFlux", "rusanovFlux"])
@pytest.mark.parametrize("precision,state", CASES)
def test_the_limits_of_the_type_give_the_ieee_forms(precision, state, flux, viscous, order):
    from ebbcfd_amd import Solver, build_mesh
    raw, cfg = channel_case(32, 8, walls="viscidWall" if viscous else "inviscidWall", flux=flux, viscosity=viscous,
                            order=order)
    mesh = build_mesh(raw)
    got = []
    for path in ("faceTiles", "split"):
        cfg["extensions"] = {"stagePath": path, "precision": precision}
        s = Solver(mesh, cfg)
        q = s.q.copy()
        STATES[precision][state](q, np.random.Generator(np.random.PCG64(5)))
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
