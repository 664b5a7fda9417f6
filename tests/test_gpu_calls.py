"""Residual and step calls on every path: the scalars that the call's last kernel leaves (new dt of the
last stage, Rmax of all, the run loop's dt) against the oracle."""
import numpy as np
import pytest

from helpers import channel_case, oracle_cfg

pytestmark = pytest.mark.gpu


# 48 cells: fewer partials than one wave; 1,584: more workgroups than lanes on the split path's tail
@pytest.mark.parametrize("nx,ny", [(8, 3), (36, 22)])
@pytest.mark.parametrize("path", ["faceTiles", "split", "fused", "gradTiles"])
@pytest.mark.parametrize("integrator", ["Euler", "RK2", "RK2_TVD", "RK4"])
def test_calls_between_runs(integrator, path, nx, ny):
    import oracle
    from ebbcfd_amd import Solver, build_mesh
    raw, cfg = channel_case(nx, ny, integrator=integrator)
    om = oracle.Mesh(raw).setup(oracle_cfg(cfg))
    cfg["extensions"] = {"stagePath": path}
    s = Solver(build_mesh(raw), cfg)
    n = om.n_interior
    h, t, dt = s.run(3)
    oh, ot, odt = om.run(3)
    for big in (0.0, 1e6):
        R, nd, rm = s.ufvm_solver(rmax=big)
        oR, ond, orm = om.residual(rmax=big)
        assert np.array_equal(R, oR) and (nd, rm) == (ond, orm)
    for k in range(2):
        assert s.step(1e-4 * (k + 1)) == om.step(1e-4 * (k + 1))
        assert np.array_equal(s.q, om.q[:n])
    h, t, dt = s.run(3)
    oh, ot, odt = om.run(3, t=ot, dt=odt)
    assert np.array_equal(h, oh) and (t, dt) == (ot, odt)
    assert np.array_equal(s.q, om.q[:n])


@pytest.mark.parametrize("path", ["faceTiles", "split", "fused", "gradTiles"])
def test_a_failed_call_does_not_reach_the_next(path):
    from ebbcfd_amd import Solver, build_mesh
    raw, cfg = channel_case(12, 5, integrator="RK2_TVD")
    cfg["extensions"] = {"stagePath": path}
    mesh = build_mesh(raw)
    s, ref = Solver(mesh, cfg), Solver(mesh, cfg)
    q = s.q
    bad = q.copy()
    bad[7, 0] = -1.0
    for call in (lambda x: x.step(1e-4), lambda x: x.ufvm_solver()):
        s.q = q
        s.step(1e-4)
        s.q = bad
        for _ in range(2):
            with pytest.raises(Exception):
                call(s)
        s.q = q
        ref.q = q
        for x, y in zip(call(s), call(ref)):
            assert np.array_equal(x, y)
        assert np.array_equal(s.q, ref.q)
