"""The states of a renumbered solver cross the host boundary without device memory of their own."""
import numpy as np
import pytest

from ebbcfd_amd import Solver, build_mesh

from helpers import mms_case, perturb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("stage_path", ["faceTiles", "gradTiles", "fused", "split"])
@pytest.mark.parametrize("integrator", ["Euler", "RK4"])
def test_states_of_a_renumbered_solver_take_no_device_memory(integrator, stage_path):
    raw, cfg = mms_case(17, integrator=integrator)
    mesh = build_mesh(raw)
    cfg["extensions"] = dict(cfg["extensions"], stagePath=stage_path)
    ref = Solver(mesh, cfg)
    cfg["extensions"]["cellOrder"] = "tiles"
    s = Solver(mesh, cfg)
    held = s.device_bytes
    q = perturb(s.q, 0.01, seed=4)
    s.q = q
    ref.q = q
    assert np.array_equal(s.q, q)
    assert s.device_bytes == held
    # no stage yet: the edges are those of the set-up, whatever crossed the boundary
    for x, y in zip(s.edge_states(), ref.edge_states()):
        assert np.array_equal(x, y)
    held = s.device_bytes                       # (with the edge states' own buffer)
    assert np.array_equal(s.q, q)
    h, _, _ = s.run(3)
    hr, _, _ = ref.run(3)
    # between the steps of a run and the edge states and gradients of its last stage
    assert np.array_equal(s.q, ref.q) and np.array_equal(s.q_all(), ref.q_all())
    for x, y in zip(s.edge_states() + s.cell_gradients(), ref.edge_states() + ref.cell_gradients()):
        assert np.array_equal(x, y)
    s.q = q
    ref.q = q
    assert np.array_equal(np.vstack([h, s.run(3)[0]]), np.vstack([hr, ref.run(3)[0]]))
    assert np.array_equal(s.q, ref.q)
    assert s.device_bytes == held
