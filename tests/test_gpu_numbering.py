"""States and residuals of a renumbered solver cross the host boundary in the reference numbering."""
import numpy as np
import pytest

from ebbcfd_amd import Solver, build_mesh

from helpers import cylinder_case, mms_case, perturb, tiny_mesh, channel_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("case", ["tri1", "mms_9", "mms_23", "cylinder"])
def test_renumbered_rows_equal_the_reference_numbering(case, precision):
    if case == "tri1":
        raw = tiny_mesh("tri1")
        _, cfg = channel_case(4, 4)
        cfg["boudaryConditions"] = [{"tag": "Farfield", "type": "fullState", "q": cfg["initialConditions"]}]
    elif case == "cylinder":
        raw, cfg = cylinder_case(52, 31)
    else:
        raw, cfg = mms_case(int(case[4:]))
    cfg["extensions"] = dict(cfg.get("extensions", {}), precision=precision)
    mesh = build_mesh(raw)
    a = Solver(mesh, cfg)
    cfg["extensions"]["cellOrder"] = "tiles"
    b = Solver(mesh, cfg)
    q = perturb(a.q, 0.01, seed=4)
    for s in (a, b):
        s.q = q
    assert np.array_equal(a.q, q) and np.array_equal(b.q, q)
    for x, y in zip(a.ufvm_solver(), b.ufvm_solver()):
        assert np.array_equal(x, y)
    a.run(3)
    b.run(3)
    assert np.array_equal(a.q, b.q) and np.array_equal(a.q_all(), b.q_all())
