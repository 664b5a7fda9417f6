"""The step epilogue: its sums at the edges of its blocks, chunks and remainder against the oracle,
and what a loop that ends inside a queued batch of steps leaves behind (the epilogue of a step runs
beside the next step's gradients)."""
import numpy as np
import pytest

from ebbcfd_amd import meshgen
from helpers import channel_case, cylinder_case, mms_case, oracle_cfg, tiny_mesh

pytestmark = pytest.mark.gpu


def bump(nx, ny, quads=False):
    raw, cfg = channel_case(nx, ny, integrator="RK2_TVD")
    if quads:
        raw = meshgen.channel_bump_quads(nx, ny, 0.06, seed=3)
    return raw, cfg


# cells with ghosts: 31 (one block, 15 over), 4 (no block), 16,198 (1,012 blocks, 6 over),
# 16,384 (one whole chunk), 16,560 (a chunk and 11 blocks), 49,152 (three whole chunks)
SHAPES = {"one_block_15_over": lambda: bump(5, 3, quads=True), "no_block": lambda: (tiny_mesh("tri1"), None),
          "below_a_chunk": lambda: mms_case(89), "one_chunk": lambda: bump(2730, 2),
          "above_a_chunk": lambda: mms_case(90), "three_chunks": lambda: bump(3510, 6)}


@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_history_at_the_edges_of_the_sums(shape):
    import oracle
    from ebbcfd_amd import Solver, build_mesh
    raw, cfg = SHAPES[shape]()
    if cfg is None:
        _, cfg = channel_case(4, 4, integrator="RK2_TVD")
        cfg["boudaryConditions"] = [{"tag": "Farfield", "type": "fullState", "q": cfg["initialConditions"]}]
        cfg["forceBoundary"] = "Farfield"
    s = Solver(build_mesh(raw), cfg)
    om = oracle.Mesh(raw).setup(oracle_cfg(cfg))
    hist, t, dt = s.run(5)
    ohist, ot, odt = om.run(5)
    assert np.array_equal(hist, ohist, equal_nan=True) and t == ot and dt == odt
    assert np.array_equal(s.q, om.q[: om.n_interior])


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("path", ["faceTiles", "split", "gradTiles"])
@pytest.mark.parametrize("integrator", ["Euler", "RK2_TVD", "RK4"])
@pytest.mark.parametrize("order", [1, 2])
def test_a_loop_that_ends_early_leaves_what_its_last_step_left(integrator, path, precision, order):
    from ebbcfd_amd import Solver, build_mesh
    raw, cfg = cylinder_case(48, 24, integrator=integrator, order=order)
    cfg["extensions"] = {"stagePath": path, "precision": precision}
    mesh = build_mesh(raw)
    a = Solver(mesh, cfg)
    h, t, dt = a.run(5)                       # ends with the queued batch
    cfg["tEnd"] = float(0.5 * (h[4, 0] + t))  # inside the fifth step
    b = Solver(mesh, cfg)
    h2, t2, dt2 = b.run(40)                   # ends five steps into it
    assert len(h2) == 5 and np.array_equal(h, h2) and (t, dt) == (t2, dt2)
    assert np.array_equal(a.q_all(), b.q_all())
    if order == 2:
        for x, y in zip(a.cell_gradients(), b.cell_gradients()):
            assert np.array_equal(x, y)
    for x, y in zip(a.edge_states(), b.edge_states()):
        assert np.array_equal(x, y)
