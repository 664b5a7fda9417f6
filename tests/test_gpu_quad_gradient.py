"""Gradients with four, two and one lane per cell (by the mesh's size): the same solve as the gradient
tiles', which form them in the tile kernel, at the edges of the blocks and of the rule."""
import numpy as np
import pytest

from ebbcfd_amd import meshgen
from helpers import channel_case

pytestmark = pytest.mark.gpu


# cells: 1 short block, 64 (a whole block of four lanes), 65, 256, 257 and, on triangles, both sides of
# the rule's lines (40,000 and 800,000) and sizes between them
@pytest.mark.parametrize("limiter", ["scalar", "venkatakrishnan"])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("nx,ny,quads", [(7, 3, 1), (64, 1, 1), (65, 1, 1), (128, 1, 0), (257, 1, 1), (200, 100, 0),
                                         (201, 100, 0), (500, 100, 0), (501, 100, 0), (1000, 400, 0), (1001, 400, 0)])
def test_lanes_per_cell_do_not_show(nx, ny, quads, precision, limiter):
    from ebbcfd_amd import Solver, build_mesh
    raw, cfg = channel_case(nx, ny, integrator="RK2_TVD")
    if quads:
        raw = meshgen.channel_bump_quads(nx, ny, 0.06, seed=3)
    mesh = build_mesh(raw)
    got = []
    for path in ("faceTiles", "gradTiles"):
        cfg["extensions"] = {"stagePath": path, "precision": precision, "limiter": limiter}
        s = Solver(mesh, cfg)
        got.append(s.run(3) + (s.q_all(),))
    for x, y in zip(*got):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("nx,ny", [(6, 3), (40, 13), (64, 16)])
def test_lp_limiter_against_the_oracle(nx, ny):
    import oracle
    from ebbcfd_amd import Solver, build_mesh
    from helpers import oracle_cfg
    raw, cfg = channel_case(nx, ny, lpThresh=1.0, CFL=0.07)
    s = Solver(build_mesh(raw), cfg)
    om = oracle.Mesh(raw).setup(oracle_cfg(cfg))
    hist, t, dt = s.run(10)
    ohist, ot, odt = om.run(10)
    assert np.array_equal(hist, ohist) and (t, dt) == (ot, odt)
    assert np.array_equal(s.q, om.q[: om.n_interior])
