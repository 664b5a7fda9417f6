"""Edges whose squared length is subnormal: the face tiles form lengths and normals from the nodes, and they
equal the ones of the mesh set-up, which the split kernels read.  A square whose corner is cut by one such
edge, the only one of the force boundary, so that drag and lift are its length times its flux."""
import numpy as np
import pytest

from ebbcfd_amd import meshgen
from helpers import base_config, oracle_cfg

pytestmark = pytest.mark.gpu


def cut_corner(n, d):
    h = 1.0 / n
    nid = lambda i, j: i * (n + 1) + j
    nodes = [[i * h, j * h] for i in range(n + 1) for j in range(n + 1)]
    nodes[0] = [d, 0.0]                       # the corner's node on the lower side
    nodes.append([0.0, d * 0.7])              # and the one on the left
    last = len(nodes) - 1
    elems = [[nid(i, j), nid(i + 1, j), nid(i + 1, j + 1), nid(i, j + 1)] for i in range(n) for j in range(n)]
    elems[0] = [0, nid(1, 0), nid(1, 1), nid(0, 1), last]
    lower = [[nid(i, 0), nid(i + 1, 0)] for i in range(n)]
    right = [[nid(n, j), nid(n, j + 1)] for j in range(n)]
    upper = [[nid(i + 1, n), nid(i, n)] for i in range(n)]
    left = [[nid(0, j + 1), nid(0, j) if j else last] for j in range(n)]
    groups = [lower + right + upper + left, [[last, 0]]]
    return meshgen.RawMesh(nodes=np.array(nodes, float),
                           elem_offsets=np.cumsum([0] + [len(e) for e in elems]).astype(np.uint32),
                           elem_nodes=np.array([v + 1 for e in elems for v in e], np.uint32),
                           bnodes=np.array([p for g in groups for p in g], np.uint32), btags=["Farfield", "Tip"],
                           bgroup_start=np.array([0, len(groups[0])], np.uint64))


@pytest.mark.parametrize("viscous", [False, True])
@pytest.mark.parametrize("d", [6.560392180538345e-162, 1.4382538534190863e-160, 3.2855147033030913e-159,
                               2.3348240771290105e-157, 4.678775301608913e-155, 1e-140, 1e-99, 1e-101, 1e-3])
def test_short_edge_forces(d, viscous):
    import oracle
    from ebbcfd_amd import Solver, build_mesh
    q = [0.3, 3.0, 1.0, 1.0]
    cfg = base_config(initialConditions=q, forceBoundary="Tip", viscosity=viscous,
                      boudaryConditions=[{"tag": t, "type": "fullState", "q": q} for t in ("Farfield", "Tip")])
    raw = cut_corner(4, d)
    om = oracle.Mesh(raw).setup(oracle_cfg(cfg))
    ohist, _, _ = om.run(3)
    for path in ("split", "faceTiles"):
        cfg["extensions"] = {"stagePath": path}
        s = Solver(build_mesh(raw), cfg)
        hist, _, _ = s.run(3)
        assert np.all(hist[:, 7:9] != 0)
        assert np.array_equal(hist, ohist), path
        assert np.array_equal(s.q, om.q[: om.n_interior])
