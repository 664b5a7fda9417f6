"""The step epilogue's sums of whole chunks at the edges of its ways to fold them: a lane's sixteen tops,
whole waves of them, and the counter beyond 1,024 (16.8M cells)."""
import numpy as np
import pytest

from helpers import base_config

from ebbcfd_amd import meshgen

pytestmark = pytest.mark.gpu

CHUNK = 16 * 1024


def trees(x, out):
    """The perfect pairwise trees of the rows of x, largest first (the binary counter's stack)."""
    n = len(x)
    while n:
        k = 1 << (n.bit_length() - 1)
        y = x[:k]
        while len(y) > 1:
            y = y[0::2] + y[1::2]
        out.append(y[0])
        x = x[k:]
        n -= k


def phobos_sum(x):
    """std.algorithm.sum over the rows: 16-element blocks, merged by a binary counter, then the rest."""
    nb = len(x) // 16
    b = x[: nb * 16].reshape(nb, 16, -1)
    while b.shape[1] > 1:
        b = b[:, 0::2] + b[:, 1::2]
    stack = []
    trees(b[:, 0], stack)
    trees(x[nb * 16:], stack)
    s = stack.pop()
    while stack:
        s = s + stack.pop()
    return s


# tops: 15, 16 and 17 (a lane's sixteen), 64 and 65; 1,024 and 1,025 (the counter) with a part chunk after
# them.  n_r x n_theta cells of the O-grid, two triangles each, and two ghosts per n_theta
@pytest.mark.parametrize("n_theta,n_r", [(1024, 120), (1024, 128), (1024, 136), (2048, 256), (2048, 260),
                                         (4096, 2048), (4096, 2050)])
def test_history_sums_of_many_chunks(n_theta, n_r):
    from ebbcfd_amd import Solver, build_mesh
    q = [0.2, 0.0, 1.0, 1.0]
    cfg = base_config(initialConditions=q, flux="rusanovFlux", order=1, forceBoundary="Wall",
                      boudaryConditions=[{"tag": "Wall", "type": "inviscidWall", "q": q},
                                         {"tag": "Farfield", "type": "fullState", "q": q}])
    mesh = build_mesh(meshgen.cylinder_ogrid(n_theta, n_r, r_far=30.0, stretch=1.003))
    print("%d cells, %d chunks" % (mesh.n_cells, mesh.n_cells // CHUNK), flush=True)
    s = Solver(mesh, cfg)
    a = s.q
    a[:, :] *= 1.0 + 0.01 * np.random.Generator(np.random.PCG64(1)).uniform(-1, 1, (len(a), 1))
    s.q = a
    hist, _, _ = s.run(1)
    b = s.q
    x = np.zeros((mesh.n_cells, 8))               # ghost slots count as zeros
    x[: len(a), :4] = (b - a) ** 2
    x[: len(a), 4:] = b
    del a, b
    tot = 0.0 + phobos_sum(x)
    assert np.array_equal(hist[0, 2:6], np.sqrt(float(s.n_interior) * tot[:4]) / tot[4:])
