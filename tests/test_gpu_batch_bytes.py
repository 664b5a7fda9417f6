"""A batched solve, whose ghost rows nobody reads, keeps no copy of them and is not charged for one."""
import numpy as np
import pytest

from ebbcfd_amd import Batch, Solver, build_mesh, estimate_device_bytes

from helpers import channel_case

pytestmark = pytest.mark.gpu


def test_a_batched_solve_is_admitted_without_its_ghosts_copy():
    raw, cfg = channel_case(6000, 1, integrator="RK2_TVD")
    mesh = build_mesh(raw)
    ghosts = mesh.n_cells - mesh.n_interior
    limit = estimate_device_bytes(mesh, cfg) - 16 * ghosts    # a copy takes 32 B per ghost
    b = Batch(device_bytes_limit=limit)
    sid = b.add(mesh, cfg)
    s = Solver(mesh, cfg)
    b.run(4)
    s.run(4)
    assert np.array_equal(b.q(sid), s.q)
    assert b.status(sid)["device_bytes"] <= limit
