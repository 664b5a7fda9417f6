"""States and residuals between the device and ordinary memory: the threaded chunked copies give the
bytes that page-locked memory gets, at the edges of their sizes, from several solvers and threads."""
import threading

import numpy as np
import pytest

from ebbcfd_amd import meshgen
from ebbcfd_amd.solver import pinned_array
from helpers import channel_case

pytestmark = pytest.mark.gpu


def solver(nx, ny, **ext):
    from ebbcfd_amd import Solver, build_mesh
    _, cfg = channel_case(8, 4, integrator="Euler")
    cfg["extensions"] = ext
    return Solver(build_mesh(meshgen.channel_bump_quads(nx, ny, 0.06, seed=3)), cfg)


# cells of 32 bytes: a small state, a row below 4 MB, at 4 MB, a row over it, an odd size, a row below
# and at 8 MB (larger chunks, two threads), 33 MB (all eight threads, a short last chunk)
@pytest.mark.parametrize("nx,ny", [(331, 99), (131071, 1), (131072, 1), (131073, 1), (443, 357), (262143, 1), (512, 512),
                                   (1021, 1013)])
@pytest.mark.parametrize("order", ["reference", "tiles"])
def test_pageable_copies_equal_page_locked_ones(nx, ny, order):
    s = solver(nx, ny, cellOrder=order)
    n = nx * ny
    rng = np.random.default_rng(7)
    q = s.q * (1.0 + 0.01 * rng.random((n, 1)))
    pin = pinned_array((n, 4))
    s.q = q
    R = s.ufvm_solver()[0]
    Rp = s.ufvm_solver(out=pinned_array((n, 4)))[0]
    assert np.array_equal(R, Rp)
    pin[:] = s.q
    assert np.array_equal(pin, q)
    s.q = 2.0 * q
    s.q = pin
    assert np.array_equal(s.q, q)
    odd = np.empty(n * 4 + 1)[1:].reshape(n, 4)   # 8-byte alignment only
    odd[:] = q
    s.q = odd
    assert np.array_equal(s.q, q)


def test_solvers_on_several_threads():
    states = []
    for k in range(4):
        s = solver(512 + k, 300)
        states.append((s, s.q * (1.0 + 0.1 * k)))
    bad = []

    def work(s, q):
        for i in range(5):
            s.q = q + i
            if not np.array_equal(s.q, q + i):
                bad.append(i)
    threads = [threading.Thread(target=work, args=x) for x in states]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
