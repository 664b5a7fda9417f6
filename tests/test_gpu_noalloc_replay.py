"""A captured ebb_residual_noalloc that is replayed on a failing state leaves its error words on the device
without the host taking part: they do not reach the next call."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from helpers import ROOT, channel_case

pytestmark = pytest.mark.gpu

# the solver's stream, which a program that captures the call has from the solver's own header
HANDLE = """
#include "solver_impl.hpp"
extern "C" void* solver_stream(ebb_solver* s) { return s->stream; }
"""


@pytest.fixture(scope="module")
def solver_stream(tmp_path_factory):
    d = tmp_path_factory.mktemp("handle")
    src = d / "handle.cpp"
    src.write_text(HANDLE)
    so = str(d / "handle.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__=1", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "ebbcfd_amd", "csrc"), "-I" + os.path.join(ROOT, "include"),
                    str(src), "-o", so, "-Wl,--unresolved-symbols=ignore-all"], check=True)
    f = C.CDLL(so).solver_stream
    f.restype, f.argtypes = C.c_void_p, [C.c_void_p]
    return f


def test_a_replayed_error_does_not_reach_the_next_call(solver_stream):
    from ebbcfd_amd import Solver, build_mesh
    from ebbcfd_amd._lib import lib
    raw, cfg = channel_case(12, 5, integrator="RK2_TVD")
    mesh = build_mesh(raw)
    s, ref = Solver(mesh, cfg), Solver(mesh, cfg)
    q = s.q
    bad = q.copy()
    bad[7, 0] = -1.0
    hip = lib()                                 # (its HIP runtime)
    R, got = C.c_void_p(), np.empty((s.n_interior, 4))
    stream, graph, run = C.c_void_p(solver_stream(s.h)), C.c_void_p(), C.c_void_p()
    ok = lambda rc: rc == 0 or pytest.fail("hip error %d" % rc)
    ok(hip.hipMalloc(C.byref(R), C.c_size_t(got.nbytes)))
    noalloc = lambda: lib().ebb_residual_noalloc(s.h, 1, 1, R, None, None)
    assert noalloc() == 0                       # looks the scratch up before the capture
    s.q = q                                     # waits for it
    ok(hip.hipStreamBeginCapture(stream, C.c_int(1)))
    assert noalloc() == 0
    ok(hip.hipStreamEndCapture(stream, C.byref(graph)))
    ok(hip.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)))
    want, _, _ = ref.ufvm_solver()
    for _ in range(3):
        s.q = q
        ok(hip.hipGraphLaunch(run, stream))
        ok(hip.hipStreamSynchronize(stream))
        ok(hip.hipMemcpy(C.c_void_p(got.ctypes.data), R, C.c_size_t(got.nbytes), C.c_int(2)))
        assert np.array_equal(got, want)
        got[:] = 0
        assert np.array_equal(s.ufvm_solver()[0], want)     # a call that leaves the words clear
        s.q = bad
        ok(hip.hipGraphLaunch(run, stream))
        s.q = q                                             # waits for it
        for call in (lambda x: x.ufvm_solver(), lambda x: x.step(1e-4)):
            ref.q = q
            s.q = q
            for x, y in zip(call(s), call(ref)):
                assert np.array_equal(x, y)
            assert np.array_equal(s.q, ref.q)
        s.q = q
        ref.q = q
    ok(hip.hipGraphExecDestroy(run))
    ok(hip.hipGraphDestroy(graph))
    ok(hip.hipFree(R))
