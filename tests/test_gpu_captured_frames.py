"""A frame captured into a HIP graph (allocation-free or ordinary, in range order) can be
replayed after its simulator ran more scan origins than a dataset keeps orders for: the
order that it names is neither given back nor replaced.

Tolerance: the graph runs the kernels of the eager frame on the same records; the 1e-6
that frames of different summation order agree to."""
import ctypes as C

import numpy as np
import pytest

from backends import rel_l2
from openbcsim_amd import _lib
from openbcsim_amd import workloads as W
from test_zz_no_alloc import frame, make

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("entry", ["bcsim_simulate_lines_device", "bcsim_simulate_lines_device_noalloc"])
def test_replay_after_other_origins(entry):
    from openbcsim_amd.hip_rt import DeviceBuffer, hip
    rt, lib = hip(), _lib.load()
    wl = W.fixed_sector_2d(20000, 64, seed=5, line_length=0.06)
    sim = make(wl)

    def at(x):
        o, d, lat, t, length = wl.scan
        sim.set_scan_sequence(o + np.float32([x, 0, 0]), d, length, lat, t, True)
        return frame(sim, "bcsim_simulate_lines_device"), "range order" in sim.get_parameter("launch_plan")

    ref, ranged = at(0.0)
    assert ranged
    L, S = sim.output_shape()
    buf, nl, ns = DeviceBuffer(L * S * 8), C.c_int(), C.c_int()
    stream, graph, run = C.c_void_p(), C.c_void_p(), C.c_void_p()
    _lib.check(lib.bcsim_get_stream(sim.handle, C.byref(stream)))
    assert rt.hipStreamBeginCapture(stream, 1) == 0
    rc = getattr(lib, entry)(sim.handle, C.c_void_p(buf.address), L * S, C.byref(nl), C.byref(ns))
    assert rt.hipStreamEndCapture(stream, C.byref(graph)) == 0
    _lib.check(rc)
    assert "range order" in sim.get_parameter("launch_plan")
    assert rt.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)) == 0
    for x in (1e-3, 2e-3, 3e-3, 4e-3, 4e-3, 5e-3, 5e-3, 6e-3, 6e-3):
        _, ranged = at(x)
    assert ranged  # the last origin took an order's place
    again, ranged = at(0.0)
    assert ranged and rel_l2(again, ref) <= 1e-6
    for _ in range(3):
        assert rt.hipGraphLaunch(run, stream) == 0
        _lib.check(lib.bcsim_synchronize(sim.handle))
        out = np.empty((L, S), np.complex64)
        buf.to_host(out)
        assert rel_l2(out, ref) <= 1e-6
        frame(sim, "bcsim_simulate_lines_device")
    assert rt.hipGraphExecDestroy(run) == 0 and rt.hipGraphDestroy(graph) == 0
    buf.close()
    sim.close()
