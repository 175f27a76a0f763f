"""The tile kernel on scans of one origin, which run in range order by default: an
accumulation set by hand keeps them on it, so that block order, chunk order and tuned
shapes are compared with something.  And host copies of every size class.

Tolerance: the same contributions in another order of summation (1e-6, as between the
tiled and the direct kernel)."""
import numpy as np
import pytest

from backends import rel_l2
from openbcsim_amd import workloads as W

pytestmark = pytest.mark.gpu


def sim(wl, **params):
    from openbcsim_amd.pyrfsim import RfSimulator
    s = RfSimulator("gpu")
    wl.apply(s)
    for k, v in params.items():
        s.set_parameter(k, v)
    return s


def tiled(s):
    iq = s.simulate_frame()
    assert "range order" not in s.get_parameter("launch_plan")
    return iq


@pytest.mark.parametrize("bins", ["float", "fixed"])
def test_tile_and_chunk_order_keep_frames(bins):
    """From the first frame (no counts yet) on, over changing numbers of blocks and several datasets."""
    wl = W.volume_lut(150_000, n_az=64, n_el=40, seed=41)
    wl.fixed.append(W.volume_lut(100_000, n_az=2, n_el=2, seed=42).fixed[0])
    on, off = (sim(wl, tile_order=m, chunk_order=m, bin_accumulation=bins) for m in ("on", "off"))
    o, d, l, t, length = wl.scan
    for keep in (2560, 2560, 2048, 2560, 640):
        for s in (on, off):
            s.set_scan_sequence(o[:keep], d[:keep], length, l[:keep], t[:keep], False)
        a, b = tiled(on), tiled(off)
        assert np.abs(b).max() > 0 and rel_l2(a, b) < 1e-6
        assert np.array_equal(np.abs(on.get_projection()) > 0, np.abs(off.get_projection()) > 0)
    on.close()
    off.close()


def test_frames_equal_those_in_range_order():
    for wl in (W.volume_lut(100_000, n_az=32, n_el=24, seed=43, phase_delay=True),
               W.fixed_sector_2d(60_000, 200, seed=44, line_length=0.08)):
        a, b = sim(wl), sim(wl, bin_accumulation="float")
        x, y = a.simulate_frame(), tiled(b)
        assert "range order" in a.get_parameter("launch_plan")
        assert np.abs(y).max() > 0 and rel_l2(x, y) < 1e-6
        a.close()
        b.close()


def test_tuned_shapes_match_the_default():
    for k, (wl, bins) in enumerate(((W.fixed_sector_2d(30_000, 48, seed=75, phase_delay=True), "fixed"),
                                    (W.fixed_sector_2d(30_000, 260, seed=76), "float"),
                                    (W.volume_lut(40_000, n_az=24, n_el=24, seed=78), "float"))):
        plain = sim(wl, bin_accumulation=bins)
        tuned = sim(wl, bin_accumulation=bins, autotune="on")
        a = tiled(plain)
        for _ in range(2):
            assert rel_l2(tiled(tuned), a) < 1e-6, k
        plain.close()
        tuned.close()


@pytest.mark.parametrize("lines,length,decimation", [(8, 0.028, 1), (8, 0.12, 1), (48, 0.12, 1), (340, 0.12, 1),
                                                     (640, 0.13, 1)])
def test_host_copies(lines, length, decimation):
    """0.1 and 0.5 MB: the runtime's copy; 3 MB: pinned pieces, moved by one thread; 21 MB: by several; 43 MB: two
    buffers by turns."""
    from openbcsim_amd.hip_rt import DeviceBuffer
    wl = W.fixed_sector_2d(3000, lines, seed=47, line_length=length, decimation=decimation)
    s = sim(wl, tile_order="off")
    host = s.simulate_frame()
    L, S = s.output_shape()
    assert (host.nbytes < 128 << 10) == (length == 0.028)
    dev = DeviceBuffer(L * S * 8)
    s.simulate_lines_device(dev.address, L * S)
    s.synchronize()
    ref = np.empty((L, S), np.complex64)
    dev.to_host(ref)
    assert np.abs(ref).max() > 0 and rel_l2(host, ref) < 1e-6
    # again, into buffers that were copied into before, and a smaller frame after a larger one
    assert rel_l2(s.simulate_frame(), ref) < 1e-6 and rel_l2(s.simulate_lines(), ref.T) < 1e-6
    o, d, l, t, ln = wl.scan
    s.set_scan_sequence(o[:5], d[:5], ln, l[:5], t[:5], False)
    assert rel_l2(s.simulate_frame(), ref[:5]) < 1e-6
    s.close()
