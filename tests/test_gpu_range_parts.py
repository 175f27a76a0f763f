"""Range order over points that crowd at some distances: blocks of bins with many points
are projected in parts (project_range_parts_kernel).  Against the tile kernel, which runs
when a launch shape is set by hand, and the FP64 oracle, at line counts around a patch and a
workgroup's patches, part counts from one to the most, blocks cut by the line's end and
points on both sides of the origin.

Tolerance: the weights are the tile kernel's; a bin is a sum of doubles, then of at most 64
floats, so frames agree to the 1e-6 that the tiled and the direct kernel agree to."""
import numpy as np
import pytest

from backends import Oracle, rel_l2
from openbcsim_amd import workloads as W

pytestmark = pytest.mark.gpu


def frame(wl, **params):
    from openbcsim_amd.pyrfsim import RfSimulator
    g = RfSimulator("gpu")
    wl.apply(g)
    for k, v in params.items():
        g.set_parameter(k, v)
    iq = g.simulate_frame()
    plan = g.get_parameter("launch_plan")
    g.close()
    return iq, plan


def check(wl, parts=True, oracle=True):
    iq, plan = frame(wl)
    assert "range order" in plan and ("in parts" in plan) == parts, plan
    tile, plan = frame(wl, tile_lines="1")
    assert "range order" not in plan
    e = rel_l2(iq, tile)
    print(f"[result] lines={wl.num_lines} points={wl.num_scatterers}: parts vs tile {e:.2e}", flush=True)
    assert np.abs(tile).max() > 0 and e < 1e-6
    if oracle:
        o = Oracle()
        wl.apply(o)
        assert rel_l2(iq, o.simulate_frame()) <= 1e-5


def shell(points, lines, radius, thickness, line_length=0.05, phase=False, seed=1, around=0.6):
    wl = W.fixed_sector_2d(points, lines, seed=seed, line_length=line_length, phase_delay=phase)
    rng = np.random.default_rng(seed)
    p = wl.fixed[0]
    r = radius + thickness * (rng.uniform(-0.5, 0.5, points))
    a, y = rng.uniform(-around, around, points), rng.uniform(-0.004, 0.004, points)
    z = np.sqrt(np.maximum(r ** 2 - y ** 2, 0))
    p[:, 0], p[:, 1], p[:, 2] = z * np.sin(a), y, z * np.cos(a)
    return wl


def table(nr, side, depth=0.05):
    ext = (0.0, depth, -0.01, 0.01, -0.01, 0.01)
    return ("lut", ext, W.gaussian_lut(nr, side, side, ext[:2], ext[2:4], ext[4:], 0.5e-3, 3e-3))


@pytest.mark.parametrize("phase", [False, True])
@pytest.mark.parametrize("lines,lut", [(16, False), (65, False), (129, False), (700, False), (16, True), (33, True),
                                       (65, True)])
def test_lines(lines, lut, phase):
    wl = shell(20011, lines, 0.03, 1e-4, phase=phase, seed=lines)
    if lut:
        wl.profile = table(40, 24)
    check(wl)


@pytest.mark.parametrize("points", [6000, 33000, 70001])
@pytest.mark.parametrize("thickness", [0.0, 3e-5])
def test_parts_of_one_block(points, thickness):
    """All points within a block or two: 12 parts, and as many as there are."""
    check(shell(points, 40, 0.03, thickness, seed=points))


def test_few_of_the_points_crowd():
    wl = W.fixed_sector_2d(60000, 80, seed=2, line_length=0.05, phase_delay=True)
    wl.fixed[0][:4000] = shell(4000, 80, 0.022, 0.0, seed=3).fixed[0]
    check(wl)
    wl.profile = table(64, 33)
    check(wl)


@pytest.mark.parametrize("radius", [0.0295, 0.02999, 0.0302])
def test_end_of_the_line(radius):
    """Points around the last bins: part of a block lies beyond the line."""
    wl = shell(30000, 70, radius, 6e-4, line_length=0.03, phase=True, seed=5)
    wl.fixed[0][:100, :3] *= np.float32(0.5)
    iq, plan = frame(wl)
    tile, _ = frame(wl, tile_lines="1")
    assert "range order" in plan and np.abs(tile).max() > 0 and rel_l2(iq, tile) < 1e-6


@pytest.mark.parametrize("lut", [False, True])
def test_around_the_origin(lut):
    rng = np.random.default_rng(11)
    wl = W.fixed_sector_2d(100, 33, seed=1, line_length=0.02, phase_delay=True)
    p = rng.uniform(-0.02, 0.02, (9000, 4)).astype(np.float32)
    p[:6000, :3] *= np.float32(1e-3)  # within 20 um: a sample is 15 um
    p[6000:6010, :3] = 0.0
    wl.fixed = [p]
    if lut:
        ext = (-0.004, 0.02, -0.01, 0.01, -0.012, 0.01)
        wl.profile = ("lut", ext, W.gaussian_lut(40, 21, 23, ext[:2], ext[2:4], ext[4:], 2e-3, 3e-3))
    check(wl)


def test_several_datasets_and_wide_volumes():
    wl = shell(20000, 70, 0.03, 1e-4, phase=True)
    wl.fixed.append(W.fixed_sector_2d(3001, 70, seed=7).fixed[0])
    check(wl)
    wl = W.volume_lut(200, n_az=27, n_el=31, seed=5, lut_shape=(64, 48, 32), line_length=0.1)
    wl.fixed = [shell(40000, 70, 0.08, 5e-5, seed=9, around=0.5).fixed[0]]
    wl.fixed[0][:, 1] *= np.float32(5.0)
    check(wl, oracle=False)


def test_counters():
    from openbcsim_amd.pyrfsim import RfSimulator
    wl = shell(20000, 70, 0.03, 1e-4)
    got = []
    for shape in ("0", "1"):
        g = RfSimulator("gpu")
        wl.apply(g)
        g.set_parameter("tile_lines", shape)
        g.set_parameter("projection_counters", "on")
        g.simulate_frame()
        got.append([g.get_debug_data(k)[0] for k in ("projection_weight_evals", "projection_lds_adds",
                                                     "projection_chunk_line_pairs")])
        g.close()
    assert abs(got[0][0] - got[1][0]) <= 1e-5 * got[1][0] + 2
    assert abs(got[0][1] - got[1][1]) <= 1e-5 * got[1][1] + 2
    assert 64 * got[0][2] >= got[0][0]


def test_batch_jobs_with_crowds_run_the_tile_kernel():
    from openbcsim_amd.batch import Batch
    from openbcsim_amd.pyrfsim import RfSimulator
    sims, want = [], []
    for wl in (shell(20011, 65, 0.03, 1e-4, phase=True), W.fixed_sector_2d(9000, 40, seed=4, line_length=0.04)):
        g = RfSimulator("gpu")
        wl.apply(g)
        sims.append(g)
        want.append(frame(wl, tile_lines="1")[0])
    batch = Batch(sims)
    for _ in range(2):
        for a, b in zip(batch.simulate(), want):
            assert np.abs(b).max() > 0 and rel_l2(a, b) < 1e-6
    for x in (batch, *sims):
        x.close()


def test_steering_without_waiting():
    """Frames of other directions enqueued one after another: each has its own patches."""
    from openbcsim_amd.hip_rt import DeviceBuffer
    from openbcsim_amd.pyrfsim import RfSimulator
    wl = W.fixed_sector_2d(20000, 96, seed=9, line_length=0.05, phase_delay=True)
    g = RfSimulator("gpu")
    wl.apply(g)
    L, S = g.output_shape()
    outs, want = [], []
    for k in range(6):
        o, d, l, t, length = W.sector_scan(96, 0.6 + 0.12 * k, 0.05)
        g.set_scan_sequence(o, d, length, l, t)
        outs.append(DeviceBuffer(L * S * 8))
        g.simulate_lines_device(outs[-1].address, L * S)
        assert "range order" in g.get_parameter("launch_plan")
    g.synchronize()
    for k, out in enumerate(outs):
        wl.scan = W.sector_scan(96, 0.6 + 0.12 * k, 0.05)
        iq = np.empty((L, S), np.complex64)
        out.to_host(iq)
        assert rel_l2(iq, frame(wl, tile_lines="1")[0]) < 1e-6, k
    g.close()
