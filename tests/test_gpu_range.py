"""Projection in range order (project_range.hip) against the tile kernel, which runs
when a launch shape is set by hand, and against the FP64 oracle, at the sizes where
the range order's patches (64 lines), runs (4 bins), windows and point batches (64)
have remainders, and where its bounds and its rule for the far side of the origin
decide.

Tolerance: both kernels evaluate the same float32 coordinates, bins and weights (a
Gaussian's within a few roundings, 1e-6 of a weight at 6 sigma) and sum them in
another order, so frames agree to the 1e-6 that the tiled and the direct kernel
agree to."""
import math

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


def check(wl, oracle=True, ranged=True):
    iq, plan = frame(wl)
    assert ("range order" in plan) == ranged, plan
    tile, plan = frame(wl, tile_lines="1")
    assert "range order" not in plan, plan
    e = rel_l2(iq, tile)
    print(f"[result] {wl.name} lines={wl.num_lines} points={wl.num_scatterers}: range vs tile {e:.2e}", flush=True)
    assert np.abs(tile).max() > 0 and e < 1e-6
    if oracle:
        o = Oracle()
        wl.apply(o)
        assert rel_l2(iq, o.simulate_frame()) <= 1e-5
    return iq


def table(nr, side, depth):
    ext = (0.0, depth, -0.01, 0.01, -0.01, 0.01)
    return ("lut", ext, W.gaussian_lut(nr, side, side, ext[:2], ext[2:4], ext[4:], 0.5e-3, 3e-3))


@pytest.mark.parametrize("lines", [16, 63, 64, 65, 131])
@pytest.mark.parametrize("phase", [False, True])
def test_lines_per_patch(lines, phase):
    check(W.fixed_sector_2d(5000, lines, seed=lines, line_length=0.0301, phase_delay=phase))


@pytest.mark.parametrize("points", [1, 63, 64, 65, 4097])
@pytest.mark.parametrize("lut", [False, True])
def test_points_per_batch(points, lut):
    wl = W.fixed_sector_2d(points, 40, seed=points, line_length=0.05, sigma=4e-3)
    wl.fixed[0][:, :3] *= np.float32(0.3)  # every point near the axis and inside the lines
    if lut:
        wl.profile = table(20, 9, 0.05)
    check(wl)


@pytest.mark.parametrize("length", [0.0002, 0.004, 0.00503, 0.15])
@pytest.mark.parametrize("lut", [0, 2, 64, 700])
def test_line_lengths_and_tables(length, lut):
    """Lines of fewer samples than a window, and tables of less and more than a radial cell per window."""
    wl = W.fixed_sector_2d(20000, 70, seed=3, line_length=length, phase_delay=True)
    wl.fixed[0][:, :3] *= np.float32(length / 0.12)
    wl.fixed[0][:, 2] -= np.float32(0.05 * length)
    if lut:
        wl.profile = table(lut, 64 if lut == 64 else 17, length)
    # tables of many cells per sample: the slices of four bins do not fit LDS
    check(wl, ranged=not (lut >= 64 and length == 0.0002))


@pytest.mark.parametrize("lut", [False, True])
@pytest.mark.parametrize("phase", [False, True])
def test_points_around_the_origin(lut, phase):
    """Points on both sides of the scan origin and within a sample of it (bin 0 is reached
    from both sides), and several at the origin itself."""
    rng = np.random.default_rng(11)
    wl = W.fixed_sector_2d(100, 33, seed=1, line_length=0.02, phase_delay=phase)
    p = rng.uniform(-0.02, 0.02, (6000, 4)).astype(np.float32)
    p[:2000, :3] *= np.float32(1e-3)   # within 20 um: a sample is 15 um
    p[2000:2010, :3] = 0.0
    p[2010:4000, :3] *= np.float32(0.1)
    wl.fixed = [p]
    if lut:
        ext = (-0.004, 0.02, -0.01, 0.01, -0.012, 0.01)
        wl.profile = ("lut", ext, W.gaussian_lut(40, 21, 23, ext[:2], ext[2:4], ext[4:], 2e-3, 3e-3))
    check(wl)


@pytest.mark.parametrize("half_angle", [80.0, 179.0])
def test_wide_scans_split_into_narrow_patches(half_angle):
    wl = W.fixed_sector_2d(20000, 48, seed=4, line_length=0.05)
    wl.scan = W.sector_scan(48, math.radians(2 * half_angle), 0.05)
    wl.fixed[0][:, 2] -= np.float32(0.06)
    check(wl)


def test_origin_away_from_zero_and_cutoff_off():
    wl = W.volume_lut(30000, n_az=9, n_el=11, seed=5, lut_shape=(64, 48, 32), line_length=0.1)
    o, d, l, t, length = wl.scan
    wl.scan = (o + np.float32([0.003, -0.002, 0.001]), d, l, t, length)
    check(wl)
    a, _ = frame(wl, weight_cutoff="0")
    b, _ = frame(wl, weight_cutoff="0", tile_lines="1")
    assert rel_l2(a, b) < 1e-6


@pytest.mark.parametrize("lut", [False, True])
def test_several_datasets_accumulate(lut):
    wl = W.fixed_sector_2d(7000, 70, seed=6, line_length=0.06, phase_delay=True)
    wl.fixed.append(W.fixed_sector_2d(3001, 70, seed=7).fixed[0])
    wl.splines = W.spline_mmode(2000, 70, seed=8).splines
    if lut:
        wl.profile = table(64, 33, 0.06)
    check(wl)


@pytest.mark.parametrize("splines,lines,lut", [(70001, 200, False), (60000, 128, True)])
def test_rendered_splines(splines, lines, lut):
    """Splines at one time are sorted for every frame: frames at several times, and a frame
    after another simulator's, equal the tile kernel's."""
    from openbcsim_amd.pyrfsim import RfSimulator
    wl = W.spline_mmode(splines, lines, seed=12, all_timestamps_equal=True, line_length=0.05, phase_delay=True)
    for s in wl.splines:
        s.control_points *= np.float32(0.45)
    if lut:
        wl.profile = table(40, 24, 0.05)
    g = RfSimulator("gpu")
    wl.apply(g)
    o, d, l, _, length = wl.scan
    for t in (0.1, 0.83, 0.1):
        ts = np.full(lines, t, np.float32)
        wl.scan = (o, d, l, ts, length)
        g.set_scan_sequence(o, d, length, l, ts, True)
        a = g.simulate_frame()
        assert "range order" in g.get_parameter("launch_plan")
        b, plan = frame(wl, tile_lines="1")
        assert "range order" not in plan and rel_l2(a, b) < 1e-6
        assert np.array_equal(g.simulate_lines(), g.simulate_frame().T) or rel_l2(g.simulate_lines(), a.T) < 1e-6
    g.close()


@pytest.mark.parametrize("lines,decimation", [(1, 1), (33, 3), (96, 1), (700, 2)])
def test_frame_by_sample_is_the_frame_turned(lines, decimation):
    """simulate_lines' (samples, lines) array is simulate_frame's transposed, for host copies
    below, at and above the sizes where they pass through pinned pieces."""
    from openbcsim_amd.pyrfsim import RfSimulator
    g = RfSimulator("gpu")
    W.fixed_sector_2d(3000, lines, seed=13, decimation=decimation).apply(g)
    a = g.simulate_frame()
    b = g.simulate_lines()
    assert b.shape == a.T.shape and b.flags.c_contiguous and b.dtype == np.complex64
    assert np.abs(a).max() > 0 and rel_l2(b, a.T) < 1e-6
    g.close()


def test_changes_between_frames():
    """New directions, time, length, origin and demodulation between frames of one simulator:
    each frame equals a new simulator's."""
    from openbcsim_amd.pyrfsim import RfSimulator
    wl = W.fixed_sector_2d(20000, 96, seed=9, line_length=0.06, phase_delay=True)
    g = RfSimulator("gpu")
    wl.apply(g)
    base = wl.scan
    scans = [W.sector_scan(96, math.radians(70), 0.06), W.sector_scan(80, math.radians(50), 0.06),
             W.sector_scan(80, math.radians(50), 0.03), W.sector_scan(80, math.radians(50), 0.03, tilt=0.2),
             (base[0] + np.float32(0.002), base[1], base[2], base[3], 0.06)] + [
             (base[0] + np.float32(0.001 * k), base[1], base[2], base[3], 0.05) for k in range(1, 6)]
    for k, (o, d, l, t, length) in enumerate(scans):
        wl.scan = (o, d, l, t, length)
        wl.demod_freq = W.FC * (1 + k % 2)
        g.set_excitation(wl.excitation, wl.center_index, wl.fs, wl.demod_freq)
        g.set_scan_sequence(o, d, length, l, t)
        a = g.simulate_frame()
        b, _ = frame(wl, tile_lines="1")
        assert rel_l2(a, b) < 1e-6, k
    g.close()


def test_counters_match_the_tile_kernel():
    from openbcsim_amd.pyrfsim import RfSimulator
    wl = W.fixed_sector_2d(20000, 70, seed=10, line_length=0.06)
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


def test_batch_jobs():
    """Fixed points of a Gaussian beam in a batch: patches of one and several, runs of two and
    four bins, phase delay, an odd last run, beside jobs of the tile kernels; equal to the tile
    kernels' bins, and the same on a second frame and after the batch's jobs change."""
    from openbcsim_amd.batch import Batch
    from openbcsim_amd.pyrfsim import RfSimulator
    sims = []
    for n, lines, length, phase in ((5000, 16, 0.03, False), (25001, 48, 0.0601, True), (90000, 65, 0.02, False),
                                    (8000, 200, 0.05, True), (3000, 9, 0.04, False)):
        g = RfSimulator("gpu")
        W.fixed_sector_2d(n, lines, seed=lines, line_length=length, phase_delay=phase).apply(g)
        sims.append(g)
    batch, tiles = Batch(sims), Batch(sims)
    tiles.set_parameter("tile_lines", "1")
    for g in sims:
        assert ("range order" in (g.simulate_frame() is not None and g.get_parameter("launch_plan"))) == (g.output_shape()[0] >= 16)
    want = tiles.simulate()
    for _ in range(2):
        for a, b in zip(batch.simulate(), want):
            assert np.abs(b).max() > 0 and rel_l2(a, b) < 1e-6
    sims[0].set_parameter("sound_speed", "1500")
    for a, b in zip(batch.simulate(), tiles.simulate()):
        assert rel_l2(a, b) < 1e-6
    for x in (batch, tiles, *sims):
        x.close()
