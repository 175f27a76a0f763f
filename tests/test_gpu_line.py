"""The one-line tile kernel (project_line_kernel: straight scans, and splines with a
time per line) against the direct kernel and the FP64 oracle, at chunk counts around a
chunk, a wave's turn and a list step, every spline degree, and both bin types.

Tolerance: the bins and weights are the direct kernel's; only the order of the sums
differs (the 1e-6 that the tiled and the direct kernel agree to)."""
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


def check(wl, **params):
    ref, _ = frame(wl, projection_mode="direct", weight_cutoff="0")
    o = Oracle()
    wl.apply(o)
    exact = o.simulate_frame()
    for bins in ("fixed", "float"):
        iq, plan = frame(wl, bin_accumulation=bins, weight_cutoff="0", **params)
        assert "lines=1 " in plan, plan
        e = rel_l2(iq, ref)
        print(f"[result] {wl.name} points={wl.num_scatterers} {bins}: vs direct {e:.2e}", flush=True)
        assert np.abs(ref).max() > 0 and e < 1e-6
        assert rel_l2(iq, exact) <= 1e-5


def straight(points, lines, arc, lut, phase):
    wl = W.fixed_sector_2d(points, lines, seed=points, line_length=0.05, arc=arc, phase_delay=phase, sigma=4e-3)
    wl.scan = W.linear_scan(lines, 0.05, 0.05)
    wl.fixed[0][:, 2] *= np.float32(0.45)
    if lut:
        ext = (0.0, 0.05, -0.01, 0.01, -0.01, 0.01)
        wl.profile = ("lut", ext, W.gaussian_lut(33, 17, 16, ext[:2], ext[2:4], ext[4:], 2e-3, 3e-3))
    return wl


@pytest.mark.parametrize("points", [1, 63, 64, 65, 1025, 70000])
@pytest.mark.parametrize("arc", [False, True])
def test_straight_scan_sizes(points, arc):
    check(straight(points, 5, arc, False, False))


@pytest.mark.parametrize("lut", [False, True])
@pytest.mark.parametrize("phase", [False, True])
def test_straight_scan_profiles(lut, phase):
    check(straight(9000, 7, False, lut, phase))
    check(straight(9000, 7, True, lut, phase), tile_windows="3", tile_lines="1")


@pytest.mark.parametrize("degree", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("phase", [False, True])
def test_spline_degrees(degree, phase):
    check(W.spline_mmode(4099, 6, seed=degree, num_cp=degree + 3, degree=degree, phase_delay=phase, sigma=3e-3))


@pytest.mark.parametrize("points", [1, 64, 200])
def test_few_splines_and_a_table(points):
    wl = W.spline_mmode(points, 9, seed=points, decimation=1, sigma=5e-3)
    wl.splines[0].control_points[:, :, :2] *= np.float32(0.1)
    check(wl)
    ext = (0.0, 0.12, -0.01, 0.01, -0.01, 0.01)
    wl.profile = ("lut", ext, W.gaussian_lut(20, 9, 9, ext[:2], ext[2:4], ext[4:], 2e-3, 3e-3))
    check(wl)
