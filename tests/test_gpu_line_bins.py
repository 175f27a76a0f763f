"""Bins of one-line tiles with a lookup table (straight scans, splines with a time per
line): the automatic choice keeps float's relative precision for lines that see only the
tails of the beam, and samples that are not finite reach the frame as in float.

Tolerance: the contributions are the same float32 products, summed in float and in
double: a line's IQ agrees to a few float roundings (1e-6)."""
import numpy as np
import pytest

from backends import rel_l2
from openbcsim_amd import workloads as W

pytestmark = pytest.mark.gpu

EXT = (0.0, 0.05, -0.01, 0.01, -0.01, 0.01)


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


def scan(splines, phase, arc):
    lines = 24
    if splines:
        wl = W.spline_mmode(3000, lines, seed=5, line_length=0.05, phase_delay=phase)
        c = wl.splines[0].control_points
        c[:, :, 0] = 0.004 + 0.2 * np.abs(c[:, :, 0])
        c[:, :, 2] *= np.float32(0.4)
        o, d, l, t, length = wl.scan
        d[:], l[:] = [0, 0, 1], [1, 0, 0]
        o[:, 0] = np.linspace(-0.0055, 0.004, lines)
    else:
        wl = W.fixed_sector_2d(3000, lines, seed=6, line_length=0.05, phase_delay=phase, arc=arc)
        wl.scan = W.linear_scan(lines, 0.0095, 0.05)
        wl.scan[0][:, 0] -= np.float32(0.00075)
        wl.fixed[0][:, 0] = 0.004 + 0.2 * np.abs(wl.fixed[0][:, 0])
        wl.fixed[0][:, 2] *= np.float32(0.4)
    wl.profile = ("lut", EXT, W.gaussian_lut(17, 65, 33, EXT[:2], EXT[2:4], EXT[4:], 1.3e-3, 1.3e-3))
    return wl


@pytest.mark.parametrize("splines,phase,arc", [(False, False, False), (False, True, True), (True, False, True),
                                               (True, True, True)])
def test_tails_of_the_beam(splines, phase, arc):
    wl = scan(splines, phase, arc)
    a, plan = frame(wl, weight_cutoff="0")
    b, plan_b = frame(wl, weight_cutoff="0", bin_accumulation="float")
    assert "lines=1 " in plan and "bins=float" in plan_b, plan
    per_line = [rel_l2(x, y) for x, y in zip(a, b)]
    dim = np.abs(b).max(1)
    print(f"[result] lines' peaks {dim.min():.1e} .. {dim.max():.1e}: {max(per_line):.2e}; {plan.splitlines()[0]}", flush=True)
    assert 0 < dim.min() < 1e-8 * dim.max()
    assert max(per_line) < 1e-6


@pytest.mark.parametrize("splines", [False, True])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_samples_that_are_not_finite(splines, bad):
    wl = scan(splines, False, True)
    wl.profile[2][9, 40, 16] = bad
    a, _ = frame(wl)
    b, _ = frame(wl, bin_accumulation="float")
    bad_lines = ~np.isfinite(b).all(1)
    assert bad_lines.any() and not bad_lines.all()
    assert np.array_equal(bad_lines, ~np.isfinite(a).all(1))
    assert rel_l2(a[~bad_lines], b[~bad_lines]) < 1e-6


def test_batch_uses_the_same_bins():
    from openbcsim_amd.batch import Batch
    from openbcsim_amd.pyrfsim import RfSimulator
    sims, want = [], []
    for splines, phase in ((False, False), (True, True), (True, False)):
        wl = scan(splines, phase, True)
        g = RfSimulator("gpu")
        wl.apply(g)
        g.set_parameter("weight_cutoff", "0")
        sims.append(g)
        want.append(frame(wl, weight_cutoff="0", bin_accumulation="float")[0])
    for tune in ("on", "off"):
        batch = Batch(sims)
        batch.set_parameter("autotune", tune)
        for _ in range(2):
            for a, b in zip(batch.simulate(), want):
                # (several lines a tile: float bins)
                assert max(rel_l2(x, y) for x, y in zip(a, b)) < 1e-6
        batch.close()
    for g in sims:
        g.close()
