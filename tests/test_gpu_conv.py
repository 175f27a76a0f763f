"""Convolution with transforms of constant length: every length, fold and kind of bins against
the kernel for any length (fft_radix 4), singly and in a batch.

Tolerance: a radix-R transform of 2^k points in float rounds each value about k log2 R / log2 R
times; with rounding errors of 2^-24 taken as all in one direction over the two transforms of up
to 14 stages each and the products between (about 32 roundings), a path is within 32 x 6e-8 =
1.9e-6 of exact, and two paths within 3.8e-6 of one another."""
import numpy as np
import pytest

from openbcsim_amd import workloads as W

pytestmark = pytest.mark.gpu
TOL = 3.8e-6


def rel_l2(a, b):
    return np.linalg.norm(a.astype(np.complex128) - b) / np.linalg.norm(b)


def setup(samples, decimation, phase, lines):
    """A sector of `lines` lines with `samples` RF samples a line (odd numbers included)."""
    from openbcsim_amd.pyrfsim import RfSimulator
    wl = W.fixed_sector_2d(4000, lines, seed=samples + decimation, decimation=decimation, phase_delay=phase)
    o, d, l, t, _ = wl.scan
    length = samples / wl.fs * float(wl.params["sound_speed"]) / 2.0
    wl.scan = (o, d, l, t, length)
    g = RfSimulator("gpu")
    wl.apply(g)
    return g, wl


@pytest.mark.parametrize("phase", [False, True])
@pytest.mark.parametrize("decimation", [1, 2, 3, 4, 6, 12])
@pytest.mark.parametrize("log2n", [11, 12, 13, 14])
def test_constant_lengths_match_any_length(log2n, decimation, phase):
    for samples, lines in (((1 << log2n) - 250, 3), ((1 << log2n) // 2 + 1, 2)):
        g, wl = setup(samples, decimation, phase, lines)
        assert wl.fft_len() == 1 << log2n
        g.set_parameter("fft_radix", "8")
        a = g.simulate_frame()
        g.set_parameter("fft_radix", "4")
        b = g.simulate_frame()
        assert a.shape == b.shape and np.abs(b).max() > 0
        assert rel_l2(a, b) < TOL
        g.close()


def test_batch_of_lengths_folds_and_kinds():
    """One batch whose jobs take different constant lengths, folds and kinds of bins, and the
    kernel for any length beside them."""
    from openbcsim_amd.batch import Batch
    jobs = [(1500, 1, False), (1500, 2, True), (3001, 2, False), (6000, 4, True), (9001, 3, False), (9001, 8, False), (700, 1, False)]
    sims = [setup(n, dec, phase, 2)[0] for n, dec, phase in jobs]
    single = []
    for g in sims:
        g.set_parameter("fft_radix", "4")
        single.append(g.simulate_frame())
        g.set_parameter("fft_radix", "8")
    batch = Batch(sims)
    for a, b in zip(batch.simulate(), single):
        assert rel_l2(a, b) < TOL
    batch.close()
    for g in sims:
        g.close()
