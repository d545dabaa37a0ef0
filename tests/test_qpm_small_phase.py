"""The z sum for mismatches near zero, whose imaginary part is sum w dk z: the
terms are of the order of w, so neither part loses digits or underflows.

Bound: phases of one sign carry a few roundings of their size and the sum one
for each run, so either part is off by (n_run + 16) 2^-53 of itself at most."""
import numpy as np
import pytest

from optifax_amd import qpm


@pytest.mark.gpu
@pytest.mark.parametrize("lengths", [[1] * 7, [4, 1, 9, 2, 3], [30]])
def test_small_mismatch(lengths):
    w = np.repeat(1e-3 * (1.0 + np.arange(len(lengths))), lengths)
    z = 1e-3 * np.arange(1, w.size + 1)
    dk = np.array([1e-9, 1e-14, 1e-15, 1e-16, 1e-100, 1e-155, 1e-200, 1e-250, 1e-290, -1e-290, 0.0])
    got = qpm.zsum(dk, z, w)
    assert qpm.zsum.last_runs == len(lengths)
    ph = dk[:, None].astype(np.longdouble) * z.astype(np.longdouble)
    re, im = (w * np.cos(ph)).sum(1), (w * np.sin(ph)).sum(1)
    eps = (len(lengths) + 16) * 2.0 ** -53
    assert np.all(np.abs(got.real - re) <= eps * np.abs(re))
    assert np.all(np.abs(got.imag - im) <= eps * np.abs(im))
