"""The z sum's shares (16, 4 or 1 per output, by the number of outputs) against
the literal sum in extended precision: sizes on both sides of each line, run
counts below, at and beyond the shares and the 512-run staging chunk, runs of
one sample, and step phases of exactly 0 and 2 pi.

Bound per output: every term's phase carries a few roundings of its size, so
|error| <= 2^-53 (4 max|k z| + 32) sum |w|."""
import numpy as np
import pytest

from optifax_amd import qpm


def grating(n_run, seed, longest):
    """Samples of n_run runs of 1..longest samples, weights alternating in sign."""
    rng = np.random.default_rng(seed)
    lens = rng.integers(1, longest + 1, n_run)
    w = np.repeat(np.where(np.arange(n_run) % 2, -1.0, 1.0), lens)
    return 1e-6 * np.arange(w.size), w * 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("n_out,n_run,longest", [
    (1, 1, 1), (15, 3, 1), (17, 15, 9), (257, 16, 9), (1000, 513, 3), (2 ** 15 - 1, 33, 5),
    (2 ** 15, 33, 5), (2 ** 15 + 3, 5, 2), (2 ** 19 - 1, 7, 3), (2 ** 19, 7, 3)])
def test_zsum_shares_match_literal_sum(n_out, n_run, longest):
    z, w = grating(n_run, n_out, longest)
    rng = np.random.default_rng(1)
    dk = rng.uniform(0.0, 8e5, n_out)
    dk[0] = 0.0
    if n_out > 2:
        dk[1], dk[2] = 2 * np.pi / 1e-6, 1e-9
    got = qpm.zsum(dk, z, w)
    pick = np.unique(np.concatenate([[0, n_out - 1], np.arange(min(n_out, 3)),
                                     rng.integers(0, n_out, 200)]))
    want = np.zeros(pick.size, np.clongdouble)
    for zk, wk in zip(z.astype(np.longdouble), w.astype(np.longdouble)):
        want += wk * np.exp(1j * dk[pick].astype(np.longdouble) * zk)
    bound = 2.0 ** -53 * (4 * np.abs(dk[pick]) * z[-1] + 32) * np.abs(w).sum()
    assert np.all(np.abs(got[pick] - want) <= bound)
