"""The fibre solver's kernel for long grids (optifax_amd/csrc/ofx_gnlse_wide.h)
against the oracle, on the device and in the emulation: FP64 grids of 2^11 and
2^12 points (whose half-length transforms end in a radix-2 and a radix-4 pass)
and the FP32 grid of 2^13, with and without the Raman term and self-steepening,
and the first grid below each line, which the general kernel runs.

Bounds: ~70 evaluations of transforms of up to 13 passes add rounding errors of
~2^-53 (2^-24) per pass and sample; with a factor 30 for their growth over 2 mm,
1e-12 (FP64) and 3e-5 (FP32)."""
import os

import numpy as np
import pytest

from optifax_amd import _lib, fibre
from test_gnlse import dudley_case, gain_case, rel
import oracle.gnlse as og

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CASES = [(1024, "double"), (2048, "double"), (4096, "double"), (4096, "single"), (8192, "single")]


def solve(c, precision, lib):
    op = fibre.operators(c["T"], c["w0"], c["gamma"], c["betas"], 0.0, c["fr"], c["RT"])
    Z, AWz, stats, _ = fibre.gnlse_batch(c["T"], [c["A"], 0.8 * c["A"]], [op] * 2, c["flength"], 5,
                                         precision, lib=lib, max_steps=20000)
    return fibre.lab_frame(Z, AWz[0], op, c["T"].size, op["dT"])[0], stats


def check(c, precision, lib, bound):
    _, want, _, _, _, st = og.gnlsefib(c["T"], c["A"], c["w0"], c["gamma"], c["betas"], 0.0, c["fr"],
                                       c["RT"], c["flength"], 5)
    got, stats = solve(c, precision, lib)
    assert stats[0].tolist() == [st["accepted"], st["rejected"], st["evaluations"], 0]
    assert stats[1, 3] == 0
    assert rel(got, want) < bound


def emu():
    path = os.path.join(ROOT, "tests", "emu", "libofx_emu.so")
    if not os.path.exists(path):
        pytest.skip("emulation library not built")
    return _lib.load(path)


@pytest.mark.parametrize("raman,shock", [(True, True), (False, True), (True, False)])
@pytest.mark.parametrize("n,precision", CASES[1:])
def test_emulated_long_grids_match_the_oracle(n, precision, raman, shock):
    c = dudley_case(n=n, raman=raman, shock=shock, flength=0.002)
    check(c, precision, emu(), 1e-12 if precision == "double" else 3e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("raman,shock", [(True, True), (False, True), (True, False)])
@pytest.mark.parametrize("n,precision", CASES)
def test_long_grids_match_the_oracle(n, precision, raman, shock):
    c = dudley_case(n=n, raman=raman, shock=shock, flength=0.002)
    check(c, precision, None, 1e-12 if precision == "double" else 3e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2048, 4096])
def test_rejected_steps_match_the_oracle(n):
    c = gain_case(n=n)
    _, want, _, _, _, st = og.gnlsefib(c["T"], c["A"], c["w0"], c["gamma"], c["betas"], c["loss"],
                                       c["fr"], c["RT"], c["flength"], 5)
    op = fibre.operators(c["T"], c["w0"], c["gamma"], c["betas"], c["loss"], c["fr"], c["RT"])
    Z, AWz, stats, _ = fibre.gnlse_batch(c["T"], [c["A"]], [op], c["flength"], 5, "double",
                                         max_steps=20000)
    assert st["rejected"] > 0
    assert stats[0].tolist() == [st["accepted"], st["rejected"], st["evaluations"], 0]
    got = fibre.lab_frame(Z, AWz[0], op, n, op["dT"])[0]
    assert rel(got, want) < 1e-9


@pytest.mark.gpu
def test_nonfinite_field_and_step_cap_are_reported():
    c = dudley_case(n=4096, flength=0.002)
    op = fibre.operators(c["T"], c["w0"], c["gamma"], c["betas"], 0.0, c["fr"], c["RT"])
    bad = c["A"].copy()
    bad[7] = np.nan
    _, _, stats, _ = fibre.gnlse_batch(c["T"], [bad, c["A"]], [op] * 2, c["flength"], 3, "double",
                                       max_steps=20000)
    assert stats[0, 3] == 3 and stats[1, 3] == 0
    _, _, stats, _ = fibre.gnlse_batch(c["T"], [c["A"]], [op], c["flength"], 3, "double", max_steps=2)
    assert stats[0, 3] == 2
