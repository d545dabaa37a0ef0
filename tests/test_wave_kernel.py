"""The wave kernel (optifax_amd/csrc/ofx_wave_impl.h) against the general one
(forced by the counter-barrier exchange): the same samples through the same
arithmetic with the same roundings, so the same step sequences and the same
bits.

Geometries: one workgroup without an exchange, one wave per workgroup, several
waves, odd and even transform lengths on either side, a partly filled wave of
rows and of columns, 1, 2 and 4 points a thread; the default geometries, whose
kernels have them fixed at compile time."""
import os

import numpy as np
import pytest

from cases import opo_case
from optifax_amd.solver import Context, OPOBatch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SMALL = [(64, 1, 64), (64, 2, 64), (128, 1, 64), (256, 1, 64), (256, 4, 64), (512, 8, 64),
         (512, 1, 128), (1024, 16, 64), (1024, 1, 256), (2048, 1, 512)]
LARGE = [(4096, 32, 128), (8192, 32, 128), (16384, 64, 256), (32768, 128, 256), (65536, 128, 512)]

FIXED_EMU = [(256, 1, 256), (512, 1, 256), (1024, 1, 512), (2048, 16, 128), (4096, 16, 256)]
FIXED = FIXED_EMU + [(8192, 32, 256)]
FIXED_F64 = [(1024, 1, 256), (65536, 128, 256)]   # (where FP64's differ from FP32's)


def both(ctx, n, C, block, precision, trips, length):
    cfg, b = opo_case(n=n, window=3e-12 * (n / 512) ** 0.5, length=length, energy=2e-9)
    ops = b["ops"]
    inst = dict(solver=b["solver"], field0=ops["field0"], pump=ops["pump"], cav=ops["cav"],
                ocm=ops["ocm"], delay=cfg.delay)
    out = []
    for exchange in ("barrier", "tags"):
        run = OPOBatch([inst], precision=precision, trip_cap=4, ctx=ctx,
                       tune=dict(cluster=C, block=block, exchange=exchange))
        run.keep_history(2)
        run.launch(trips)
        run.sync()
        r = run.read(0)
        r["hist"], r["hist_sm"] = run.read_history(0, trips - 1)
        r["avg"], r["xavg"], _ = run.read_average(0)
        r["lds"] = run.geometry(0)["lds_bytes"]
        run.close()
        out.append(r)
    return out


def check(general, wave):
    assert wave["lds"] != general["lds"]          # (another kernel's workspace)
    assert (wave["attempts"], wave["accepted"], wave["status"]) == \
        (general["attempts"], general["accepted"], general["status"])
    assert np.array_equal(wave["stepmods"], general["stepmods"])
    assert np.array_equal(wave["hist_sm"], general["hist_sm"])
    for k in ("field", "oc_spec", "apft", "hist", "avg", "xavg"):
        assert np.array_equal(wave[k], general[k]), k


@pytest.fixture(scope="module")
def emu():
    path = os.path.join(ROOT, "tests", "emu", "libofx_emu.so")
    if not os.path.exists(path):
        pytest.skip("emulation library not built")
    old = os.environ.get("OFX_EMU_CUS")
    os.environ["OFX_EMU_CUS"] = "64"
    ctx = Context(0, lib_path=path)
    if old is None:
        del os.environ["OFX_EMU_CUS"]
    else:
        os.environ["OFX_EMU_CUS"] = old
    yield ctx
    ctx.close()


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("n,C,block", SMALL + FIXED_EMU)
def test_emulated_wave_kernel_matches_general(emu, n, C, block, precision):
    check(*both(emu, n, C, block, precision, 2, 6e-6))


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("n,C,block", SMALL + LARGE + FIXED + FIXED_F64)
def test_wave_kernel_matches_general(n, C, block, precision):
    ctx = Context(0)
    check(*both(ctx, n, C, block, precision, 2, 20e-6))
    ctx.close()
