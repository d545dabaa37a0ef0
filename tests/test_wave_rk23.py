"""The wave kernel's RK23 pass (optifax_amd/csrc/ofx_wave_rk23.h) against the
general one (forced by the counter-barrier exchange): the same step sequences
and, as every rounding is the same, the same bits.

Geometries: one workgroup without an exchange, one wave and several waves per
workgroup, with and without waves that have no row, the fewest own columns (4:
every column is a boundary column), 1, 2 and 4 points a thread; the default
geometries, whose kernels have them fixed at compile time.  Strong pumping, so
that steps are rejected and K1 is formed again."""
import numpy as np
import pytest

from cases import opo_case
from optifax_amd.solver import Context, OPOBatch
from test_wave_kernel import check, emu  # noqa: F401  (emu: fixture)

SMALL = [(64, 1, 64), (64, 2, 64), (128, 1, 64), (256, 1, 64), (256, 4, 64), (256, 1, 256),
         (512, 1, 128), (512, 1, 256), (512, 8, 64), (1024, 1, 256), (1024, 8, 128),
         (2048, 16, 64), (2048, 2, 256)]
LARGE = [(4096, 16, 128), (4096, 16, 256), (4096, 8, 128), (8192, 32, 64), (8192, 32, 256),
         (16384, 32, 128), (16384, 32, 256), (32768, 64, 256), (32768, 32, 256)]
# grids with their default geometry
FIXED = [(2 ** lg, 0, 0) for lg in range(8, 17)]


def both(ctx, n, C, block, precision, trips, length, energy=2e-9, cavity=True):
    cfg, b = opo_case(n=n, window=3e-12 * (n / 512) ** 0.5, length=length, energy=energy)
    ops = b["ops"]
    inst = dict(solver=b["solver"], field0=ops["field0"], delay=cfg.delay, method="rk23")
    if cavity:
        inst.update(pump=ops["pump"], cav=ops["cav"], ocm=ops["ocm"])
    out = []
    for exchange in ("barrier", "tags"):
        tune = dict(exchange=exchange, cluster=C, block=block)
        if not C:
            tune = dict(exchange=exchange) if exchange == "barrier" else None
        run = OPOBatch([inst], precision=precision, trip_cap=4, ctx=ctx, tune=tune)
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


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("n,C,block", SMALL)
def test_emulated_rk23_wave_kernel_matches_general(emu, n, C, block, precision):  # noqa: F811
    general, wave = both(emu, n, C, block, precision, 2, 6e-6)
    check(general, wave)


def test_emulated_rk23_rejections(emu):  # noqa: F811
    general, wave = both(emu, 256, 4, 64, "single", 2, 10e-6, energy=2e-8)
    check(general, wave)
    assert wave["attempts"] > wave["accepted"]


@pytest.mark.parametrize("n", [256, 1024, 4096])
def test_emulated_fixed_rk23_matches_general(emu, n):  # noqa: F811
    check(*both(emu, n, 0, 0, "single", 1, 6e-6))


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("n,C,block", SMALL + LARGE + FIXED)
def test_rk23_wave_kernel_matches_general(n, C, block, precision):
    if precision == "double" and (n, C) in ((65536, 0), (32768, 32)):
        pytest.skip("does not fit LDS in one of the kernels")
    ctx = Context(0)
    check(*both(ctx, n, C, block, precision, 2, 20e-6))
    ctx.close()


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["single", "double"])
def test_rk23_rejections(precision):
    ctx = Context(0)
    general, wave = both(ctx, 8192, 0, 0, precision, 2, 20e-6, energy=2e-8)
    check(general, wave)
    assert wave["attempts"] > wave["accepted"]
    ctx.close()
