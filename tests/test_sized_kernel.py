"""The general kernel with fixed grid splits (optifax_amd/csrc/ofx_backend_sized.hip:
512 threads, counter barrier, no RK23 in the launch) against the general one at
256 threads: the same bits.  Splits with a compiled form, one without (2^11), a
split the caller gives, one workgroup to many, and grids of several sizes in one
launch."""
import numpy as np
import pytest

from cases import opo_case
from optifax_amd.solver import Context, OPOBatch
from test_wave_kernel import emu  # noqa: F401  (fixture)

KEYS = ("field", "oc_spec", "apft", "stepmods")
SHAPES = [(2048, 4, 0), (4096, 1, 0), (4096, 8, 0), (8192, 4, 0), (16384, 16, 0), (16384, 8, 256),
          (32768, 16, 0), (65536, 32, 0)]


def instance(n, length, cluster=0, n1=0):
    cfg, b = opo_case(n=n, window=3e-12 * (n / 512) ** 0.5, length=length, energy=2e-9)
    ops = b["ops"]
    inst = dict(solver=b["solver"], field0=ops["field0"], pump=ops["pump"], cav=ops["cav"],
                ocm=ops["ocm"], delay=cfg.delay)
    if cluster:
        inst["cluster"] = cluster
    if n1:
        inst["n1"] = n1
    return inst


def trips(ctx, insts, precision, block, count=2):
    run = OPOBatch(insts, precision=precision, trip_cap=4, ctx=ctx,
                   tune=dict(block=block, exchange="barrier"))
    run.launch(count)
    run.sync()
    out = [run.read(i) for i in range(len(insts))]
    run.close()
    return out


def same(x, y):
    for a, b in zip(x, y):
        assert (a["attempts"], a["accepted"], a["status"]) == (b["attempts"], b["accepted"], b["status"])
        for k in KEYS:
            assert np.array_equal(a[k], b[k]), k


@pytest.mark.parametrize("precision", ["single", "double"])
def test_emulated_sized_kernel(emu, precision):  # noqa: F811
    for n, C in ((2048, 4), (4096, 8), (8192, 8)):
        insts = [instance(n, 6e-6, C)]
        same(trips(emu, insts, precision, 512, 1), trips(emu, insts, precision, 256, 1))


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("n,C,n1", SHAPES)
def test_sized_kernel_matches_general(n, C, n1, precision):
    if precision == "double" and (n, C) in ((4096, 1), (65536, 32)):
        pytest.skip("the share does not fit LDS in FP64")
    ctx = Context(0)
    insts = [instance(n, 20e-6, C, n1)]
    same(trips(ctx, insts, precision, 512), trips(ctx, insts, precision, 256))
    ctx.close()


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["single", "double"])
def test_sized_kernel_in_a_mixed_launch(precision):
    ctx = Context(0)
    insts = [instance(n, 20e-6, n // 1024) for n in (2048, 4096, 8192, 16384, 32768, 65536)]
    same(trips(ctx, insts, precision, 512), trips(ctx, insts, precision, 256))
    ctx.close()
