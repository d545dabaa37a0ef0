"""A batch of uneven instances (ofx_opo_create's uneven shares): each runs on a
cluster of its own size, and grids of different sizes follow each other in one
cluster.  Results are those of the instance alone on the general kernel, to the
last bit (the sums over a trip, whose order is the members', to rounding)."""
import os

import numpy as np
import pytest

from cases import opo_case
from optifax_amd.solver import Context, OPOBatch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def instances(sizes):
    out = []
    for n, length in sizes:
        cfg, b = opo_case(n=n, window=3e-12 * (n / 512) ** 0.5, length=length, energy=2e-9)
        ops = b["ops"]
        out.append(dict(solver=b["solver"], field0=ops["field0"], pump=ops["pump"],
                        cav=ops["cav"], ocm=ops["ocm"], delay=cfg.delay))
    return out


def read(run, i):
    r = run.read(i)
    r["avg"], r["xavg"], _ = run.read_average(i)
    return r


def check(ctx, sizes, precision, uneven):
    insts = instances(sizes)
    run = OPOBatch(insts, precision=precision, trip_cap=4, ctx=ctx)
    used = [run.geometry(i)["cluster"] for i in range(len(insts))]
    run.launch(2)
    run.sync()
    got = [read(run, i) for i in range(len(insts))]
    run.close()
    assert uneven(used), used
    for i, inst in enumerate(insts):
        alone = OPOBatch([inst], precision=precision, trip_cap=4, ctx=ctx,
                         tune=dict(exchange=2))
        alone.launch(2)
        alone.sync()
        want = read(alone, 0)
        alone.close()
        assert (got[i]["attempts"], got[i]["status"]) == (want["attempts"], want["status"])
        for k in ("field", "oc_spec", "apft", "avg", "xavg", "stepmods"):
            assert np.array_equal(got[i][k], want[k]), (i, k)
        # sums of n terms in another order: n rounding errors at most
        np.testing.assert_allclose(got[i]["trip_log"][:2], want["trip_log"][:2],
                                   rtol=sizes[i][0] * 2.0 ** -52)


@pytest.mark.parametrize("precision", ["single", "double"])
def test_emulated_uneven_batch(precision):
    path = os.path.join(ROOT, "tests", "emu", "libofx_emu.so")
    if not os.path.exists(path):
        pytest.skip("emulation library not built")
    old = os.environ.get("OFX_EMU_CUS")
    os.environ["OFX_EMU_CUS"] = "8"
    ctx = Context(0, lib_path=path)
    if old is None:
        del os.environ["OFX_EMU_CUS"]
    else:
        os.environ["OFX_EMU_CUS"] = old
    # two clusters of four and more instances than clusters
    sizes = [(2048, 30e-6), (1024, 6e-6), (2048, 6e-6), (4096, 4e-6), (512, 20e-6)]
    check(ctx, sizes, precision, lambda used: True)
    ctx.close()


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("count,lo,hi", [(40, 13, 15), (12, 13, 15), (24, 14, 16), (9, 11, 13)])
def test_uneven_batch(count, lo, hi, precision):
    ctx = Context(0)
    sizes = [(2 ** (lo + i % (hi - lo + 1)), 5e-6 + 25e-6 * ((i * 0.618) % 1.0))
             for i in range(count)]
    check(ctx, sizes, precision, lambda used: len(set(used)) > 1)
    ctx.close()
