"""Uneven batches whose schedule is shown: cluster sizes that differ from equal
shares, and clusters of several workgroups in which grids of different sizes
follow each other (stale tags, offsets of the exchange buffers), for every
kernel that takes such launches.  Results are those of the instance alone on
the general kernel, bit for bit."""
import os

import numpy as np
import pytest

from cases import opo_case
from emu_launch import kernel, last_launch
from optifax_amd.solver import Context, OPOBatch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
KEYS = ("field", "oc_spec", "apft", "avg", "xavg", "stepmods")


@pytest.fixture(scope="module")
def ctx16():
    path = os.path.join(ROOT, "tests", "emu", "libofx_emu.so")
    if not os.path.exists(path):
        pytest.skip("emulation library not built")
    old = os.environ.get("OFX_EMU_CUS")
    os.environ["OFX_EMU_CUS"] = "16"
    ctx = Context(0, lib_path=path)
    if old is None:
        del os.environ["OFX_EMU_CUS"]
    else:
        os.environ["OFX_EMU_CUS"] = old
    yield ctx
    ctx.close()


def instance(n, length, method):
    cfg, b = opo_case(n=n, window=3e-12 * (n / 512) ** 0.5, length=length, energy=2e-9)
    ops = b["ops"]
    return dict(solver=b["solver"], field0=ops["field0"], pump=ops["pump"], cav=ops["cav"],
                ocm=ops["ocm"], delay=cfg.delay, method=method)


def read(run, i):
    r = run.read(i)
    r["avg"], r["xavg"], _ = run.read_average(i)
    return r


def sizes(ctx, insts, precision, tune):
    run = OPOBatch(insts, precision=precision, ctx=ctx, tune=tune)
    out = [run.geometry(i)["cluster"] for i in range(len(insts))]
    run.close()
    return out


def check(ctx, insts, precision):
    """Runs two trips of the batch against each instance alone; its cluster sizes."""
    run = OPOBatch(insts, precision=precision, trip_cap=4, ctx=ctx)
    used = [run.geometry(i)["cluster"] for i in range(len(insts))]
    run.launch(2)
    run.sync()
    got = [read(run, i) for i in range(len(insts))]
    run.close()
    assert used != sizes(ctx, insts, precision, dict(exchange="tags"))   # (equal shares)
    for i, inst in enumerate(insts):
        alone = OPOBatch([inst], precision=precision, trip_cap=4, ctx=ctx,
                         tune=dict(exchange="barrier"))
        alone.launch(2)
        alone.sync()
        want = read(alone, 0)
        alone.close()
        assert (got[i]["attempts"], got[i]["status"]) == (want["attempts"], want["status"])
        for k in KEYS:
            assert np.array_equal(got[i][k], want[k]), (i, k)
    return used


# (grid, crystal length [um], method) of every instance
HEUN, RK23 = "heun", "rk23"
EMULATED = [
    ("wave", "single", [(4096, 2, HEUN), (4096, 16, HEUN), (2048, 4, HEUN), (2048, 16, HEUN)]),
    ("wave", "double", [(2048, 4, HEUN), (2048, 8, HEUN), (4096, 16, HEUN), (4096, 2, HEUN),
                        (2048, 16, HEUN)]),
    ("wave rk23", "single", [(2048, 16, RK23), (4096, 2, RK23), (2048, 2, RK23), (2048, 4, RK23),
                             (4096, 16, RK23)]),
    ("wave rk23", "double", [(4096, 16, RK23), (2048, 8, RK23), (2048, 16, RK23),
                             (4096, 2, RK23)]),
    ("sized", "single", [(4096, 16, HEUN), (2048, 16, HEUN), (4096, 8, HEUN), (8192, 2, HEUN),
                         (8192, 16, HEUN)]),
    ("general barrier", "double", [(2048, 16, HEUN), (2048, 4, RK23), (4096, 2, HEUN),
                                   (8192, 2, HEUN), (4096, 16, HEUN), (4096, 8, RK23)])]


@pytest.mark.parametrize("name,precision,batch", EMULATED)
def test_emulated_schedule(ctx16, name, precision, batch):
    insts = [instance(n, um * 1e-6, method) for n, um, method in batch]
    run = OPOBatch(insts, precision=precision, ctx=ctx16)
    run.launch(0)
    run.sync()
    mode, schedule = last_launch(ctx16)
    run.close()
    assert kernel(mode) == name
    grids = {}
    for n, c in schedule:
        grids.setdefault(c, set()).add(n)
    assert max(len(g) for g in grids.values()) > 1
    assert min(check(ctx16, insts, precision)) > 1


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("methods", [(HEUN,), (RK23,), (HEUN, RK23)])
@pytest.mark.parametrize("count,lo,hi", [(9, 11, 13), (10, 12, 15)])
def test_schedule(count, lo, hi, methods, precision):
    ctx = Context(0)
    insts = [instance(2 ** (lo + i % (hi - lo + 1)), 5e-6 + 25e-6 * ((i * 0.618) % 1.0),
                      methods[(i // 2) % len(methods)]) for i in range(count)]
    check(ctx, insts, precision)
    ctx.close()
