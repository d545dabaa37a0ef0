"""The general kernel's tagged exchange, which runs where the wave kernel cannot:
RK23 beside Heun, workgroup sizes that are no power of two, more than 4 points a
thread, transforms of more than 256.  Against its counter barrier: the same
bits."""
import numpy as np
import pytest

from emu_launch import kernel, last_launch
from test_uneven_schedule import KEYS, instance, read
from test_wave_kernel import emu  # noqa: F401  (fixture)

from optifax_amd.solver import Context, OPOBatch


def trips(ctx, insts, precision, tune):
    run = OPOBatch(insts, precision=precision, trip_cap=4, ctx=ctx, tune=tune)
    lds = run.geometry(0)["lds_bytes"]
    run.launch(2)
    run.sync()
    out = [read(run, i) for i in range(len(insts))]
    run.close()
    return out, lds


def same_as_barrier(ctx, insts, precision, tune):
    tags, lds = trips(ctx, insts, precision, dict(tune, exchange="tags"))
    mode = last_launch(ctx)[0] if hasattr(ctx.lib, "ofx_emu_last_launch") else None
    barrier, other = trips(ctx, insts, precision, dict(tune, exchange="barrier"))
    assert lds == other                      # the general kernel's workspace both times
    for x, y in zip(tags, barrier):
        assert (x["attempts"], x["status"]) == (y["attempts"], y["status"])
        for k in KEYS:
            assert np.array_equal(x[k], y[k]), k
    return mode


ONE = [("general tags", "heun", 512, dict(cluster=4, block=192)),
       ("general tags", "heun", 2048, dict(cluster=4, block=64)),       # 8 points a thread
       ("general tags", "heun", 2048, dict(cluster=4, n1=512)),
       ("rk23 tags", "rk23", 512, dict(cluster=4, block=192)),
       ("rk23 tags", "rk23", 2048, dict(cluster=4, block=64)),
       ("rk23 tags", "rk23", 2048, dict(cluster=4, n1=512))]


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("name,method,n,tune", ONE)
def test_emulated_tags(emu, name, method, n, tune, precision):  # noqa: F811
    mode = same_as_barrier(emu, [instance(n, 6e-6, method)], precision, tune)
    assert kernel(mode) == name


@pytest.mark.parametrize("precision", ["single", "double"])
def test_emulated_rk23_beside_heun(emu, precision):  # noqa: F811
    insts = [instance(512, 6e-6, "heun"), instance(1024, 6e-6, "rk23"),
             instance(512, 8e-6, "rk23")]
    assert kernel(same_as_barrier(emu, insts, precision, dict(cluster=4))) == "general tags"


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("method,n,tune", [c[1:] for c in ONE] + [
    ("heun", 16384, dict(cluster=16, block=192)), ("rk23", 16384, dict(cluster=32, block=192)),
    ("heun", 8192, dict(cluster=16, n1=512)), ("rk23", 8192, dict(cluster=8, block=64))])
def test_tags(method, n, tune, precision):
    ctx = Context(0)
    same_as_barrier(ctx, [instance(n, 20e-6, method)], precision, tune)
    ctx.close()


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["single", "double"])
def test_rk23_beside_heun(precision):
    """Both on 64 workgroups or more: tags by default, too."""
    ctx = Context(0)
    insts = [instance(65536, 6e-6, "heun"),
             instance(32768, 6e-6, "rk23")]
    same_as_barrier(ctx, insts, precision, dict(cluster=64))
    run = OPOBatch(insts, precision=precision, ctx=ctx)
    assert min(run.geometry(i)["cluster"] for i in range(2)) >= 64
    run.close()
    default, _ = trips(ctx, insts, precision, None)
    barrier, _ = trips(ctx, insts, precision, dict(exchange="barrier"))
    for x, y in zip(default, barrier):
        for k in KEYS:
            assert np.array_equal(x[k], y[k]), k
    ctx.close()
