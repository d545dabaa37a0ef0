"""Cluster sizes follow the kernel that runs.  A launch that the wave kernel
cannot take (RK23 beside Heun, a workgroup size that is no power of two, a grid
that it does not fit) has the general kernel's cluster sizes, which the counter
barrier's launches always have."""
import os

import pytest

from cases import opo_case
from optifax_amd.solver import Context, OPOBatch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def ctx256():
    path = os.path.join(ROOT, "tests", "emu", "libofx_emu.so")
    if not os.path.exists(path):
        pytest.skip("emulation library not built")
    old = os.environ.get("OFX_EMU_CUS")
    os.environ["OFX_EMU_CUS"] = "256"
    ctx = Context(0, lib_path=path)
    if old is None:
        del os.environ["OFX_EMU_CUS"]
    else:
        os.environ["OFX_EMU_CUS"] = old
    yield ctx
    ctx.close()


def clusters(ctx, grids, precision="single", tune=None):
    insts = []
    for n, method in grids:
        _, b = opo_case(n=n, window=3e-12 * (n / 512) ** 0.5, length=6e-6)
        insts.append(dict(solver=b["solver"], field0=b["ops"]["field0"], method=method))
    run = OPOBatch(insts, precision=precision, ctx=ctx, tune=tune)
    out = [run.geometry(i)["cluster"] for i in range(len(insts))], run.geometry(0)["lds_bytes"]
    run.close()
    return out


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("n", [512, 1024, 4096])
@pytest.mark.parametrize("pairs", [1, 4])
def test_heun_beside_rk23(ctx256, n, pairs, precision):
    grids = [(n, "heun"), (n, "rk23")] * pairs
    assert clusters(ctx256, grids, precision) == \
        clusters(ctx256, grids, precision, dict(exchange="barrier"))


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("method", ["heun", "rk23"])
@pytest.mark.parametrize("n", [512, 1024, 4096])
def test_odd_workgroup_size(ctx256, n, method, precision):
    assert clusters(ctx256, [(n, method)], precision, dict(block=192)) == \
        clusters(ctx256, [(n, method)], precision, dict(block=192, exchange="barrier"))


@pytest.mark.parametrize("method", ["heun", "rk23"])
@pytest.mark.parametrize("n", [4096, 8192, 32768])
def test_f64_workgroups_of_512_threads(ctx256, n, method):
    """FP64 fields in clusters of 512-thread workgroups: the general kernel (its
    workspace and clusters), also with the tagged exchange unless the caller
    gives the threads too."""
    general = clusters(ctx256, [(n, method)], "double", dict(block=512, exchange="barrier"))
    assert clusters(ctx256, [(n, method)], "double", dict(block=512)) == general
    assert clusters(ctx256, [(n, method)], "double",
                    dict(block=512, cluster=general[0][0])) == general
    both = dict(block=512, exchange="tags", cluster=general[0][0])
    assert clusters(ctx256, [(n, method)], "double", both)[1] != general[1]


def test_f64_large_shares_with_tags(ctx256):
    """Shares above the wave kernel's default: the tagged exchange alone brings
    the general kernel (FP64, 512 threads)."""
    many = [(32768, "heun")] * 16
    assert clusters(ctx256, many, "double", dict(exchange="tags")) == \
        clusters(ctx256, many, "double", dict(exchange="barrier"))


def test_f64_one_workgroup_of_512_threads(ctx256):
    """One workgroup without an exchange keeps the wave kernel."""
    got = clusters(ctx256, [(512, "heun")], "double", dict(block=512))
    general = clusters(ctx256, [(512, "heun")], "double",
                       dict(block=512, cluster=1, exchange="barrier"))
    assert got[0] == [1] and got[1] != general[1]


def test_f64_batch_of_16384_points(ctx256):
    """40 FP64 instances of 2^14: a step of the wave kernel at 1024 points a
    workgroup takes 22 us there, so three rounds of it (66) are no gain over two of
    the general kernel (60)."""
    many = [(16384, "heun")] * 40
    got, lds = clusters(ctx256, many, "double")
    assert got == [8] * 40 and lds == clusters(ctx256, many, "double", dict(exchange="barrier"))[1]


@pytest.mark.parametrize("block", [64, 128, 192, 512])
def test_given_threads_with_clusters_of_the_wave_kernel(ctx256, block):
    """Shares that fit LDS in the wave kernel only: with threads that it does not
    take, the general kernel has larger clusters of its own."""
    many = [(16384, "rk23")] * 10
    got, _ = clusters(ctx256, many, "double", dict(block=block))
    assert got == clusters(ctx256, many, "double", dict(block=block, exchange="barrier"))[0]


def test_f64_threads_that_only_the_wave_kernel_fits():
    """512 threads given: where the general kernel's clusters do not fit the
    device (a part of 32 CUs), the wave kernel runs."""
    path = os.path.join(ROOT, "tests", "emu", "libofx_emu.so")
    if not os.path.exists(path):
        pytest.skip("emulation library not built")
    os.environ["OFX_EMU_CUS"] = "32"
    try:
        ctx = Context(0, lib_path=path)
    finally:
        del os.environ["OFX_EMU_CUS"]
    got = clusters(ctx, [(16384, "rk23"), (2048, "rk23")], "double", dict(block=512))
    ctx.close()
    assert sum(got[0]) <= 32
