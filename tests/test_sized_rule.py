"""When a launch has the general kernel with fixed grid splits: 512 threads, the
counter barrier, no RK23, and an instance whose split and columns have a form;
and FP64 fields on it, whose stages take 2 columns at a time, give the general
kernel's bits down to the fewest columns."""
import pytest

from emu_launch import kernel, last_launch
from test_sized_kernel import instance, same, trips
from test_wave_kernel import emu  # noqa: F401  (fixture)

from optifax_amd.solver import Context


@pytest.mark.parametrize("n,C,n1,block,want", [
    (4096, 4, 0, 512, "sized"), (4096, 16, 0, 512, "sized"), (8192, 8, 0, 512, "sized"),
    (2048, 4, 0, 512, "general barrier"),      # 64 x 32: no form
    (4096, 32, 0, 512, "general barrier"),     # 2 columns
    (4096, 4, 128, 512, "general barrier"),    # 128 x 32
    (4096, 4, 0, 256, "general barrier")])
def test_rule(emu, n, C, n1, block, want):  # noqa: F811
    trips(emu, [instance(n, 2e-6, C, n1)], "double", block, 1)
    assert kernel(last_launch(emu)[0]) == want


def test_rule_with_several_instances(emu):  # noqa: F811
    trips(emu, [instance(2048, 2e-6, 4), instance(4096, 2e-6, 4)], "single", 512, 1)
    assert kernel(last_launch(emu)[0]) == "sized"
    rk23 = dict(instance(2048, 2e-6, 4), method="rk23")
    trips(emu, [rk23, instance(4096, 2e-6, 4)], "single", 512, 1)
    assert kernel(last_launch(emu)[0]) == "general barrier"


@pytest.mark.gpu
@pytest.mark.parametrize("n,C", [(4096, 16), (4096, 2), (8192, 4), (32768, 64), (65536, 64)])
def test_f64_columns(n, C):
    ctx = Context(0)
    insts = [instance(n, 20e-6, C)]
    same(trips(ctx, insts, "double", 512), trips(ctx, insts, "double", 256))
    ctx.close()
