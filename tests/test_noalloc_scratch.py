"""The no-allocation pass at the limit of the library's array: a call whose
buffers fit with the general kernel's clusters is accepted where the wave
kernel's need more.  (NSteps sizes the G table; sel beyond it leaves no step to
run.)"""
import re

import numpy as np

from emu_launch import kernel, last_launch
from noalloc_cases import OFX_E_ARG, call_noalloc, host_ptrs, raw_case

CAP = 16 << 20


def call(ctx, c, nsteps):
    c["p"].nsteps, c["p"].sel = nsteps, 4.0 * nsteps
    c["G"] = np.zeros(nsteps, np.float32)
    c["stepMods"] = np.zeros((c["batch"], 1), np.float32)
    keep = []
    c["ApFT"] = c["ApFT"][:, :0]
    ptrs = host_ptrs(keep)
    rc = ctx.lib.ofx_crystal_pass_noalloc(
        ctx.h, c["p"], c["batch"], ptrs("Et", c["Et"])[0], ptrs("alpha", c["alpha"])[0],
        ptrs("G", c["G"])[0], 1, ptrs("beta", c["beta"])[0], None, None, None)
    return rc, ctx.lib.ofx_last_error(ctx.h)


def test_limit(emu_ctx):
    """One instance of 2^11: up to 2070176 steps fit on the general kernel's 8
    workgroups, 2069152 on the wave kernel's 16."""
    c = raw_case(2048, 1, False)
    c["p"].n_cols = 0
    rc, err = call(emu_ctx, c, 3_000_000)
    assert rc == OFX_E_ARG
    need = int(re.search(rb"needs (\d+) bytes", err).group(1))
    fits = 3_000_000 - (need - CAP) // 8
    assert fits > 2_070_000
    assert call(emu_ctx, c, fits - 64)[0] == 0
    assert kernel(last_launch(emu_ctx)[0]) == "general barrier"
    assert call(emu_ctx, c, fits + 64)[0] == OFX_E_ARG
    assert call(emu_ctx, c, fits - 2048)[0] == 0
    assert kernel(last_launch(emu_ctx)[0]) == "wave"
