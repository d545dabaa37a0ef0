"""Several host threads read one surrogate handle at once: every result is the
one that a single thread gets, bit for bit.  Vectors of more transfer chunks
than pinned buffers, first use (which makes the buffers) among them."""
import threading

import numpy as np
import pytest

from optifax_amd.surrogate import SurrogateMLP, num_params


def together(*calls):
    """The calls' results, each from a thread of its own, all started at once."""
    gate, out = threading.Barrier(len(calls)), [None] * len(calls)

    def body(i):
        gate.wait()
        out[i] = calls[i]()

    threads = [threading.Thread(target=body, args=(i,)) for i in range(len(calls))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    return out


@pytest.mark.gpu
def test_threads_read_one_handle():
    dims = (767, 1024, 512)                       # 17.7 MB: 17 chunks of 1 MB
    rng = np.random.default_rng(5)
    p = rng.standard_normal(num_params(*dims)).astype(np.float32) * np.float32(0.02)
    x = rng.standard_normal((64, dims[0])).astype(np.float32)
    t = rng.standard_normal((64, dims[2])).astype(np.float32)
    alone = SurrogateMLP(*dims, max_batch=64, params=p)
    loss, grads = alone.gradients(x, t)
    alone.close()
    net = SurrogateMLP(*dims, max_batch=64, params=p)
    for _ in range(4):
        for q in together(*[net.get_params] * 4):
            assert np.array_equal(q, p)
        q, (got_loss, got), r = together(net.get_params, lambda: net.gradients(x, t),
                                         net.get_params)
        assert np.array_equal(q, p) and np.array_equal(r, p)
        assert got_loss == loss and np.array_equal(got, grads)
    net.close()
