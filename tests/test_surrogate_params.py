"""Parameter transfers of the surrogate: what set_params loads, get_params
returns, bit for bit, for layer-0 widths with and without padding and vectors
of less than one transfer chunk (2^18 floats), of exactly whole chunks and of
chunks with a remainder."""
import numpy as np
import pytest

from optifax_amd.surrogate import num_params


@pytest.mark.gpu
@pytest.mark.parametrize("n_in,width,n_out", [(1, 64, 64), (64, 64, 64), (101, 128, 192),
                                              (2050, 512, 256), (767, 512, 512), (2112, 1024, 64)])
def test_parameters_round_trip(n_in, width, n_out):
    from optifax_amd.surrogate import SurrogateMLP
    p = np.random.default_rng(3).standard_normal(num_params(n_in, width, n_out)).astype(np.float32)
    net = SurrogateMLP(n_in, width, n_out, max_batch=64, params=p)
    for _ in range(2):
        assert np.array_equal(net.get_params(), p)
        p = p[::-1].copy()
        net.set_params(p)
    net.close()

