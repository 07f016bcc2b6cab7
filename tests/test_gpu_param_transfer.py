"""Parameters through the pinned staging buffer: uploads in quick succession
(the second waits for the first), read back bit for bit, the FP32 copy
refreshed with them, a change of network size in between, and a host array
that is overwritten right after the call."""
import numpy as np
import pytest

from _helpers import ising, random_keys
from nqhip import Context, _lib

pytestmark = pytest.mark.gpu


def test_uploads_and_downloads(gpu_ok):
    rng = np.random.default_rng(5)
    ctx, other = Context(0, 1), Context(0, 2)
    for N, nh, na in ((1, 1, 1), (4, 7, 5), (16, 64, 64), (3, 2, 2)):
        for c in (ctx, other):
            c.set_ndm(N, nh, na)
            c.set_precision(_lib.PREC_FP32, _lib.PREC_FP32)
        keys = random_keys(N, 33, seed=N)
        for k in range(20):
            host = rng.normal(0.0, 0.1, ctx.np_)
            keep = host.copy()
            ctx.set_params(np.full(ctx.np_, 0.5))
            ctx.set_params(host)
            host[:] = np.nan            # the call has taken its copy
            if k % 5 == 0:
                other.set_params(keep)
                assert np.array_equal(other.get_params(), keep)
                assert np.array_equal(ctx.logpsi(keys), other.logpsi(keys))
            assert np.array_equal(ctx.get_params(), keep)
    ctx.close()
    other.close()
