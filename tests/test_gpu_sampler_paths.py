"""The sampler's dispatch: chains by products of the units' factors, one to
four units per lane, copies of a lane group for few chains, and the chains by
sums of f that take over where the weights leave the products' range; every
route against the oracle's trajectories, drawn from the same streams, bit for
bit."""
import numpy as np
import pytest

from _helpers import ising, params
from nqhip import Context, _lib
from oracle import nqref

pytestmark = pytest.mark.gpu

# (N, nh, na, sigma, chains): lane groups of 8, 16, 32 and 64 with full and ragged units; few chains
# (copies of a group), more than one wave per SIMD (two and four units per lane); and weights whose
# products leave e^(+-600) (sigma 3 at nh = 64: the range is about 0.5 (N + 1) 0.8 sigma nh)
SHAPES = [(3, 1, 1, 0.5, 2), (4, 8, 5, 0.5, 37), (4, 9, 3, 0.5, 40), (5, 16, 17, 0.4, 33), (3, 33, 20, 0.3, 21),
          (4, 64, 64, 0.2, 9), (3, 18, 32, 0.3, 2060), (3, 32, 18, 0.3, 4100), (3, 40, 12, 0.3, 2060),
          (4, 64, 64, 3.0, 9), (3, 18, 32, 6.0, 2060)]


@pytest.mark.parametrize("act", [0, 1])
@pytest.mark.parametrize("N,nh,na,sigma,chains", SHAPES)
def test_fp64_chains_follow_the_oracle(gpu_ok, act, N, nh, na, sigma, chains):
    ref = nqref.Ref(act=act)
    flat, _, _ = ising(N)
    p = params(ref.ndm_np(N, nh, na), seed=17 * nh + na, sigma=sigma)
    ctx = Context(0, 991)
    ctx.set_problem(flat)
    ctx.set_ndm(N, nh, na, act)
    ctx.set_params(p)
    ctx.set_precision(_lib.PREC_FP64, _lib.PREC_FP64)
    length, passes, burn = (2, 5, 1) if chains > 1000 else (4, 37, 3)
    ctx.set_sampler(chains, length, passes, burn)
    ctx.set_iteration(5)
    keys, acc = ctx.sample()
    keys_r, acc_r = ref.metropolis(N, nh, na, p, chains, length, passes, burn, 991, it=5)
    assert np.array_equal(keys, keys_r)
    assert acc == acc_r
    ctx.close()
