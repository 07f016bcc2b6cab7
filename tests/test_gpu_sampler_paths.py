"""The sampler's dispatch: chains by products of the units' factors, one to
four units per lane, copies of a lane group for few chains, and the chains by
sums of f that take over where the weights leave the products' range; every
route against the oracle's trajectories, drawn from the same streams, bit for
bit."""
import numpy as np
import pytest

from _helpers import ising, params
from nqhip import Context, _lib, hilbert, operators
from oracle import nqref, obs_ref

pytestmark = pytest.mark.gpu

# (N, nh, na, sigma, chains): lane groups of 8, 16, 32 and 64 with full and ragged units; few chains
# (copies of a group), more than one wave per SIMD (two and four units per lane); and weights whose
# products leave e^(+-600) (sigma 3 at nh = 64: the range is about 0.5 (N + 1) 0.8 sigma nh)
SHAPES = [(3, 1, 1, 0.5, 2), (4, 8, 5, 0.5, 37), (4, 9, 3, 0.5, 40), (5, 16, 17, 0.4, 33), (3, 33, 20, 0.3, 21),
          (4, 64, 64, 0.2, 9), (3, 18, 32, 0.3, 2060), (3, 32, 18, 0.3, 4100), (3, 40, 12, 0.3, 2060),
          (4, 64, 64, 3.0, 9), (3, 18, 32, 6.0, 2060), (6, 6, 6, 20.0, 16)]


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


# one unit (a pair for logcosh) beyond what its kept factor or its table entries hold in FP64, every other weight small:
# K m = 520 over all sites (the factor of the far side would be e^(-1.5 K m) = 0), and a single weight of
# 360 / K (a table entry e^(+-2 K w) beyond e^709); K = 2 for logcosh
def outlier(ref, N, nh, na, act, block, kind):
    p = params(ref.ndm_np(N, nh, na), seed=41, sigma=0.2)
    K = 2.0 if act else 1.0
    first, count = nqref.ndm_layout(N, nh, na)[0][block]
    rows = nh if block == "w_la" else na
    w = p[first:first + count].reshape(N, rows)          # column-major [unit, site]
    w[:, 0] = 520.0 / (K * N) if kind == "factor" else 0.0
    if kind == "table":
        w[0, 0] = 360.0 / K
    if act:         # the units' linear parts, which join the visible biases, cancel in another unit
        first, count = nqref.ndm_layout(N, nh, na)[0]["w_la"]
        p[first:first + count].reshape(N, nh)[:, 1] = -w[:, 0]
    return p


@pytest.mark.parametrize("act", [0, 1])
@pytest.mark.parametrize("block", ["w_la", "u_la"])
@pytest.mark.parametrize("kind", ["factor", "table"])
def test_one_unit_out_of_range(gpu_ok, act, block, kind):
    ref = nqref.Ref(act=act)
    N, nh, na, chains, length, passes, burn = 4, 3, 2, 21, 4, 9, 2
    p = outlier(ref, N, nh, na, act, block, kind)
    ctx = Context(0, 77)
    ctx.set_problem(ising(N)[0])
    ctx.set_ndm(N, nh, na, act)
    ctx.set_params(p)
    ctx.set_precision(_lib.PREC_FP64, _lib.PREC_FP64)
    ctx.set_sampler(chains, length, passes, burn)
    ctx.set_iteration(3)
    keys, acc = ctx.sample()
    keys_r, acc_r = ref.metropolis(N, nh, na, p, chains, length, passes, burn, 77, it=3)
    assert np.array_equal(keys, keys_r)
    assert acc == acc_r
    h = hilbert.HomogeneousSpin(N)
    ctx.set_iteration(0)
    ctx.observable(operators.flatten(1.0 * operators.sigmaz(h, 1)), 9, 3, passes, burn)
    keys, _ = ctx.observable_samples()
    keys_r, _ = obs_ref.diag_metropolis(lambda k: ref.logpsi(N, nh, na, p, k), N, 9, 3, passes, burn, seed=77, it=0,
                                        philox=ref.philox)
    assert np.array_equal(keys, keys_r)
    ctx.close()
