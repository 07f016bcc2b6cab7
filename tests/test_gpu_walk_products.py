"""The FP64 walk by products of the units' factors against the oracle at the
edges of its tiles (16 units), both activations, and where the weights leave
the products' range (the sums of f): log rho, L_loc and, through the gradient,
the recorded connections.  1e-10 relative, the bar of the FP64 path."""
import numpy as np
import pytest

from _helpers import ising, params, random_keys, rel_err, xyz
from nqhip import Context, _lib
from oracle import nqref

pytestmark = pytest.mark.gpu

# (model, N, nh, na, sigma): one unit, full and ragged tiles, both unit rows (2 nh > 64), each by
# differences and by factors (sum over the units of |K w|^2 times the flipped sites above 24.5: the last
# two of the small ones for softplus, sigma 0.2 and 0.3 for logcosh), and a range beyond e^(+-600) (sigma 4 at 64 units: a site's sum over the units is about 2 x 0.8 sigma (2 nh + na))
SHAPES = [("ising", 2, 1, 1, 0.5), ("ising", 5, 15, 16, 0.3), ("ising", 5, 16, 17, 0.3), ("xyz", 4, 17, 15, 0.3),
          ("xyz", 6, 32, 33, 0.2), ("ising", 4, 33, 31, 0.2), ("xyz", 6, 64, 64, 0.1),
          ("xyz", 4, 17, 15, 0.6), ("ising", 4, 33, 31, 0.4), ("ising", 3, 64, 48, 4.0)]


# the out-of-range shape with softplus only: the oracle's log cosh drops up to 3.8e-11 per unit beyond
# |x| = 12, which at these weights is more than the bar allows in |L_loc|^2
@pytest.mark.parametrize("model,N,nh,na,sigma,act",
                         [s + (act,) for s in SHAPES for act in (0, 1) if not (act == 1 and s[4] > 1.0)])
def test_walk_matches_the_oracle(gpu_ok, model, N, nh, na, sigma, act):
    ref = nqref.Ref(act=act)
    flat, tab, _ = xyz(2, N // 2) if model == "xyz" else ising(N)
    p = params(ref.ndm_np(N, nh, na), seed=nh + 3 * na, sigma=sigma)
    ctx = Context(0, 1)
    ctx.set_problem(flat)
    ctx.set_ndm(N, nh, na, act)
    ctx.set_params(p)
    ctx.set_precision(_lib.PREC_FP64, _lib.PREC_FP64)
    chains, length = 9, 5
    keys = random_keys(N, chains * length, seed=7)
    L = ctx.local_estimator(keys)
    L_r, dL_r = ref.local_estimator(tab, nh, na, p, keys)
    assert rel_err(L, L_r) < 1e-10
    st, _, F, _ = ctx.grad_from_samples(keys, chains, length)
    _, O_r = ref.logpsi_grad(N, nh, na, p, keys)
    _, F_r, _, st_r = ref.grad_step(chains, length, O_r, L_r, dL_r)
    assert rel_err(st, st_r) < 1e-10
    # the exact force sums take addends below 2^30 a sample and read as NaN beyond (eight samples together
    # at the latest from 2^33)
    if np.max(np.abs((np.conj(L_r)[:, None] * dL_r).real)) / len(keys) > 2.0 ** 33:
        assert np.all(np.isnan(F))
    else:
        assert rel_err(F, F_r) < 1e-10
    ctx.close()


def test_route_at_the_threshold_is_one(gpu_ok):
    """A site whose sum over the units stands at the products' bound, where the
    order of the sum decides: every workgroup, and every call, takes the same
    route, so equal configurations give equal L_loc bit for bit."""
    N, nh, na = 4, 32, 32
    ref = nqref.Ref()
    p = np.zeros(ref.ndm_np(N, nh, na))
    off = nqref.ndm_layout(N, nh, na)[0]
    for block, rows in (("w_la", nh), ("w_mu", nh), ("u_la", na)):
        first, count = off[block]
        p[first:first + count].reshape(N, rows)[0] = 1.0e-14     # 2 w below half a unit in the last place of 300
    p[off["w_la"][0]] = 150.0                                     # two flips of 2 |w| reach the bound of 600
    ctx = Context(0, 1)
    ctx.set_problem(ising(N)[0])
    ctx.set_ndm(N, nh, na)
    ctx.set_params(p)
    ctx.set_precision(_lib.PREC_FP64, _lib.PREC_FP64)
    base = random_keys(N, 16, seed=8)
    first = ctx.local_estimator(base)
    for _ in range(3):
        assert np.array_equal(ctx.local_estimator(np.tile(base, 1024)), np.tile(first, 1024))
    ctx.close()


def test_visible_bias_against_a_unit(gpu_ok):
    """A visible bias of 720 on one site against a Pi unit that takes 70 of it
    back: e^650 is in range although e^720 is not.  1e-10 relative."""
    N, nh, na = 3, 2, 2
    ref = nqref.Ref()
    flat, tab, _ = ising(N)
    p = params(ref.ndm_np(N, nh, na), seed=61, sigma=0.1)
    off = nqref.ndm_layout(N, nh, na)[0]
    p[off["b_la"][0]] = 720.0
    p[off["d_la"][0]] = 70.0
    p[off["u_la"][0]] = -70.0
    ctx = Context(0, 1)
    ctx.set_problem(flat)
    ctx.set_ndm(N, nh, na)
    ctx.set_params(p)
    ctx.set_precision(_lib.PREC_FP64, _lib.PREC_FP64)
    keys = np.arange(1 << (2 * N), dtype=np.uint64)
    L = ctx.local_estimator(keys)
    L_r, _ = ref.local_estimator(tab, nh, na, p, keys)
    assert np.all(np.isfinite(L_r)) and np.max(np.abs(L_r)) > 1e270
    assert np.max(np.abs(L - L_r) / np.maximum(np.abs(L_r), 1.0)) < 1e-10
    ctx.close()
