"""The FP64 forces at the ends of their range: entries whose samples stay
below the accumulator's bound of 2^30 although eight of them together do not,
connection tables whose records fit in LDS only beside fewer waves, and f' at
the angles themselves, where the factor tables do not fit in LDS or a unit
leaves their range."""
import dataclasses

import numpy as np
import pytest

from _helpers import ising, params, random_keys, rel_err
from nqhip import Context, _lib
from oracle import nqref

pytestmark = pytest.mark.gpu


def context(flat, N, nh, na, p):
    ctx = Context(0, 1)
    ctx.set_problem(flat)
    ctx.set_ndm(N, nh, na)
    ctx.set_params(p)
    ctx.set_precision(_lib.PREC_FP64, _lib.PREC_FP64)
    return ctx


def test_samples_below_the_bound_whose_sum_is_not(gpu_ok, ref):
    """2048 samples x 2 on 3 sites with a transverse field of 6e5: the bias
    entries are about |L_loc|^2 / Ns, 2^26 to 2^29 a sample and above 2^30
    over a wave's eight.  1e-10 relative, the bar of the FP64 path."""
    N, chains, length = 3, 2048, 2
    flat, tab, _ = ising(N, g=6e5)
    p = params(ref.ndm_np(N, 2, 2), seed=3, sigma=0.3)
    keys = random_keys(N, chains * length, seed=4)
    L_r, dL_r = ref.local_estimator(tab, 2, 2, p, keys)
    _, O_r = ref.logpsi_grad(N, 2, 2, p, keys)
    per_sample = np.max(np.abs(np.conj(L_r)[:, None] * dL_r), axis=1) / len(keys)
    assert 2.0 ** 27 < per_sample.max() < 2.0 ** 30
    ctx = context(flat, N, 2, 2, p)
    st, _, F, _ = ctx.grad_from_samples(keys, chains, length)
    _, F_r, _, st_r = ref.grad_step(chains, length, O_r, L_r, dL_r)
    assert rel_err(st, st_r) < 1e-10
    assert rel_err(F, F_r) < 1e-10
    ctx.close()


def test_long_records(gpu_ok):
    """The chain's table of 16 sites repeated until a configuration has 1280
    connections, with nh = 1 and na = 33 (tiles of 64 units of each kind):
    four waves' records fit beside the parameters (up to 1417 connections),
    but not beside the tiles (1156).  L_loc grows by the number of repeats and
    the force by its square."""
    N, nh, na, lo, hi = 16, 1, 33, 1157, 1417
    flat, _, _ = ising(N)
    k = hi // flat.max_connections()
    assert lo <= k * flat.max_connections() <= hi
    rep = dataclasses.replace(flat, **{f: np.tile(getattr(flat, f), k) for f in ("term_kind", "term_op_l", "term_op_r")})
    keys = random_keys(N, 40, seed=5)
    out = []
    for t in (flat, rep):
        ctx = Context(0, 1)
        ctx.set_problem(t)
        ctx.set_ndm(N, nh, na)
        ctx.set_params(params(ctx.np_, seed=6, sigma=0.1))
        ctx.set_precision(_lib.PREC_FP64, _lib.PREC_FP64)
        L = ctx.local_estimator(keys)
        _, _, F, _ = ctx.grad_from_samples(keys, 20, 2)
        out.append((L, F))
        ctx.close()
    assert rel_err(out[1][0], k * out[0][0]) < 1e-12
    assert rel_err(out[1][1], k * k * out[0][1]) < 1e-12


# 16 sites with 64 units of each kind: the tables alone take 98 KB beside an accumulator of 68; and a
# hidden bias of 320 (softplus) on a unit of small weights
@pytest.mark.parametrize("N,nh,na,sigma,bias", [(16, 64, 64, 0.03, 0.0), (3, 5, 4, 0.1, 320.0)])
def test_forces_at_the_angles(gpu_ok, ref, N, nh, na, sigma, bias):
    flat, tab, _ = ising(N)
    p = params(ref.ndm_np(N, nh, na), seed=7, sigma=sigma)
    p[nqref.ndm_layout(N, nh, na)[0]["h_la"][0] + 1] += bias
    keys = random_keys(N, 24, seed=8)
    ctx = context(flat, N, nh, na, p)
    st, _, F, _ = ctx.grad_from_samples(keys, 12, 2)
    L_r, dL_r = ref.local_estimator(tab, nh, na, p, keys)
    _, O_r = ref.logpsi_grad(N, nh, na, p, keys)
    _, F_r, _, st_r = ref.grad_step(12, 2, O_r, L_r, dL_r)
    assert rel_err(st, st_r) < 1e-10
    assert rel_err(F, F_r) < 1e-10
    ctx.close()
