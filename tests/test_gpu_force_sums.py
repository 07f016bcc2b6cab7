"""The FP64 forces' exact sums and records at the ends of their range:
entries whose samples stay below the accumulator's bound of 2^30 although
eight of them together do not, and connection tables whose records fit in LDS
only beside fewer waves."""
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
