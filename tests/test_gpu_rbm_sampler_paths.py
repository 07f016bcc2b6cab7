"""The complex RBMs' FP64 sampler: chains by products of the units' factors
(groups of 8, 16, 32 and 64 lanes, one and two units per lane, few chains with
copies of a group, many chains) and, where the weights leave their range, by
sums of f, against the oracle's trajectories bit for bit."""
import numpy as np
import pytest

from _helpers import ising
from nqhip import Context, _lib, operators, problems
from oracle import nqref, rbm_ref

pytestmark = pytest.mark.gpu

# sigma 2 at 70 units leaves the range (sum over the units of (2 N + 1) 0.8 sigma + 1.4 > 600)
SHAPES = [(2, 1, 0.3, 3), (3, 9, 0.3, 5), (2, 17, 0.3, 4), (2, 33, 0.2, 4), (2, 70, 0.1, 3), (2, 128, 0.05, 2),
          (2, 18, 0.3, 2060), (2, 70, 2.0, 3)]


@pytest.mark.parametrize("ket", [False, True])
@pytest.mark.parametrize("N,nh,sigma,chains", SHAPES)
def test_chains_follow_the_oracle(gpu_ok, ref, ket, N, nh, sigma, chains):
    rng = np.random.default_rng(nh)
    n = rbm_ref.ket_n_params(N, nh) if ket else rbm_ref.n_params(N, nh)
    p = sigma * (rng.standard_normal(n) + 1j * rng.standard_normal(n)) / np.sqrt(2)
    ctx = Context(0, 23)
    if ket:
        ctx.set_problem(operators.flatten(problems.ising_hamiltonian(N, 1.0, 2.0)[1]))
        ctx.set_rbm(N, nh)
    else:
        ctx.set_problem(ising(N)[0])
        ctx.set_rbmsplit(N, nh)
    ctx.set_precision(_lib.PREC_FP64, _lib.PREC_FP64)
    ctx.set_params(p.view(np.float64))
    length, passes, burn = (2, 3, 0) if chains > 1000 else (2, 35, 1)
    ctx.set_sampler(chains, length, passes, burn)
    ctx.set_iteration(2)
    keys, acc = ctx.sample()
    if ket:
        keys_r, acc_r = rbm_ref.ket_metropolis(p, N, nh, chains, length, passes, burn, 23, 2, ref.philox)
    else:
        keys_r, _, acc_r = rbm_ref.metropolis(p, N, nh, chains, length, passes, burn, 23, 2, ref.philox)
    assert np.array_equal(keys, keys_r)
    assert acc == acc_r
    ctx.close()
