"""The complex RBMs' FP64 sampler: chains by products of the units' factors
(groups of 8, 16, 32 and 64 lanes, one to four units per lane, few chains with
copies of a group, many chains) and, where the weights leave their range, by
sums of f, against the oracle's trajectories bit for bit."""
import numpy as np
import pytest

from _helpers import ising
from nqhip import Context, _lib, hilbert, operators, problems
from oracle import obs_ref, rbm_ref

pytestmark = pytest.mark.gpu

# sigma 2 at 70 units leaves the range (sum over the units of (2 N + 1) 0.8 sigma + 1.4 > 600)
SHAPES = [(2, 1, 0.3, 3), (3, 9, 0.3, 5), (2, 17, 0.3, 4), (2, 33, 0.2, 4), (2, 70, 0.1, 3), (2, 128, 0.05, 2),
          (2, 18, 0.3, 2060), (2, 70, 2.0, 3),
          # four units per lane, full and ragged (groups of 8, 16 and 32), and the largest tables (132 KB of LDS)
          (2, 32, 0.2, 4100), (2, 40, 0.2, 2060), (2, 70, 0.1, 1100), (16, 128, 0.02, 3)]


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


# one unit alone beyond what its kept factor or its table entries hold in FP64: Re W = 520 over all
# sites, or 360 on one (e^720) with a bias that keeps the angle itself within e^(+-709)
@pytest.mark.parametrize("ket", [False, True])
@pytest.mark.parametrize("kind", ["factor", "table"])
def test_one_unit_out_of_range(gpu_ok, ref, ket, kind):
    N, nh, chains, length, passes, burn = 3, 5, 13, 3, 9, 2
    rng = np.random.default_rng(43)
    n = rbm_ref.ket_n_params(N, nh) if ket else rbm_ref.n_params(N, nh)
    p = 0.2 * (rng.standard_normal(n) + 1j * rng.standard_normal(n))
    sites = N if ket else 2 * N
    w = p[sites + nh:].reshape(sites, nh)
    w[:, 1] = 520.0 / sites if kind == "factor" else 0.0
    if kind == "table":
        w[0, 1], p[sites + 1] = 360.0, -200.0
    ctx = Context(0, 29)
    if ket:
        ctx.set_problem(operators.flatten(problems.ising_hamiltonian(N, 1.0, 2.0)[1]))
        ctx.set_rbm(N, nh)
    else:
        ctx.set_problem(ising(N)[0])
        ctx.set_rbmsplit(N, nh)
    ctx.set_precision(_lib.PREC_FP64, _lib.PREC_FP64)
    ctx.set_params(p.view(np.float64))
    ctx.set_sampler(chains, length, passes, burn)
    ctx.set_iteration(4)
    keys, acc = ctx.sample()
    if ket:
        keys_r, acc_r = rbm_ref.ket_metropolis(p, N, nh, chains, length, passes, burn, 29, 4, ref.philox)
    else:
        keys_r, _, acc_r = rbm_ref.metropolis(p, N, nh, chains, length, passes, burn, 29, 4, ref.philox)
    assert np.array_equal(keys, keys_r)
    assert acc == acc_r
    if not ket:
        ctx.set_iteration(0)
        h = hilbert.HomogeneousSpin(N)
        ctx.observable(operators.flatten(1.0 * operators.sigmaz(h, 1)), 7, 3, passes, burn)
        keys, _ = ctx.observable_samples()
        keys_r, _ = obs_ref.diag_metropolis(lambda k: rbm_ref.logpsi(p, k, N, nh), N, 7, 3, passes, burn, seed=29, it=0,
                                            philox=ref.philox)
        assert np.array_equal(keys, keys_r)
    ctx.close()
