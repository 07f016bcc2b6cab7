"""What a user of nqhip has it do: the workloads whose time is watched.

The library runs variational Monte Carlo loops, so most cases are one SR
iteration at the parameters that the program holds: they are uploaded, the
iteration samples, estimates, solves and steps, and the stepped parameters
are read back (what a driver does that keeps the canonical copy of its
network, as the VMC API of the package does).  Beside them stand the calls
that are made between iterations: observables and exact sums.

    kind "step"     Context.set_params, sr_iteration, get_params; one hipGraph
                    replay per iteration (with a matrix-free solver: eager)
    kind "loop"     the VMC API as the reference's example writes it: sample_,
                    compute_observables, precondition_, update_
    kind "batch"    "step" for many problems of uneven size in one Batch
    kind "observe"  compute_observables on a density matrix
    kind "exact"    Context.exact over every doubled configuration

Models: "ising" (dissipative Ising chain), "xyz" (dissipative XYZ on a square
lattice of lx x ly sites) and "tfim" (the closed Ising chain, on kets).
Precision: the pairs of the VMC API, "fp64", "fp32" (FP32 network and S
build) and "mixed" (FP32 network, BF16 S build).  What a network evaluated in
32 bits gives leaves `run` as 32-bit numbers: the width of its computation,
not of the doubles that carry it over the C ABI.

`exact` restates all of it in 64 bits with plain torch: the Philox streams of
the sampler, the networks, the local estimators and the SR solve.
"""
from __future__ import annotations

import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "neuralquantum.jl_amd"))

from nqhip import (  # noqa: E402
    NDM, SR, Batch, BatchedSampler, Context, Descent, LocalRule, MetropolisSampler, RBMSplit, _lib,
    add_observable_, compute_observables, hilbert, operators, precondition_, problems, sample_, update_)

PREC = {"fp64": (_lib.PREC_FP64, _lib.PREC_FP64), "fp32": (_lib.PREC_FP32, _lib.PREC_FP32),
        "mixed": (_lib.PREC_FP32, _lib.PREC_BF16)}
SOLVERS = {"cholesky": _lib.SOLVER_CHOLESKY, "cg": _lib.SOLVER_CG}
ACTS = {"softplus": _lib.ACT_SOFTPLUS, "logcosh": _lib.ACT_LOGCOSH}
CG_TOL = 1e-4


# ---------------------------------------------------------------- the cases
def _case(kind, **kw):
    c = dict(kind=kind, model="ising", lx=6, ly=1, periodic=True, g=1.0, net="ndm", act="softplus", alpha_h=1,
             alpha_a=1, sigma=0.01, precision="fp64", chains=256, length=8, passes=13, burn=50, persistent=False,
             solver="cholesky", eps=0.01, lr=0.01, instances=1)
    c.update(kw)
    return c


def listed():
    return [
        # the smallest system anyone runs, through the VMC API in its default precision: a chain of
        # six sites, few long chains, observables every iteration (the reference's example loop)
        _case("loop", name="ising6_loop", lx=6, periodic=False, chains=16, length=125, passes=13, burn=100,
              sigma=0.1),
        # the working size on one chain, 32-bit throughout, chains kept between iterations
        _case("step", name="ising12_fp32", lx=12, alpha_h=2, alpha_a=2, chains=1024, length=16, passes=25,
              precision="fp32", persistent=True),
        # the same system in 64 bits on the reference's schedule (restart and burn in every iteration)
        _case("step", name="ising12_fp64", lx=12, alpha_h=2, alpha_a=2, chains=1024, length=16, passes=25,
              sigma=0.05),
        # the two forms of the headline workload, the 4x4 XYZ lattice: plain 64 bits ...
        _case("step", name="xyz44_fp64", model="xyz", lx=4, ly=4, alpha_h=2, alpha_a=2, chains=4096, length=4,
              passes=33, lr=0.005),
        # ... and FP32 network with BF16 S build and persistent chains
        _case("step", name="xyz44_mixed", model="xyz", lx=4, ly=4, alpha_h=2, alpha_a=2, chains=4096, length=4,
              passes=33, lr=0.005, precision="mixed", persistent=True),
        # sizes that fill no tile: nine sites, nh = 27, na = 9, the other activation, 1000 x 5 samples
        _case("step", name="xyz33_ragged_mixed", model="xyz", lx=3, ly=3, act="logcosh", alpha_h=3, alpha_a=1,
              chains=1000, length=5, passes=19, sigma=0.05, precision="mixed", persistent=True),
        # a parameter sweep: 64 chains of 6 to 16 sites, one packed launch per kernel
        _case("batch", name="ising64_batch", instances=64, chains=256, length=8, passes=0, precision="mixed",
              persistent=True),
        # SR without forming S: conjugate gradients on the O rows of the headline system
        _case("step", name="xyz44_cg", model="xyz", lx=4, ly=4, alpha_h=2, alpha_a=2, chains=4096, length=4,
              passes=33, lr=0.005, solver="cg", persistent=True),
        # the other density matrix, complex parameters and a complex SR system
        _case("step", name="rbmsplit8", net="rbmsplit", lx=8, alpha_h=2, alpha_a=0, chains=256, length=16,
              passes=17, sigma=0.1),
        # a ground state: the ket RBM on the closed chain
        _case("step", name="rbm16_energy", model="tfim", net="rbm", lx=16, alpha_h=2, alpha_a=0, chains=1024,
              length=8, passes=17, sigma=0.1, persistent=True),
        # three observables of a 12-site density matrix
        _case("observe", name="ising12_observe", lx=12, alpha_h=2, alpha_a=2, chains=1024, length=16, passes=25,
              sigma=0.05),
        # the loss of a network without sampling noise, over all 2^20 doubled configurations
        _case("exact", name="ising10_exact", lx=10, sigma=0.05),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["step"] * 8 + ["loop", "batch", "observe", "exact"])
    sigma = rng.choice([0.01, 0.05, 0.1])
    if kind == "exact":
        return _case(kind, lx=rng.randint(5, 9), alpha_h=rng.randint(1, 2), alpha_a=rng.randint(1, 2),
                     precision=rng.choice(["fp64", "fp32"]), sigma=sigma, g=round(rng.uniform(0.5, 2.0), 3))
    if kind == "batch":
        return _case(kind, instances=_log_int(rng, 4, 48), chains=_log_int(rng, 32, 256), length=rng.randint(4, 8),
                     passes=0, precision="mixed", persistent=True, sigma=sigma)
    net = rng.choice(["ndm"] * 6 + ["rbmsplit", "rbm"]) if kind == "step" else "ndm"
    model, lx, ly = "ising", rng.randint(4, 16), 1
    if net == "rbm":
        model = "tfim"
    elif net == "rbmsplit":
        lx = rng.randint(4, 9)
    elif kind == "step" and rng.random() < 0.4:
        model, (lx, ly) = "xyz", rng.choice([(2, 3), (3, 3), (3, 4), (2, 5), (4, 4)])
    n = lx * ly
    alpha = [a for a in (1, 2, 3) if a * n <= 32]
    length = _log_int(rng, 2, 64)
    precision = "fp64" if net != "ndm" else rng.choice(["fp64", "fp32", "mixed"])
    return _case(kind, model=model, lx=lx, ly=ly, net=net, act=rng.choice(["softplus", "softplus", "logcosh"])
                 if net == "ndm" else "softplus", alpha_h=rng.choice(alpha),
                 alpha_a=rng.choice(alpha) if net == "ndm" else 0, sigma=sigma, g=round(rng.uniform(0.5, 2.0), 3),
                 precision=precision, chains=_log_int(rng, 16, max(16, 12000 // length)), length=length,
                 passes=2 * n + 1, burn=rng.randint(10, 50), persistent=kind == "step" and rng.random() < 0.5,
                 solver="cg" if net == "ndm" and kind == "step" and rng.random() < 0.15 else "cholesky")


# ---------------------------------------------------------------- what a program has in hand
@functools.lru_cache(maxsize=None)
def _problem(model, lx, ly, periodic, g):
    """(operator of the loop, its flat table)"""
    if model == "xyz":
        op = problems.dissipative_xyz(lx, ly, Jx=0.9, Jy=1.0, Jz=1.1, gamma=1.0, periodic=periodic)[3]
    elif model == "tfim":
        op = problems.ising_hamiltonian(lx, g, 2.0, periodic)[1]
    else:
        op = problems.dissipative_ising_chain(lx, V=2.0, g=g, gamma=1.0, periodic=periodic)[3]
    return op, operators.flatten(op)


@functools.lru_cache(maxsize=None)
def _magnetisations(n):
    """The observables of the reference's example: Sx, Sy, Sz per site."""
    h, out = hilbert.HomogeneousSpin(n), {}
    for name, site in (("Sx", operators.sigmax), ("Sy", operators.sigmay), ("Sz", operators.sigmaz)):
        op = operators.LocalOperator(h)
        for i in range(1, n + 1):
            op = op + (1.0 / n) * site(h, i)
        out[name] = op
    return out


def _sites(case):
    return case["lx"] * case["ly"]


def _members(case):
    """A batch's problems: N ~ U{6..16}, g ~ U[0.5, 2] as its own cases of one instance."""
    rng = np.random.default_rng(2024)
    ns, gs = rng.integers(6, 17, size=case["instances"]), rng.uniform(0.5, 2.0, size=case["instances"])
    return [dict(case, kind="step", lx=int(n), g=round(float(g), 3), passes=2 * int(n) + 1, instances=1)
            for n, g in zip(ns, gs)]


def _seeds(seed, i=0):
    """(parameter seed, sampler seed) of member i"""
    return 100003 * int(seed) + 2 * i + 1, (7919 * int(seed) + 104729 * i + 4321) & 0x7fffffff


def _params(case, seed):
    """The flat parameter vector: normal with standard deviation sigma (complex ones per component)."""
    n, nh = _sites(case), int(case["alpha_h"] * _sites(case))
    na = int(case["alpha_a"] * n)
    count = {"ndm": 2 * n + 2 * nh + na + 2 * nh * n + 2 * na * n, "rbmsplit": 2 * (2 * n + nh + 2 * nh * n),
             "rbm": 2 * (n + nh + nh * n)}[case["net"]]
    return np.random.default_rng(seed).standard_normal(count) * case["sigma"]


def _narrow(case, a):
    a = np.asarray(a, dtype=np.float64)
    return a if case["precision"] == "fp64" else a.astype(np.float32)


def _context(case, pseed, sseed):
    n = _sites(case)
    ctx = Context(0, sseed)
    ctx.set_problem(_problem(case["model"], case["lx"], case["ly"], case["periodic"], case["g"])[1])
    nh = int(case["alpha_h"] * n)
    if case["net"] == "rbm":
        ctx.set_rbm(n, nh)
    elif case["net"] == "rbmsplit":
        ctx.set_rbmsplit(n, nh)
    else:
        ctx.set_ndm(n, nh, int(case["alpha_a"] * n), ACTS[case["act"]])
    ctx.set_precision(*PREC[case["precision"]])
    p = _params(case, pseed)
    ctx.set_params(p)
    if case["kind"] == "step":
        ctx.set_sampler(case["chains"], case["length"], case["passes"], case["burn"],
                        _lib.SAMPLER_PERSISTENT if case["persistent"] else 0)
        ctx.set_sr_solver(SOLVERS[case["solver"]], CG_TOL, 0)
        ctx.set_graph(case["solver"] == "cholesky")
        if case["persistent"]:
            ctx.sample()          # the chains of a running loop are thermalised
    return ctx, p


def prepare(case, seed):
    state = {"case": case}
    if case["kind"] == "batch":
        made = [_context(m, *_seeds(seed, i)) for i, m in enumerate(_members(case))]
        state["members"], state["p"] = [c for c, _ in made], [p for _, p in made]
        state["batch"] = Batch(state["members"])
        return state
    pseed, sseed = _seeds(seed)
    if case["kind"] in ("loop", "observe"):
        n = _sites(case)
        net = NDM(n, case["alpha_h"], case["alpha_a"], act=case["act"]) if case["net"] == "ndm" \
            else RBMSplit(n, case["alpha_h"])
        net.flat[:] = _params(case, pseed)
        algo = SR(case["eps"])
        is_ = BatchedSampler(net, MetropolisSampler(LocalRule(), case["length"], case["passes"] | 1,
                                                    burn=case["burn"], seed=sseed),
                             _problem(case["model"], case["lx"], case["ly"], case["periodic"], case["g"])[0], algo,
                             batch_sz=case["chains"], precision=case["precision"])
        for name, op in _magnetisations(n).items():
            add_observable_(is_, name, op)
        state.update(net=net, p=net.flat.copy(), algo=algo, sampler=is_, opt=Descent(case["lr"]))
        return state
    state["ctx"], state["p"] = _context(case, pseed, sseed)
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "step":
        ctx = state["ctx"]
        ctx.set_params(state["p"])
        st = ctx.sr_iteration(case["eps"], case["lr"])
        return {"stats": _narrow(case, st), "params": _narrow(case, ctx.get_params())}
    if kind == "batch":
        for ctx, p in zip(state["members"], state["p"]):
            ctx.set_params(p)
        st = state["batch"].sr_iteration(case["eps"], case["lr"])
        return {"stats": _narrow(case, st),
                "params": _narrow(case, np.concatenate([ctx.get_params() for ctx in state["members"]]))}
    if kind == "exact":
        loss, mean, logz = state["ctx"].exact()
        return {"sums": _narrow(case, [loss, mean.real, mean.imag, logz])}
    if kind == "observe":
        return {"observables": _observables(case, compute_observables(state["sampler"]))}
    net = state["net"]
    net.flat[:] = state["p"]
    loss, prec = sample_(state["sampler"])
    obs = compute_observables(state["sampler"])
    grad = precondition_(prec, state["algo"], 0)
    update_(state["opt"], net, grad)
    return {"stats": _narrow(case, [loss.mean, loss.error, loss.variance, loss.tau, loss.R]),
            "observables": _observables(case, obs), "step": _narrow(case, grad), "params": _narrow(case, net.flat)}


def _observables(case, obs):
    return _narrow(case, [[m.mean.real, m.mean.imag, m.error, m.variance, m.tau, m.R]
                          for m in (obs[k] for k in ("Sx", "Sy", "Sz"))])


# ---------------------------------------------------------------- work
def work(case):
    """Inputs are the parameters (and the chains of a running loop), outputs the
    stepped parameters, statistics and samples; an activation counts as eight
    operations.  The S build is its non-zero lower triangles, a matrix-free
    solve is counted as 20 products (two passes of arithmetic over the rows)."""
    if case["kind"] == "batch":
        each = [work(m) for m in _members(case)]
        return {k: sum(w[k] for w in each) for k in ("bytes", "flops")}
    n, nh = _sites(case), case["alpha_h"] * _sites(case)
    na = case["alpha_a"] * n
    np_ = len(_params(case, 0))
    act = 8.0
    unit = {"ndm": nh + 2 * na, "rbmsplit": 2 * nh, "rbm": 2 * nh}[case["net"]] * (2 + act)   # one flip
    edges = {"ising": n, "tfim": n, "xyz": 2 * n}[case["model"]]
    conns = {"ising": 3 * n, "tfim": n, "xyz": 2 * edges + n}[case["model"]]
    pair = conns * {"ndm": 2 * nh + 2 * na, "rbmsplit": 2 * nh, "rbm": 2 * nh}[case["net"]] * (2 + act)
    if case["kind"] == "exact":
        ns = 4.0 ** n
        return {"bytes": 8.0 * np_, "flops": ns * (pair + 2 * n * (nh + na))}
    ns = case["chains"] * case["length"]
    calls = case["length"] + (0 if case["persistent"] else case["burn"])
    diag = 3 * (case["chains"] * calls * case["passes"] * unit + ns * n * unit)   # three observables
    if case["kind"] == "observe":
        return {"bytes": 8.0 * np_, "flops": float(diag)}
    flops = case["chains"] * calls * case["passes"] * unit + ns * pair
    if case["net"] == "ndm":
        nl, npi = n + nh + nh * n, na + 2 * na * n
        force, rows, tri = 8 * nh * n + 4 * na * n, 2 * nl + 2 * npi, float(nl + npi) ** 2
    elif case["net"] == "rbmsplit":
        force, rows, tri = 8 * nh * n, np_, 2.0 * (np_ / 2) ** 2
    else:
        force, rows, tri = 0, np_, 2.0 * (np_ / 2) ** 2
    flops += ns * conns * force + 2.0 * ns * rows
    flops += 20 * 4.0 * ns * rows if case["solver"] == "cg" else 2.0 * ns * tri + np_ ** 3 / 3.0
    if case["kind"] == "loop":
        flops += diag
    return {"bytes": 16.0 * np_ + 8.0 * ns, "flops": float(flops)}


# ---------------------------------------------------------------- the same in 64 bits, plain torch
DEV = "cuda" if torch.cuda.is_available() else "cpu"
M32 = 0xFFFFFFFF


def _philox(c0, c1, c2, c3, key):
    """Philox4x32-10 on broadcast int64 tensors of 32-bit words: four tensors of 32-bit words."""
    c = [torch.as_tensor(x, dtype=torch.int64, device=DEV) for x in (c0, c1, c2, c3)]
    k0, k1 = key & M32, (key >> 32) & M32
    for _ in range(10):
        a, b = c[0] * 0xD2511F53, c[2] * 0xCD9E8D57          # the low 64 bits, read as unsigned words below
        c = [((b >> 32) & M32) ^ c[1] ^ k0, b & M32, ((a >> 32) & M32) ^ c[3] ^ k1, a & M32]
        k0, k1 = (k0 + 0x9E3779B9) & M32, (k1 + 0xBB67AE85) & M32
    return torch.broadcast_tensors(*c)


def _spins(keys, bits):
    return (((keys[..., None] >> torch.arange(bits, device=DEV)) & 1) * 2 - 1).double()


def _f(act, x):
    if act == "logcosh":
        return x.abs() + torch.log1p(torch.exp(-2 * x.abs())) - math.log(2.0)
    return torch.nn.functional.softplus(x, threshold=50.0)


def _f_complex(act, a, b):
    """f(a + ib) as (real, imaginary)"""
    if act == "logcosh":
        t, s, c = torch.tanh(a), torch.sin(b), torch.cos(b)
        return _f(act, a) + 0.5 * torch.log(c * c + t * t * s * s), torch.atan2(t * s, c)
    e = torch.exp(a)
    return 0.5 * torch.log1p(e * (2 * torch.cos(b) + e)), torch.atan2(e * torch.sin(b), 1 + e * torch.cos(b))


def _amplitude(case, re, im, x, only_real=False):
    """log of the network at spins x [..., N or 2N] as (real, imaginary); parameters as real and imaginary parts."""
    n, nh = _sites(case), int(case["alpha_h"] * _sites(case))
    na, act = int(case["alpha_a"] * n), case["act"]
    if case["net"] == "ndm":
        bm, hm, wm, um, bl, hl, dl, wl, ul = torch.split(re, [n, nh, nh * n, na * n, n, nh, na, nh * n, na * n])
        wm, um, wl, ul = wm.view(n, nh), um.view(n, na), wl.view(n, nh), ul.view(n, na)
        s, e = x[..., :n], x[..., n:]
        p, m = s + e, s - e
        zr, zi = _f_complex(act, dl + 0.5 * p @ ul, 0.5 * m @ um)
        real = 0.5 * (_f(act, hl + s @ wl).sum(-1) + _f(act, hl + e @ wl).sum(-1) + p @ bl) + zr.sum(-1)
        if only_real:
            return real, None
        return real, 0.5 * (_f(act, hm + s @ wm).sum(-1) - _f(act, hm + e @ wm).sum(-1) + m @ bm) + zi.sum(-1)
    v = n if case["net"] == "rbm" else 2 * n       # visible units: a (ar, ac), b, W (Wr, Wc), column-major
    ar, br, wr = re[:v], re[v:v + nh], re[v + nh:].view(v, nh)
    ai, bi, wi = im[:v], im[v:v + nh], im[v + nh:].view(v, nh)
    fr, fi = _f_complex("softplus", br + x @ wr, bi + x @ wi)
    return x @ ar + fr.sum(-1), x @ ai + fi.sum(-1)


def _complexed(case, flat):
    """The flat vector as (real, imaginary) parts of the parameters."""
    t = torch.tensor(flat, dtype=torch.float64, device=DEV)
    return (t, torch.zeros_like(t)) if case["net"] == "ndm" else (t[0::2].contiguous(), t[1::2].contiguous())


def _sample(case, re, im, seed, it, start, burn, diag=False):
    """(stored keys [length, chains], last keys); proposals as the sampler's streams draw them."""
    n, chains, passes = _sites(case), case["chains"], case["passes"]
    ket = case["net"] == "rbm"
    bits, tag = n if ket else 2 * n, 16 if diag else 0
    chain = torch.arange(chains, device=DEV)
    if start is None:
        w = _philox(0, it, chain, tag, seed)
        start = (w[0] | (w[1] << 32)) & ((1 << (n if diag else bits)) - 1)
        start = start | (start << n) if diag else start
    count = (burn + case["length"]) * passes
    w = _philox(torch.arange(count, device=DEV)[:, None], it, chain[None, :], tag + 1, seed)
    site = (w[0] * (n if diag else bits)) >> 32
    if case["precision"] == "fp64":
        u = ((w[1] >> 5).double() * 67108864.0 + (w[2] >> 6).double()) / 9007199254740992.0
    else:
        u = (w[1] >> 8).double() / 16777216.0
    flip = 1.0 - 2.0 * torch.eye(n if diag else bits, dtype=torch.float64, device=DEV)
    flip = torch.cat([flip, flip], 1) if diag else flip
    factor, x, out = 1.0 if diag else 2.0, _spins(start, bits), []
    lp = factor * _amplitude(case, re, im, x, True)[0]
    for t in range(count):
        xn = x * flip[site[t]]
        ln = factor * _amplitude(case, re, im, xn, True)[0]
        ok = u[t] < torch.exp(ln - lp)
        x, lp = torch.where(ok[:, None], xn, x), torch.where(ok, ln, lp)
        if (t + 1) % passes == 0 and (t + 1) // passes > burn:
            out.append(x)
    weights = 1 << torch.arange(bits, device=DEV)
    keys = ((torch.stack(out) > 0) * weights).sum(-1)
    return keys, keys[-1]


def _bonds(case):
    if case["model"] != "xyz":
        n = case["lx"]
        return [(i, i + 1) for i in range(n - 1)] + ([(n - 1, 0)] if case["periodic"] and n > 1 else [])
    return [(i - 1, j - 1) for i, j in _lattice_edges(case["lx"], case["ly"], case["periodic"])]


def _lattice_edges(lx, ly, periodic):
    """Nearest neighbours of the lattice, each once, 1-based."""
    es = set()
    for y in range(ly):
        for x in range(lx):
            for nx, ny in ((x + 1, y), (x, y + 1)):
                if not periodic and (nx >= lx or ny >= ly):
                    continue
                i, j = 1 + x + lx * y, 1 + nx % lx + lx * (ny % ly)
                if i != j:
                    es.add((min(i, j), max(i, j)))
    return sorted(es)


def _half(case, s):
    """The Hamiltonian at spins s [B, N]: (diagonal element, [(sites flipped, element)])."""
    bonds = _bonds(case)
    zz = sum(s[:, i] * s[:, j] for i, j in bonds)
    if case["model"] == "xyz":
        return 1.1 * zz, [((i, j), 0.9 - 1.0 * s[:, i] * s[:, j]) for i, j in bonds]
    return 0.5 * zz, [((i,), torch.full_like(s[:, 0], 0.5 * case["g"])) for i in range(s.shape[1])]


def _connections(case, x):
    """[(spins flipped or None, complex element [B])] of the loop's operator at x."""
    n = _sites(case)
    if case["net"] == "rbm":
        d, off = _half(case, x)
        return [(None, d + 0j)] + [(f, m + 0j) for f, m in off]
    s, e = x[:, :n], x[:, n:]
    ds, os_ = _half(case, s)
    de, oe = _half(case, e)
    decay = ((s < 0).double() + (e < 0).double()).sum(1)      # sigma^- takes bit 0 (v = -1) to bit 1
    out = [(None, -1j * (ds - de) - 0.5 * decay)]
    out += [(f, -1j * m) for f, m in os_] + [(tuple(i + n for i in f), 1j * m) for f, m in oe]
    out += [((i, i + n), ((s[:, i] > 0) & (e[:, i] > 0)).double() + 0j) for i in range(n)]
    return out


def _flipped(x, sites):
    if sites is None:
        return x
    x = x.clone()
    x[:, list(sites)] *= -1
    return x


def _local(case, re, im, x, conns):
    """(local values, their addends) at spins x"""
    lr, li = _amplitude(case, re, im, x)
    parts = []
    for sites, mel in conns:
        r, i = _amplitude(case, re, im, _flipped(x, sites))
        parts.append(mel * torch.exp(torch.complex(r - lr, i - li)))
    return sum(parts), parts


def _chain_stats(v):
    """[mean, error, variance, tau, R] of values [length, chains] (real or complex; the mean's real part first)."""
    L, B = v.shape
    m = v.mean(0)
    mu = m.mean()
    var_in = ((v - m).abs() ** 2).sum(0).div(L - 1).mean()
    var_m = ((m - mu).abs() ** 2).sum() / (B - 1)
    t = var_m / (((v - mu).abs() ** 2).sum() / (B * L - 1))
    vals = [mu.real, torch.sqrt(var_m / B), var_in, torch.clamp(0.5 * (t * L - 1), min=0.0),
            torch.sqrt((L - 1) / L + t), mu.imag if v.is_complex() else torch.zeros_like(t)]
    return torch.stack(vals).cpu().numpy()


def _rows(case, re, im, x):
    """The log-derivatives [B, parameters], complex: derivatives along the parameters' real directions."""
    def one(k):
        return lambda q, y: _amplitude(case, q, im, y)[k]
    parts = []
    for y in x.split(2048):
        d = [torch.func.vmap(torch.func.grad(one(k)), (None, 0))(re, y) for k in (0, 1)]
        parts.append(torch.complex(*d))
    return torch.cat(parts)


def _solve(case, keys, re, im):
    """(statistics, step) of one SR iteration on stored keys [length, chains]"""
    ket = case["net"] == "rbm"
    x = _spins(keys.reshape(-1), _sites(case) * (1 if ket else 2))
    ns = len(x)
    conns = _connections(case, x)
    local, parts = _local(case, re, im, x, conns)
    O = _rows(case, re, im, x)
    mean = O.mean(0)
    O -= mean
    if ket:
        stats = _chain_stats(local.view(keys.shape))
        F = (local @ O.conj()) / ns
    else:
        stats = _chain_stats((local.abs() ** 2).view(keys.shape))
        coef, G = local.conj() / ns, []
        for k in (0, 1):
            q, total = re.clone().requires_grad_(True), torch.zeros_like(re)
            for (sites, _), w in zip(conns, parts):
                r, i = _amplitude(case, q, im, _flipped(x, sites))
                c = coef * w
                val = (c.real * r - c.imag * i if k == 0 else c.real * i + c.imag * r).sum()
                total += torch.autograd.grad(val, q)[0]
            G.append(total)
            if case["net"] == "ndm":
                G.append(torch.zeros_like(total))
                break
        F = torch.complex(*G) - stats[0] * mean
    if case["net"] == "ndm":
        F, S = F.real, (O.real.T @ O.real + O.imag.T @ O.imag) / ns
    else:
        S = O.conj().T @ O / ns
    S.diagonal().add_(case["eps"])
    step = torch.linalg.solve(S, F)
    if case["net"] != "ndm":
        step = torch.view_as_real(step).reshape(-1)
    return stats[:5], step.cpu().numpy()


def _iteration(case, seeds):
    """(statistics, step, parameters before) of the first pass on a prepared state"""
    p = _params(case, seeds[0])
    re, im = _complexed(case, p)
    if case["kind"] == "step" and case["persistent"]:
        _, last = _sample(case, re, im, seeds[1], 0, None, case["burn"])
        keys, _ = _sample(case, re, im, seeds[1], 1, last, 0)
    else:
        keys, _ = _sample(case, re, im, seeds[1], 0, None, case["burn"])
    return (*_solve(case, keys, re, im), p)


def _magnetisation_stats(case, seeds, it):
    """[3, 6] statistics of Sx, Sy, Sz on the diagonal chain of iteration `it`"""
    n = _sites(case)
    re, im = _complexed(case, _params(case, seeds[0]))
    keys, _ = _sample(case, re, im, seeds[1], it, None, case["burn"], diag=True)
    x = _spins(keys.reshape(-1), 2 * n)
    lr, li = _amplitude(case, re, im, x)
    sx = sy = 0
    for i in range(n):
        r, m = _amplitude(case, re, im, _flipped(x, (i,)))
        w = torch.exp(torch.complex(r - lr, m - li)) / n
        sx, sy = sx + w, sy + 1j * x[:, i] * w
    out = []
    for v in (sx, sy, -x[:, :n].sum(1) / n + 0j):     # sigma^z is +1 on v = -1
        st = _chain_stats(v.view(keys.shape))
        out.append([st[0], st[5], *st[1:5]])
    return np.array(out)


def exact(case, seed):
    kind, seeds = case["kind"], _seeds(seed)
    if kind == "exact":
        re, im = _complexed(case, _params(case, seeds[0]))
        bits, lps, ls = 2 * _sites(case), [], []
        for keys in torch.arange(1 << bits, device=DEV).split(1 << 18):
            x = _spins(keys, bits)
            lps.append(2 * _amplitude(case, re, im, x)[0])
            ls.append(_local(case, re, im, x, _connections(case, x))[0])
        lp, local = torch.cat(lps), torch.cat(ls)
        logz = torch.logsumexp(lp, 0)
        w = torch.exp(lp - logz)
        mean = (w * local).sum()
        return {"sums": np.array([(w * local.abs() ** 2).sum().item(), mean.real.item(), mean.imag.item(),
                                  logz.item()])}
    if kind == "observe":
        return {"observables": _magnetisation_stats(case, seeds, 0)}
    if kind == "batch":
        done = [_iteration(m, _seeds(seed, i)) for i, m in enumerate(_members(case))]
        return {"stats": np.stack([d[0] for d in done]),
                "params": np.concatenate([p - case["lr"] * step for _, step, p in done])}
    stats, step, p = _iteration(case, seeds)
    out = {"stats": stats, "params": p - case["lr"] * step}
    if kind == "loop":
        out.update(step=step, observables=_magnetisation_stats(case, seeds, 1))
    return out
