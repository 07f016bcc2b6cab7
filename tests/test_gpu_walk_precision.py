"""How far the FP64 walk's L_loc by products is from the exact values: not
further than L_loc by the sums of f, which the parity mode (per-sample
gradients) evaluates on the same device.  Both against an 80-bit evaluation;
weights on either side of the walk's two forms."""
import numpy as np
import pytest

from _helpers import ising, params, random_keys, xyz
from nqhip import Context, _lib, problems

pytestmark = pytest.mark.gpu
T = np.longdouble


def exact(model, lx, ly, nh, na, act, p, keys):
    """L_loc (real, imaginary) of the dissipative Ising chain (V = 2, g = 1)
    or XYZ lattice (0.9, 1, 1.1) in 80 bits."""
    N, half = lx * ly, T(0.5)
    sizes = np.cumsum([N, nh, nh * N, na * N, N, nh, na, nh * N])
    bm, hm, wm, um, bl, hl, dl, wl, ul = np.split(p.astype(T), sizes)
    wm, um, wl, ul = wm.reshape(N, nh), um.reshape(N, na), wl.reshape(N, nh), ul.reshape(N, na)
    x = (((keys[:, None] >> np.arange(2 * N, dtype=np.uint64)) & np.uint64(1)).astype(np.int64) * 2 - 1).astype(T)

    def mul(a, w):
        return sum(a[:, i:i + 1] * w[i] for i in range(len(w)))

    def f(y):
        return np.abs(y) + np.log1p(np.exp(-2 * np.abs(y))) - np.log(T(2)) if act else np.log1p(np.exp(y))

    def fc(a, b):
        if act:
            t, s, c = np.tanh(a), np.sin(b), np.cos(b)
            return f(a) + half * np.log(c * c + t * t * s * s), np.arctan2(t * s, c)
        e = np.exp(a)
        return half * np.log1p(e * (2 * np.cos(b) + e)), np.arctan2(e * np.sin(b), 1 + e * np.cos(b))

    def logrho(x):
        s, e = x[:, :N], x[:, N:]
        zr, zi = fc(dl + mul((s + e) * half, ul), mul((s - e) * half, um))
        return (half * ((f(hl + mul(s, wl)) + f(hl + mul(e, wl))).sum(1) + mul(s + e, bl[:, None])[:, 0]) + zr.sum(1),
                half * ((f(hm + mul(s, wm)) - f(hm + mul(e, wm))).sum(1) + mul(s - e, bm[:, None])[:, 0]) + zi.sum(1))

    def hamiltonian(s):
        if model == "ising":
            zz = sum(s[:, i] * s[:, (i + 1) % N] for i in range(N))
            return half * zz, [((i,), half + 0 * zz) for i in range(N)]
        bonds = [(i - 1, j - 1) for i, j in problems.square_edges(lx, ly)]
        return (T(1.1) * sum(s[:, i] * s[:, j] for i, j in bonds),
                [((i, j), T(0.9) - s[:, i] * s[:, j]) for i, j in bonds])

    s, e = x[:, :N], x[:, N:]
    (ds, fs), (de, fe), zero = hamiltonian(s), hamiltonian(e), np.zeros(len(x), T)
    conns = [((), -half * ((s < 0).astype(T) + (e < 0)).sum(1), de - ds)]
    conns += [(q, zero, -m) for q, m in fs] + [(tuple(i + N for i in q), zero, m) for q, m in fe]
    conns += [((i, i + N), ((s[:, i] > 0) & (e[:, i] > 0)).astype(T), zero) for i in range(N)]
    r0, i0 = logrho(x)
    L = np.zeros((2, len(x)), T)
    for sites, mr, mi in conns:
        y = x.copy()
        y[:, list(sites)] *= -1
        r, i = logrho(y)
        q, u = np.exp(r - r0) * np.cos(i - i0), np.exp(r - r0) * np.sin(i - i0)
        L += np.stack([mr * q - mi * u, mr * u + mi * q])
    return L


@pytest.mark.parametrize("model,lx,ly,nh,na,act,sigma", [
    ("ising", 6, 1, 6, 6, 0, 0.1), ("ising", 6, 1, 6, 6, 1, 0.1), ("ising", 12, 1, 24, 24, 0, 0.05),
    ("xyz", 2, 3, 18, 18, 0, 0.1), ("xyz", 3, 3, 27, 9, 1, 0.05), ("ising", 8, 1, 16, 33, 0, 0.1),
    ("ising", 8, 1, 64, 64, 1, 0.1), ("ising", 10, 1, 20, 10, 0, 0.3), ("xyz", 2, 3, 12, 12, 1, 0.6)])
def test_no_further_than_the_sums_of_f(gpu_ok, model, lx, ly, nh, na, act, sigma):
    N = lx * ly
    ctx = Context(0, 1)
    ctx.set_problem((xyz(lx, ly) if model == "xyz" else ising(N))[0])
    ctx.set_ndm(N, nh, na, act)
    ctx.set_precision(_lib.PREC_FP64, _lib.PREC_FP64)
    p = params(ctx.np_, seed=19, sigma=sigma)
    ctx.set_params(p)
    keys = random_keys(N, 800, seed=20)
    L = exact(model, lx, ly, nh, na, act, p, keys)
    off = []
    for got in (ctx.local_estimator(keys), ctx.local_estimator(keys, grad=True)[0]):
        off.append(float(np.sqrt(((np.stack([got.real, got.imag]) - L) ** 2).sum() / (L ** 2).sum())))
    ctx.close()
    assert off[0] <= off[1], off
