"""The BF16 S build (split-K Gram on the matrix cores) against the same Gram
computed on the CPU from the same BF16-rounded centred O rows: only FP32
accumulation error remains, so the bound is tight, at shapes that use many
128 x 128 tiles (edges not multiples of 128) and many sample chunks."""
import numpy as np
import pytest

from _helpers import ising, params, random_keys, rel_err
from nqhip import Context, _lib

pytestmark = pytest.mark.gpu


def to_bf16(x):
    """Round float32 values to BF16 (nearest, ties to even), returned as float64."""
    u = np.ascontiguousarray(x, dtype=np.float32).view(np.uint32).astype(np.uint64)
    u = (u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000
    return u.astype(np.uint32).view(np.float32).astype(np.float64)


@pytest.mark.parametrize("N,alpha,chains,Lc", [(12, 2, 256, 8), (8, 1, 100, 7)])
def test_bf16_gram_matches_cpu_gram_of_rounded_rows(gpu_ok, ref, N, alpha, chains, Lc):
    nh = na = alpha * N
    flat, _, _ = ising(N)
    p = params(ref.ndm_np(N, nh, na), seed=21, sigma=0.1)
    keys = random_keys(N, chains * Lc, seed=22)
    ctx = Context(0, 1)
    ctx.set_problem(flat)
    ctx.set_ndm(N, nh, na)
    ctx.set_params(p)
    ctx.set_precision(_lib.PREC_FP32, _lib.PREC_BF16)
    _, O = ctx.logpsi_grad(keys)                  # FP32 network values, reference order
    _, S, _, _ = ctx.grad_from_samples(keys, chains, Lc)
    Ns = len(keys)
    Oc = O - O.mean(axis=0)
    Re = to_bf16(Oc.real.astype(np.float32))
    Im = to_bf16(Oc.imag.astype(np.float32))
    S_cpu = (Re.T @ Re + Im.T @ Im) / Ns
    assert rel_err(S, S_cpu) < 2e-5
    assert np.array_equal(S, S.T)                 # mirrored exactly
    ctx.close()


# samples: fewer than a k-step of the FP64 (16) and FP32 (32) tiles, one past it, several chunks with
# a ragged last k-step; nA = 15, 78, 210 columns (one tile of 64, ragged, several)
@pytest.mark.parametrize("sprec", [_lib.PREC_FP64, _lib.PREC_FP32])
@pytest.mark.parametrize("N,alpha,chains,Lc", [(2, 1, 2, 2), (5, 1, 3, 5), (5, 1, 11, 3), (8, 1, 2, 8), (8, 1, 125, 16),
                                               (4, 3, 77, 9)])
def test_gram_chunks_match_cpu_gram(gpu_ok, sprec, N, alpha, chains, Lc):
    """The FP64 and FP32 Gram of the FP64 network's rows against the CPU Gram
    of the same rows in FP64: rounding of the sums only (FP64: 1e-12; FP32:
    the centred rows rounded to 24 bits, 2 x 6e-8 per product, and sums of at
    most 2000 addends in FP32, below 1e-5 of the largest element)."""
    flat, _, _ = ising(N)
    ctx = Context(0, 1)
    ctx.set_problem(flat)
    ctx.set_ndm(N, alpha * N, alpha * N)
    ctx.set_params(params(ctx.np_, seed=31, sigma=0.2))
    ctx.set_precision(_lib.PREC_FP64, sprec)
    keys = random_keys(N, chains * Lc, seed=32)
    _, O = ctx.logpsi_grad(keys)
    _, S, _, _ = ctx.grad_from_samples(keys, chains, Lc)
    Oc = O - O.mean(axis=0)
    S_cpu = (Oc.real.T @ Oc.real + Oc.imag.T @ Oc.imag) / len(keys)
    assert rel_err(S, S_cpu) < (1e-12 if sprec == _lib.PREC_FP64 else 1e-5)
    assert np.array_equal(S, S.T)
    ctx.close()


def test_fp32_rows_are_centred_in_fp64(gpu_ok):
    """An FP32 network's rows are centred in FP64 and rounded once, as an FP64
    network's are: with every parameter zero the rows of both are the same
    numbers (halves, quarters and zeros), so S is the same bit for bit; six
    and fourteen samples give means that no float holds."""
    N, out = 4, []
    for chains in (3, 7):
        keys = random_keys(N, 2 * chains, seed=90 + chains)
        for prec in (_lib.PREC_FP64, _lib.PREC_FP32):
            ctx = Context(0, 1)
            ctx.set_problem(ising(N)[0])
            ctx.set_ndm(N, 2 * N, N)
            ctx.set_params(np.zeros(ctx.np_))
            ctx.set_precision(prec, _lib.PREC_FP32)
            _, O = ctx.logpsi_grad(keys)
            _, S, _, _ = ctx.grad_from_samples(keys, chains, 2)
            out.append((O, S))
            ctx.close()
        (O64, S64), (O32, S32) = out[-2:]
        assert np.array_equal(O64, O32)
        assert np.array_equal(S64, S32)
