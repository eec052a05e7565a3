"""W8A32 on the bf16 matrix cores: fp32 activations in three exact pieces.

Against a 64-bit product with a bound of fp32 sums: the pieces' products are
exact and a sum of K of them in any order is within K * 2^-24 * sum|a b| of
the exact one (the scale, bias and output rounding add three more)."""
import numpy as np
import pytest
import torch

import oracle
from luisaml_amd import capi, synth

pytestmark = pytest.mark.gpu


def run(dev, a, qw, sw, bias, pad=0, shift=0, out_dtype=torch.float32, mfma=True):
    M, K = a.shape
    buf = torch.zeros(shift + M * (K + pad), dtype=torch.float32, device=dev)
    va = buf[shift:].view(M, K + pad)[:, :K]
    va.copy_(torch.from_numpy(a))
    bp = capi.pack_weight(torch.from_numpy(qw).to(dev), True)
    capi.kernel_trace()
    y = capi.gemm_w8a32(va, bp, torch.from_numpy(sw).to(dev), qw.shape[0], K, c=torch.from_numpy(bias).to(dev),
                        out_dtype=out_dtype)
    assert capi.kernel_trace() == ["gemm_w8a32_mfma" if mfma else "gemv_valu_w8a32"]
    return y


def weights(N, K, seed):
    w = synth.normal(seed, (N, K), std=0.05)
    sw = oracle.channel_scales(w, axis=0)
    return oracle.quantize(w, sw, axis=0), sw


def check(y, a, qw, sw, bias):
    K = a.shape[1]
    B = oracle.e4m3_to_float(qw).astype(np.float64) * sw.astype(np.float64)[:, None]
    ref = a.astype(np.float64) @ B.T + bias
    bound = (K + 3) * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(B).T + np.abs(bias))
    assert np.all(np.abs(y.astype(np.float64) - ref) <= bound)


# 16x1, 16x2 and 32x3 tiles with row, column and K remainders (K at the edges
# of a 16-k chunk, a 64-k step, a 128-k block and the parts), and the
# vector-ALU kernel's sizes
@pytest.mark.parametrize("M,N,K", [(1, 64, 100), (17, 4100, 1000), (65, 1030, 65), (33, 11000, 127), (40, 11008, 129),
                                   (129, 6000, 200), (100, 11007, 64), (127, 8200, 1), (96, 12300, 528)])
@pytest.mark.parametrize("pad,shift", [(0, 0), (4, 4), (3, 1)])
def test_w8a32_against_64_bits(dev, M, N, K, pad, shift):
    a = synth.normal(M, (M, K)) * np.exp(synth.normal(M + 1, (M, K), std=3.0)).astype(np.float32)
    qw, sw = weights(N, K, N)
    bias = synth.normal(3, (N,), std=0.01)
    check(run(dev, a, qw, sw, bias, pad, shift, mfma=M > 1).cpu().numpy(), a, qw, sw, bias)


def check_unscaled(y, a, B):
    """check() for unit scales; at most 8 parts' sums, their sum and the result
    are each rounded to a multiple of 2^-149."""
    K = a.shape[1]
    ref = a.astype(np.float64) @ B.T
    bound = (K + 3) * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(B).T) + 17 * 2.0 ** -150
    assert np.all(np.abs(y.astype(np.float64) - ref) <= bound)


@pytest.mark.parametrize("scale", [1e-43, 1e-40, 1e-38, 1e-36, 1e-33, 1e-30, 1e30, 1e34])
@pytest.mark.parametrize("M,N", [(40, 2048), (40, 11008), (128, 11008)])
def test_w8a32_ends_of_the_range(dev, M, N, scale):
    """Subnormal activations and pieces, and values near the largest: the same bound."""
    K = 256
    a = (synth.normal(1, (M, K)) * scale).astype(np.float32)
    qw, sw = weights(N, K, 2)
    y = run(dev, a, qw, np.ones_like(sw), np.zeros(N, np.float32)).cpu().numpy()
    check_unscaled(y, a, oracle.e4m3_to_float(qw).astype(np.float64))


@pytest.mark.parametrize("big", [2.0 ** 111, 2.0 ** 112, 2.0 ** 113, 2.0 ** 118, np.inf])
def test_w8a32_small_beside_large(dev, big):
    """Activations at the ends of the range in one workgroup, in other rows and
    in one row whose large values meet zero weights: the small ones keep their
    bits, and an infinity's row has none to keep."""
    M, N, K = 40, 2048, 256
    a = (synth.normal(1, (M, K)) * np.float32(1e-38)).astype(np.float32)
    qw, _ = weights(N, K, 2)
    qw[:N // 2, 7] = 0
    a[3, 7] = a[30, 7] = np.float32(big)
    a[5, 9] = np.float32(big)
    y = run(dev, a, qw, np.ones(N, np.float32), np.zeros(N, np.float32)).cpu().numpy()
    B = oracle.e4m3_to_float(qw).astype(np.float64)
    if np.isinf(big):
        ref = oracle.gemm(a, oracle.e4m3_to_float(qw), transB=1)
        for r in (3, 5, 30):
            assert np.array_equal(np.isnan(y[r]), np.isnan(ref[r])) and not np.isfinite(y[r]).any()
        fin = [r for r in range(M) if r not in (3, 5, 30)]
        y, a = y[fin], a[fin]
    check_unscaled(y, a, B)


@pytest.mark.parametrize("M,N", [(40, 2048), (40, 11008), (128, 11008)])
def test_w8a32_infinities_and_nan(dev, M, N):
    """inf and NaN activations (a NaN whose upper half is an infinity's among
    them) give what the oracle's fma chain gives, in their own rows only."""
    K = 130
    a = synth.normal(5, (M, K))
    a[3, 7], a[20, 129], a[21, 1] = np.inf, -np.inf, np.array(0x7F800001, np.uint32).view(np.float32)
    a[22, 4], a[22, 5] = np.inf, -np.inf
    qw, sw = weights(N, K, 6)
    bias = np.zeros(N, np.float32)
    y = run(dev, a, qw, sw, bias).cpu().numpy()
    ref = oracle.gemm(a, oracle.dequantize(qw, sw, axis=0), transB=1)
    assert np.array_equal(np.isnan(y), np.isnan(ref)) and np.array_equal(np.isinf(y), np.isinf(ref))
    assert np.array_equal(np.sign(y[np.isinf(y)]), np.sign(ref[np.isinf(ref)]))
    fin = np.isfinite(ref).all(1)
    check(y[fin], a[fin], qw, sw, bias)


def test_w8a32_more_row_groups_than_a_grid(dev):
    """One column, 2^27 rows: more row groups than one grid dimension has workgroups."""
    M = (1 << 27) + 16
    a = torch.empty((M, 1), device=dev).normal_(generator=torch.Generator(device=dev).manual_seed(3))
    qw, sw = np.array([[0x42]], np.uint8), np.array([0.5], np.float32)
    y = torch.full((M, 1), np.nan, device=dev)
    capi.gemm_w8a32(a, capi.pack_weight(torch.from_numpy(qw).to(dev), True), torch.from_numpy(sw).to(dev), 1, 1, out=y)
    assert torch.equal(y, a * float(oracle.e4m3_to_float(qw)[0, 0]) * 0.5)


# the choice of the kernel: rows and panels up to 512 on the vector ALU but for
# a few rows of many panels over a long K; up to 1024 with little work, whose
# bound depends on the activations' alignment; and next to no work
@pytest.mark.parametrize("M,N,K,mfma", [(56, 212, 6722, False), (30, 982, 4333, False), (9, 2900, 3550, False), (8, 2900, 4628, True),
                                        (4, 4100, 7312, True), (1, 11008, 4096, False), (2, 11008, 4096, True),
                                        (61, 1007, 730, False), (61, 1007, 732, True), (339, 170, 200, False), (39, 2500, 16, False),
                                        (391, 152, 60, True), (16, 4096, 512, True)])
def test_w8a32_kernel(dev, M, N, K, mfma):
    a = synth.normal(M, (M, K))
    qw, sw = weights(N, K, N)
    bias = synth.normal(3, (N,), std=0.01)
    y = run(dev, a, qw, sw, bias, mfma=mfma)
    check(y.cpu().numpy(), a, qw, sw, bias)
