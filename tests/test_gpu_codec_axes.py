"""Quantize / dequantize with a scale per axis element, dynamic quantisation of
odd sizes and packing of [N, K] weights: equal to the oracle byte for byte at
the remainders of the four-element accesses, in every layout of the axis."""
import numpy as np
import pytest
import torch

import oracle
from luisaml_amd import capi, synth

pytestmark = pytest.mark.gpu


def special(x):
    f = x.reshape(-1)
    for i, v in enumerate([np.nan, np.inf, -np.inf, 0.0, -0.0, 1e-40, 3e38]):
        f[(i * 7919) % f.size] = v
    return x


# shape, axis: the last axis with lengths 0..3 mod 4 (periods of one, two and
# four rows), fewer and more rows than a period, more groups than the grid; an
# inner run of 1, 2, 3, more and odd, outer repeats; n below 4
SHAPES = [((5, 8), 1), ((9, 1000), 1), ((7, 1002), 1), ((13, 1001), 1), ((1, 3), 1), ((2, 5003), 1), ((3000, 2051), 1),
          ((17, 1), 0), ((1001, 7), 0), ((33, 1023), 0), ((64, 4095), 0), ((2, 3), 0), ((3, 5, 2), 1), ((4, 6, 9), 1),
          ((2, 3, 7, 13), 1), ((3, 130, 4), 1), ((3, 4, 11, 5), 2), ((2100, 2051), 0)]


@pytest.mark.parametrize("shape,axis", SHAPES)
@pytest.mark.parametrize("shift", [0, 1])
def test_per_axis(dev, shape, axis, shift):
    x = special(synth.normal(sum(shape), shape))
    s = np.abs(synth.normal(axis + 1, (shape[axis],), std=0.05)) + np.float32(1e-4)
    s[0] = 1e-25  # outside the reciprocal's range
    n = x.size
    xb = torch.empty(n + shift, device=dev)
    yb = torch.empty(n + shift, dtype=torch.uint8, device=dev)
    dx, q = xb[shift:].view(shape), yb[shift:].view(shape)
    dx.copy_(torch.from_numpy(x))
    capi.quantize(dx, torch.from_numpy(s).to(dev), axis=axis, out=q)
    ref = oracle.quantize(x, s, axis=axis)
    assert np.array_equal(q.cpu().numpy(), ref)
    back = capi.dequantize(q, torch.from_numpy(s).to(dev), axis=axis, out=xb[shift:].view(shape))
    assert np.array_equal(back.cpu().numpy(), oracle.dequantize(ref, s, axis=axis), equal_nan=True)


# the smallest tensors of the four-at-a-time kernels and the largest scalar
# ones: last-axis lengths 0..3 mod 4, one row, short rows; runs of 2, 3, 5, 7,
# just under and over 256 and longer, whole vectors, outer repeats
@pytest.mark.parametrize("shape,axis,quant,dequant", [
    ((656, 1000), 1, "cols", "cols"), ((655, 1002), 1, "cols", "cols"), ((656, 1001), 1, "cols", "cols"), ((1, 655363), 1, "cols", "cols"),
    ((218455, 3), 1, "cols", "cols"), ((2, 327681), 1, "cols", "cols"), ((655, 1000), 1, "scalar", "cols"),
    ((1048577, 2), 0, "axis", "axis"), ((699053, 3), 0, "axis", "axis"), ((699050, 3), 0, "scalar", "axis"), ((7, 42801, 7), 1, "axis", "axis"),
    ((2, 3, 70001, 5), 2, "axis", "axis"), ((3, 2100, 255), 1, "scalar", "axis"), ((3, 2743, 255), 1, "axis", "axis"), ((3, 1361, 257), 1, "axis", "axis"),
    ((3, 1360, 257), 1, "scalar", "scalar"), ((1026, 1023), 0, "axis", "axis"), ((5, 7, 12), 1, "axis", "axis")])
def test_per_axis_kernel(dev, shape, axis, quant, dequant):
    x = special(synth.normal(sum(shape), shape))
    s = np.abs(synth.normal(axis + 1, (shape[axis],), std=0.05)) + np.float32(1e-4)
    s[0] = 1e-25  # outside the reciprocal's range
    ds = torch.from_numpy(s).to(dev)
    capi.kernel_trace()
    q = capi.quantize(torch.from_numpy(x).to(dev), ds, axis=axis)
    back = capi.dequantize(q, ds, axis=axis)
    assert capi.kernel_trace() == ["quantize_" + quant, "dequantize_" + dequant]
    ref = oracle.quantize(x, s, axis=axis)
    assert np.array_equal(q.cpu().numpy(), ref)
    assert np.array_equal(back.cpu().numpy(), oracle.dequantize(ref, s, axis=axis), equal_nan=True)


@pytest.mark.parametrize("shape", [(1 << 10, (1 << 12) + 1, 1 << 10), (1 << 16, (1 << 16) + 1, 1), (3, 21, 68191747)])
def test_per_axis_beyond_32_bits(dev, shape):
    """2^32 elements and more, with an inner run and without, whole vectors and not."""
    x = torch.empty(shape, device=dev).normal_(generator=torch.Generator(device=dev).manual_seed(1))
    s = np.abs(synth.normal(1, (shape[1],), std=0.05)) + np.float32(1e-4)
    ds = torch.from_numpy(s).to(dev)
    capi.kernel_trace()
    q = capi.quantize(x, ds, axis=1)
    # first, last, and either side of element 2^32
    inner, n = shape[2], x.numel()
    xf, qf = x.view(-1), q.view(-1)
    at = torch.cat([torch.arange(0, 5000), torch.arange((1 << 32) - 5000, min(n, (1 << 32) + 5000)), torch.arange(n - 5000, n)])
    ref = oracle.quantize(xf[at.to(dev)].cpu().numpy(), s[(at // inner % shape[1]).numpy()], axis=0)
    assert np.array_equal(qf[at.to(dev)].cpu().numpy(), ref)
    capi.dequantize(q, ds, axis=1, out=x)
    back = oracle.dequantize(ref, s[(at // inner % shape[1]).numpy()], axis=0)
    assert np.array_equal(xf[at.to(dev)].cpu().numpy(), back)
    kind = "cols" if inner == 1 else "axis"
    assert capi.kernel_trace() == ["quantize_" + kind, "dequantize_" + kind]


@pytest.mark.parametrize("n", [1, 3, 4, 5, 4097, 5003, 16387, 65533, 65537, 262147, 2097155, 9000001])
@pytest.mark.parametrize("shift", [0, 1])
def test_dynamic_odd_sizes(dev, n, shift):
    """The largest magnitude in the last element, so the tail sets the scale."""
    x = synth.normal(n, (n,))
    x[-1] = -9.0
    buf = torch.empty(n + shift, device=dev)
    buf[shift:].copy_(torch.from_numpy(x))
    q, s = capi.quantize_dynamic(buf[shift:])
    ref = oracle.dynamic_scale(x)
    assert float(s.item()) == ref
    assert np.array_equal(q.cpu().numpy(), oracle.quantize(x, ref))
    back = capi.dequantize(q, s)
    assert np.array_equal(back.cpu().numpy(), oracle.dequantize(oracle.quantize(x, ref), ref))


@pytest.mark.parametrize("n,kernel", [(1, "_small"), (255, "_small"), (4097, "_small"), (4999, "_small"), (5001, "_spread"), (4, "_spread"),
                                      (4996, "_spread"), (65535, "_spread"), (65537, "")])
def test_dynamic_kernel(dev, n, kernel):
    x = synth.normal(n, (n,))
    x[-1] = -9.0
    capi.kernel_trace()
    q, s = capi.quantize_dynamic(torch.from_numpy(x).to(dev))
    assert capi.kernel_trace() == ["quantize_dynamic" + kernel]
    ref = oracle.dynamic_scale(x)
    assert float(s.item()) == ref and np.array_equal(q.cpu().numpy(), oracle.quantize(x, ref))


@pytest.mark.parametrize("N,K", [(1, 1), (3, 15), (65, 16), (64, 17), (130, 255), (70, 1001), (33, 128), (5, 4099)])
@pytest.mark.parametrize("shift", [0, 1, 2, 3])
def test_pack_nk_bytes(dev, N, K, shift):
    w = (np.arange(N * K, dtype=np.int64) * 2654435761 >> 7).astype(np.uint8).reshape(N, K)
    buf = torch.empty(N * K + shift, dtype=torch.uint8, device=dev)
    buf[shift:].copy_(torch.from_numpy(w.reshape(-1)))
    p = capi.pack_weight(buf[shift:].view(N, K), True).cpu().numpy()
    Kp, Np = -(-K // 128) * 128, -(-N // 64) * 64
    full = np.zeros((Np, Kp), np.uint8)
    full[:N, :K] = w
    ref = full.reshape(Np // 64, 64, Kp // 16, 16).transpose(0, 2, 1, 3).reshape(-1)
    assert np.array_equal(p, ref)
