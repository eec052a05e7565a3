"""The fp32 Gemm and convolution on the fp32 matrix instruction: every output
is the oracle's sequential fma chain, bit for bit (the order and the single
rounding per product leave no tolerance), at the edges of the tiles, of the
16-k groups and of the staged parts, in every operand layout, aligned or not."""
import numpy as np
import pytest
import torch

import oracle
from luisaml_amd import capi, synth

pytestmark = pytest.mark.gpu


def place(a, dev, pitch, shift):
    """a on the device as rows of `pitch` elements, `shift` elements into its buffer."""
    buf = torch.zeros(shift + a.shape[0] * pitch, dtype=torch.float32, device=dev)
    v = buf[shift:].view(a.shape[0], pitch)
    v[:, :a.shape[1]] = torch.from_numpy(a).to(dev)
    return buf, v


def sgemm(dev, a, b, ta, tb, bias, pad, shift):
    M, K = (a.shape[1], a.shape[0]) if ta else a.shape
    N = b.shape[0] if tb else b.shape[1]
    _, va = place(a, dev, a.shape[1] + pad, shift)
    _, vb = place(b, dev, b.shape[1] + pad, shift)
    c = torch.from_numpy(bias).to(dev)
    y = torch.full((M, N), 7.0, dtype=torch.float32, device=dev)
    capi._check(capi.lib().lcml_fp8_sgemm(M, N, K, va.data_ptr(), va.stride(0), int(ta), vb.data_ptr(), vb.stride(0),
                                          int(tb), 1.0, c.data_ptr(), 1, N, 0, 1.0, capi.ACT_RELU, y.data_ptr(),
                                          capi.DTYPE_FLOAT, N, capi._stream()))
    return y.cpu().numpy()


# 16-row tiles, 32-row tiles (more than 256 of the smaller ones), 64-row
# tiles; K at the edges of a 4-k step, a 16-k group and a chunk
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (16, 40, 129), (17, 1000, 300), (130, 560, 64), (515, 530, 67),
                                   (1030, 1028, 36), (1024, 1100, 33)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("pad,shift", [(0, 0), (4, 4), (3, 1)])
def test_sgemm_is_the_fma_chain(dev, M, N, K, ta, tb, pad, shift):
    a = synth.normal(M + K, (K, M) if ta else (M, K))
    b = synth.normal(N + K, (N, K) if tb else (K, N))
    bias = synth.normal(3, (N,))
    ref = oracle.gemm(a, b, bias, transA=ta, transB=tb, act=oracle.ACT_RELU)
    assert np.array_equal(sgemm(dev, a, b, ta, tb, bias, pad, shift), ref)


@pytest.mark.parametrize("tb", [0, 1])
def test_sgemm_infinities_stay_in_their_row(dev, tb):
    """K and the tiles are padded inside: nothing but row 3 meets the infinity."""
    M, N, K = 20, 50, 77
    a, b = synth.normal(1, (M, K)), synth.normal(2, (N, K) if tb else (K, N))
    a[3, K - 1] = np.inf
    bias = np.zeros(N, np.float32)
    ref = oracle.gemm(a, b, bias, transB=tb, act=oracle.ACT_RELU)
    assert np.array_equal(sgemm(dev, a, b, 0, tb, bias, 0, 0), ref, equal_nan=True)


# few k, also with many outputs, take the general kernel; either side of the lines
@pytest.mark.parametrize("M,N,K,general", [(1, 1, 1, True), (59, 1, 1, True), (70, 130, 6, True), (70, 130, 7, False),
                                           (723, 725, 7, False), (725, 724, 10, True), (725, 724, 11, False)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_sgemm_few_k(dev, M, N, K, general, ta, tb):
    a, b = synth.normal(M + K, (K, M) if ta else (M, K)), synth.normal(N + K, (N, K) if tb else (K, N))
    bias = synth.normal(3, (N,))
    capi.kernel_trace()
    y = sgemm(dev, a, b, ta, tb, bias, 0, 0)
    assert capi.kernel_trace() == ["lcml_fp8_sgemm_any" if general else "lcml_fp8_sgemm"]
    assert np.array_equal(y, oracle.gemm(a, b, bias, transA=ta, transB=tb, act=oracle.ACT_RELU))


def test_sgemm_more_tiles_than_a_grid(dev):
    """One row by 2^29 columns: more tiles than one grid dimension has workgroups."""
    N, K = (1 << 29) + 5, 25
    b = torch.empty((N, K), device=dev).normal_(generator=torch.Generator(device=dev).manual_seed(3))
    a = synth.normal(1, (1, K))
    da, y = torch.from_numpy(a).to(dev), torch.full((1, N), np.nan, device=dev)
    capi._check(capi.lib().lcml_fp8_sgemm(1, N, K, da.data_ptr(), K, 0, b.data_ptr(), K, 1, 1.0, None, 0, 0, 0, 0.0,
                                          capi.ACT_NONE, y.data_ptr(), capi.DTYPE_FLOAT, N, capi._stream()))
    assert not bool(torch.isnan(y).any())
    for at in (slice(0, 999), slice((1 << 29) - 500, N)):
        assert np.array_equal(y[:, at].cpu().numpy(), oracle.gemm(a, b[at].cpu().numpy(), transB=1))


# n, c, h, w, cout, kh, kw, stride, pad, dilation, group: one, two and four
# 16-channel blocks with and without a remainder, one and two pixels per lane
# (few and many pixels, odd planes), K of one part (160), just over it and
# several, images of fewer pixels than a wavefront, the direct kernel (fewer
# than four channels per group)
CONVS = [(1, 3, 28, 28, 8, 3, 3, 1, 1, 1, 1), (2, 3, 61, 57, 64, 7, 7, 2, 3, 1, 1), (9, 3, 119, 121, 24, 5, 5, 1, 2, 1, 1),
         (16, 1, 90, 90, 10, 3, 3, 1, 1, 1, 1), (2, 20, 31, 29, 37, 3, 3, 1, 1, 1, 1), (1, 20, 30, 31, 70, 7, 7, 2, 1, 1, 1),
         (3, 18, 3, 3, 130, 3, 3, 1, 1, 1, 1), (40, 32, 40, 41, 64, 1, 1, 1, 0, 1, 2), (2, 12, 33, 35, 24, 3, 3, 1, 2, 2, 3),
         (2, 16, 21, 20, 16, 3, 3, 1, 1, 1, 16)]


@pytest.mark.parametrize("case", CONVS)
@pytest.mark.parametrize("weight", [None, np.inf, np.nan])
def test_conv_f32_is_the_fma_chain(dev, case, weight):
    """A weight that is not finite meets no padding tap: the reference skips those."""
    n, c, h, w, cout, kh, kw, st, pd, dl, group = case
    x = synth.normal(c + h, (n, c, h, w))
    wt = synth.normal(cout + kh, (cout, c // group, kh, kw), std=0.2)
    if weight is not None:
        wt[cout // 2, -1, -1, 0] = weight
    b = synth.normal(3, (cout,), std=0.1)
    y = capi.conv2d_f32(torch.from_numpy(x).to(dev), torch.from_numpy(wt).to(dev), torch.from_numpy(b).to(dev),
                        (st, st), (pd, pd), (dl, dl), group, act=capi.ACT_RELU)
    ref = oracle.conv2d(x, wt, b, strides=(st, st), pads=(pd, pd), dilations=(dl, dl), group=group, act=oracle.ACT_RELU)
    assert np.array_equal(y.cpu().numpy(), ref, equal_nan=True)


def test_conv_f32_many_small_images(dev):
    """More images than one grid dimension has workgroups: every output is written."""
    n, c, cout = (1 << 24) + 3, 4, 4
    x = torch.randn(n, c, 1, 1, device=dev, generator=torch.Generator(device=dev).manual_seed(5))
    wt = synth.normal(1, (cout, c, 1, 1))
    w = torch.from_numpy(wt).to(dev)
    y = torch.full((n, cout, 1, 1), np.nan, device=dev)
    capi._check(capi.lib().lcml_fp8_conv2d_f32(x.data_ptr(), w.data_ptr(), None, y.data_ptr(), n, c, 1, 1, cout, 1, 1, 1, 1,
                                               0, 0, 1, 1, 1, 1, 1, capi.ACT_NONE, capi._stream()))
    assert not bool(torch.isnan(y).any())
    for at in (slice(0, 999), slice((1 << 24) - 500, n)):
        assert np.array_equal(y[at].cpu().numpy(), oracle.conv2d(x[at].cpu().numpy(), wt, np.zeros(cout, np.float32)))


def test_conv_f32_more_outputs_than_a_grid(dev):
    """2^32 outputs and more of the direct kernel (fewer than four channels a group)."""
    n, cout = (1 << 31) // 3 + 7, 6
    x = torch.empty((n, 3, 1, 1), device=dev).normal_(generator=torch.Generator(device=dev).manual_seed(6))
    wt = synth.normal(2, (cout, 1, 1, 1))
    w = torch.from_numpy(wt).to(dev)
    y = torch.full((n, cout, 1, 1), np.nan, device=dev)
    capi._check(capi.lib().lcml_fp8_conv2d_f32(x.data_ptr(), w.data_ptr(), None, y.data_ptr(), n, 3, 1, 1, cout, 1, 1, 1, 1,
                                               0, 0, 1, 1, 3, 1, 1, capi.ACT_NONE, capi._stream()))
    assert y.numel() > 1 << 32 and not bool(torch.isnan(y.view(-1)[-1000:]).any())
    for at in (slice(0, 999), slice((1 << 32) // cout - 500, (1 << 32) // cout + 7), slice(n - 500, n)):
        assert np.array_equal(y[at].cpu().numpy(), oracle.conv2d(x[at].cpu().numpy(), wt, np.zeros(cout, np.float32), group=3))


# the choice of the kernel: small planes, single pixels, taps that mostly lie
# in the padding and few products go to the direct kernel, the rest by their
# channels and K to the other two
@pytest.mark.parametrize("case,kernel", [((512, 16, 1, 1, 24, 1, 1, 1, 0, 1, 1), "direct"), ((300, 8, 4, 4, 9, 1, 1, 1, 0, 1, 1), "direct"),
                                         ((40, 20, 1, 1, 20, 7, 7, 1, 3, 1, 1), "direct"), ((200, 12, 2, 2, 40, 3, 3, 1, 1, 1, 2), "direct"),
                                         ((2, 30, 10, 10, 48, 1, 1, 1, 0, 1, 2), "direct"), ((3, 2, 30, 30, 3, 3, 3, 1, 1, 1, 1), "direct"),
                                         ((4, 3, 57, 58, 40, 3, 3, 1, 1, 1, 1), "patch"), ((2, 24, 20, 21, 12, 3, 3, 1, 1, 1, 1), "mfma"),
                                         ((1, 60, 4, 4, 70, 5, 5, 1, 2, 1, 1), "mfma")])
def test_conv_f32_kernel(dev, case, kernel):
    n, c, h, w, cout, kh, kw, st, pd, dl, group = case
    x, b = synth.normal(c + h, (n, c, h, w)), synth.normal(3, (cout,), std=0.1)
    wt = synth.normal(cout + kh, (cout, c // group, kh, kw), std=0.2)
    capi.kernel_trace()
    y = capi.conv2d_f32(torch.from_numpy(x).to(dev), torch.from_numpy(wt).to(dev), torch.from_numpy(b).to(dev),
                        (st, st), (pd, pd), (dl, dl), group, act=capi.ACT_RELU)
    assert capi.kernel_trace() == ["conv2d_f32_" + kernel]
    ref = oracle.conv2d(x, wt, b, strides=(st, st), pads=(pd, pd), dilations=(dl, dl), group=group, act=oracle.ACT_RELU)
    assert np.array_equal(y.cpu().numpy(), ref)
