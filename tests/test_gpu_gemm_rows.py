"""Medium M behind a dynamic quantisation: codes in 16-row blocks, read by the
kernel made for them, for each of its tile shapes and every remainder of the
rows, columns and K.  The route depends on sizes alone, so the kernel trace says
that it was taken; the scale is the oracle's, the sums are within its bound."""
import numpy as np
import pytest
import torch

import oracle
from luisaml_amd import capi, synth

from .gemm_cases import assert_close

pytestmark = pytest.mark.gpu


ROWS_CASES = [(17, 1000, 1040), (32, 4096, 1040), (33, 2049, 2064), (47, 4100, 1168), (50, 6001, 1024), (63, 4096, 4112),
              (64, 3000, 1936), (100, 4099, 2064), (100, 11008, 2048), (113, 12290, 2192), (129, 4096, 2064),
              (200, 2050, 4096), (200, 4096, 2064), (250, 4096, 4112), (340, 4090, 2064), (384, 4096, 4096)]


def case(dev, M, N, K):
    x = synth.normal(M + K, (M, K))
    x[M - 1, K - 1] = 7.0  # the last row of the last block sets the scale
    w = synth.normal(N, (K, N), std=0.05)
    sw = oracle.channel_scales(w, axis=1)
    qw = oracle.quantize(w, sw, axis=1)
    bias = synth.normal(3, (N,), std=0.01)
    bp = capi.pack_weight(torch.from_numpy(qw).to(dev), False)
    s = oracle.dynamic_scale(x)
    ref, A, B = oracle.qlinear(oracle.quantize(x, s), s, qw, sw, bias=bias, act=oracle.ACT_RELU)
    return x, bp, sw, bias, s, ref, oracle.gemm_abs_bound(A, B, bias)


# 32x16 .. 96x64 tiles (by M and N), blocks of 1 to 16 rows at the end, odd N,
# K one chunk over a 64-k quad, a 128-k block and the 8 parts
@pytest.mark.parametrize("M,N,K", ROWS_CASES)
def test_rows_match_oracle(dev, M, N, K):
    x, bp, sw, bias, s, ref, bound = case(dev, M, N, K)
    capi.kernel_trace()
    sx = torch.empty(1, device=dev)
    y, _ = capi.gemm_dynamic_ex(torch.from_numpy(x).to(dev), bp, torch.from_numpy(sw).to(dev), N, K,
                                c=torch.from_numpy(bias).to(dev), act=capi.ACT_RELU, scale_out=sx)
    assert capi.kernel_trace() == ["amax_partials", "quantize_rows", "gemm_rows"]
    assert float(sx.item()) == s
    assert_close(y.cpu().numpy(), ref, bound)


def test_rows_partials_strides_and_alignment(dev):
    """Partial maxima in and out as the other kernels'; an x that is not 16-byte
    aligned keeps the row-major route; a row pitch of y above N; NaN and
    infinite activations as the standalone quantiser gives them."""
    M, N, K = 70, 2048, 1040
    x, bp, sw, bias, s, ref, bound = case(dev, M, N, K)
    d = [torch.from_numpy(v).to(dev) for v in (x, sw, bias)]
    xp, yp = capi.amax_parts_buffer(M, K, dev), capi.amax_parts_buffer(M, N, dev)
    xp.zero_()
    xp[:2] = torch.tensor([1.0, float(np.abs(x).max())]).view(torch.int32).to(dev)
    y, n = capi.gemm_dynamic_ex(d[0], bp, d[1], N, K, c=d[2], act=capi.ACT_RELU, x_amax=(xp, 2), y_amax_part=yp)
    assert_close(y.cpu().numpy(), ref, bound)
    assert yp[:n].cpu().view(torch.float32).max() == y.abs().max().cpu()
    wide = torch.full((M, N + 8), 5.0, device=dev)
    capi.gemm_dynamic(d[0], bp, d[1], N, K, c=d[2], act=capi.ACT_RELU, out=wide[:, :N])
    assert torch.equal(wide[:, :N], y) and bool((wide[:, N:] == 5.0).all())
    buf = torch.empty(M * K + 1, device=dev)
    buf[1:].copy_(d[0].reshape(-1))
    capi.kernel_trace()
    y1 = capi.gemm_dynamic(buf[1:].view(M, K), bp, d[1], N, K, c=d[2], act=capi.ACT_RELU)
    assert "gemm_rows" not in capi.kernel_trace()
    assert_close(y1.cpu().numpy(), ref, bound)
    for v in (np.nan, np.inf):
        x2 = x.copy()
        x2[69, 3] = v
        d2 = torch.from_numpy(x2).to(dev)
        q, s2 = capi.quantize_dynamic(d2)
        a = capi.gemm(q, s2, bp, d[1], N, K).cpu().numpy()
        b = capi.gemm_dynamic(d2, bp, d[1], N, K).cpu().numpy()
        assert np.array_equal(np.isnan(a), np.isnan(b))
        ok = ~np.isnan(a)
        assert np.allclose(a[ok], b[ok], rtol=1e-4, atol=1e-5 * np.abs(a[ok]).max())


# either side of the sizes where the row-major choice turns from the small-M
# kernel to the tiles, and sizes well inside either
@pytest.mark.parametrize("M,N,K", [(17, 1000, 1040), (64, 12288, 2048), (100, 4096, 2064), (100, 11008, 4096),
                                   (160, 11008, 2048), (161, 11008, 2048), (200, 11008, 4096), (512, 4096, 1024),
                                   (513, 4096, 1024), (600, 4096, 2048), (300, 8192, 1024), (180, 12288, 2048),
                                   (1100, 2048, 1024), (2100, 1024, 1024)])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
def test_one_call_equals_two(dev, M, N, K, out_dtype):
    """gemm_dynamic is quantize_dynamic followed by gemm bit for bit, whatever
    kernels either takes, and whether or not x is 16-byte aligned."""
    g = torch.Generator(device=dev).manual_seed(M + N)
    buf = torch.empty(M * K + 1, device=dev).normal_(generator=g)
    x, xm = buf[:M * K].view(M, K), buf[1:].view(M, K)
    q = torch.empty((N, K), device=dev).normal_(0.0, 0.05, generator=g)
    bp = capi.pack_weight(capi.quantize(q, torch.full((1,), 2.0 ** -11, device=dev)), True)
    sw = torch.empty(N, device=dev).uniform_(1e-4, 1e-3, generator=g)
    kw = dict(c=torch.empty(N, device=dev).normal_(generator=g), act=capi.ACT_GELU_ERF, out_dtype=out_dtype)
    for v in (x, xm):
        codes, s = capi.quantize_dynamic(v)
        two = capi.gemm(codes, s, bp, sw, N, K, **kw)
        assert torch.equal(capi.gemm_dynamic(v, bp, sw, N, K, **kw), two)


# either side of what the choice counts: the second launch for a small x, and a
# short K under few rows of many panels
@pytest.mark.parametrize("M,N,K,rows", [(32, 8192, 512, False), (65, 4096, 512, False), (100, 4096, 1024, True), (17, 8192, 3072, False),
                                        (17, 8192, 4096, True), (32, 8128, 2048, True), (33, 8192, 2048, True), (200, 11008, 4096, False)])
def test_rows_choice(dev, M, N, K, rows):
    x = torch.ones((M, K), device=dev)
    bp = torch.zeros(capi.packed_weight_bytes(K, N), dtype=torch.uint8, device=dev)
    capi.kernel_trace()
    y = capi.gemm_dynamic(x, bp, torch.ones(N, device=dev), N, K)
    assert ("gemm_rows" in capi.kernel_trace()) == rows
    assert bool((y == 0).all())
