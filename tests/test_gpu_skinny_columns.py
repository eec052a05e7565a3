"""Small M on a quarter, half or whole 64-column panel per workgroup: an output
is the same sum in the same order whichever its workgroup's width, so the first
columns of a wide weight (whole panels) and a narrow weight of those columns
agree bit for bit, with E4M3 and with fp32 activations, for each way that the
fused quantiser holds its activations; and the wide one matches the oracle."""
import numpy as np
import pytest
import torch

import oracle
from luisaml_amd import capi, synth

from .gemm_cases import assert_close

pytestmark = pytest.mark.gpu

WIDE = 8256  # 129 panels


# K: one block per wavefront and fewer, 4 and 8 slots, 16 slots, more
@pytest.mark.parametrize("M,K", [(1, 16), (1, 4096), (2, 4112), (1, 11008), (1, 16384), (2, 8192), (4, 4096), (5, 528),
                                 (7, 1040), (16, 1024), (16, 2320)])
@pytest.mark.parametrize("kernel", [capi.KERNEL_SKINNY, capi.KERNEL_SKINNY_FP8, capi.KERNEL_AUTO])
def test_columns_agree(dev, M, K, kernel):
    x = synth.normal(M + K, (M, K))
    w = synth.normal(K, (K, WIDE), std=0.05)
    sw = oracle.channel_scales(w, axis=1)
    qw = oracle.quantize(w, sw, axis=1)
    bias = synth.normal(3, (WIDE,), std=0.01)
    dx = torch.from_numpy(x).to(dev)
    qx, sx = capi.quantize_dynamic(dx)
    full = {}
    for n in (WIDE, 8192, 4098, 4096, 1000, 17, 16, 1):
        bp = capi.pack_weight(torch.from_numpy(np.ascontiguousarray(qw[:, :n])).to(dev), False)
        args = (bp, torch.from_numpy(sw[:n].copy()).to(dev), n, K)
        kw = dict(c=torch.from_numpy(bias[:n].copy()).to(dev), act=capi.ACT_RELU, kernel=kernel)
        for name, y in (("gemm", capi.gemm(qx, sx, *args, **kw)), ("dynamic", capi.gemm_dynamic(dx, *args, **kw))):
            y = y.cpu().numpy()
            if n == WIDE:
                full[name] = y
            assert np.array_equal(y, full[name][:, :n]), (name, n)
    assert np.array_equal(full["gemm"], full["dynamic"])
    if kernel != capi.KERNEL_SKINNY_FP8:
        s = oracle.dynamic_scale(x)
        ref, A, B = oracle.qlinear(oracle.quantize(x, s), s, qw, sw, bias=bias, act=oracle.ACT_RELU)
        assert_close(full["gemm"], ref, oracle.gemm_abs_bound(A, B, bias))


@pytest.mark.parametrize("N,K,part", [(64, 1024, False), (4096, 2048, False), (4096, 2064, True), (4097, 16, True), (8192, 1024, True),
                                      (8193, 4096, False)])
@pytest.mark.parametrize("M", [1, 16])
def test_part_panels(dev, M, N, K, part):
    """Quarters of a panel for a long K only, halves for 65 to 128 panels."""
    a = torch.zeros((M, K), dtype=torch.uint8, device=dev)
    bp = torch.zeros(capi.packed_weight_bytes(K, N), dtype=torch.uint8, device=dev)
    one = torch.ones(1, device=dev)
    capi.kernel_trace()
    y = capi.gemm(a, one, bp, one, N, K)
    assert capi.kernel_trace() == ["gemm_skinny_part" if part else "gemm_skinny"]
    assert bool((y == 0).all())
