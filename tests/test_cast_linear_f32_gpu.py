"""cast_linear's one-call form (fp32 rows cast in the same entry) gives the
bits of the separate casts for every layout: odd row counts, both weight
layouts, with and without bias, values outside the 16-bit range, infinities
and NaN, rows that are a view at an unaligned address (which take the separate
casts), rows in another type and lazily negated views."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", [(1, 32, 64), (16, 96, 192), (17, 128, 128), (179, 320, 640)])
def test_one_call_equals_separate_casts(dev, dtype, M, N, K):
    from hackathon_amd import kernels as hk

    g = torch.Generator(device=dev).manual_seed(M + K)
    w = ((torch.rand(N, K, generator=g, device=dev) * 2 - 1) * K ** -0.5).to(dtype)
    b = torch.rand(N, generator=g, device=dev).to(dtype)
    x = torch.randn(M, K, generator=g, device=dev)
    special = x.clone()
    special[0, :6] = torch.tensor([1e30, -1e30, float("inf"), float("-inf"), float("nan"), 1e-30])
    buf = torch.empty(M * K + 1, device=dev)
    shifted = buf[1:].view(M, K).copy_(x)
    packed = hk.pack_cast_weight(w)
    for bias in (None, b):
        for weight, p in ((w, False), (packed, True)):
            for rows in (x, special):
                # float64 rows hold the same values and take the separate casts
                want = hk.cast_linear(rows.double(), weight, bias, packed=p)
                assert torch.equal(hk.cast_linear(rows, weight, bias, packed=p).nan_to_num(),
                                   want.nan_to_num())
            want = hk.cast_linear(x, weight, bias, packed=p)
            assert torch.equal(hk.cast_linear(shifted, weight, bias, packed=p), want)
            assert torch.equal(hk.cast_linear(x.view(1, M, K), weight, bias, packed=p)[0], want)
    want = hk.cast_linear(-x, w, -b)
    assert torch.equal(hk.cast_linear(torch._neg_view(x), w, -b), want)
    assert torch.equal(hk.cast_linear(-x, w, torch._neg_view(b)), want)
