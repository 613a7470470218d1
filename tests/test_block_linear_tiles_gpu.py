"""BlockLinear at the edges of its kernels' dispatch (hk_block_linear): row
counts around the 16-row kernel (16, 17), every tile of the short-K kernel
(few to many rows, rows and columns past the last tile, K below one step per
wave), both sides of the line where the 64x64-tile kernel takes over and of
the lines where 64-row tiles would be more than one to a CU, against float64. Bound: a sum of K products in fp32 in any order is within
K * 2^-24 * sum |x w| of the exact one; sums split over waves stay within
sixteen rounding steps of it."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,blocks,bs", [
    (16, 4, 512), (17, 4, 512), (33, 4, 512), (64, 4, 512), (65, 4, 512), (129, 4, 512),
    (256, 4, 512), (321, 4, 512), (383, 4, 512), (385, 4, 512), (40, 16, 512), (200, 4, 256),
    (257, 4, 512), (257, 2, 512), (512, 4, 256), (513, 4, 256), (577, 2, 256), (1100, 1, 256), (145, 1, 512),
    (257, 1, 512), (500, 4, 128), (70, 3, 48), (19, 1, 16), (100, 1, 80), (31, 2, 528)])
def test_block_linear_tiles(dev, rows, blocks, bs):
    from hackathon_amd import kernels as hk

    g = torch.Generator(device=dev).manual_seed(rows * bs)
    x = torch.randn(rows, blocks * bs, generator=g, device=dev)
    w = (torch.rand(blocks, bs, bs, generator=g, device=dev) * 2 - 1) * bs ** -0.5
    b = torch.rand(blocks * bs, generator=g, device=dev)
    for bias in (None, b):
        got = hk.block_linear(x, w, bias).double().cpu()
        for k in range(blocks):
            s = slice(k * bs, (k + 1) * bs)
            xk, wk = x[:, s].double().cpu(), w[k].double().cpu()
            want, mag = xk @ wk.T, xk.abs() @ wk.abs().T
            if bias is not None:
                want, mag = want + b[s].double().cpu(), mag + b[s].double().cpu()
            assert bool(((got[:, s] - want).abs() <= 16 * 2.0 ** -24 * mag).all())
