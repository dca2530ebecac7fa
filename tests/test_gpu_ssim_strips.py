"""SSIM kernels at the edges of their strips of 64 channel elements: rows shorter than a strip, a last strip of a
few elements, fewer image rows than the window, and heights that leave a short last part of a strip."""
import numpy as np
import pytest
import torch

import oracle
from gaussian_splatting.rasterizer import _get_rasterizer

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("height,width", [(1, 1), (2, 5), (3, 21), (5, 22), (9, 43), (1, 500), (700, 1), (13, 128), (131, 75),
                                          (257, 320)])
def test_ssim_at_strip_edges(height, width):
    g = torch.Generator().manual_seed(1000 * height + width)
    gt = torch.rand(height, width, 3, generator=g)
    rendered = (gt + 0.1 * torch.randn(height, width, 3, generator=g)).clamp(0, 1)
    ext = _get_rasterizer()
    got = ext.ssim_forward(rendered.to(DEV), gt.to(DEV))
    want = oracle.ssim_forward(rendered.numpy(), gt.numpy())
    # The forward rounds every product and sum as the oracle does.
    for name, a, b in zip(("map", "d_mu", "d_aa", "d_ab"), got, want):
        np.testing.assert_allclose(a.cpu().numpy(), b, rtol=1e-6, atol=1e-7, err_msg=name)
    grad = ext.ssim_backward(torch.tensor([0.7], device=DEV), rendered.to(DEV), gt.to(DEV), *got[1:])
    want_grad = oracle.ssim_backward(0.7, rendered.numpy(), gt.numpy(), *want[1:])
    # 22 sums of two blurs in another order: 22 * 2^-24 of the sum of the terms' sizes, bounded per image.
    size = 0.7 / (3 * height * width) * sum(np.abs(w).max() * f for w, f in zip(want[1:], (1, 2, 1)))
    np.testing.assert_allclose(grad.cpu().numpy(), want_grad, rtol=0, atol=32 * 2.0 ** -24 * size)
