"""The blend forward at the edges of its groups, against the CPU oracle: numbers of hits around 4, 16 and the 64
entries tested together, blocks that few entries reach, pixels that stop inside a group, frames that cut blocks, colours
that are not finite, and a range cleared beside the walk."""
import numpy as np
import pytest
import torch

import oracle
from gaussian_splatting.rasterizer import _get_rasterizer
from tests.scenes import flat_scene

pytestmark = pytest.mark.gpu
DEV = "cuda"


def np_(t):
    return None if t is None else t.detach().cpu().numpy()


def forward_both(inputs, width, height, channels=0, clear=None):
    m2, d, r, c, col, op = inputs
    bg = torch.tensor([0.2, 0.6, 0.4], device=DEV)
    feats = torch.randn(m2.shape[0], channels, generator=torch.Generator().manual_seed(7)).to(DEV) if channels else None
    ext = _get_rasterizer()
    values, ranges, conic4, color4 = ext.bin(m2, d, r, c, col, op, width, height)
    image, fimg, T, nc = ext.render(m2, conic4, color4, values, ranges, width, height, bg, feats, clear=clear)
    o_image, o_T, o_nc, o_fimg = oracle.render_forward(width, height, np_(ranges), np_(values), np_(m2), np_(c), np_(op),
                                                       np_(col), np_(bg), np_(feats))
    return [np_(t) for t in (image, T, nc, fimg)], [o_image, o_T, o_nc, o_fimg], feats


def check(inputs, width, height, channels=0):
    got, want, feats = forward_both(inputs, width, height, channels)
    for name, a, b in zip(("image", "final_T", "n_contrib"), got, want):
        np.testing.assert_array_equal(a, b, err_msg=name)
    if channels:
        # Weights sum to at most 1; both operands carry 16 bits: 3 * 2^-16 of the largest feature.
        np.testing.assert_allclose(got[3], want[3], rtol=0, atol=3 * 2.0 ** -16 * float(feats.abs().max()))


@pytest.mark.parametrize("channels", [0, 32, 64, 128])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 15, 16, 17, 63, 64, 65, 79, 80, 81, 150])
def test_hits_around_groups_and_batches(n, channels):
    """n gaussians over one block, faint, so that every pixel blends the whole list."""
    g = torch.Generator().manual_seed(n)
    centre = (torch.tensor([12.0, 12.0]) + 2 * torch.rand(n, 2, generator=g)).tolist()
    check(flat_scene(centre, (1 + torch.rand(n, generator=g)).tolist(), [3.0] * n,
                     (0.005 + 0.02 * torch.rand(n, generator=g)).tolist(), device=DEV), 24, 24, channels)


@pytest.mark.parametrize("every", [2, 7, 40, 100])
def test_few_entries_reach_a_block(every):
    """A tile of 700 entries of which one in `every` lies in the first block and the rest in the last one."""
    g = torch.Generator().manual_seed(every)
    n = 700
    centre = torch.where((torch.arange(n) % every == 0)[:, None], torch.tensor([4.0, 4.0]), torch.tensor([12.0, 12.0]))
    check(flat_scene((centre + torch.rand(n, 2, generator=g)).tolist(), (1 + torch.arange(n) / n).tolist(), [0.8] * n,
                     (0.005 + 0.05 * torch.rand(n, generator=g)).tolist(), device=DEV), 16, 16, 32)


@pytest.mark.parametrize("channels", [0, 128, 512])
@pytest.mark.parametrize("width,height", [(8, 8), (9, 3), (50, 41)])
def test_pixels_stop_inside_a_group(width, height, channels):
    g = torch.Generator().manual_seed(width)
    n = 600
    rand = lambda *s: torch.rand(*s, generator=g)  # noqa: E731
    check(flat_scene((rand(n, 2) * torch.tensor([width, height])).tolist(), (1 + rand(n)).tolist(), (0.7 + 4 * rand(n)).tolist(),
                     (0.05 + 0.94 * rand(n)).tolist(), device=DEV), width, height, channels)


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_a_colour_that_is_not_finite_reaches_only_its_pixels(value):
    """A pixel that the gaussian does not blend into keeps its colour, in a block that the gaussian reaches."""
    inputs = list(flat_scene([[2.0, 2.0], [4.0, 4.0], [5.0, 3.0]], [1.0, 2.0, 3.0], [0.6, 3.0, 2.0], [0.9, 0.5, 0.4], device=DEV))
    inputs[4][0, 1] = value
    got, want, _ = forward_both(inputs, 8, 8)
    np.testing.assert_array_equal(got[0], want[0])
    assert not np.isfinite(got[0][2, 2, 1]) and np.isfinite(got[0][6, 6]).all() and np.isfinite(got[0][..., [0, 2]]).all()


@pytest.mark.parametrize("words", [4, 1024, 4 * 255, 4 * 257, 100_004])
def test_cleared_range(words):
    buf = torch.full((words + 8,), 3.0, device=DEV)
    inputs = flat_scene([[5.0, 5.0]], [1.0], [2.0], [0.5], device=DEV)
    forward_both(inputs, 70, 20, 32, clear=buf[4:4 + words])
    assert (buf[4:4 + words] == 0).all() and (buf[:4] == 3).all() and (buf[4 + words:] == 3).all()
