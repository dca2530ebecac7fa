"""The blend backward through stored gradient rows (hds_render_backward_rows), against the CPU oracle.

Where it can go wrong: list lengths around its groups of 16 gaussians and rounds of 32, frames that cut
8x8 blocks and tiles, every channel slicing, gaussians with more rows than are summed in one piece,
rows past the storage (added atomically by a second launch), and non-finite upstream gradients.
Tolerances are the suite's gradient bars (assert_grads_close).
"""
import numpy as np
import pytest
import torch

import oracle
from gaussian_splatting.rasterizer import _get_rasterizer
from tests.scenes import flat_scene
from tests.tolerances import assert_grads_close

pytestmark = pytest.mark.gpu

DEV = "cuda"
NAMES = ("means2D", "conics", "colors", "opacities", "features")


def np_(t):
    return None if t is None else t.detach().cpu().numpy()


def random_scene(seed, n, width, height, sigma=(0.6, 4.0)):
    g = torch.Generator().manual_seed(seed)
    rand = lambda *s: torch.rand(*s, generator=g)  # noqa: E731
    means = (rand(n, 2) * torch.tensor([width + 8.0, height + 8.0]) - 4.0).tolist()
    sig = (sigma[0] + (sigma[1] - sigma[0]) * rand(n)).tolist()
    return flat_scene(means, (1 + rand(n)).tolist(), sig, (0.02 + 0.9 * rand(n)).tolist(), device=DEV)


def backward_both(inputs, width, height, channels, rgb=True, want_features=True, slice_width=None, grads=None):
    """(GPU gradients, oracle gradients) of one frame, each (means2D, conics, colors, opacities, features)."""
    m2, d, r, c, col, op = inputs
    n = m2.shape[0]
    g = torch.Generator().manual_seed(7)
    bg = torch.tensor([0.2, 0.6, 0.4], device=DEV)
    feats = torch.randn(n, channels, generator=g).to(DEV) if channels else None
    gi = torch.randn(height, width, 3, generator=g).to(DEV)
    gf = torch.randn(height, width, channels, generator=g).to(DEV) if channels else None
    if grads is not None:
        gi, gf = grads(gi, gf)
    ext = _get_rasterizer()
    values, ranges, conic4, color4 = ext.bin(m2, d, r, c, col, op, width, height)
    _, _, T, nc = ext.render(m2, conic4, color4, values, ranges, width, height, bg, feats)
    got = ext.render_backward(m2, conic4, color4, values, ranges, T, nc, width, height, grad_image=gi if rgb else None,
                              background=bg, features=feats, grad_feature_image=gf, slice_width=slice_width,
                              want_feature_grad=want_features)
    o = [np_(t) for t in (m2, c, op, col)]
    want = oracle.render_backward(width, height, np_(ranges), np_(values), *o, np_(bg), np_(T), np_(nc),
                                  np_(gi if rgb else torch.zeros_like(gi)), np_(feats), np_(gf))
    return [np_(t) for t in got], want


def compare(got, want, names=NAMES):
    kept = [(n, a, b) for n, a, b in zip(names, got, want) if a is not None]
    assert_grads_close([k[0] for k in kept], [k[1] for k in kept], [np.asarray(k[2]).reshape(k[1].shape) for k in kept])


@pytest.mark.parametrize("n", [1, 15, 16, 17, 31, 32, 33, 65, 300])
def test_list_lengths_around_groups_and_rounds(n):
    """n gaussians that all reach one block (sigma 3 about its centre): one list of n entries."""
    g = torch.Generator().manual_seed(n)
    centre = (torch.tensor([12.0, 12.0]) + 2 * torch.rand(n, 2, generator=g)).tolist()
    inputs = flat_scene(centre, (1 + torch.rand(n, generator=g)).tolist(), [3.0] * n,
                        (0.02 + 0.1 * torch.rand(n, generator=g)).tolist(), device=DEV)
    got, want = backward_both(inputs, 24, 24, 32)
    compare(got, want)


@pytest.mark.parametrize("channels,slice_width", [(0, None), (32, 32), (64, 32), (64, 64), (128, 128), (256, 128), (512, 64)])
@pytest.mark.parametrize("width,height", [(8, 8), (33, 7), (61, 45)])
def test_frames_that_cut_blocks_and_every_slicing(channels, slice_width, width, height):
    inputs = random_scene(width, 400, width, height)
    got, want = backward_both(inputs, width, height, channels, slice_width=slice_width)
    compare(got, want)


@pytest.mark.parametrize("rgb,want_features", [(False, True), (False, False), (True, False)])
@pytest.mark.parametrize("channels", [32, 64, 128])
def test_features_alone_and_frozen_features(rgb, want_features, channels):
    got, want = backward_both(random_scene(3, 500, 50, 40), 50, 40, channels, rgb=rgb, want_features=want_features)
    assert (got[2] is None) == (not rgb) and (got[4] is None) == (not want_features)
    compare(got, want)


@pytest.mark.parametrize("channels", [0, 64, 256])
def test_gaussians_with_more_rows_than_one_piece(channels):
    """A few gaussians over all 256 blocks of the frame (more than 64 rows each) among small ones."""
    width = height = 128
    small = random_scene(5, 300, width, height)
    big = flat_scene([[40.0, 60.0], [90.0, 70.0], [64.0, 64.0]], [0.5, 0.6, 3.0], [60.0, 70.0, 80.0], [0.05, 0.04, 0.5], device=DEV)
    inputs = tuple(torch.cat([a, b]).contiguous() for a, b in zip(big, small))
    got, want = backward_both(inputs, width, height, channels)
    compare(got, want)


@pytest.mark.parametrize("channels", [0, 32, 128])
@pytest.mark.parametrize("stored", [0, 100, 1000])
def test_rows_past_the_storage_are_added_atomically(channels, stored, monkeypatch):
    ext = _get_rasterizer()
    monkeypatch.setattr(ext, "ROWS_MAX_BYTES", stored * (4 * channels + 64))
    got, want = backward_both(random_scene(9, 1500, 96, 80), 96, 80, channels)
    compare(got, want)


def test_a_second_call_gives_the_same_gradients():
    """Nothing is left in the workspace's memory that a later call would add to."""
    inputs = random_scene(2, 800, 64, 64)
    first, want = backward_both(inputs, 64, 64, 128)
    second, _ = backward_both(inputs, 64, 64, 128)
    compare(first, want)
    compare(second, want)


@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_a_non_finite_pixel_gradient_reaches_only_the_gaussians_it_sees(value):
    """One pixel's dL/dRGB is not finite: the geometry gradients of gaussians that do not touch that pixel's block
    are the oracle's, and those of gaussians in the block that do not contribute to the pixel stay finite."""
    width = height = 32
    # The third gaussian reaches 0.5 sqrt(2 ln(255 * 0.6)) = 1.6 pixels, so one block: its gradient is a single row, the
    # same bits in both runs (the rows of several tiles are summed in the order they were counted in).
    inputs = flat_scene([[3.5, 3.5], [6.5, 6.5], [20.0, 20.0]], [1.0, 2.0, 3.0], [0.5, 0.5, 0.5], [0.8, 0.7, 0.6], device=DEV)

    def poison(gi, gf):
        gi = gi.clone()
        gi[3, 3, 0] = value
        return gi, gf

    got, _ = backward_both(inputs, width, height, 0, grads=poison)
    clean, want = backward_both(inputs, width, height, 0)
    compare(clean, want)
    for k in (0, 1, 3):
        assert np.isfinite(got[k][1:]).all(), NAMES[k]
        np.testing.assert_array_equal(got[k][2], clean[k][2])


@pytest.mark.parametrize("width,height,n", [(8, 8, 40), (33, 7, 300), (61, 45, 900), (16, 16, 3000)])
def test_marks_of_the_render(width, height, n):
    """The render marks what blends into each block, and the backward gives the oracle's gradients from the marks."""
    m2, d, r, c, col, op = random_scene(n, n, width, height)
    bg = torch.tensor([0.2, 0.6, 0.4], device=DEV)
    g = torch.Generator().manual_seed(3)
    feats = torch.randn(n, 32, generator=g).to(DEV)
    gi, gf = torch.randn(height, width, 3, generator=g).to(DEV), torch.randn(height, width, 32, generator=g).to(DEV)
    ext = _get_rasterizer()
    values, ranges, conic4, color4 = ext.bin(m2, d, r, c, col, op, width, height)
    plain = ext.render(m2, conic4, color4, values, ranges, width, height, bg, feats)
    marks = torch.full((4 * values.numel(),), 7, device=DEV, dtype=torch.uint8)
    image, fimg, T, nc = ext.render(m2, conic4, color4, values, ranges, width, height, bg, feats, contributes=marks)
    for a, b in zip(plain, (image, fimg, T, nc)):
        assert torch.equal(a, b)
    marked, lists, tiles, last = np_(marks), np_(values), np_(ranges), np_(nc)
    mean, con, opac = (np_(t).astype(np.float64) for t in (m2, c, op))
    tiles_x = (width + 15) // 16
    for t, (begin, end) in enumerate(tiles):
        gids = lists[begin:end]
        for b in range(4):
            x0, y0 = t % tiles_x * 16 + b % 2 * 8, t // tiles_x * 16 + b // 2 * 8
            if x0 >= width or y0 >= height:
                continue
            ys, xs = np.mgrid[y0:min(y0 + 8, height), x0:min(x0 + 8, width)]
            dx, dy = xs.ravel() + 0.5 - mean[gids, :1], ys.ravel() + 0.5 - mean[gids, 1:]
            alpha = opac[gids] * np.exp(-0.5 * (con[gids, :1] * dx * dx + 2 * con[gids, 1:2] * dx * dy + con[gids, 2:] * dy * dy))
            walked = np.arange(len(gids))[:, None] < last[y0:y0 + 8, x0:x0 + 8].ravel()
            # Away from 1/255 by more than the rounding of alpha (a few ulp of the exponent's argument).
            sure = (walked & (alpha > 1.0001 / 255)).any(1)
            never = ~(walked & (alpha > 0.9999 / 255)).any(1)
            deepest = int(last[y0:y0 + 8, x0:x0 + 8].max())
            got = marked[4 * begin + b * len(gids):][:deepest]
            assert (got <= 1).all() and (got[sure[:deepest]] == 1).all() and (got[never[:deepest]] == 0).all()
    got = ext.render_backward(m2, conic4, color4, values, ranges, T, nc, width, height, grad_image=gi, background=bg,
                              features=feats, grad_feature_image=gf, contributes=marks)
    want = oracle.render_backward(width, height, tiles, lists, *[np_(t) for t in (m2, c, op, col)], np_(bg), np_(T), last,
                                  np_(gi), np_(feats), np_(gf))
    compare([np_(t) for t in got], want)
