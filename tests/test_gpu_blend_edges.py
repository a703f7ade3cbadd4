"""The blend kernels against the oracle where their tests and their exponential
change regime: opacities at and beyond the representable range, exponents past
the end of the exponential, centres on pixel centres and conics that are not
positive definite."""

import numpy as np
import pytest
import torch

import oracle
from oracle_pipeline import check_gradient
from dsl_splat_amd.gs3d import render as grender
from dsl_splat_amd.runtime import native
from test_gpu_stages import assert_two_pixels

pytestmark = pytest.mark.gpu

DEV = "cuda"

OPACITIES = [float("nan"), float("inf"), 3.0e38, 1.4e36, 1.3e36, 2.0, 1.0, 0.99, 0.5, 0.0040, 0.0039, 1e-30, 0.0,
             -0.0, -1.0]


def _np(t):
    return t.detach().cpu().numpy()


def _lists(n, width, height, per_tile, g):
    """Tile lists that are not derived from footprints: each tile lists
    `per_tile` Gaussians, most of them far outside it.  Frames of 1300x1300
    stand for the two-pixel kernels."""
    if (width, height) == (1300, 1300):
        assert_two_pixels(width, height)
    tiles = ((width + 15) // 16) * ((height + 15) // 16)
    ids = torch.stack([torch.randperm(n, generator=g)[:per_tile] for _ in range(tiles)]).int().flatten()
    first = torch.arange(tiles, dtype=torch.int32) * per_tile
    return ids.to(DEV), torch.stack([first, first + per_tile], 1).to(DEV)


def _scene(width, height, n, channels, extreme):
    g = torch.Generator().manual_seed(31)
    centers = torch.rand((1, n, 2), generator=g) * torch.tensor([width, height])
    centers[:, ::3] = centers[:, ::3].round()              # on pixel centres: zero exponents
    a, c = (torch.exp(torch.rand(n, generator=g) * 7 - 5) for _ in range(2))
    b = (torch.rand(n, generator=g) * 2 - 1) * (a * c).sqrt() * 0.98
    conics = torch.stack([a, b, c, torch.rand(n, generator=g)], 1)[None]
    if extreme:
        values = torch.tensor(OPACITIES)
        conics[0, :, 3] = torch.where(torch.rand(n, generator=g) < 0.25,
                                      values[torch.randint(0, len(values), (n,), generator=g)], conics[0, :, 3])
        conics[0, 5::17, 0] *= -1.0                          # not positive definite
        conics[0, 6::17, :3] = 0.0
        conics[0, 7::17, 1] *= 3.0
        conics[0, 8::17, 2] = 3.3                            # exponents far past -86
        centers[0, 9::50] = -1.0e7
    return centers.to(DEV), conics.to(DEV), torch.randn((n, channels), generator=g).to(DEV), g


# Fewer than 6144 tiles: one pixel per lane; more: two.  Channels: every
# compiled width of the forward.
@pytest.mark.parametrize("width,height,channels", [(75, 43, 3), (75, 43, 7), (75, 43, 13), (75, 43, 18),
                                                   (75, 43, 34), (75, 43, 41), (75, 43, 60),
                                                   (1300, 1300, 3), (1300, 1300, 6)])
def test_forward_at_extreme_opacities(width, height, channels):
    print("forward extreme opacities", width, height, channels, flush=True)
    centers, conics, feats, g = _scene(width, height, 400, channels, extreme=True)
    ids, ranges = _lists(400, width, height, 150, g)
    out = grender.render_views(ranges, ids, centers, conics, feats, width, height)
    image, final_t, contributors = oracle.render_fwd(width, height, _np(ranges), _np(ids), _np(centers), _np(conics),
                                                     _np(feats))
    np.testing.assert_array_equal(_np(out.contributors), contributors)
    np.testing.assert_array_equal(_np(out.transmittance), final_t)
    np.testing.assert_array_equal(_np(out.stacked()), image)
    assert contributors.max() > 64  # more than one chunk


def _backward(width, height, ranges, ids, centers, conics, feats, up, tail=True):
    """Kernel gradients, the oracle's and their bounds.  Without the constant
    alpha channel the oracle, which always blends one, gets a zero upstream
    gradient for it."""
    out = grender.render_views(ranges, ids, centers, conics, feats, width, height, one_tail=tail)
    record, grad_features, _ = grender.backward_views(ranges, ids, centers, conics, feats, out.transmittance,
                                                      out.contributors, up, width, height, absgrad=True,
                                                      one_tail=tail)
    up = _np(up) if tail else np.concatenate([_np(up), np.zeros(up.shape[:-1] + (1,), np.float32)], -1)
    args = (width, height, _np(ranges), _np(ids), _np(centers), _np(conics), _np(feats), _np(out.transmittance),
            _np(out.contributors), up)
    rec = _np(record)
    return (dict(centers=rec[..., 0:2], conics=rec[..., 2:6], abs=rec[..., 6:8], features=_np(grad_features)),
            oracle.render_bwd(*args, absgrad=True), oracle.render_bwd_bound(*args))


# Gradients of every compiled width of the backward, with and without the
# constant channel, at one and two pixels per lane, through lists whose
# Gaussians mostly miss the tile: groups of four end anywhere in a batch.
@pytest.mark.parametrize("width,height,channels,tail", [
    (75, 43, 1, True), (75, 43, 3, True), (75, 43, 4, False), (75, 43, 7, True), (75, 43, 8, False),
    (75, 43, 13, True), (75, 43, 16, False), (75, 43, 18, True), (75, 43, 20, False), (75, 43, 34, True),
    (75, 43, 41, True), (75, 43, 44, False), (75, 43, 36, False),
    (1300, 1300, 3, True), (1300, 1300, 4, False), (1300, 1300, 6, True)])
def test_backward_in_groups(width, height, channels, tail):
    print("backward in groups", width, height, channels, tail, flush=True)
    centers, conics, feats, g = _scene(width, height, 400, channels, extreme=False)
    ids, ranges = _lists(400, width, height, 150, g)
    up = torch.randn((1, height, width, channels + tail), generator=g).to(DEV)
    got, ref, bound = _backward(width, height, ranges, ids, centers, conics, feats, up, tail)
    for name in got:
        check_gradient(name, got[name], ref[name], bound[name])
        assert np.abs(got[name]).max() > 0


# Grids of 4096 to 6143 tiles: two pixels per lane beyond 40 list entries per
# Gaussian or where their count is not given, one up to 40, and 8 channels in a
# further window after 56.
@pytest.mark.parametrize("n,channels,counted", [(400, 3, True), (17_000, 3, True), (17_000, 3, False),
                                                (400, 58, True), (17_000, 58, True)])
def test_backward_of_mid_size_grids(n, channels, counted, monkeypatch):
    width, height = 1152, 960
    print("backward mid-size grid", n, channels, counted, flush=True)
    if not counted:
        real, calls = native.call, []

        def call(name, *args):
            if name == "gs3d_render_bwd_lists":
                calls.append(name)
                return real("gs3d_render_bwd", args[0], args[2])
            return real(name, *args)
        monkeypatch.setattr(native, "call", call)
    centers, conics, feats, g = _scene(width, height, n, channels, extreme=False)
    ids, ranges = _lists(n, width, height, 150, g)
    assert 4096 <= len(ranges) < 6144 and (ids.numel() > 40 * n) == (n == 400)
    up = torch.randn((1, height, width, channels + 1), generator=g).to(DEV)
    got, ref, bound = _backward(width, height, ranges, ids, centers, conics, feats, up)
    assert counted or len(calls) == 1
    for name in got:
        check_gradient(name, got[name], ref[name], bound[name])


@pytest.mark.parametrize("width,height,channels", [(75, 43, 3), (75, 43, 13), (75, 43, 34), (1300, 1300, 3),
                                                   (1300, 1300, 6)])
def test_backward_at_extreme_opacities(width, height, channels):
    print("backward extreme opacities", width, height, channels, flush=True)
    centers, conics, feats, g = _scene(width, height, 400, channels, extreme=True)
    # Opacities near the end of the range overflow or not by the order of the
    # products; NaN and infinite ones do not depend on it.
    o = conics[..., 3]
    conics[..., 3] = torch.where((o > 1e30) & (o < float("inf")), torch.full_like(o, 2.0), o)
    ids, ranges = _lists(400, width, height, 150, g)
    up = torch.randn((1, height, width, channels + 1), generator=g).to(DEV)
    got, ref, bound = _backward(width, height, ranges, ids, centers, conics, feats, up)
    for name in got:
        finite = np.isfinite(ref[name])
        np.testing.assert_array_equal(np.isfinite(got[name]), finite, err_msg=name)
        check_gradient(name, got[name][finite], ref[name][finite],
                       np.broadcast_to(bound[name], ref[name].shape)[finite])


# Finite opacities to the end of the range with small upstream gradients: no
# product overflows, but e^power is as small as 1e-38 and its product with the
# upstream gradient alone would lose its bits below the normal range.
@pytest.mark.parametrize("width,height,channels", [(75, 43, 3), (75, 43, 13), (75, 43, 18), (75, 43, 34),
                                                   (75, 43, 50), (1300, 1300, 3)])
def test_backward_at_huge_opacities(width, height, channels):
    print("backward huge opacities", width, height, channels, flush=True)
    centers, conics, feats, g = _scene(width, height, 400, channels, extreme=False)
    o = conics[0, :, 3].cpu()
    o[::2] = 10.0 ** (torch.arange(200) % 39).float()
    conics[0, :, 3] = o.to(DEV)
    ids, ranges = _lists(400, width, height, 150, g)
    up = torch.randn((1, height, width, channels + 1), generator=g).to(DEV) * 1e-6
    got, ref, bound = _backward(width, height, ranges, ids, centers, conics, feats, up)
    for name in got:
        # The absolute tolerance scaled by the upstream gradients.
        finite = np.isfinite(ref[name])
        np.testing.assert_array_equal(np.isfinite(got[name]), finite, err_msg=name)
        check_gradient(name, got[name][finite], ref[name][finite],
                       np.broadcast_to(bound[name], ref[name].shape)[finite], atol=1e-11)


# Conics far sharper than projection's (its 0.3 px dilation keeps entries below
# 3.4), to the end of the range, on or just beside pixel centres: one pixel of
# a lane blends the Gaussian, its neighbours' products with the conic overflow
# or are many orders larger than the blending pixel's.
@pytest.mark.parametrize("width,height,channels", [(75, 43, 3), (75, 43, 13), (75, 43, 18), (75, 43, 34),
                                                   (75, 43, 41), (75, 43, 50), (1300, 1300, 3)])
def test_backward_at_extreme_conics(width, height, channels):
    print("backward extreme conics", width, height, channels, flush=True)
    centers, conics, feats, g = _scene(width, height, 400, channels, extreme=False)
    centers, conics = centers.cpu(), conics.cpu()
    m = 200
    scale = 10.0 ** (torch.arange(m) % 20 * 2.0)           # 1 to 1e38
    a, c = (scale * (1.0 + torch.rand(m, generator=g)) for _ in range(2))
    conics[0, :m, 0], conics[0, :m, 2] = a, c
    conics[0, :m, 1] = (torch.rand(m, generator=g) * 2 - 1) * a.sqrt() * c.sqrt() * 0.9
    conics[0, :m, 3] = 0.5
    # Within one standard deviation of a pixel of the first rows and columns,
    # where small offsets are representable; a third exactly on it.
    centers[0, :m] = torch.randint(0, 3, (m, 2), generator=g) + \
        (torch.rand((m, 2), generator=g) - 0.5) / scale.sqrt()[:, None]
    centers[0, :m:3] = centers[0, :m:3].round()
    centers, conics = centers.to(DEV), conics.to(DEV)
    ids, ranges = _lists(400, width, height, 150, g)
    up = torch.randn((1, height, width, channels + 1), generator=g).to(DEV)
    got, ref, bound = _backward(width, height, ranges, ids, centers, conics, feats, up)
    for name in got:
        finite = np.isfinite(ref[name])
        np.testing.assert_array_equal(np.isfinite(got[name]), finite, err_msg=name)
        # The absolute tolerance is of the magnitude of 1: entries of sharp
        # Gaussians' centres reach 1e19 and only rtol and the bound apply.
        check_gradient(name, got[name][finite], ref[name][finite],
                       np.broadcast_to(bound[name], ref[name].shape)[finite])
    blended = np.abs(ref["features"][:m]).max(-1) > 0
    assert blended.reshape(-1, 20).any(0).all()            # every scale reaches a pixel


@pytest.mark.parametrize("width,height,channels", [(75, 43, 3), (75, 43, 7), (75, 43, 13), (75, 43, 18), (75, 43, 34),
                                                   (75, 43, 41), (75, 43, 60), (1300, 1300, 3), (1300, 1300, 6)])
def test_non_finite_channels_and_gradients(width, height, channels):
    # One and two pixels per lane: a non-finite channel or upstream gradient
    # reaches what blended it and nothing else, in every compiled width.
    print("non-finite", width, height, channels, flush=True)
    centers, conics, feats, g = _scene(width, height, 400, channels, extreme=False)
    ids, ranges = _lists(400, width, height, 150, g)
    feats[11, 0] = float("nan")
    feats[12, channels - 1] = float("inf")
    out = grender.render_views(ranges, ids, centers, conics, feats, width, height)
    image, _, _ = oracle.render_fwd(width, height, _np(ranges), _np(ids), _np(centers), _np(conics), _np(feats))
    np.testing.assert_array_equal(_np(out.stacked()), image)
    up = torch.randn((1, height, width, channels + 1), generator=g).to(DEV)
    up[0, height // 2, width // 3, 0] = float("nan")
    up[0, height // 3, width // 2, channels - 1] = float("-inf")
    got, ref, bound = _backward(width, height, ranges, ids, centers, conics, feats, up)
    for name in got:
        finite = np.isfinite(ref[name])
        np.testing.assert_array_equal(np.isfinite(got[name]), finite, err_msg=name)
        check_gradient(name, got[name][finite], ref[name][finite],
                       np.broadcast_to(bound[name], ref[name].shape)[finite])
