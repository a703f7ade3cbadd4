"""The blend kernels against the oracle where their tests and their exponential
change regime: opacities at and beyond the representable range, exponents past
the end of the exponential, centres on pixel centres and conics that are not
positive definite."""

import numpy as np
import pytest
import torch

import oracle
from dsl_splat_amd.gs3d import render as grender

pytestmark = pytest.mark.gpu

DEV = "cuda"

OPACITIES = [float("nan"), float("inf"), 3.0e38, 1.4e36, 1.3e36, 2.0, 1.0, 0.99, 0.5, 0.0040, 0.0039, 1e-30, 0.0,
             -0.0, -1.0]


def _np(t):
    return t.detach().cpu().numpy()


def _lists(n, width, height, per_tile, g):
    """Tile lists that are not derived from footprints: each tile lists
    `per_tile` Gaussians, most of them far outside it."""
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


# Fewer than 4096 tiles: one pixel per lane; more: two.  Channels: every
# compiled width of the forward.
@pytest.mark.parametrize("width,height,channels", [(75, 43, 3), (75, 43, 7), (75, 43, 13), (75, 43, 34),
                                                   (1030, 1027, 3), (1030, 1027, 6)])
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

