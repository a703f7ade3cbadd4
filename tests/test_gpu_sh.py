"""Standalone SH evaluation and its VJP over the row lengths, alignments and
row counts that choose its kernels, against the oracle."""

import numpy as np
import pytest
import torch

import oracle
from oracle_pipeline import check_gradient
from dsl_splat_amd.primitives.spherical_harmonics import spherical_harmonics

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _np(t):
    return t.detach().cpu().numpy()


@pytest.mark.parametrize("degree,rows,n,offset", [
    (0, 16, 1, 0), (1, 16, 63, 0), (2, 16, 64, 0), (3, 16, 65, 0), (3, 16, 129, 1), (1, 4, 1000, 0), (1, 4, 191, 3),
    (0, 1, 257, 0), (2, 9, 300, 0), (2, 12, 130, 0), (3, 17, 200, 0), (3, 20, 200, 0), (0, 3, 100, 2)])
def test_row_lengths_and_alignments(degree, rows, n, offset):
    print("sh", degree, rows, n, offset, flush=True)
    g = torch.Generator().manual_seed(rows + n)
    storage = torch.randn(n * rows * 3 + offset, generator=g) * 0.3
    # `offset` floats into an allocation: rows off the 16-byte grid.
    leaf = storage.to(DEV).requires_grad_(True)
    coef = leaf[offset:].view(n, rows, 3)
    assert (coef.data_ptr() % 16 == 0) == (offset % 4 == 0)
    dirs = torch.randn((n, 3), generator=g).to(DEV).requires_grad_(True)
    up = torch.randn((n, 3), generator=g).to(DEV)
    colors = spherical_harmonics(coef, dirs, degree)
    colors.backward(up)
    ref, active = oracle.sh_fwd(_np(coef), _np(dirs), degree)
    np.testing.assert_array_equal(_np(colors), ref)
    gco, gdir = oracle.sh_bwd(_np(coef), _np(dirs), degree, active, _np(up))
    bco, bdir = oracle.sh_bwd_bound(_np(coef), _np(dirs), degree, active, _np(up))
    got = _np(leaf.grad)[offset:].reshape(n, rows, 3)
    assert np.all(got[:, (degree + 1) ** 2:] == 0)
    check_gradient("coefficients", got, gco, bco)
    if degree > 0:
        check_gradient("directions", _np(dirs.grad), gdir, bdir)
