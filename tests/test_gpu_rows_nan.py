"""Boxes that are not finite, in the growing-row modes: no bound (NaN, so UNKNOWN), and
the boxes beside them as without them.  The base of such a box is NaN, or its error
terms are, and both stay NaN through every layer."""
import numpy as np
import pytest
import torch

from niq import implicit_mlp_utils, models

pytestmark = pytest.mark.gpu

MODES = [("affine_all", {}), ("affine_truncate", {"affine_n_truncate": 8, "affine_truncate_policy": "absolute"}),
         ("affine_append", {"affine_n_append": 4})]
NETS = [([32] * 3, "relu"), ([100, 128], "tanh"), ([256] * 2, "elu"), ([300], "relu")]


@pytest.mark.parametrize("mode,kw", MODES, ids=[m for m, _ in MODES])
@pytest.mark.parametrize("hidden,act", NETS, ids=[f"{a}{h[-1]}" for h, a in NETS])
def test_boxes_that_are_not_finite(hidden, act, mode, kw):
    f, p = implicit_mlp_utils.implicit_from_params(models.random_mlp(hidden, activation=act, init="xavier", seed=7),
                                                   mode, **kw)
    g = np.random.default_rng(3)
    lo = g.uniform(-1, 1, (40, 3)).astype(np.float32)
    up = lo + g.uniform(0, .2, (40, 3)).astype(np.float32)
    want_c, want_b = f.classify_box(p, torch.tensor(lo).cuda(), torch.tensor(up).cuda(), return_bounds=True)
    bad = np.zeros(40, bool)
    bad[[0, 13, 39]] = True
    lo[0, 1] = np.nan
    lo[13], up[13] = -np.inf, np.inf
    up[39, 2] = np.inf
    codes, bounds = f.classify_box(p, torch.tensor(lo).cuda(), torch.tensor(up).cuda(), return_bounds=True)
    ok = torch.tensor(~bad).cuda()
    assert torch.equal(codes[ok], want_c[ok])
    assert torch.equal(bounds[ok], want_b[ok])
    assert torch.isnan(bounds[~ok]).all()
    assert (codes[~ok] == 0).all()
