"""affine_append with more than 64 rows an activation.  With n_append at least the
layer's width every delta gets its own row, so the bounds are affine_all's up to
rounding."""
import numpy as np
import pytest
import torch

from niq import implicit_mlp_utils, models
from oracle import affine as oaff

pytestmark = pytest.mark.gpu

U = 2. ** -24


@pytest.mark.parametrize("width,n_append", [(64, 64), (65, 65), (100, 512), (128, 128), (257, 257), (512, 512)])
def test_append_of_every_delta_equals_affine_all(width, n_append):
    p = models.random_mlp([width], activation="relu", init="he", seed=width)
    g = np.random.default_rng(width)
    c = g.uniform(-.5, .5, (50, 3)).astype(np.float32)
    h = g.uniform(.2, 1., (50, 3)).astype(np.float32)
    lo, up = torch.tensor(c - h).cuda(), torch.tensor(c + h).cuda()

    def bounds(mode, **kw):
        f, q = implicit_mlp_utils.implicit_from_params(p, mode, **kw)
        return f.classify_box(q, lo, up, return_bounds=True)[1].cpu().numpy().astype(np.float64)

    every, rows = bounds("affine_all"), bounds("affine_append", affine_n_append=n_append)
    # The two sum the same deltas' rows in another order: 2 (width + 6) U of the radius.
    # affine_append then adds sum(delta) - sum(kept) to the interval part of every
    # feature: zero but for the rounding of two sums of at most n terms, 2 n U
    # sum(delta), which the last layer multiplies by its sum of |weights|.
    mats = [np.asarray(v, np.float64) for k, v in sorted(p.items()) if k.endswith(".A")]
    bias = [np.asarray(v, np.float64) for k, v in sorted(p.items()) if k.endswith(".b")]
    base = c.astype(np.float64) @ mats[0] + bias[0]
    rad = h.astype(np.float64) @ np.abs(mats[0])
    delta = np.abs(oaff.relu_rule(base - rad, base + rad)[2]).sum(1)
    n = -(-width // 16) * 16
    radius = (every[:, 1] - every[:, 0]) / 2
    tol = 2 * (n + 6) * U * radius + 2 * n * U * delta * np.abs(mats[-1]).sum() + 4 * U * np.abs(every).max(1)
    assert (delta > 0).all() and (np.abs(rows - every) <= tol[:, None]).all()
    # the bar is well below the share of the rows after the 64th
    assert (tol < 0.05 * radius).all() and (width > 65 or (tol < 0.005 * radius).all())
