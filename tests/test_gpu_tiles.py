"""Tiles of the classify pass at their edges: nets up to 32 wide (a tile of one
wave, four to a workgroup), 64 and 128 wide (16-box tiles), the activation-only
kernels and the rolled transcendental rules, at batch sizes around a tile, a
workgroup and the switch from the small-launch tile.

Bars: bounds within 1e-5 * max |oracle32| + 2 |oracle32 - oracle64| per cell
(the parity suite's); the same box gives the same bits in every tile and at
every place in a batch (each box's sums have one order)."""
import numpy as np
import pytest
import torch

from oracle import funcs as ofuncs
from niq import models, implicit_mlp_utils

pytestmark = pytest.mark.gpu

NETS = [([32, 32], "relu"), ([17, 32, 5], "tanh"), ([32, 32, 32], "elu"), ([9], "sin"), ([33, 64], "tanh"),
        ([64, 64], "elu"), ([64, 50], "relu"), ([128, 100], "tanh"), ([65, 128], "elu"), ([256, 130], "tanh"),
        ([30, 20], "sin")]


@pytest.mark.parametrize("hidden,act", NETS)
@pytest.mark.parametrize("mode", ["interval", "affine_fixed", "slope_interval"])
def test_tile_edges(hidden, act, mode):
    p = models.random_mlp(hidden, activation=act, init="he" if act in ("relu", "elu") else "xavier", seed=5)
    f, _ = implicit_mlp_utils.implicit_from_params(p, mode)
    n_all = 32 * 256 + 17   # past the small-launch tile, ragged
    rng = np.random.default_rng(4)
    c = rng.uniform(-1, 1, size=(n_all, 3))
    h = rng.uniform(0.002, 0.2, size=(n_all, 3))
    lo, up = (c - h).astype(np.float32), (c + h).astype(np.float32)
    dlo, dup = torch.as_tensor(lo, device="cuda"), torch.as_tensor(up, device="cuda")
    codes, bounds = [t.cpu().numpy() for t in f.classify_box(p, dlo, dup, return_bounds=True)]
    for variant in (2, 3, 4):
        f.cfg.variant = variant
        c2, b2 = [t.cpu().numpy() for t in f.classify_box(p, dlo, dup, return_bounds=True)]
        assert np.array_equal(codes, c2) and np.array_equal(bounds, b2), variant
    f.cfg.variant = 1
    for n in (1, 15, 16, 17, 63, 64, 65, 1000):
        for off in (0, 5):
            c2, b2 = [t.cpu().numpy() for t in f.classify_box(p, dlo[off:off + n], dup[off:off + n],
                                                              return_bounds=True)]
            assert np.array_equal(codes[off:off + n], c2) and np.array_equal(bounds[off:off + n], b2), (n, off)
    m = 400
    r32 = np.stack(ofuncs.OracleFunc(p, mode, np.float32).bounds_box(lo[:m], up[:m]), 1)
    r64 = np.stack(ofuncs.OracleFunc(p, mode, np.float64).bounds_box(lo[:m], up[:m]), 1)
    assert np.all(np.abs(bounds[:m] - r32) <= 1e-5 * np.max(np.abs(r32)) + 2 * np.abs(r32 - r64))


@pytest.mark.parametrize("hidden,act", NETS)
def test_point_tile_edges(hidden, act):
    p = models.random_mlp(hidden, activation=act, init="xavier", seed=6)
    f, _ = implicit_mlp_utils.implicit_from_params(p, "affine_fixed")
    x = torch.as_tensor(np.random.default_rng(2).uniform(-1, 1, size=(2100, 3)).astype(np.float32), device="cuda")
    ref = f(p, x).cpu().numpy()
    for n in (1, 31, 32, 33, 63, 64, 65):
        assert np.array_equal(f(p, x[7:7 + n]).cpu().numpy(), ref[7:7 + n]), n
    o32 = ofuncs.OracleFunc(p, "affine_fixed", np.float32)(x.cpu().numpy()).reshape(-1)
    assert np.all(np.abs(ref - o32) <= 1e-5 * np.max(np.abs(o32)))
