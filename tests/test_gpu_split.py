"""Trees of wide ReLU nets, whose classification runs on bf16 matrix
instructions with the near-threshold boxes left to the plain kernel, against
the plain kernel's trees (eval cfg variant 3): the same lists, order and counts
included, since every code is the plain kernel's.  And point values of wide nets
on the same instructions: within 1e-5 * max |oracle32| (the parity suite's bar),
no further from float64 than the float32 oracle in the mean square (the split is
exact; its sums round less often), and the plain rules for points outside the
split's range."""
import numpy as np
import pytest
import torch

from oracle import mlp as omlp
from niq import models, implicit_mlp_utils, kd_tree

pytestmark = pytest.mark.gpu

ONE = (np.array([-1., -1., -1.], np.float32), np.array([1., 1., 1.], np.float32))
SKEW = (np.array([-1.3, -0.4, -1.], np.float32), np.array([0.7, 1.1, 2.], np.float32))
# far from the origin beside its size: the small boxes take the plain kernel
FAR = (np.array([0.5, 0.5, 0.5], np.float32), np.array([1.25, 1.25, 1.25], np.float32))


def tree(p, root, variant, **kw):
    f, _ = implicit_mlp_utils.implicit_from_params(p, "affine_fixed")
    f.cfg.variant = variant
    out, st = kd_tree.build_tree(f, p, *root, with_interior_nodes=True, with_exterior_nodes=True, **kw)
    return {k: v.cpu().numpy() for k, v in out.items()}, st


@pytest.mark.parametrize("hidden,init,seed", [([256, 256], "he", 1), ([250, 256, 241], "he", 2),
                                              ([256] * 4, "xavier", 3), ([512, 512], "he", 4),
                                              ([500, 512, 481], "xavier", 5)])
@pytest.mark.parametrize("root,kw", [(ONE, {"split_depth": 17}), (ONE, {"split_depth": 5}),
                                     (SKEW, {"split_depth": 15, "offset": 0.05}), (FAR, {"split_depth": 16}),
                                     (ONE, {"node_terminate_thresh": 20000}),
                                     (ONE, {"split_depth": 14, "batch_process_size": 512})])
def test_split_tree_is_the_plain_tree(hidden, init, seed, root, kw):
    p = models.random_mlp(hidden, init=init, seed=seed)
    a, sa = tree(p, root, 0, **kw)
    b, sb = tree(p, root, 3, **kw)
    assert sa == sb
    for k in b:
        assert np.array_equal(a[k], b[k]), k


def test_deep_split_tree_is_the_plain_tree():
    # below level 21 the boxes are too small for the split contraction
    p = models.random_mlp([256] * 3, seed=6)
    a, sa = tree(p, ONE, 0, split_depth=23)
    b, sb = tree(p, ONE, 3, split_depth=23)
    assert sa == sb
    for k in b:
        assert np.array_equal(a[k], b[k]), k


def test_large_biases_take_the_plain_kernel():
    p = models.random_mlp([256, 256], seed=7)
    p["0000.dense.b"] = p["0000.dense.b"] + np.float32(100.0)
    a, sa = tree(p, ONE, 0, split_depth=13)
    b, sb = tree(p, ONE, 3, split_depth=13)
    assert sa == sb
    for k in b:
        assert np.array_equal(a[k], b[k]), k


POINT_NETS = [([256, 256], "relu"), ([255, 250, 256], "tanh"), ([512], "elu"), ([512, 500, 512], "relu"),
              ([256] * 3, "sin")]


@pytest.mark.parametrize("hidden,act", POINT_NETS)
def test_split_points(hidden, act):
    p = models.random_mlp(hidden, activation=act, init="xavier", seed=8)
    f, _ = implicit_mlp_utils.implicit_from_params(p, "affine_fixed")
    x = np.random.default_rng(3).uniform(-1, 1, size=(3001, 3)).astype(np.float32)
    got = f(p, torch.as_tensor(x, device="cuda")).cpu().numpy()
    r32, r64 = omlp.eval_points(p, x, np.float32).reshape(-1), omlp.eval_points(p, x, np.float64).reshape(-1)
    assert np.all(np.abs(got - r32) <= 1e-5 * np.max(np.abs(r32)))
    assert np.linalg.norm(got - r64) <= np.linalg.norm(r32 - r64)
    for n in (1, 15, 16, 17, 63, 64, 65):   # the same bits at every place in a batch
        part = f(p, torch.as_tensor(x[5:5 + n], device="cuda")).cpu().numpy()
        assert np.array_equal(part, got[5:5 + n]), n


@pytest.mark.parametrize("width", [256, 512])
def test_points_outside_the_split_range(width):
    p = models.random_mlp([width, width], init="he", seed=9)
    f, _ = implicit_mlp_utils.implicit_from_params(p, "affine_fixed")
    x = np.random.default_rng(5).uniform(-1, 1, size=(200, 3)).astype(np.float32)
    odd = {0: (np.inf, 0, 0), 7: (0, -np.inf, 1), 63: (np.nan, 0, 0), 64: (1e7, 2, 3), 70: (1, 1e20, -1e20),
           199: (-2e6, 0.5, 0)}
    for i, v in odd.items():
        x[i] = v
    got = f(p, torch.as_tensor(x, device="cuda")).cpu().numpy()
    # the kernels' rules in float64: relu(x) = x > 0 ? x : 0 (NaN gives 0)
    h = x.astype(np.float64)
    with np.errstate(invalid="ignore"):
        for i in range(0, 6, 2):
            h = np.stack([np.sum(h[:, :, None] * p[f"{i:04d}.dense.A"].astype(np.float64)[None], axis=1)])[0]
            h = h + p[f"{i:04d}.dense.b"].astype(np.float64)
            if i < 4:
                h = np.where(h > 0, h, 0.0)
    ref = h[:, 0]
    assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(np.isinf(got), np.isinf(ref))
    fin = np.isfinite(ref)
    # float32 sums of up to 512 terms of the point's own magnitude
    scale = np.maximum(1.0, np.max(np.abs(np.nan_to_num(x, posinf=0, neginf=0)), axis=1))
    assert np.all(np.abs(got[fin] - ref[fin]) <= 1e-4 * scale[fin])
