"""Trees of wide ReLU nets, whose classification runs on bf16 matrix
instructions with the near-threshold boxes left to the plain kernel, against
the plain kernel's trees (eval cfg variant 3): the same lists, order and counts
included, since every code is the plain kernel's."""
import numpy as np
import pytest

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
