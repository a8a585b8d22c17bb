"""Nets whose float32 rounding is large beside what they resolve: one hidden layer's
biases are raised and the next layer's take the change back, so pre-activations are
large and their differences small.  The first looks of the wide nets' trees (split
contraction), of the growing-row trees (corner signs) and of the ray caster (certified
segments) keep clear of that rounding, or leave the work to the paths that they
shorten: the results are those paths' results."""
import numpy as np
import pytest
import torch

from niq import implicit_mlp_utils, kd_tree, models, queries
from test_gpu_ray_pool import compare as compare_casts
from test_gpu_rows_signs import nodes, plain

pytestmark = pytest.mark.gpu

ONE = (np.array([-1., -1., -1.], np.float32), np.array([1., 1., 1.], np.float32))
TINY = (1e-3 * ONE[0], 1e-3 * ONE[1])


def raised(hidden, layer, by, seed, feature=None, **kw):
    """Hidden layer `layer`'s biases (or one of them) raised by `by`, the next layer's
    lowered by what that adds there."""
    p = dict(models.random_mlp(hidden, seed=seed, **kw))
    A = [k for k in sorted(p) if k.endswith("dense.A")]
    b = [k for k in sorted(p) if k.endswith("dense.b")]
    up = np.zeros(hidden[layer])
    up[slice(None) if feature is None else feature] = by
    p[b[layer]] = (p[b[layer]] + up).astype(np.float32)
    p[b[layer + 1]] = (p[b[layer + 1]] - up @ p[A[layer + 1]].astype(np.float64)).astype(np.float32)
    return p


def tree(p, root, variant, depth):
    f, _ = implicit_mlp_utils.implicit_from_params(p, "affine_fixed")
    f.cfg.variant = variant
    out, st = kd_tree.build_tree(f, p, *root, split_depth=depth, with_interior_nodes=True, with_exterior_nodes=True)
    return {k: v.cpu().numpy() for k, v in out.items()}, st


@pytest.mark.parametrize("hidden,layer,by,feature", [([256] * 3, 1, 10., None), ([256] * 3, 1, 1e3, None),
                                                     ([256] * 3, 1, 3e4, None), ([256] * 3, 1, 1e5, None),
                                                     ([256] * 3, 1, 1e6, 17), ([256] * 2, 1, 1e5, None),
                                                     ([256] * 4, 0, 1e3, None), ([512] * 2, 0, 3e4, None)])
@pytest.mark.parametrize("root,depth", [(ONE, 13), (ONE, 21), (TINY, 18)])
def test_wide_tree_is_the_plain_tree(hidden, layer, by, feature, root, depth):
    p = raised(hidden, layer, by, 5, feature)
    a, sa = tree(p, root, 0, depth)
    b, sb = tree(p, root, 3, depth)
    assert sa == sb
    for k in b:
        assert np.array_equal(a[k], b[k]), k


@pytest.mark.parametrize("hidden,layer,by", [([32] * 3, 1, 1e3), ([32] * 3, 1, 1e5), ([64] * 4, 0, 1e4),
                                             ([128] * 2, 0, 1e5), ([256] * 3, 1, 1e5)])
@pytest.mark.parametrize("mode", ["affine_fixed", "interval"])
def test_pooled_cast_is_the_plain_cast(hidden, layer, by, mode):
    compare_casts(raised(hidden, layer, by, 6), mode, 2000, seed=3, n_max_step=200)


@pytest.mark.parametrize("hidden,layer,by,depth", [([32] * 3, 1, 1e3, 14), ([32] * 3, 1, 1e5, 13), ([64] * 3, 0, 1e4, 12),
                                                   ([128] * 2, 0, 1e5, 12), ([256] * 2, 0, 1e5, 11)])
@pytest.mark.parametrize("mode,kw", [("affine_all", {}),
                                     ("affine_truncate", {"affine_n_truncate": 8,
                                                          "affine_truncate_policy": "absolute"})])
def test_rows_tree_has_the_nodes_of_the_bounds(hidden, layer, by, depth, mode, kw):
    p = raised(hidden, layer, by, 7)
    f, _ = implicit_mlp_utils.implicit_from_params(p, mode, **kw)
    out, _ = kd_tree.build_tree(f, p, *ONE, split_depth=depth, with_interior_nodes=True, with_exterior_nodes=True)
    lo, up, leaves = plain(f, p, ONE, depth, 0.0)
    got = {k: v.cpu().numpy() for k, v in out.items()}

    def valid(kind):
        keep = got[kind + "_node_valid"].astype(bool)
        return nodes(got[kind + "_node_lower"][keep], got[kind + "_node_upper"][keep])

    assert np.array_equal(valid("unknown"), nodes(lo, up))
    for kind, c in (("exterior", 1), ("interior", 2)):
        assert np.array_equal(valid(kind), nodes(leaves[c][:, :3], leaves[c][:, 3:])), kind
