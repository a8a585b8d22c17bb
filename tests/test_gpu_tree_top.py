"""The one-workgroup build of a tree's top levels against the per-level kernels
(which a build with the FP64 re-test runs; its band here is too narrow to list
a cell): the same lists, order included, and the same counts."""
import numpy as np
import pytest
import torch

from niq import models, implicit_mlp_utils, kd_tree

pytestmark = pytest.mark.gpu


def build(p, lo, up, tol, **kw):
    f, _ = implicit_mlp_utils.implicit_from_params(p, "affine_fixed", recheck_tol=tol)
    out, st = kd_tree.build_tree(f, p, lo, up, with_interior_nodes=True, with_exterior_nodes=True, **kw)
    st.pop("n_recheck")
    return {k: v.cpu().numpy() for k, v in out.items()}, st


@pytest.mark.parametrize("batch", [1, 8, 512, 2048, 8192])
@pytest.mark.parametrize("end", [{"split_depth": d} for d in (2, 3, 7, 11, 12, 13, 14)] +
                         [{"node_terminate_thresh": t} for t in (1, 100, 2048, 4096, 5000)] +
                         [{"split_depth": 9, "node_terminate_thresh": 64}])
def test_top_matches_levels(batch, end):
    p = models.random_mlp([24, 24], activation="tanh", init="xavier", seed=3)
    lo, up = np.array([-1, -1.2, -0.9], np.float32), np.array([1.1, 1, 1], np.float32)
    kw = dict(end, batch_process_size=batch, offset=0.01)
    a, sa = build(p, lo, up, 0.0, **kw)
    b, sb = build(p, lo, up, 1e-30, **kw)
    assert sa == sb
    assert sorted(a) == sorted(b)
    for k in a:
        assert np.array_equal(a[k], b[k]), k


def test_top_of_an_empty_tree():
    # every box has one sign: the lists end at the root
    p = models.random_mlp([24, 24], activation="tanh", init="xavier", seed=3)
    lo, up = np.array([0.5, 0.5, 0.5], np.float32), np.array([0.5001, 0.5001, 0.5001], np.float32)
    a, sa = build(p, lo, up, 0.0, split_depth=12)
    b, sb = build(p, lo, up, 1e-30, split_depth=12)
    assert sa == sb and sa["n_unknown"] == 0 and sa["n_interior"] + sa["n_exterior"] == 1
    for k in a:
        assert np.array_equal(a[k], b[k]), k
