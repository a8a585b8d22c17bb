"""The serving loop's merging does not depend on how fast requests are submitted or
how long a build takes, as long as they wait in the queue together; and merged builds
of wide ReLU nets, whose levels run by the split contraction, equal lone builds bit for
bit, also where a captured graph was first built for another root box."""
import time

import numpy as np
import pytest

from niq import implicit_mlp_utils, kd_tree, models, serve
from test_gpu_rounding import raised
import test_gpu_serve as base

pytestmark = pytest.mark.gpu

LO, UP = base.LO, base.UP
FAR = (np.array([6., 6., 6.], np.float32), np.array([6.5, 6.5, 6.5], np.float32))


def test_casts_merge_however_slow_the_submits(monkeypatch):
    submit_rays = serve.Server.submit_rays

    def slow(self, *args, **kw):
        time.sleep(0.01)   # a descheduled host
        return submit_rays(self, *args, **kw)

    monkeypatch.setattr(serve.Server, "submit_rays", slow)
    base.test_rays_of_different_models_and_options_share_a_cast()


def wide_nets():
    return [models.random_mlp([256, 256], seed=1), models.random_mlp([250, 256, 241], init="xavier", seed=2),
            raised([256] * 3, 1, 3e4, 5), models.random_mlp([256] * 2, activation="tanh", init="xavier", seed=3)]


@pytest.mark.parametrize("depth", [2, 5, 12, 14])
def test_wide_trees_merge(depth):
    kw = dict(split_depth=depth, with_interior_nodes=True, with_exterior_nodes=True)
    skew = (np.array([-1.3, -0.4, -1.], np.float32), np.array([0.7, 1.1, 2.], np.float32))
    plan = [(p, root) for p in wide_nets() for root in ((LO, UP), skew, FAR)]
    fs = [implicit_mlp_utils.implicit_from_params(p, "affine_fixed")[0] for p, _ in plan]
    alone = [kd_tree.construct_uniform_unknown_levelset_tree(f, p, *root, **kw) for f, (p, root) in zip(fs, plan)]
    with serve.Server(n_streams=1) as srv:
        busy = srv.submit_tree(fs[0], plan[0][0], LO, UP, split_depth=3)
        reqs = [srv.submit_tree(f, p, *root, **kw) for f, (p, root) in zip(fs, plan)]
        busy.result()
        got = [r.result() for r in reqs]
        sizes = [r.info["n_batched"] for r in reqs]
    print(sizes, flush=True)
    assert max(sizes) >= 3
    for i, (a, g) in enumerate(zip(alone, got)):
        assert base.same_tree(a, g), f"tree request {i}"


def test_wide_512_trees_merge():
    kw = dict(split_depth=12, with_interior_nodes=True, with_exterior_nodes=True)
    ps = [models.random_mlp([512, 512], seed=s) for s in (1, 2)]
    fs = [implicit_mlp_utils.implicit_from_params(p, "affine_fixed")[0] for p in ps]
    alone = [kd_tree.construct_uniform_unknown_levelset_tree(f, p, LO, UP, **kw) for f, p in zip(fs, ps)]
    with serve.Server(n_streams=1) as srv:
        reqs = [srv.submit_tree(f, p, LO, UP, **kw) for _ in range(4) for f, p in zip(fs, ps)]
        got = [r.result() for r in reqs]
    for a, g in zip(alone * 4, got):
        assert base.same_tree(a, g)


@pytest.mark.parametrize("first", ["near", "far"])
def test_graph_of_a_near_root_is_not_a_far_roots(first):
    """A cached graph holds the levels that take the split contraction, which the root
    box decides: near and far roots keep a graph each, and both are lone builds."""
    p = models.random_mlp([256, 256], seed=1)
    f, _ = implicit_mlp_utils.implicit_from_params(p, "affine_fixed")
    kw = dict(split_depth=13, with_interior_nodes=True, with_exterior_nodes=True)
    roots = {"near": (LO, UP), "far": FAR, "half": (LO, 0.5 * UP)}
    alone = {k: kd_tree.construct_uniform_unknown_levelset_tree(f, p, *r, **kw) for k, r in roots.items()}
    order = ["near", "far"] if first == "near" else ["far", "near"]
    reused = {}
    with serve.Server(n_streams=1) as srv:
        for k in order + ["half", "far", "near"]:
            r = srv.submit_tree(f, p, *roots[k], **kw)   # one at a time: never merged
            assert base.same_tree(alone[k], r.result()), k
            reused.setdefault(k, []).append(r.info["graph_reused"])
    # the second of near and far is captured anew; near's graph serves another near root
    assert reused["near"] == [False, True] and reused["far"] == [False, True] and reused["half"] == [True]
