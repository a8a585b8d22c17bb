"""A tuned function keeps what only the default variant runs: trees of wide ReLU nets by
the split contraction, frustum casts of 32-wide nets in one launch an iteration."""
import numpy as np
import pytest

from niq import autotune, implicit_mlp_utils, kd_tree, models

pytestmark = pytest.mark.gpu

LO, UP = np.full(3, -1.0, np.float32), np.full(3, 1.0, np.float32)


@pytest.mark.parametrize("hidden", [[256] * 3, [512] * 2, [32] * 3])
@pytest.mark.parametrize("mode", ["affine_fixed", "interval"])
def test_default_is_kept_unless_a_tree_gains(hidden, mode):
    p = models.random_mlp(hidden, seed=21)
    f, _ = implicit_mlp_utils.implicit_from_params(p, mode)
    autotune._cache.clear()
    res = autotune.tune(f, p, split_depth=15, n_boxes=1 << 13, reps=1)
    autotune._cache.clear()
    assert f.cfg.variant == res["best"] and 0 in res["ms"]
    if hidden[0] == 32:
        assert res["best"] == 0, res
    elif mode == "affine_fixed":   # variants 0 and 1 both take the split contraction
        assert res["best"] in (0, 1), res
    elif res["best"] != 0:
        assert res["tree_ms"][res["best"]] < res["tree_ms"][0]


def test_a_faster_tile_on_boxes_alone_does_not_win(monkeypatch):
    """Whatever the boxes say, a wide ReLU net's tree decides."""
    p = models.random_mlp([256] * 3, seed=22)
    f, _ = implicit_mlp_utils.implicit_from_params(p, "affine_fixed")
    real = autotune._time
    boxes = iter([5.0, 5.0, 5.0, 5.0, 1.0])   # variant 4 five times as fast

    def timed(fn, reps):
        return next(boxes, None) or real(fn, reps)

    monkeypatch.setattr(autotune, "_time", timed)
    autotune._cache.clear()
    res = autotune.tune(f, p, split_depth=15, n_boxes=1 << 10, reps=2)
    autotune._cache.clear()
    assert res["best"] == 0 and res["tree_ms"][0] < res["tree_ms"][4], res
    out = {}
    for v in (0, 4):
        f.cfg.variant = v
        out[v] = kd_tree.build_tree(f, p, LO, UP, split_depth=12)[1]
    assert out[0] == out[4]
