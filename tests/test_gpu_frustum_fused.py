"""Frustum casts of 32-wide nets, whose iterations evaluate boxes and points in one
launch, against the same casts with the two launches of another classify tile (eval
cfg variant 1): every box and point sums in the same order, so the images and the
number of evaluations are identical."""
import numpy as np
import pytest
import torch

from niq import implicit_mlp_utils, models, queries

pytestmark = pytest.mark.gpu

NETS = {
    "relu32": ([32] * 3, "relu", "he"),
    "relu20": ([20, 32], "relu", "he"),
    "tanh32": ([32] * 4, "tanh", "xavier"),
    "sin32": ([32] * 2, "sin", "he"),
    "elu64": ([64] * 2, "elu", "he"),
}
CAM = (np.float32([0.3, -0.2, 3.]), np.float32([0., 0., -1.]), np.float32([0., 1., 0.]), np.float32([-1., 0., 0.]))


def compare(nets, mode, res, **kw):
    ps = tuple(models.random_mlp(*NETS[n][:1], activation=NETS[n][1], init=NETS[n][2], seed=i)
               for i, n in enumerate(nets))
    opts = queries.get_default_cast_opts()
    opts["max_dist"] = 6.0
    opts.update(kw)
    out = []
    for variant in (0, 1):
        fs = tuple(implicit_mlp_utils.implicit_from_params(p, mode)[0] for p in ps)
        for f in fs:
            f.cfg.variant = variant
        out.append(queries.cast_rays_frustum(fs, ps, (*CAM, 60.0, 50.0, *res), opts))
    (t, h, c, ev), (t2, h2, c2, ev2) = out
    assert torch.equal(t, t2) and torch.equal(h, h2) and torch.equal(c, c2) and ev == ev2


# one frustum, fewer frusta than a tile, ragged tiles, enough to fill the chip
@pytest.mark.parametrize("net", ["relu32", "relu20", "tanh32", "sin32"])
@pytest.mark.parametrize("mode", ["affine_fixed", "interval"])
@pytest.mark.parametrize("res,side", [((1, 1), 1), ((5, 3), 3), ((67, 41), 16), ((190, 211), 32)])
def test_fused_iteration_is_the_two_launches(net, mode, res, side):
    compare([net], mode, res, n_side_init=side)


@pytest.mark.parametrize("nets", [("relu32", "tanh32"), ("elu64", "relu32")])
@pytest.mark.parametrize("kw", [{"n_substeps": 2}, {"n_max_step": 9}])
def test_fused_iteration_of_several_functions(nets, kw):
    compare(nets, "affine_fixed", (64, 64), n_side_init=16, **kw)
