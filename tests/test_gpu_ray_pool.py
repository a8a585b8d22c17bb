"""The pooled ray caster (casts of one function) against the caster that gives
every ray its column and evaluates every hit test, which a cast of the same
function twice runs: bit-identical distances, the same hits, counts and number of
evaluations.  A skipped test could only have reported a hit where float32 rounding
exceeds the margin that the bound leaves, so no ray may differ."""
import pytest
import torch

from niq import implicit_mlp_utils, models, queries

pytestmark = pytest.mark.gpu

NETS = {
    "relu32": lambda: models.random_mlp([32] * 3, seed=1),
    "relu64": lambda: models.random_mlp([64, 50, 64], seed=2),
    "relu128": lambda: models.random_mlp([100, 128], seed=3),
    "relu256": lambda: models.random_mlp([256, 241, 256], seed=4),
    "relu512": lambda: models.random_mlp([512, 500], seed=5),
    "tanh32": lambda: models.random_mlp([32] * 4, "tanh", "xavier", seed=6),
    "tanh200": lambda: models.random_mlp([200] * 2, "tanh", "xavier", seed=7),
    "elu64": lambda: models.random_mlp([64] * 3, "elu", seed=8),
}


def rays(n, seed):
    g = torch.Generator().manual_seed(seed)
    roots = torch.randn(n, 3, generator=g) * 1.5
    dirs = torch.rand(n, 3, generator=g) * 1.6 - 0.8 - roots
    return roots.cuda(), torch.nn.functional.normalize(dirs, dim=1).cuda()


def compare(p, mode, n, seed, **kw):
    f, _ = implicit_mlp_utils.implicit_from_params(p, mode)
    opts = queries.get_default_cast_opts()
    opts["max_dist"] = 6.0
    opts.update(kw)
    roots, dirs = rays(n, seed)
    t, hit, cnt, ev = queries.cast_rays((f,), (p,), roots, dirs, opts)
    t2, hit2, cnt2, ev2 = queries.cast_rays((f, f), (p, p), roots, dirs, opts)
    assert torch.equal(t, t2) and torch.equal(cnt, cnt2) and ev == ev2
    assert torch.equal(hit, hit2.clamp(max=1))


# 1 ray, half a tile and one more, a tile, some hundred, and enough to fill every
# pool of the narrow nets more than once
@pytest.mark.parametrize("net", list(NETS))
@pytest.mark.parametrize("mode", ["affine_fixed", "interval", "slope_interval"])
def test_pooled_cast_is_the_plain_cast(net, mode):
    p = NETS[net]()
    for n in (1, 9, 16, 33, 700, 9001):
        compare(p, mode, n, seed=n)


@pytest.mark.parametrize("net", ["relu32", "relu256", "elu64"])
@pytest.mark.parametrize("kw", [{"n_substeps": 3}, {"n_max_step": 7}, {"hit_eps": 1e-5}, {"hit_eps": 0.2},
                                {"interval_init_size": 1e-6}, {"interval_init_size": 1.0, "safety_factor": 1.0},
                                {"max_dist": 0.5}])
def test_pooled_cast_options(net, kw):
    compare(NETS[net](), "affine_fixed", 3000, seed=11, **kw)


def test_pooled_cast_fills_the_pools_of_narrow_nets():
    compare(NETS["relu32"](), "affine_fixed", 250007, seed=12)
