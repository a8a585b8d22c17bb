"""Casts at the ray counts where the caster's launch changes: one workgroup a compute
unit, twice as many, a pool of several rays a column, and the nets whose bounds exclude
few tests, which leave the pool early.  The same rays as the caster that evaluates every
test (a cast of the function twice)."""
import pytest

from niq import models
from test_gpu_ray_pool import compare

pytestmark = pytest.mark.gpu

NETS = {
    "relu64": lambda: models.random_mlp([64] * 2, seed=2),
    "elu64x8": lambda: models.random_mlp([64] * 8, "elu", seed=8),
    "relu128": lambda: models.random_mlp([100, 128], seed=3),
    "tanh128x6": lambda: models.random_mlp([128] * 6, "tanh", "xavier", seed=6),
    "relu256": lambda: models.random_mlp([256, 241], seed=4),
    "tanh256x5": lambda: models.random_mlp([200] * 5, "tanh", "xavier", seed=7),
    "relu512": lambda: models.random_mlp([512], seed=5),
}


# compute units (256) times half a tile's, a tile's and two tiles' columns (16 or 32),
# one more of each, and past a full pool
@pytest.mark.parametrize("net,sizes", [("relu64", (4096, 8193, 32769)), ("elu64x8", (4096, 8193)),
                                       ("relu128", (4096, 8193, 16385)), ("tanh128x6", (4096, 4097, 16385)),
                                       ("relu256", (2048, 4097, 8192, 8193)), ("tanh256x5", (2048, 2049, 8193)),
                                       ("relu512", (3072, 3073, 4097))])
@pytest.mark.parametrize("mode", ["affine_fixed", "interval", "slope_interval"])
def test_pooled_cast_at_launch_sizes(net, sizes, mode):
    p = NETS[net]()
    for n in sizes:
        compare(p, mode, n, seed=n, n_max_step=40)


@pytest.mark.parametrize("n", [1, 300, 5000])
def test_several_activations_and_sin(n):
    for act in ("sin", "tanh"):
        p = models.random_mlp([256, 200], act, "xavier", seed=9)
        if act == "tanh":   # TanH, then ELU
            p = {k.replace("0003.tanh", "0003.elu"): v for k, v in p.items()}
        for mode in ("affine_fixed", "interval", "slope_interval"):
            compare(p, mode, n, seed=n, n_max_step=40)
