"""The FP64 re-test behind the tile that nets of several activations (or Sin) take at width
256: the codes of the default tile with its own re-test."""
import numpy as np
import pytest
import torch

from niq import implicit_mlp_utils, models

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden", [[256, 256], [200, 241]])
@pytest.mark.parametrize("act", ["sin", "mixed"])
def test_retest_codes(hidden, act):
    p = models.random_mlp(hidden, activation="sin" if act == "sin" else "tanh", init="xavier", seed=4)
    if act == "mixed":
        p = {k.replace("0003.tanh", "0003.elu"): v for k, v in p.items()}
    f, _ = implicit_mlp_utils.implicit_from_params(p, "affine_fixed", recheck_tol=0.05)
    for n in (1, 17, 8192, 8193, 20011):
        c = np.random.default_rng(n).uniform(-1, 1, size=(n, 3)).astype(np.float32)
        lo, up = torch.as_tensor(c - 0.02).cuda(), torch.as_tensor(c + 0.02).cuda()
        codes = {}
        for v in (0, 1, 3):
            f.cfg.variant = v
            codes[v] = f.classify_box(p, lo, up)
        assert torch.equal(codes[0], codes[1]) and torch.equal(codes[0], codes[3]), n
