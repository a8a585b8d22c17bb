"""Trees in the growing-row modes, where the corners of a box decide some of its
levels' codes, against the same tree split here with codes from classify calls,
which compute every box's bound: the same nodes, since a bound contains f's values
in the box."""
import numpy as np
import pytest
import torch

from niq import implicit_mlp_utils, kd_tree, models

pytestmark = pytest.mark.gpu

MODES = [("affine_all", {}), ("affine_truncate", {"affine_n_truncate": 8, "affine_truncate_policy": "absolute"}),
         ("affine_append", {"affine_n_append": 4})]
NETS = [([32] * 3, "relu", "he", 14), ([64, 50, 64], "elu", "he", 12), ([128] * 3, "tanh", "xavier", 13),
        ([200, 256], "relu", "he", 11), ([512, 300], "tanh", "xavier", 10), ([32] * 2, "sin", "he", 12)]
ONE = (np.float32([-1, -1, -1]), np.float32([1, 1, 1]))
SKEW = (np.float32([-1.3, -0.4, -1.]), np.float32([0.7, 1.1, 2.]))
# far from the origin beside its size: the small boxes are not judged by corners
FAR = (np.float32([0.5, 0.5, 0.5]), np.float32([0.75, 0.75, 0.75]))


def nodes(lo, up):
    a = np.concatenate([np.asarray(lo), np.asarray(up)], axis=1)
    return a[np.lexsort(a.T)]


def plain(f, p, root, depth, offset):
    lo, up = (torch.tensor(x[None]).cuda() for x in root)
    leaves = {1: [], 2: []}
    for level in range(depth + 1):
        codes = f.classify_box(p, lo, up, offset=offset)
        for c in leaves:
            leaves[c].append(torch.cat([lo[codes == c], up[codes == c]], dim=1))
        lo, up = lo[codes == 0], up[codes == 0]
        if level < depth:
            d = (up - lo).argmax(1, keepdim=True)
            mid = 0.5 * (lo + up).gather(1, d)
            lo, up = torch.cat([lo, lo.scatter(1, d, mid)]), torch.cat([up.scatter(1, d, mid), up])
    return lo.cpu(), up.cpu(), {c: torch.cat(v).cpu() for c, v in leaves.items()}


@pytest.mark.parametrize("hidden,act,init,depth", NETS)
@pytest.mark.parametrize("mode,kw", MODES)
@pytest.mark.parametrize("root,offset", [(ONE, 0.0), (SKEW, 0.05), (FAR, 0.0)])
def test_tree_has_the_nodes_of_the_bounds(hidden, act, init, depth, mode, kw, root, offset):
    p = models.random_mlp(hidden, activation=act, init=init, seed=len(hidden) + hidden[0])
    f, _ = implicit_mlp_utils.implicit_from_params(p, mode, **kw)
    out, _ = kd_tree.build_tree(f, p, *root, split_depth=depth, offset=offset, with_interior_nodes=True,
                                with_exterior_nodes=True)
    lo, up, leaves = plain(f, p, root, depth, offset)
    got = {k: v.cpu().numpy() for k, v in out.items()}

    def valid(kind):
        keep = got[kind + "_node_valid"].astype(bool)
        return nodes(got[kind + "_node_lower"][keep], got[kind + "_node_upper"][keep])

    assert np.array_equal(valid("unknown"), nodes(lo, up))
    for kind, c in (("exterior", 1), ("interior", 2)):
        assert np.array_equal(valid(kind), nodes(leaves[c][:, :3], leaves[c][:, 3:])), kind
