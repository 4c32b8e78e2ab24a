"""PhyloLik's likelihood and root posterior (lib/CamlPaml/PhyloLik.ml:46-138; paths
relative to the mlin/PhyloCSF tree) on both sides of the number of columns at which
an alphabet goes from a column per wave to a column per lane: the two routes give
the same values up to the order of k <= 24 terms per node (1e-12 relative, as the
other PhyloLik tests), and the first columns are the oracle's.
"""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import phylocsf_amd as P  # noqa: E402
from oracle import oracle as O  # noqa: E402


@pytest.fixture(scope="module")
def ctx():
    return P.Context(0)


@pytest.mark.parametrize("name,k,edge", [("12flies", 20, 2048 + 48 * 11), ("58mammals", 24, 4784),
                                         ("120mammals", 17, 6144), ("58mammals", 12, 2048),
                                         ("120mammals", 16, 2048), ("120mammals", 5, 1024)])
def test_routes_agree(ctx, params_dir, name, k, edge):
    print("PhyloLik routes: %s, k = %d, %d columns" % (name, k, edge), flush=True)
    text = open(os.path.join(params_dir, name + ".nh")).read()
    tree, otree = P.newick_tree(text), O.newick_tree(text)
    rng = np.random.default_rng([k, tree.n])
    Pm = 0.1 * rng.random((tree.n - 1, k, k)) + 0.9 * np.eye(k)
    Pm /= Pm.sum(axis=2, keepdims=True)
    prior = rng.dirichlet(np.ones(k))
    leaves = rng.integers(0, k, (1, 1)) + (rng.random((edge + 1, tree.nl)) < 0.1)
    leaves = (leaves % k).astype(np.int32)
    leaves[rng.random(leaves.shape) < 0.2] = -1
    z0, post0, _ = O.lik_posteriors(otree, Pm, prior, leaves[:70])
    got = []
    for ncols in (edge - 1, edge, edge + 1):
        it = P.PhyloLik(ctx).prepare(tree, Pm, prior, leaves[:ncols])
        got.append((it.likelihood(), it.node_posterior(tree.n - 1)))
        assert np.allclose(got[-1][0][:70], z0, rtol=1e-12, atol=0)
        assert np.allclose(got[-1][1][:70], post0[:, -1, :], rtol=1e-12, atol=1e-300)
    for z, post in got[1:]:
        assert np.allclose(z[:edge - 1], got[0][0], rtol=1e-12, atol=0)
        assert np.allclose(post[:edge - 1], got[0][1], rtol=1e-12, atol=1e-300)
