"""PhyloLik over small alphabets (one column per lane) against the oracle's
restatement of PhyloLik.prepare / likelihood / node_posterior at the root
(lib/CamlPaml/PhyloLik.ml:46-138; paths relative to the mlin/PhyloCSF tree),
at every padded width and on both sides of it, at column counts around a
wave's 64, with every leaf kind, and on a tree whose leaf rows do not fit LDS.
The sums are those of the oracle up to the order of k <= 24 terms per node:
1e-12 relative, as the other PhyloLik tests.
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


def _problem(k, n, nl, ncols):
    rng = np.random.default_rng([k, ncols])
    Pm = rng.random((n - 1, k, k)) + 0.05
    Pm /= Pm.sum(axis=2, keepdims=True)
    prior = rng.dirichlet(np.ones(k))
    leaves = rng.integers(0, k, (ncols, nl)).astype(np.int32)
    r = rng.random(leaves.shape)
    leaves[r < 0.2] = -1
    leaves[(r >= 0.2) & (r < 0.21)] = k + 2  # beyond the alphabet: a vector of zeros
    return Pm, prior, leaves, rng


@pytest.mark.parametrize("k", [1, 2, 4, 5, 8, 9, 16, 20, 24, 25])
@pytest.mark.parametrize("ncols", [1, 63, 64, 65, 700])
def test_columns_match_oracle(ctx, params_dir, k, ncols):
    print("PhyloLik k = %d, %d columns" % (k, ncols), flush=True)
    text = open(os.path.join(params_dir, "12flies.nh")).read()
    tree, otree = P.newick_tree(text), O.newick_tree(text)
    Pm, prior, leaves, rng = _problem(k, tree.n, tree.nl, ncols)
    z0, post0, _ = O.lik_posteriors(otree, Pm, prior, leaves)
    it = P.PhyloLik(ctx).prepare(tree, Pm, prior, leaves)
    assert np.allclose(it.likelihood(), z0, rtol=1e-12, atol=0)
    assert np.allclose(it.node_posterior(tree.n - 1), post0[:, -1, :], rtol=1e-12, atol=1e-300)


def test_wide_tree(ctx):
    print("PhyloLik on 300 leaves", flush=True)
    text = "a0:0.1"
    for i in range(1, 300):
        text = "(%s,a%d:0.1)%s" % (text, i, ":0.1" if i < 299 else "")
    tree, otree = P.newick_tree(text + ";"), O.newick_tree(text + ";")
    Pm, prior, leaves, _ = _problem(4, tree.n, tree.nl, 130)
    leaves[leaves > 3] = 0
    Pm = 0.2 * Pm + 0.8 * np.eye(4)
    z0, post0, _ = O.lik_posteriors(otree, Pm, prior, leaves)
    it = P.PhyloLik(ctx).prepare(tree, Pm, prior, leaves)
    assert np.allclose(it.likelihood(), z0, rtol=1e-12, atol=0)
    assert np.allclose(it.node_posterior(tree.n - 1), post0[:, -1, :], rtol=1e-12, atol=1e-300)


def test_states_are_checked(ctx, params_dir):
    print("PhyloLik state checks", flush=True)
    tree = P.newick_tree(open(os.path.join(params_dir, "12flies.nh")).read())
    Pm, prior, leaves, _ = _problem(4, tree.n, tree.nl, 200)
    for state in (-2, -3):
        bad = leaves.copy()
        bad[150, 3] = state
        with pytest.raises(P.InvalidArgument):
            P.PhyloLik(ctx).prepare(tree, Pm, prior, bad)
    assert np.isfinite(P.PhyloLik(ctx).prepare(tree, Pm, prior, leaves).likelihood()).all()
