"""The FP64 outside pass at the edges of its 16-column tiles and of its trees:
two leaves (no product), three (one product), caterpillars (every node's
message and w pass through registers) and random trees (w of the second
internal child waits in memory), a tree too large for the arrays in LDS, and
regions around a tile's and a block's edge, gaps included.  Against the
oracle's gradient through branch posteriors, at the bounds of the gradient's
other tests (1e-9 relative for d lpr / d rho, 1e-8 for a branch: FP64 sums
over up to 130 columns in another order).
"""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import phylocsf_amd as P  # noqa: E402
from oracle import oracle as O  # noqa: E402

EDGES = np.array([1, 15, 16, 17, 0, 33, 64, 65, 130])


@pytest.fixture(scope="module")
def ctx():
    return P.Context(0)


def _newick(kind, nl, branch):
    rng = np.random.default_rng(nl)
    parts = ["s%d:%g" % (i, branch) for i in range(nl)]
    while len(parts) > 1:
        i = 0 if kind == "caterpillar" else int(rng.integers(0, len(parts) - 1))
        parts[i:i + 2] = ["(%s,%s):%g" % (parts[i], parts[i + 1], branch * rng.uniform(0.5, 2))]
    return parts[0].rsplit(":", 1)[0] + ";"


@pytest.mark.parametrize("kind,nl,branch,lengths", [
    ("random", 2, 0.3, EDGES), ("caterpillar", 3, 0.3, EDGES), ("caterpillar", 12, 0.1, EDGES),
    ("random", 40, 0.05, EDGES), ("caterpillar", 700, 0.002, np.array([3, 17]))])
def test_gradient_against_oracle(ctx, params_dir, kind, nl, branch, lengths):
    print("outside pass, %s tree of %d leaves" % (kind, nl), flush=True)
    prefix = os.path.join(params_dir, "29mammals")
    text = _newick(kind, nl, branch)
    m = P.PhyloCSFModel(ctx, P.newick_tree(text), [P.import_parameters(prefix + "_coding.ECM"),
                                                   P.import_parameters(prefix + "_noncoding.ECM")])
    ecm = [O.ecm_read(prefix + "_%s.ECM" % s) for s in ("coding", "noncoding")]
    om = O.Model(O.newick_tree(text), [e[0] for e in ecm], [e[1] for e in ecm])
    codes, off = m.simulate(lengths, np.arange(len(lengths)) % 2, np.ones(len(lengths)),
                            gap_p=0.15, n_p=0.02, seed=9)
    rho = np.random.default_rng(3).uniform(0.3, 3.0, (len(lengths), 2))
    b = P.Batch(m, codes, off)
    b.forward(rho, P.PCSF_FP64M, per_region=True)
    grho, gbr = b.backward(np.ones_like(rho), branches=True)
    only_rho, _ = b.backward(np.ones_like(rho))
    assert np.allclose(only_rho, grho, rtol=1e-12, atol=1e-12)
    for r in range(len(lengths)):
        for q in range(2):
            _, d, g = om.lpr_grad(q, rho[r, q], codes[off[r]:off[r + 1]])
            assert abs(grho[r, q] - d) <= 1e-9 * max(1.0, abs(d)), (r, q)
            assert np.allclose(gbr[r, q], g, rtol=1e-8, atol=1e-9), (r, q)
