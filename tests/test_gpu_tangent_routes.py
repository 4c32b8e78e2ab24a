"""The tangent pass on trees without a generated program at one and at two workgroups
per CU: a region's gradient is the same bits in a small batch and in a large one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import phylocsf_amd as P  # noqa: E402


@pytest.fixture(scope="module")
def ctx():
    return P.Context(0)


def _balanced(levels, first=0):
    """A balanced tree of 2^levels leaves: the deepest programs, six live tiles at 64."""
    if levels == 0:
        return "s%d:0.06" % first
    return "(%s,%s):0.05" % (_balanced(levels - 1, first),
                             _balanced(levels - 1, first + 2 ** (levels - 1)))


def _model(ctx, name):
    if name != "balanced64":
        return P.PhyloCSFModel.from_paramset(ctx, name)
    prefix = P.paramset_prefix("58mammals")
    ecms = [P.import_parameters(prefix + "_%s.ECM" % w) for w in ("coding", "noncoding")]
    return P.PhyloCSFModel(ctx, P.newick_tree(_balanced(6).rsplit(":", 1)[0] + ";"), ecms)


@pytest.mark.parametrize("name", ["7yeast", "23flies", "53birds", "balanced64"])
def test_gradients_do_not_depend_on_the_batch(ctx, name):
    print("tangent routes: " + name, flush=True)
    m = _model(ctx, name)
    lengths = np.array([1, 15, 64, 65, 200])
    rng = np.random.default_rng(3)
    got = []
    for filler in (0, 64 * 150):  # 18 and 318 blocks over both models
        n = np.append(lengths, filler)
        codes, off = m.simulate(n, np.zeros(len(n), int), np.ones(len(n)), gap_p=0.15, seed=6)
        b = P.Batch(m, codes, off)
        if not got:
            rho = rng.uniform(0.2, 3.0, (len(n), 2))
        b.forward(rho, P.PCSF_FP16S, per_region=True)
        got.append(b.backward(np.ones((len(n), 2)))[0][:-1])
    assert np.array_equal(got[0], got[1])
    # and they are derivatives: the FP64 outside pass's, to the tangent's own tolerance
    b.forward(rho, P.PCSF_FP64M, per_region=True)
    want = b.backward(np.ones((len(n), 2)))[0][:-1]
    assert np.all(np.abs(got[0] - want) <= 2e-4 * np.maximum(1.0, np.abs(want)))
