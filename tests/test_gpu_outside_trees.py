"""The FP64 outside pass on trees of hundreds of leaves, whose arrays take up to the
60 KB of LDS beside the kernel's own, and the first that does not: the gradient in
tree scale against the oracle's, at the bound of the pass's other tests.
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


# LDS of the arrays: 16 bytes per leaf, 40 per branch, 8 per inner node
@pytest.mark.parametrize("nl", [440, 500, 591, 592])
def test_gradient_against_oracle(ctx, params_dir, nl):
    print("outside pass, %d leaves, %d bytes" % (nl, 16 * nl + 40 * (2 * nl - 2) + 8 * (nl - 1)),
          flush=True)
    prefix = os.path.join(params_dir, "29mammals")
    text = "s0:0.002"
    for i in range(1, nl):
        text = "(%s,s%d:0.002):0.002" % (text, i)
    text = text.rsplit(":", 1)[0] + ";"
    m = P.PhyloCSFModel(ctx, P.newick_tree(text), [P.import_parameters(prefix + "_coding.ECM"),
                                                   P.import_parameters(prefix + "_noncoding.ECM")])
    ecm = [O.ecm_read(prefix + "_%s.ECM" % s) for s in ("coding", "noncoding")]
    om = O.Model(O.newick_tree(text), [e[0] for e in ecm], [e[1] for e in ecm])
    codes, off = m.simulate([3], [0], [1.0], gap_p=0.15, n_p=0.02, seed=9)
    rho = np.array([[0.7, 1.6]])
    b = P.Batch(m, codes, off)
    b.forward(rho, P.PCSF_FP64M, per_region=True)
    grho, _ = b.backward(np.ones_like(rho))
    for q in range(2):
        d = om.lpr_grad(q, rho[0, q], codes)[1]
        assert abs(grho[0, q] - d) <= 1e-9 * max(1.0, abs(d)), q
