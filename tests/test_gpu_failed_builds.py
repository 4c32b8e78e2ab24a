"""A forward whose P(t) fails (Q.Diag.real_to_Pt, lib/CamlPaml/Q.ml:226-247; paths
relative to the mlin/PhyloCSF tree) leaves the batch as the last good forward left
it: results on the device and the scales that pcsf_backward differentiates; and the
next good call is as one on a fresh batch.  The model's Q has a negative
off-diagonal entry -q: exp(Qt) there is about -q t, within the clamp (1e-6) at tiny
tree scales and below it at ordinary ones.
"""
import ctypes as C
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import phylocsf_amd as P  # noqa: E402
from hip_runtime import D2H, runtime  # noqa: E402
from phylocsf_amd import _lib  # noqa: E402

GOOD, BAD = 1e-5, 1.0


@pytest.fixture(scope="module")
def model(params_dir):
    ctx = P.Context(0)
    prefix = os.path.join(params_dir, "12flies")
    ecms = [P.import_parameters(prefix + "_%s.ECM" % w) for w in ("coding", "noncoding")]
    S = ecms[0][0].copy()
    S[10, 14] = S[14, 10] = -0.05
    tree = P.newick_tree(open(prefix + ".nh").read())
    return P.PhyloCSFModel(ctx, tree, [(S, ecms[0][1]), ecms[1]])


def _batch(model):
    # one codon in all species: ordinary likelihoods at tiny scales
    codes = np.repeat(np.arange(90, dtype=np.uint8)[:, None] % 60, model.tree.nl, axis=1)
    return P.Batch(model, codes, np.array([0, 20, 90]))


def _on_device(b):
    ptr = C.c_void_p()
    assert _lib.lib().pcsf_batch_device_results(b.h, C.byref(ptr), None) == 0
    out = np.zeros((2, 2))
    assert runtime().hipMemcpy(out.ctypes.data, ptr, out.nbytes, D2H) == 0
    return out


@pytest.mark.parametrize("precision", [P.PCSF_FP64M, P.PCSF_FP64, P.PCSF_FP32])
@pytest.mark.parametrize("per_region", [False, True])
def test_failed_forward_leaves_the_last_good_one(model, precision, per_region):
    print("failed forward: precision %d, per region %d" % (precision, per_region), flush=True)
    scales = lambda x: np.full((2, 2), x) if per_region else x  # noqa: E731
    fresh = _batch(model)
    want, _ = fresh.forward(scales(GOOD), precision, per_region=per_region)
    want_g = fresh.backward(np.ones((2, 2)))[0]
    assert np.isfinite(want).all() and np.isfinite(want_g).all()
    b = _batch(model)
    assert np.array_equal(b.forward(scales(GOOD), precision, per_region=per_region)[0], want)
    for _ in range(2):
        with pytest.raises(P.Failure):
            b.forward(scales(BAD), precision, per_region=per_region)
        assert np.array_equal(_on_device(b), want)
    assert np.allclose(b.backward(np.ones((2, 2)))[0], want_g, rtol=1e-12, atol=0)
    assert np.array_equal(b.forward(scales(GOOD), precision, per_region=per_region)[0], want)


@pytest.mark.parametrize("strategy", ["fixed", "mle", "mle_grad"])
def test_failed_score_then_a_good_call(model, strategy):
    print("failed score: " + strategy, flush=True)
    b = _batch(model)
    want = _batch(model).forward(GOOD, P.PCSF_FP64M)[0]
    for _ in range(2):
        with pytest.raises(P.Failure):
            P.score(b, strategy, P.PCSF_FP64M)
        assert np.array_equal(b.forward(GOOD, P.PCSF_FP64M)[0], want)
        with pytest.raises(P.Failure):
            model.transition(0, BAD)
