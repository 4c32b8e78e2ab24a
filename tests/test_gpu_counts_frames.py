"""Edges of the E-step's column tiles and of the reading-frame kernel's steps.

* Expected counts over 1 to 130 columns (around a 16-column tile and a 64-column
  block), on two leaves (no product: only the root's prior and leaf tables), three,
  and a random tree, with `Marginalize leaves, states beyond the alphabet and
  weights, against the oracle (FP64 sums of at most 130 posteriors in another
  order: 1e-10 relative, as the E-step's other tests).
* Reading frames of regions around 256 codons (a workgroup's step through its
  (leaf, codon) pairs), of every byte value, in few regions (shared out by
  leaves) and in many, against numpy: whole numbers, equal.
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


@pytest.mark.parametrize("nl", [2, 3, 19])
def test_estep_edges(ctx, params_dir, nl):
    print("E-step edges, %d leaves" % nl, flush=True)
    rng = np.random.default_rng(nl)
    parts = ["s%d:0.2" % i for i in range(nl)]
    while len(parts) > 1:
        i = int(rng.integers(0, len(parts) - 1))
        parts[i:i + 2] = ["(%s,%s):%g" % (parts[i], parts[i + 1], rng.uniform(0.05, 0.4))]
    text = parts[0].rsplit(":", 1)[0] + ";"
    tree, otree = P.newick_tree(text), O.newick_tree(text)
    S, pi = O.ecm_read(os.path.join(params_dir, "12flies_coding.ECM"))
    Q = O.build_q(S, pi)
    Pm = np.stack([O.pt(Q, pi, t) for t in otree.branch[:-1]])
    for ncols in (1, 15, 16, 17, 63, 64, 65, 130):
        leaves = rng.integers(0, 64, (ncols, nl)).astype(np.int32)
        leaves[rng.random(leaves.shape) < 0.2] = -1
        leaves[rng.random(leaves.shape) < 0.02] = 64
        w = rng.uniform(0.5, 2.0, ncols)
        z0, _, ec0 = O.lik_posteriors(otree, Pm, pi, leaves, None, w, posteriors=False)
        ec = np.zeros((tree.n - 1, 64, 64))
        z = P.collect_sufficient_statistics(ctx, tree, Pm, pi, leaves, ec, weights=w)
        assert np.allclose(z, z0, rtol=1e-11, atol=0), ncols
        assert np.allclose(ec, ec0, rtol=1e-10, atol=1e-13), ncols


@pytest.mark.parametrize("regions", [1, 5, 400])
def test_frames_edges(ctx, regions):
    print("frames, %d regions" % regions, flush=True)
    m = P.PhyloCSFModel.from_paramset(ctx, "12flies")
    rng = np.random.default_rng(regions)
    lens = rng.choice([0, 2, 3, 4, 5, 63 * 3, 255 * 3 + 2, 256 * 3, 257 * 3 + 1], regions)
    if regions == 1:
        lens[:] = 257 * 3 + 1
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    letters = np.frombuffer(b"ACGTacgt" * 30 + bytes(range(256)), np.uint8)
    nuc = rng.choice(letters, (m.tree.nl, off[-1])).astype(np.uint8)
    index = np.full(256, 4)
    for i, c in enumerate(b"ACGT"):
        index[c] = index[c + 32] = i
    want = []
    for r in range(regions):
        fwd = index[nuc[:, off[r]:off[r + 1]]]
        rev = np.where(fwd == 4, 4, 3 - fwd)[:, ::-1]
        for f in range(6):
            x = (fwd if f < 3 else rev)[:, f % 3:]
            k = x.shape[1] // 3
            x = x[:, :3 * k].reshape(m.tree.nl, k, 3)
            want.append(np.where((x == 4).any(2), 255, x @ np.array([16, 4, 1])).T)
    codes, foff = P.Batch.frames(m, np.ascontiguousarray(nuc), off, 6).codes()
    assert np.array_equal(np.diff(foff), [len(x) for x in want])
    assert np.array_equal(codes, np.concatenate(want).astype(np.uint8))
