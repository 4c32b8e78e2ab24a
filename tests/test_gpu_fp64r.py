"""The FP64M forward's three routes by amount of work (one 16-column tile per
workgroup with rows split over its waves, two tiles, the tree's generated
program) give the same bits: every element is the same sum in the same order.

Regions at the edges of a 16-, 32- and 64-column tile are scored alone (the
first route), beside a filler region that takes the batch to the second, and
beside one that takes it to the third; a region's value must not change, at
the shared scale and at scales of its own.  The small batch is also held to
the plain FP64 kernel (another summation order: 1e-12 relative, the bound of
its own tests).  The route's program reads ops in pairs, which the CPU test
checks for every shipped tree and for random ones.
"""
import os

import numpy as np
import pytest

import phylocsf_amd as P
from phylocsf_amd.api import program

OP_GEMM, OP_ROOT, OP_END = 2, 5, 6
EDGES = np.array([1, 15, 16, 17, 31, 33, 48, 63, 64, 65, 0, 129])


def _check_pairs(ops):
    op = ops[:, 0] & 0xFF
    assert op[-1] == OP_END and op[-2] == OP_ROOT and len(op) % 2 == 1
    assert (op[1:-2:2] == OP_GEMM).all()
    assert not np.isin(op[0:-1:2], (OP_GEMM, OP_ROOT)).any()


@pytest.mark.parametrize("name", ["7yeast", "12flies", "23flies", "29mammals", "53birds",
                                  "58mammals", "100vertebrates", "120mammals"])
def test_program_alternates_nodes_and_products(params_dir, name):
    text = open(os.path.join(params_dir, name + ".nh")).read()
    _check_pairs(program(P.newick_tree(text))[0])


def test_program_alternates_on_random_trees():
    rng = np.random.default_rng(4)
    for nl in (2, 3, 4, 9, 40, 200):
        parts = ["s%d:0.1" % i for i in range(nl)]
        while len(parts) > 1:
            i = int(rng.integers(0, len(parts) - 1))
            parts[i:i + 2] = ["(%s,%s):0.1" % (parts[i], parts[i + 1])]
        _check_pairs(program(P.newick_tree(parts[0].rsplit(":", 1)[0] + ";"))[0])


@pytest.fixture(scope="module")
def ctx():
    return P.Context(0)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["12flies", "53birds", "58mammals", "120mammals"])
def test_routes_give_the_same_bits(ctx, name):
    print("FP64M routes: " + name, flush=True)
    m = P.PhyloCSFModel.from_paramset(ctx, name)
    rng = np.random.default_rng(8)
    rho = rng.uniform(0.1, 4.0, (len(EDGES) + 1, 2))
    got = []
    for filler in (0, 64 * 100, 64 * 520):  # 30, 230 and 1070 blocks over both models
        lengths = np.append(EDGES, filler)
        codes, off = m.simulate(lengths, np.zeros(len(lengths), int), np.ones(len(lengths)),
                                gap_p=0.15, n_p=0.02, seed=6)
        b = P.Batch(m, codes, off)
        fixed = b.forward(0.8, P.PCSF_FP64M)
        own = b.forward(rho, P.PCSF_FP64M, per_region=True)
        got.append([x[:-1] for x in fixed + own])
        if filler == 0:
            plain = b.forward(0.8, P.PCSF_FP64) + b.forward(rho, P.PCSF_FP64, per_region=True)
            for x, y in zip(got[0], plain):
                assert np.all(np.abs(x - y[:-1]) <= 1e-12 * np.maximum(1.0, np.abs(y[:-1])))
    for other in got[1:]:
        for x, y in zip(got[0], other):
            assert np.array_equal(x, y)


@pytest.mark.gpu
def test_two_leaves(ctx, params_dir):
    """A tree of two leaves has no product at all."""
    print("FP64M, two leaves", flush=True)
    m = P.PhyloCSFModel.from_paramset(ctx, "12flies", ["dmel", "dsim"])
    codes, off = m.simulate([1, 40, 200], [0, 1, 0], [1.0, 1.0, 1.0], gap_p=0.2, seed=2)
    b = P.Batch(m, codes, off)
    for x, y in zip(b.forward(1.0, P.PCSF_FP64M), b.forward(1.0, P.PCSF_FP64)):
        assert np.all(np.abs(x - y) <= 1e-12 * np.maximum(1.0, np.abs(y)))
