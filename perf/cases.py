"""The work that users of phylocsf_amd have it do, as cases that can be timed and checked.

Twelve listed cases and a draw over the ranges that they stand for.  A case names a `kind`:

  score      a new alignment set scored once: leaf codes on the host -> Batch -> score (or score_omega),
             the way the command line scores each set of candidate regions
  frames     the same from nucleotide rows: Batch.frames in every reading frame, then score_fixed
  forward    lpr and elpr of a resident batch at the tree's own scale (a genome kept on the GPU)
  gradient   lpr at per-region tree scales and its gradient in every branch length, as a fitting
             loop over a resident batch takes them
  counts     PhyloEM's E-step: expected substitution counts of every branch over many columns
  columns    PhyloLik.prepare: likelihood and root posterior of every column for caller-made P matrices

Alignments are simulated here with torch (root ~ pi, children ~ rows of P, then gaps and N codons), so
that the inputs depend on the seed alone.  Parameter sets are the shipped ones; lengths, gap rates and
tree scales are those of the repository's scoring workloads.
"""
from __future__ import annotations

import functools
import math
import random
import re

import numpy as np
import torch

import phylocsf_amd as P

FP32, FP16S, FP64, FP64M = P.PCSF_FP32, P.PCSF_FP16S, P.PCSF_FP64, P.PCSF_FP64M
GAP = 255
BASES = np.frombuffer(b"ACGT", dtype=np.uint8)
DEVICE = "cuda" if torch.cuda.is_available() else "cpu"


# ---- the cases ---------------------------------------------------------------------------------


def _case(kind, paramset, **more):
    """A case with the options of its kind spelled out: `species` 0 = every leaf of the tree, else that
    many of them (--species); regions of lo..hi codons; `strategy` and `precision` as score() takes them."""
    c = dict(kind=kind, paramset=paramset, species=0, regions=1, lo=100, hi=100, strategy="fixed",
             precision=FP64M, gap=0.1, run=0.0, rho=False, states=64)
    c.update(more)
    return c


def listed():
    return [
        # one short exon, fixed score: an interactive query, the smallest call there is (all latency)
        dict(_case("score", "12flies", precision=FP32, gap=0.0), name="exon_fixed_fp32"),
        # one exon by maximum likelihood at the command line's default precision: what PhyloCSF does
        # for each alignment file (the published ALDH2 exon has 37 codons in 29 mammals)
        dict(_case("score", "29mammals", strategy="mle", lo=37, hi=37), name="exon_mle_fp64m"),
        # a gene's candidate exons with --species: a pruned tree, for which no kernel was generated
        dict(_case("score", "58mammals", species=20, regions=24, lo=30, hi=400, strategy="mle"),
             name="gene_species_mle_fp64m"),
        # a genome's regions kept on the GPU, fixed strategy: the headline workload's lengths
        dict(_case("forward", "58mammals", regions=4000, lo=50, hi=2000, precision=FP16S, gap=0.11),
             name="genome_fixed_fp16s"),
        # an ordinary set in FP64 on a tree without generated kernels
        dict(_case("forward", "53birds", regions=300, lo=50, hi=1500), name="birds_fixed_fp64m"),
        # an ORF scan: six reading frames of every region from nucleotide rows, gaps in runs
        dict(_case("frames", "120mammals", regions=500, lo=20, hi=600, precision=FP32, gap=0.25, run=5.0),
             name="frames6_fixed_fp32"),
        # maximum likelihood over a set of transcripts, searched in split FP16
        dict(_case("score", "100vertebrates", regions=300, lo=30, hi=1500, strategy="mle", precision=FP16S,
                   gap=0.0, rho=True), name="transcripts_mle_fp16s"),
        # the same by gradient (forward-mode tangent pass), long regions with gaps
        dict(_case("score", "100vertebrates", regions=120, lo=100, hi=3000, strategy="mle_grad",
                   precision=FP16S, gap=0.15), name="transcripts_mlegrad_fp16s"),
        # a branch-length fit: FP64 forward and outside pass per step
        dict(_case("gradient", "100vertebrates", regions=60, lo=100, hi=1500, gap=0.15, rho=True),
             name="branch_gradients_fp64m"),
        # the omega (dN/dS) test of a gene family's regions
        dict(_case("score", "58mammals", regions=40, lo=150, hi=600, strategy="omega"), name="omega_fp64m"),
        # one E-step of an ECM re-estimation
        dict(_case("counts", "58mammals", regions=120, lo=50, hi=2000), name="estep_codons"),
        # a nucleotide model through PhyloLik (the library's other alphabet), every alignment column
        dict(_case("columns", "58mammals", regions=60, lo=200, hi=2000, states=4), name="lik_nucleotides"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    trees = ["12flies", "23flies", "29mammals", "53birds", "58mammals", "100vertebrates", "120mammals"]
    kind = rng.choice(["exon", "mle", "mle", "grad", "omega", "forward", "forward", "frames", "gradient",
                       "counts", "columns"])
    lo = rng.randint(20, 120)
    hi = lo + _log_int(rng, 1, 1500)
    gap = round(rng.uniform(0.0, 0.3), 3)
    if kind == "exon":
        return _case("score", rng.choice(trees), lo=lo, hi=lo + rng.randint(0, 200), gap=gap,
                     strategy=rng.choice(["fixed", "mle"]), precision=rng.choice([FP32, FP16S, FP64M]))
    if kind == "mle":
        tree = rng.choice(trees)
        return _case("score", tree, species=rng.choice([0, 0, rng.randint(5, 12)]), lo=lo, hi=hi, gap=gap,
                     regions=_log_int(rng, 1, 120), strategy="mle", precision=rng.choice([FP16S, FP64M, FP64M]),
                     rho=rng.random() < 0.5)
    if kind == "grad":
        return _case("score", rng.choice(trees), regions=_log_int(rng, 1, 100), lo=lo, hi=hi, gap=gap,
                     strategy="mle_grad", precision=FP16S, rho=rng.random() < 0.5)
    if kind == "omega":
        return _case("score", rng.choice(["12flies", "29mammals", "58mammals"]), regions=_log_int(rng, 1, 40),
                     lo=150, hi=150 + _log_int(rng, 1, 450), strategy="omega", gap=gap)
    if kind == "forward":
        return _case("forward", rng.choice(trees), regions=_log_int(rng, 1, 1500), lo=lo, hi=hi, gap=gap,
                     precision=rng.choice([FP32, FP16S, FP16S, FP64M]))
    if kind == "frames":
        return _case("frames", rng.choice(trees), regions=_log_int(rng, 1, 400), lo=20, hi=20 + _log_int(rng, 1, 580),
                     gap=gap, run=5.0, precision=rng.choice([FP32, FP16S]))
    if kind == "gradient":
        return _case("gradient", rng.choice(trees), regions=_log_int(rng, 1, 60), lo=lo, hi=hi, gap=gap, rho=True)
    if kind == "counts":
        return _case("counts", rng.choice(trees), regions=_log_int(rng, 1, 100), lo=lo, hi=hi, gap=gap)
    return _case("columns", rng.choice(trees[:5]), regions=_log_int(rng, 1, 50), lo=lo, hi=hi, gap=gap, states=4)


# ---- trees and rate models, from the parameter files --------------------------------------------


def _prune(node, keep):
    """Newick.subtree: the tree over the species in `keep` (None where nothing is left)."""
    kids, label, bl = node
    if label and label not in keep:
        return None
    if not kids:
        return node
    left = [k for k in (_prune(x, keep) for x in kids) if k]
    if len(left) == 1:
        return left[0][0], left[0][1], bl + left[0][2]
    return (left, label, bl) if left else None


@functools.lru_cache(maxsize=None)
def _tree(paramset, species):
    """(children [n_internal, 2], branch [n - 1], names of the kept species or None): leaves left to
    right, then internal nodes in post-order, the root last."""
    text = open(P.paramset_prefix(paramset) + ".nh").read()
    tokens = re.findall(r"[(),:;]|[^(),:;\s]+", text)
    pos = 0

    def node():
        nonlocal pos
        kids, label, bl = [], "", 0.0
        if tokens[pos] == "(":
            while tokens[pos] != ")":
                pos += 1
                kids.append(node())
            pos += 1
        if pos < len(tokens) and tokens[pos] not in "(),:;":
            label, pos = tokens[pos], pos + 1
        if pos < len(tokens) and tokens[pos] == ":":
            bl, pos = float(tokens[pos + 1]), pos + 2
        return kids, label, bl

    root, names = node(), None
    if species:
        labels = [t for t in tokens if re.match(r"[A-Za-z_]", t)]
        names = [labels[(i * len(labels)) // species] for i in range(species)]
        root = _prune(root, set(names))
    leaves, inner = [], []

    def number(x):
        if not x[0]:
            leaves.append(x[2])
            return len(leaves) - 1
        kids = [number(k) for k in x[0]]
        inner.append((kids, x[2]))
        return -len(inner)

    number(root)
    nl = len(leaves)
    children = np.array([[k if k >= 0 else nl - 1 - k for k in kids] for kids, _ in inner], dtype=np.int32)
    return children, np.array(leaves + [b for _, b in inner[:-1]]), names


@functools.lru_cache(maxsize=None)
def _eigen(paramset, which, states):
    """(U, lambda, pi) of Pi^1/2 Q Pi^-1/2, mean rate one: a shipped ECM, or a four-state model."""
    if states == 4:
        pi = np.array([0.29, 0.21, 0.21, 0.29])
        s = np.ones((4, 4))
        s[0, 2] = s[2, 0] = s[1, 3] = s[3, 1] = 3.2
    else:
        numbers = []
        for t in open("%s_%s.ECM" % (P.paramset_prefix(paramset), ("coding", "noncoding")[which])).read().split():
            if t[0].isalpha():
                break
            numbers.append(float(t))
        s = np.zeros((64, 64))
        s[np.tril_indices(64, -1)] = numbers[:2016]
        s, pi = s + s.T, np.array(numbers[2016:2080])
    q = s * pi
    np.fill_diagonal(q, 0.0)
    np.fill_diagonal(q, -q.sum(1))
    q /= -(pi * np.diag(q)).sum()
    root = np.sqrt(pi)
    a = root[:, None] * q / root
    lam, u = np.linalg.eigh((a + a.T) / 2)
    return u, lam, pi, q


def _transitions(paramset, which, states, t):
    """P(t) for every t: [len(t), k, k], tiny negatives set to 0 and the diagonal 1 - the others."""
    u, lam, pi, _ = _eigen(paramset, which, states)
    root = np.sqrt(pi)
    p = np.einsum("im,tm,jm->tij", u / root[:, None], np.exp(np.outer(t, lam)), u * root[:, None], optimize=True)
    p = np.maximum(p, 0.0)
    i = np.arange(states)
    p[:, i, i] = 0.0
    p[:, i, i] = 1.0 - p.sum(2)
    return p


# ---- inputs -------------------------------------------------------------------------------------


def _regions(case, seed):
    """Offsets [R + 1], generating model and tree scale of every region; the lengths are the case's own,
    so that outputs of every seed have the same shapes."""
    lengths = np.random.default_rng([case["regions"], case["lo"], case["hi"]]).integers(
        case["lo"], case["hi"] + 1, case["regions"])
    rng = np.random.default_rng([seed, 17])
    model = rng.permutation(np.arange(case["regions"]) % 2)
    scales = np.array([0.3, 0.5, 0.8, 1.0, 1.4, 1.9, 2.4, 3.0])
    rho = rng.choice(scales, case["regions"]) if case["rho"] else np.ones(case["regions"])
    return np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64), model, rho


def _alignment(case, seed):
    """Leaf states [n_cols, n_leaves] (uint8, GAP = no codon) and region offsets."""
    children, branch, _ = _tree(case["paramset"], case["species"])
    nl, k = len(children) + 1, case["states"]
    off, model, rho = _regions(case, seed)
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)
    ncols = int(off[-1])
    col_class = np.repeat(model + 2 * (rho * 10).round().astype(np.int64), np.diff(off))
    out = torch.empty((nl, ncols), dtype=torch.uint8, device=DEVICE)
    for c in np.unique(col_class):
        at = torch.from_numpy(np.flatnonzero(col_class == c)).to(DEVICE)
        p = _transitions(case["paramset"], int(c % 2), k, branch * ((c // 2) / 10.0))
        # row r of a branch's cumulative P, moved to [r, r + 1]: one sorted table per branch
        rows = np.ascontiguousarray(np.cumsum(p, 2) + np.arange(k)[None, :, None]).reshape(len(branch), k * k)
        steps = torch.from_numpy(rows).to(DEVICE)
        pi = torch.from_numpy(np.cumsum(_eigen(case["paramset"], int(c % 2), k)[2])).to(DEVICE)
        uniform = lambda: torch.rand(len(at), generator=gen, device=DEVICE, dtype=torch.float64)  # noqa: E731
        state = {len(branch): torch.searchsorted(pi, uniform()).clamp_(max=k - 1)}
        for i in range(len(branch), nl - 1, -1):
            above = state.pop(i)
            for child in children[i - nl]:
                got = torch.searchsorted(steps[child], above + uniform()) - above * k
                got = got.clamp_(0, k - 1)
                if child < nl:
                    out[child, at] = got.to(torch.uint8)
                else:
                    state[int(child)] = got
    if case["gap"] > 0 and ncols:  # the reference species (leaf 0) has no gaps
        draws = torch.rand((nl - 1, ncols), generator=gen, device=DEVICE)
        absent = draws < case["gap"]
        if case["run"] > 0:  # a run ends with probability 1 / run at each column, then gap or not anew
            new = torch.rand((nl - 1, ncols), generator=gen, device=DEVICE) < 1.0 / case["run"]
            last = torch.where(new, torch.arange(ncols, device=DEVICE), torch.zeros((), dtype=torch.int64, device=DEVICE))
            absent = absent.gather(1, last.cummax(1).values)
        out[1:][absent] = GAP
    return out.t().contiguous().cpu().numpy(), off


def _nucleotides(codes, off):
    """The alignment as nucleotide rows [n_leaves, 3 n_cols] and nucleotide offsets."""
    c = codes.T.astype(np.int16)
    n = np.stack([BASES[(c >> s) & 3] for s in (4, 2, 0)], axis=2)
    n[c == GAP] = ord("-")
    return np.ascontiguousarray(n.reshape(codes.shape[1], -1)), 3 * off


@functools.lru_cache(maxsize=None)
def _context():
    return P.Context(0)


def _newick(case):
    names = _tree(case["paramset"], case["species"])[2]
    return P.newick_tree(open(P.paramset_prefix(case["paramset"]) + ".nh").read(), names), names


def prepare(case, seed):
    """What a program holds before the call: the context, the model of the tree, and the alignment."""
    codes, off = _alignment(case, seed)
    ctx = _context()
    tree, names = _newick(case)
    state = {"case": case, "ctx": ctx, "tree": tree}
    if case["kind"] in ("counts", "columns"):
        which = 0
        branch = _tree(case["paramset"], case["species"])[1]
        state["P"] = _transitions(case["paramset"], which, case["states"], branch)
        state["pi"] = _eigen(case["paramset"], which, case["states"])[2]
        state["leaves"] = np.where(codes == GAP, -1, codes.astype(np.int32))
        state["lik"] = P.PhyloLik(ctx)
        return state
    if case["strategy"] == "omega":
        state["model"] = P.PhyloCSFModel.tree_only(ctx, tree)
    else:
        state["model"] = P.PhyloCSFModel.from_paramset(ctx, case["paramset"], names)
    if case["kind"] == "frames":
        state["nuc"], state["off"] = _nucleotides(codes, off)
    elif case["kind"] == "score":
        state["codes"], state["off"] = codes, off
    else:  # resident on the GPU
        state["batch"] = P.Batch(state["model"], codes, off)
        rho = _regions(case, seed)[2]
        state["rho"] = np.repeat(rho[:, None], 2, axis=1) * np.array([1.0, 1.1])
        state["weights"] = np.ones((case["regions"], 2))
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "score":
        batch = P.Batch(state["model"], state["codes"], state["off"])
        if case["strategy"] == "omega":
            return P.score_omega(batch, precision=case["precision"])
        return P.score(batch, case["strategy"], case["precision"])
    if case["kind"] == "frames":
        batch = P.Batch.frames(state["model"], state["nuc"], state["off"], 6)
        return P.score_fixed(batch, case["precision"])
    if case["kind"] == "forward":
        lpr, elpr = state["batch"].forward(1.0, case["precision"])
        return {"lpr": lpr, "elpr": elpr}
    if case["kind"] == "gradient":
        lpr, elpr = state["batch"].forward(state["rho"], case["precision"], per_region=True)
        drho, dbranch = state["batch"].backward(state["weights"], branches=True)
        return {"lpr": lpr, "elpr": elpr, "drho": drho, "dbranch": dbranch}
    if case["kind"] == "counts":
        k = case["states"]
        counts = np.zeros((state["tree"].n - 1, k, k))
        z = P.collect_sufficient_statistics(state["ctx"], state["tree"], state["P"], state["pi"],
                                            state["leaves"], counts)
        return {"z": z, "counts": counts}
    it = state["lik"].prepare(state["tree"], state["P"], state["pi"], state["leaves"])
    return {"z": it.likelihood(), "root": it.node_posterior(state["tree"].n - 1)}


# ---- the work that a pass cannot do without -----------------------------------------------------


def work(case):
    """Each input byte read once and each result written once; one k x k product per internal branch and
    column (two for a gradient or the counts, and the product's derivative or the rank-one update)."""
    children, branch, _ = _tree(case["paramset"], case["species"])
    nl, k = len(children) + 1, case["states"]
    ncols = case["regions"] * (case["lo"] + case["hi"]) / 2.0
    nreg, models, passes, inner = case["regions"], 2, 1, nl - 2
    product = 2.0 * k * k
    if case["kind"] == "counts":
        return {"bytes": ncols * (4 * nl + 8) + 3 * len(branch) * k * k * 8,
                "flops": ncols * product * (2 * inner + len(branch))}
    if case["kind"] == "columns":
        return {"bytes": ncols * (4 * nl + 8 + 8 * k) + len(branch) * k * k * 8, "flops": ncols * product * inner}
    if case["kind"] == "gradient":
        return {"bytes": ncols * nl + nreg * models * 8 * (len(branch) + 4),
                "flops": ncols * models * product * (3 * inner + inner)}
    if case["kind"] == "frames":
        return {"bytes": ncols * 3 * nl + 6 * nreg * 32, "flops": 6 * ncols * models * product * inner}
    # evaluations of a fit: find_init's four and about ten Brent steps; a root search's grid and gradients;
    # three rounds of two such fits for the omega test's hypotheses
    passes = {"fixed": 1, "mle": 14, "mle_grad": 14, "omega": 65}[case["strategy"]]
    return {"bytes": ncols * nl + nreg * 80, "flops": passes * ncols * models * product * inner}


# ---- the same results in 64 bits, by plain torch ------------------------------------------------


def _messages(children, p, prior, states):
    """(z [c], alpha and message tensors per node, each [k, c]) of columns `states` [nl, c]; GAP = all."""
    nl, k = len(children) + 1, len(prior)
    ones = torch.ones((k, 1), dtype=torch.float64, device=DEVICE)
    eye = torch.cat([torch.eye(k, dtype=torch.float64, device=DEVICE), ones], 1)
    at = torch.where(states == GAP, torch.full_like(states, k), states).long()
    alpha, message = {}, {}
    for i in range(nl, 2 * nl - 1):
        alpha[i] = 1.0
        for c in children[i - nl]:
            c = int(c)
            message[c] = (p[c] @ eye)[:, at[c]] if c < nl else p[c] @ alpha[c]
            alpha[i] = alpha[i] * message[c]
    root = alpha[2 * nl - 2] * prior[:, None]
    return root.sum(0), root, alpha, message


def exact(case, seed):
    if case["kind"] == "score" and case["strategy"] != "fixed":
        return None  # a maximiser's estimates depend on its steps
    codes, off = _alignment(case, seed)
    children, branch, _ = _tree(case["paramset"], case["species"])
    nl, k = len(children) + 1, case["states"]
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEVICE)  # noqa: E731
    if case["kind"] == "counts":
        return _exact_counts(case, codes, children, branch, to)
    if case["kind"] == "columns":
        pi = to(_eigen(case["paramset"], 0, k)[2])
        p = to(_transitions(case["paramset"], 0, k, branch))
        z, root = torch.empty(len(codes), dtype=torch.float64), torch.empty((len(codes), k), dtype=torch.float64)
        for a in range(0, len(codes), 1 << 16):
            zz, r, _, _ = _messages(children, p, pi, to(codes[a:a + (1 << 16)].T))
            z[a:a + (1 << 16)], root[a:a + (1 << 16)] = zz.cpu(), (r / zz).t().cpu()
        return {"z": z, "root": root}
    if case["kind"] == "gradient":
        return _exact_gradient(case, seed, codes, off, children, branch, to)
    if case["kind"] == "frames":
        codes, off = _frames(codes, off)
    lpr, elpr = np.zeros((len(off) - 1, 2)), np.zeros((len(off) - 1, 2))
    for m in range(2):
        pi = to(_eigen(case["paramset"], m, k)[2])
        p = to(_transitions(case["paramset"], m, k, branch))
        lz, el = [], []
        for a in range(0, len(codes), 1 << 16):
            z, r, _, _ = _messages(children, p, pi, to(codes[a:a + (1 << 16)].T))
            lz.append(z.log())
            el.append((r * pi.log()[:, None]).sum(0) / z)
        for per_col, into in ((lz, lpr), (el, elpr)):
            total = np.concatenate([[0.0], torch.cat(per_col).cpu().numpy()])
            into[:, m] = [math.fsum(total[1 + a:1 + b]) for a, b in zip(off[:-1], off[1:])]
    if case["kind"] == "forward":
        return {"lpr": lpr, "elpr": elpr}
    score, anc = P.DB * (lpr[:, 0] - lpr[:, 1]), P.DB * (elpr[:, 0] - elpr[:, 1])
    if case["kind"] == "frames":
        return {"score": score, "anc_comp": anc, "lpr_c": lpr[:, 0], "lpr_n": lpr[:, 1]}
    return {"score": score, "anc_comp": anc, "lpr": lpr, "elpr": elpr, "rho": np.ones_like(lpr)}


def _frames(codes, off):
    """Codes of the six reading frames of every region, region by region."""
    nuc, noff = _nucleotides(codes, off)
    index = np.full(256, -1, dtype=np.int64)
    index[BASES] = np.arange(4)
    rows, lengths = [], []
    for a, b in zip(noff[:-1], noff[1:]):
        fwd = index[nuc[:, a:b]]
        rev = np.where(fwd[:, ::-1] < 0, -1, 3 - fwd[:, ::-1])
        for strand in (fwd, rev):
            for f in range(3):
                n = max(0, (strand.shape[1] - f) // 3)
                x = strand[:, f:f + 3 * n].reshape(len(strand), n, 3)
                code = x @ np.array([16, 4, 1])
                rows.append(np.where((x < 0).any(2), GAP, code).T.astype(np.uint8))
                lengths.append(n)
    return np.concatenate(rows), np.concatenate([[0], np.cumsum(lengths)]).astype(np.int64)


def _exact_counts(case, codes, children, branch, to):
    nl, k = len(children) + 1, case["states"]
    pi = to(_eigen(case["paramset"], 0, k)[2])
    p = to(_transitions(case["paramset"], 0, k, branch))
    counts = torch.zeros((len(branch), k, k), dtype=torch.float64, device=DEVICE)
    eye = torch.cat([torch.eye(k, device=DEVICE), torch.ones((k, 1), device=DEVICE)], 1).double()
    z = []
    for a in range(0, len(codes), 1 << 15):
        states = to(codes[a:a + (1 << 15)].T)
        zz, _, alpha, message = _messages(children, p, pi, states)
        z.append(zz)
        beta = {2 * nl - 2: pi[:, None].expand(-1, len(zz))}
        for i in range(2 * nl - 2, nl - 1, -1):
            above = beta.pop(i)
            for c, s in (children[i - nl], children[i - nl][::-1]):
                c, w = int(c), above * message[int(s)]
                v = alpha[c] if c >= nl else eye[:, torch.where(states[c] == GAP, k, states[c].long())]
                counts[c] += p[c] * ((w / zz) @ v.t())
                if c >= nl:
                    beta[c] = p[c].t() @ w
    return {"z": torch.cat(z).cpu(), "counts": counts.cpu()}


def _exact_gradient(case, seed, codes, off, children, branch, to):
    nl, k = len(children) + 1, case["states"]
    rho = np.repeat(_regions(case, seed)[2][:, None], 2, axis=1) * np.array([1.0, 1.1])
    lpr, elpr, drho = (np.zeros(rho.shape) for _ in range(3))
    dbranch = torch.zeros((len(rho), 2, len(branch)), dtype=torch.float64, device=DEVICE)
    for m in range(2):
        pi, q = to(_eigen(case["paramset"], m, k)[2]), to(_eigen(case["paramset"], m, k)[3])
        for r in range(len(rho)):
            p = to(_transitions(case["paramset"], m, k, branch * rho[r, m]))
            z, root, _, message = _messages(children, p, pi, to(codes[off[r]:off[r + 1]].T))
            lpr[r, m] = float(z.log().sum())
            elpr[r, m] = float(((root * pi.log()[:, None]).sum(0) / z).sum())
            beta = {2 * nl - 2: pi[:, None].expand(-1, len(z))}
            for i in range(2 * nl - 2, nl - 1, -1):
                above = beta.pop(i)
                for c, s in (children[i - nl], children[i - nl][::-1]):
                    c, w = int(c), above * message[int(s)]
                    dbranch[r, m, c] = ((w * (q @ message[c])).sum(0) / z).sum()
                    if c >= nl:
                        beta[c] = p[c].t() @ w
    dbranch = dbranch.cpu().numpy()
    drho[:] = (dbranch * branch).sum(2)
    return {"lpr": lpr, "elpr": elpr, "drho": drho, "dbranch": dbranch}
