"""The host path of the C ABI (devices, memory, waits, error paths) on a runtime
without a GPU (fake_hip.cpp)."""
import pytest

from fake_hip import on_fake  # noqa: F401


def test_scores_use_the_contexts_device(on_fake):
    """With another device current, a batch's memory and launches stay on its context's."""
    on_fake("""
    ctx = P.Context(1)
    m = P.PhyloCSFModel.from_paramset(ctx, "12flies")
    before = fake.fake_used(0)
    for strategy in ("fixed", "mle", "mle_grad"):
        b = batch(m, 2, 70)
        fake.hipSetDevice(0)
        P.score(b, strategy, P.PCSF_FP64M)
    fake.hipSetDevice(0)
    m.transition(0, 1.7)
    assert fake.fake_used(0) == before and fake.fake_count(FOREIGN) == 0
    """)


def test_destroy_waits_for_readers_of_device_results(on_fake):
    """A batch whose device results were handed out goes back to the driver, which waits
    for readers on other streams; its arrays are aligned as allocations are."""
    on_fake("""
    ctx = P.Context(0)
    m = P.PhyloCSFModel.from_paramset(ctx, "12flies")
    for regions in (1, 3, 40):
        b = batch(m, regions, 70)
        b.forward(1.0, P.PCSF_FP64M)
        ll, el = C.c_void_p(), C.c_void_p()
        assert L.pcsf_batch_device_results(b.h, C.byref(ll), C.byref(el)) == 0
        assert ll.value % 256 == 0 and el.value % 256 == 0
        got = np.ctypeslib.as_array(C.cast(ll, C.POINTER(C.c_double)), (regions, 2)).copy()
        assert (got == b.forward(1.0, P.PCSF_FP64M)[0]).all()
        fake.fake_reset()
        del b
        assert fake.fake_count(FREES) == 1  # which waits
    b = batch(m, 3, 70)
    b.forward(1.0, P.PCSF_FP64M)
    fake.fake_reset()
    del b
    assert fake.fake_count(FREES) == 0 and fake.fake_count(WAITS) == 0
    """)


@pytest.mark.parametrize("kernel,nth", [("region_reduce", 2), ("prune", 3)])
def test_error_between_passes_leaves_no_failure_record(on_fake, kernel, nth):
    """A launch that fails after a failed build of the same call: the next calls, at good
    scales, are not told of that build."""
    on_fake("""
    ctx = P.Context(0)
    m = P.PhyloCSFModel.from_paramset(ctx, "12flies")
    for strategy in ("mle", "mle_grad"):
        b = batch(m, 2, 70)
        fake.fake_fail_rho(0.01 if strategy == "mle" else float(np.exp(-2.0)))
        fake.fake_fail_launch(%r, %d)
        try:
            P.score(b, strategy, P.PCSF_FP64M)
        except P.Failure:
            raise
        except P.PcsfError as e:
            assert e.code == _lib.PCSF_EDEVICE
        else:
            raise AssertionError("no error")
        b.forward(1.0, P.PCSF_FP64M)
        b.forward(np.full((2, 2), 1.5), P.PCSF_FP64M, per_region=True)
        m.transition(0, 1.0)
    """ % (kernel.encode(), nth))


def test_refused_forward_leaves_no_built_sets(on_fake):
    """FP64 on a tree whose workspace exceeds LDS is refused; a failed build in front of it
    must not count as built."""
    on_fake("""
    ctx = P.Context(0)
    text = "a0:0.1"
    for i in range(1, 200):
        text = "(%s,a%d:0.1)%s" % (text, i, ":0.1" if i < 199 else "")
    prefix = P.paramset_prefix("12flies")
    ecms = [P.import_parameters(prefix + "_%s.ECM" % w) for w in ("coding", "noncoding")]
    m = P.PhyloCSFModel(ctx, P.newick_tree(text + ";"), ecms)
    b = batch(m, 2, 5)
    fake.fake_fail_rho(2.5)
    for per_region in (False, True):
        try:
            b.forward(np.full((2, 2), 2.5) if per_region else 2.5, P.PCSF_FP64, per_region=per_region)
        except P.InvalidArgument as e:
            assert "LDS" in str(e)
        else:
            raise AssertionError("not refused")
        for _ in range(2):
            try:
                m.transition(0, 2.5)
            except P.Failure:
                continue
            raise AssertionError("a failed build passed for a good one")
        m.transition(0, 1.0)
    """)


@pytest.mark.parametrize("column", [0, -1])
def test_bad_state_writes_nothing(on_fake, column):
    """A leaf state that PhyloLik's columns refuse, in the first or in a later chunk of the
    columns: no output has been written."""
    on_fake("""
    ctx = P.Context(0)
    nl, ncols = 2000, 70000  # 512 MB a chunk: two
    kids = [[0, 1]] + [[nl + i, i + 2] for i in range(nl - 2)]
    kids = np.array(kids, np.int32)
    Pm = np.zeros((2 * nl - 2, 4, 4))
    prior = np.full(4, 0.25)
    leaves = np.zeros((ncols, nl), np.int32)
    z, post = np.full(ncols, -7.0), np.full((ncols, 4), -7.0)
    dp, ip = C.POINTER(C.c_double), C.POINTER(C.c_int32)

    def call():
        return L.pcsf_lik_columns(ctx.h, 4, 2 * nl - 1, kids.ctypes.data_as(ip), Pm.ctypes.data_as(dp),
                                  prior.ctypes.data_as(dp), leaves.ctypes.data_as(ip), ncols,
                                  z.ctypes.data_as(dp), post.ctypes.data_as(dp))

    leaves[%d, 3] = -2
    assert call() == _lib.PCSF_EINVAL
    assert (z == -7.0).all() and (post == -7.0).all()
    leaves[:, 3] = 1
    assert call() == 0 and (z == 1.0).all() and launches("lik_small") >= 2
    """ % column)


@pytest.mark.parametrize("k,nl,ncols", [(20, 1000, 20000), (4, 5000, 30000), (20, 300, 100000),
                                        (4, 300, 100000), (20, 4000, 300)])
def test_small_alphabet_memory_is_bounded(on_fake, k, nl, ncols):
    """PhyloLik's columns hold at most the 512 MB of a chunk, 2 GiB of workspace (or the
    column kernel's 2,048 columns) and the tree's P, however large the tree."""
    on_fake("""
    k, nl, ncols = %d, %d, %d
    ctx = P.Context(0)
    kids = np.array([[0, 1]] + [[nl + i, i + 2] for i in range(nl - 2)], np.int32)
    n = 2 * nl - 1
    Pm, prior, z = np.zeros((n - 1, k, k)), np.full(k, 1.0 / k), np.zeros(ncols)
    leaves = np.zeros((ncols, nl), np.int32)
    dp, ip = C.POINTER(C.c_double), C.POINTER(C.c_int32)
    before = fake.fake_used(0)
    fake.fake_reset()
    assert L.pcsf_lik_columns(ctx.h, k, n, kids.ctypes.data_as(ip), Pm.ctypes.data_as(dp),
                              prior.ctypes.data_as(dp), leaves.ctypes.data_as(ip), ncols,
                              z.ctypes.data_as(dp), None) == 0
    assert launches("lik_small") + launches("lik_columns") > 0
    bound = (512 << 20) + max(2 << 30, 2048 * 2 * n * k * 8) + 2 * Pm.nbytes
    assert fake.fake_peak(0) - before <= 1.15 * bound, fake.fake_peak(0) - before
    """ % (k, nl, ncols))


@pytest.mark.parametrize("first,then", [("FP16S", "FP64M"), ("FP64M", "FP32"), ("FP64", "FP64M")])
def test_set_budget_bounds_all_kinds_together(on_fake, first, then):
    """A pass that adds a kind of transition matrix to sets that fill the budget goes through
    in more chunks, not in twice the memory."""
    on_fake("""
    ctx = P.Context(0)
    m = P.PhyloCSFModel.from_paramset(ctx, "12flies")
    b = batch(m, 60, 3)
    rho = np.full((60, 2), 1.5)
    assert b.forward(rho, P.PCSF_%s, per_region=True)[0].shape == (60, 2)
    assert launches("region_reduce_aligned") == 1
    fake.fake_reset()
    got = b.forward(rho, P.PCSF_%s, per_region=True)[0]
    assert launches("region_reduce_aligned") == 2
    assert (abs(got[:, 0] + 100 * (np.log(1.5) - 0.3) ** 2) < 1e-9).all()
    """ % (first, then), env={"PHYLOCSF_SET_BUDGET_MB": "100"})


def test_large_omega_call_goes_through_in_one_chunk(on_fake):
    """3,000 regions of 58mammals, 24 GB of sets with rate models of their own, take as many
    passes as ten regions: one chunk, in which a pass starts from the last one's
    eigensystems."""
    on_fake("""
    ctx = P.Context(0)
    tree = P.newick_tree(open(P.paramset_prefix("58mammals") + ".nh").read())
    m = P.PhyloCSFModel.tree_only(ctx, tree)
    passes = []
    for regions in (10, 3000):
        fake.fake_reset()
        P.score_omega(batch(m, regions, 1), precision=P.PCSF_FP64M)
        passes.append(launches("region_reduce_aligned"))
    assert passes[0] == passes[1] > 20, passes
    """)


def test_alternating_precisions_keep_the_sets(on_fake):
    """Forwards at one tree scale in FP64 and at an MFMA precision, and transition matrices in
    between, build each kind once."""
    on_fake("""
    ctx = P.Context(0)
    m = P.PhyloCSFModel.from_paramset(ctx, "12flies")
    b = batch(m, 2, 70)

    def turn():
        b.forward(1.0, P.PCSF_FP16S)
        b.forward(1.0, P.PCSF_FP64M)
        m.transition(0, 1.0)
        b.forward(1.0, P.PCSF_FP64)

    turn()
    fake.fake_reset()
    turn()
    assert launches("pbuild") == 0 and launches("cherry_table") == 0
    b.forward(1.0, P.PCSF_FP32)  # another tile format: the tiles alone
    assert launches("pbuild") == 1 and launches("cherry_table") == 0
    """)


def test_pool_keeps_the_latest_blocks(on_fake):
    """Calls that repeat find their memory kept, also after larger or other ones: of more
    than 16 GiB the blocks freed first go back to the driver."""
    on_fake("""
    ctx = P.Context(0)
    m = P.PhyloCSFModel.from_paramset(ctx, "58mammals")

    def call(regions):
        b = batch(m, regions, 1)
        for precision in (P.PCSF_FP16S, P.PCSF_FP64M):
            b.forward(np.full((regions, 2), 1.5), precision, per_region=True)

    base = fake.fake_used(0)
    for regions in (150, 700, 290, 800):  # 2.3, 10.6, 4.4 and 12.2 GB of sets
        for turn in range(4):
            fake.fake_reset()
            call(regions)
            if turn > 1:
                assert fake.fake_count(MALLOCS) == fake.fake_count(FREES) == 0, (regions, turn)
        assert fake.fake_used(0) - base <= 16 << 30
    ctx2 = P.Context(0)  # another context does not get this one's
    m2 = P.PhyloCSFModel.from_paramset(ctx2, "12flies")
    fake.fake_reset()
    batch(m2, 1, 1).forward(1.0, P.PCSF_FP64M)
    assert fake.fake_count(MALLOCS) > 0
    """)


def test_pool_gives_back_when_memory_runs_out(on_fake):
    """An allocation that fails empties every context's kept memory and is tried again; a
    context's end gives back what it kept."""
    on_fake("""
    ctx, ctx2 = P.Context(0), P.Context(0)
    m = P.PhyloCSFModel.from_paramset(ctx, "58mammals")
    m2 = P.PhyloCSFModel.from_paramset(ctx2, "58mammals")

    def call(m, regions):
        b = batch(m, regions, 1)
        return b.forward(np.full((regions, 2), 1.5), P.PCSF_FP64M, per_region=True)

    call(m, 1200)
    fake.fake_capacity(fake.fake_used(0) + (1 << 30))
    want = call(m2, 600)
    assert fake.fake_used(0) < 8 << 30  # the first context's 9 GB went back
    try:
        call(m2, 1400)  # 10.6 GB do not fit: everything kept goes back, and it still fails
        fake.fake_capacity(0)
    except P.PcsfError as e:
        assert e.code == _lib.PCSF_ENOMEM
    fake.fake_capacity(288 << 30)
    assert (call(m2, 600)[0] == want[0]).all()
    L.pcsf_model_destroy(m2.h)
    m2.h = None
    before = fake.fake_used(0)
    L.pcsf_ctx_destroy(ctx2.h)
    ctx2.h = None
    assert fake.fake_used(0) <= before - (4 << 30)
    """)


def test_model_memory(on_fake):
    """A model holds of its fixed sets what forwards and pcsf_model_transition read (per
    branch two tiles of FP32, two of FP64), no transposes for the outside pass, which
    runs on a batch's sets."""
    on_fake("""
    ctx = P.Context(0)
    before = fake.fake_used(0)
    m = P.PhyloCSFModel.from_paramset(ctx, "100vertebrates")
    nbr = m.tree.n - 1
    sets = 2 * nbr * (65 * 64 * 4 + 4160 * 4 + 65 * 8 + 4096 * 8 + 65 * 64 * 8)
    tables = 2 * 65 * 65 * (64 * 4 + 8)  # per cherry
    kids = np.asarray(m.tree.children).reshape(-1, 2)
    cherries = int((kids < m.tree.nl).all(axis=1).sum())
    assert fake.fake_used(0) - before <= 1.07 * (sets + cherries * tables)
    """)


def test_pinned_ring_wraps(on_fake):
    """Uploads that go round the context's 1 MB ring: what is still to be copied is not
    overwritten (the fake's streams copy as late as they may)."""
    on_fake("""
    ctx = P.Context(0)
    m = P.PhyloCSFModel.from_paramset(ctx, "58mammals")
    nl = m.tree.nl
    rng = np.random.default_rng(2)
    made = []
    fake.fake_reset()
    for k in range(45):  # 0.9 KB to 64 KB each, 1.5 MB in all, some past the small size
        codes = rng.integers(0, 64, (25 * k + 16, nl)).astype(np.uint8)
        made.append((P.Batch(m, codes, np.array([0, 7, len(codes)])), codes))
    assert 1 <= fake.fake_count(WAITS) <= 3
    for b, codes in made:
        assert (b.codes()[0] == codes).all()
    """)


def test_results_larger_than_the_ring(on_fake):
    """Shared scales together (one wait) and one by one where their results do not fit the
    ring, results and set parameters beyond it: the same values."""
    on_fake("""
    ctx = P.Context(0)
    tree = P.newick_tree(open(P.paramset_prefix("12flies") + ".nh").read(), ["dmel", "dsim"])
    prefix = P.paramset_prefix("12flies")
    ecms = [P.import_parameters(prefix + "_%s.ECM" % w) for w in ("coding", "noncoding")]
    m = P.PhyloCSFModel(ctx, tree, ecms)
    want = [-100 * (np.log(1.5) - 0.3 - 0.01 * q) ** 2 for q in range(2)]
    for strategy in ("mle", "mle_grad"):
        small = P.score(batch(m, 3, 1), strategy, P.PCSF_FP64M)
        large = P.score(batch(m, 12000, 1), strategy, P.PCSF_FP64M)  # 4 x 384 KB
        for key in ("lpr", "rho", "elpr"):
            assert (large[key] == small[key][0]).all(), key
    b = batch(m, 70000, 1)  # 2.2 MB of results, 1.3 MB of scales and flags
    assert np.allclose(b.forward(1.5, P.PCSF_FP64M)[0], want)
    fake.fake_reset()
    got = b.forward(np.full((70000, 2), 1.5), P.PCSF_FP64M, per_region=True)[0]
    assert launches("region_reduce_aligned") == 1 and np.allclose(got, want)
    """, env={"PHYLOCSF_SET_BUDGET_MB": "30000"})


def test_interpreter_keeps_its_launch_shape(on_fake):
    """FP32 on a shipped tree loads leaf rows ahead in the tree's own program; where that is
    forbidden the interpreter runs without (<..., waves, per SIMD, ahead, ...>), unless a
    shape was chosen."""
    on_fake("""
    ctx = P.Context(0)
    m = P.PhyloCSFModel.from_paramset(ctx, "58mammals")
    b = batch(m, 2, 70)
    ahead, plain = "Li4ELi3ELb1E", "Li4ELi3ELb0E"

    def shapes():
        fake.fake_reset()
        b.forward(1.0, P.PCSF_FP32)
        b.forward(np.full((2, 2), 1.5), P.PCSF_FP32, per_region=True)
        return launches(ahead), launches(plain)

    assert shapes() == (2, 0)
    m.specialized(False)
    assert shapes() == (0, 2) and launches("Interp") == 2
    m.set_variant(5, P.PCSF_FP32)
    assert shapes() == (2, 0) and launches("Interp") == 2
    """)
