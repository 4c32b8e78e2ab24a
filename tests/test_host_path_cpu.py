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
