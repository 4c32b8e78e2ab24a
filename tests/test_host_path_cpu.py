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
