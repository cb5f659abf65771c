"""Grouping of assignments by expert over several workgroups: the stable order, at the sizes where portions and runs begin and end."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 1023, 1024, 1025, 2047, 2048, 2049, 5000, 16384, 32768, 33000, 70001])
@pytest.mark.parametrize("experts", [1, 7, 128, 1024])
def test_stable_order(hip, n, experts):
    from rmlx_amd import ops, runtime as rt
    rng = np.random.default_rng(n + experts)
    idx = rng.integers(0, experts, size=n).astype(np.uint32)
    idx[rng.random(n) < 0.3] = experts // 2  # one expert with a third of them, over every portion
    bad = rng.random(n) < 0.05
    idx[bad] = rng.choice(np.array([experts, 0xFFFFFFFF], np.uint32), size=int(bad.sum()))
    order, offsets = ops.moe_sort(rt.DeviceBuffer.from_numpy(idx), experts)
    good = int((~bad).sum())
    counts = np.bincount(idx[~bad], minlength=experts)
    assert np.array_equal(offsets.numpy(), np.concatenate([[0], np.cumsum(counts)]).astype(np.uint32))
    assert np.array_equal(order.numpy()[:good], np.argsort(np.where(bad, experts, idx), kind="stable")[:good].astype(np.uint32))
