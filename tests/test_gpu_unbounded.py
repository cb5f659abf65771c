"""Infinite activations of a few rows, on whatever kernel the library picks, give what the sums of their products are."""
import numpy as np
import pytest

from oracle import model
from tests.helpers import assert_close, make_weight, make_x, x_as_f64
from tests.test_gpu_ring import _assert_same_class, _unbounded

pytestmark = pytest.mark.gpu


# Shapes that the slot-streaming kernel and the multi-row GEMVs share among them, both sides of the lines: equal shares of the weight rows per CU (with
# whole and with clamped loads, two and three tiles, one and two waves' tiles beside each other), and the slot-streaming kernel.
@pytest.mark.parametrize("m,n,k,gs,dtype", [(8, 11008, 3840, 64, "f16"), (8, 12288, 3200, 128, "bf16"), (8, 9001, 4096, 64, "f32"), (8, 24001, 1984, 64, "bf16"),
                                            (7, 9216, 2880, 64, "f16"), (6, 9216, 2880, 64, "f32"), (5, 16001, 1088, 64, "f16"), (6, 12001, 4032, 64, "bf16"),
                                            (4, 16001, 1984, 64, "f16"), (3, 9001, 4096, 128, "f16"), (4, 22528, 3328, 64, "f16"), (3, 28672, 3200, 128, "bf16"),
                                            (4, 28672, 3328, 64, "f32"), (3, 23040, 2816, 64, "f32"), (6, 15680, 1088, 64, "f16"), (4, 9216, 4096, 64, "f16"),
                                            (8, 9216, 4096, 128, "bf16"), (8, 9216, 2880, 64, "f16"), (6, 12288, 4032, 64, "f16")])
def test_infinite_activations(hip, m, n, k, gs, dtype):
    from rmlx_amd import ops, runtime as rt
    rng = np.random.default_rng(m + n + k)
    w = make_weight(rng, n, k, 4, gs)
    x = make_x(rng, m, k).astype(np.float32)
    big = np.inf if dtype == "f16" else 1e6  # (a value that f16 does not hold is an infinity too)
    x[0, 7] = x[m - 1, k - 1] = big
    x[m - 1, k // 2] = -big
    x[1, 5], x[1, k - 130] = np.nan, big
    raw = model.f32_to_bf16_bits(x) if dtype == "bf16" else x.astype(np.float16 if dtype == "f16" else np.float32)
    xd = rt.DeviceBuffer.from_numpy(raw, rt.BF16) if dtype == "bf16" else rt.DeviceBuffer.from_numpy(raw)
    out = ops.affine_quantized_matmul_batched(xd, ops.QuantizedWeight.from_numpy(*w, gs, 4)).numpy()
    cols = np.unique(np.concatenate([np.arange(80), np.arange(0, n, 61), np.arange(n - 80, n)]))
    part = tuple(a[cols] for a in w)
    with np.errstate(over="ignore"):
        x16 = x_as_f64(raw, dtype).astype(np.float16)
    _assert_same_class(out[:, cols], _unbounded(x16.astype(np.float64), part, gs, 4))
    rest = np.isfinite(x16).all(axis=1)
    if rest.any():
        assert_close(out[np.ix_(rest, cols)], model.qmm(x16[rest].astype(np.float64), *part, gs, 4))


@pytest.mark.parametrize("m,n,k,gs", [(8, 9001, 4096, 64), (4, 9216, 4096, 128), (6, 9216, 2880, 64), (4, 22528, 3328, 64), (3, 28672, 3200, 128)])
def test_infinite_scales_and_biases(hip, m, n, k, gs):
    from rmlx_amd import ops, runtime as rt
    rng = np.random.default_rng(n)
    words, scales, biases = make_weight(rng, n, k, 4, gs)
    words |= 0x11111111  # (no value of zero)
    x = rt.DeviceBuffer.from_numpy(np.abs(make_x(rng, m, k)) + np.float16(0.1))
    run = lambda s, b: ops.affine_quantized_matmul_batched(x, ops.QuantizedWeight.from_numpy(words, s, b, gs, 4)).numpy()
    clean = run(scales, biases)
    scales, biases = scales.copy(), biases.copy()
    scales[3, 2], scales[n // 2, 0], biases[n - 1, -1] = np.inf, -np.inf, -np.inf
    out = run(scales, biases)
    assert np.isposinf(out[:, 3]).all() and np.isneginf(out[:, n // 2]).all() and np.isneginf(out[:, n - 1]).all()
    rest = np.setdiff1d(np.arange(n), [3, n // 2, n - 1])
    assert np.array_equal(out[:, rest].view(np.uint16), clean[:, rest].view(np.uint16))
