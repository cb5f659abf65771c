"""Calls whose weights are multiplied exactly (scale * q + bias in f32, not rounded to f16): the error against 64 bits is that of
rounding the result, on every route that such calls take."""
import numpy as np
import pytest

from oracle import model
from tests.helpers import assert_close, make_weight, make_x, x_as_f64

pytestmark = pytest.mark.gpu


def _ratio(out, ref):
    """2-norm of the error over that of rounding the exact result to f16.  f32 sums and weights kept to 21 bits add about 1e-5 of the
    result to the 2.1e-4 of that rounding (1.001); weights rounded to f16 add 1.8e-4 (1.3)."""
    out, ref = np.asarray(out, np.float64), np.asarray(ref, np.float64)
    return np.linalg.norm(out - ref) / np.linalg.norm(ref.astype(np.float16).astype(np.float64) - ref)


def _linear(m, n, k, bits, gs, dtype="f16", kernel=0):
    from rmlx_amd import ops
    from rmlx_amd.runtime import BF16, DeviceBuffer
    rng = np.random.default_rng(m + n + k + bits + gs)
    w = make_weight(rng, n, k, bits, gs)
    x = make_x(rng, m, k, dtype)
    xd = DeviceBuffer.from_numpy(x, BF16) if dtype == "bf16" else DeviceBuffer.from_numpy(x)
    out = ops.affine_quantized_matmul_batched(xd, ops.QuantizedWeight.from_numpy(*w, gs, bits), kernel=kernel).numpy()
    x64 = x_as_f64(x, dtype)
    return out, model.qmm(x64 if dtype != "f32" else x64.astype(np.float16).astype(np.float64), *w, gs, bits)


# an N off the multiples of 8, group sizes and K's without a GEMM, and rows that stay on the streaming kernels
@pytest.mark.parametrize("m,n,k,bits,gs,dtype", [(1, 3001, 2880, 4, 64, "f16"), (8, 3301, 2880, 4, 64, "bf16"), (20, 1030, 4096, 4, 64, "f32"),
                                                 (70, 1031, 1088, 4, 32, "f16"), (300, 515, 2048, 8, 64, "bf16"), (5, 3001, 1152, 8, 128, "f16"),
                                                 (600, 130, 1088, 4, 64, "f16"), (12, 1408, 1984, 4, 64, "f16"), (10, 3360, 12160, 4, 64, "f16"),
                                                 (24, 2048, 4096, 4, 64, "f16"), (12, 1024, 8192, 8, 64, "f16"), (40, 96, 96, 4, 32, "f16")])
def test_linear_calls_with_exact_weights(hip, m, n, k, bits, gs, dtype):
    out, ref = _linear(m, n, k, bits, gs, dtype)
    assert _ratio(out, ref) < 1.05


@pytest.mark.parametrize("bits,gs", [(4, 64), (4, 32), (4, 128), (8, 64), (8, 32), (8, 128)])
@pytest.mark.parametrize("m,n,groups", [(1, 515, 8), (31, 127, 9), (33, 129, 21), (65, 300, 17), (130, 257, 11), (300, 1027, 8), (600, 70, 45), (40, 9, 1)])
def test_tile_gemm_with_exact_weights(hip, bits, gs, m, n, groups):
    """Remainders in each dimension."""
    from rmlx_amd import runtime as rt
    out, ref = _linear(m, n, groups * gs, bits, gs, kernel=rt.KERNEL_QMM_TILE_EXACT)
    assert_close(out, ref)
    assert _ratio(out, ref) < 1.05


# every tile, number of wave groups along k and kind of k split that the plans hold, at the smallest sizes that take them
@pytest.mark.parametrize("m,n,k,bits", [(1, 54, 256, 4), (1, 1454, 8448, 4), (69, 5723, 512, 4), (48, 2739, 6848, 4), (36, 8704, 384, 4), (1, 55, 6080, 4),
                                        (34, 9398, 320, 4), (1, 55, 2048, 4), (38, 8787, 256, 4), (1, 56, 4096, 4), (66, 11423, 832, 4), (37, 2860, 6720, 4),
                                        (141, 11085, 320, 4), (141, 11859, 448, 4), (68, 6039, 6784, 4), (531, 7694, 256, 4), (1500, 9001, 320, 4),
                                        (1, 59, 4224, 8), (68, 5815, 320, 8), (69, 1134, 8256, 8), (36, 8193, 320, 8), (1, 55, 4992, 8), (33, 9645, 320, 8),
                                        (1, 54, 2624, 8), (1, 6954, 256, 8), (1, 55, 4032, 8), (73, 8449, 576, 8), (33, 4362, 4096, 8), (194, 8507, 320, 8),
                                        (71, 2617, 3968, 8), (131, 11332, 256, 8), (75, 6171, 6016, 8), (1096, 3618, 256, 8), (649, 11094, 320, 8)])
@pytest.mark.parametrize("exact", [True, False])
def test_tile_gemm_plans(hip, m, n, k, bits, exact):
    from rmlx_amd import ops, runtime as rt
    from rmlx_amd.runtime import DeviceBuffer
    gs = 64
    rng = np.random.default_rng(m + n + k + bits)
    w = make_weight(rng, n, k, bits, gs)
    x = make_x(rng, m, k)
    out = ops.affine_quantized_matmul_batched(DeviceBuffer.from_numpy(x), ops.QuantizedWeight.from_numpy(*w, gs, bits),
                                              kernel=rt.KERNEL_QMM_TILE_EXACT if exact else rt.KERNEL_QMM_TILE).numpy()
    rows = np.unique(np.concatenate([np.arange(0, m, 19), [m - 1]]))
    cols = np.unique(np.concatenate([np.arange(0, n, 7), [n - 1]]))
    ref = model.qmm(x[rows].astype(np.float64), *(a[cols] for a in w), gs, bits)
    got = out[rows][:, cols]
    assert_close(got, ref)
    if exact and got.size > 300:
        assert _ratio(got, ref) < 1.05


@pytest.mark.parametrize("gs", [64, 128])
@pytest.mark.parametrize("dtype", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("m,n,groups", [(1, 1, 1), (3, 17, 3), (4, 33, 45), (5, 127, 64), (8, 8200, 5), (9, 515, 67), (16, 40, 129), (33, 16397, 9)])
def test_multi_row_gemv_off_its_multiples(hip, gs, dtype, m, n, groups):
    """Fewer weight rows than a tile, one more than a tile, K that ends in the middle of a slab of 128 or in the first of a pass, several
    passes over K, chunks of eight rows with a remainder; workgroups of one and two tiles per wave."""
    from rmlx_amd import runtime as rt
    if gs == 128 and n % 16 == 0:
        n += 1  # (the plain kernel takes whole tiles)
    out, ref = _linear(m, n, groups * gs, 4, gs, dtype, kernel=rt.KERNEL_QMV_RAGGED)
    assert_close(out, ref)
    if out.size > 500:
        assert _ratio(out, ref) < 1.05


# a few rows per expert below the GEMMs' thresholds, dimensions without a grouped GEMM, dimensions off the multiples of 64
@pytest.mark.parametrize("tokens,experts,top_k,hidden,inter,bits,gs", [(64, 32, 4, 512, 512, 4, 32), (20, 8, 1, 1088, 448, 4, 64), (96, 16, 2, 768, 896, 4, 128),
                                                                       (300, 8, 2, 768, 640, 4, 128), (40, 8, 2, 544, 544, 4, 32), (640, 4, 2, 544, 288, 4, 32),
                                                                       (90, 8, 2, 544, 544, 8, 32), (30, 4, 2, 1056, 544, 8, 32)])
def test_routed_block_with_exact_weights(hip, tokens, experts, top_k, hidden, inter, bits, gs):
    """(the hidden activations are rounded to f16 between the two products: about 1.08)"""
    from rmlx_amd import ops
    from rmlx_amd.runtime import DeviceBuffer
    rng = np.random.default_rng(tokens + hidden)
    gate, up = (make_weight(rng, inter, hidden, bits, gs, (experts,)) for _ in range(2))
    down = make_weight(rng, hidden, inter, bits, gs, (experts,))
    g, u, d = (ops.QuantizedWeight.from_numpy(*w, gs, bits) for w in (gate, up, down))
    x = make_x(rng, tokens, hidden)
    logits = rng.standard_normal((tokens, experts)).astype(np.float32)
    out = ops.moe_forward(g, u, d, DeviceBuffer.from_numpy(x), DeviceBuffer.from_numpy(logits), top_k).numpy()
    idx, w, _, _ = model.topk_route(logits, top_k)
    assert _ratio(out, model.moe_forward(x, idx, w, gate, up, down, gs, top_k, bits=bits)) < 1.2


@pytest.mark.parametrize("batch,rows,n,k,gs", [(8, 4, 1440, 2880, 64), (5, 30, 130, 1056, 32), (3, 70, 1001, 1088, 64), (64, 3, 1344, 1600, 64),
                                               (8, 12, 768, 896, 128), (3, 300, 260, 1024, 128), (2, 9, 7, 1024, 64)])
def test_gather_with_exact_weights(hip, batch, rows, n, k, gs):
    from rmlx_amd import ops
    from rmlx_amd.runtime import DeviceBuffer
    rng = np.random.default_rng(batch + rows + n)
    w = make_weight(rng, n, k, 4, gs, (4,))
    idx = rng.integers(0, 4, size=batch).astype(np.uint32)
    x = make_x(rng, batch * rows, k).reshape(batch, rows, k)
    out = ops.gather_qmm(DeviceBuffer.from_numpy(x), *(DeviceBuffer.from_numpy(a) for a in w), DeviceBuffer.from_numpy(idx), batch, rows, n, k, 4, gs).numpy()
    ref = np.stack([model.qmm(x[i].astype(np.float64), *(a[idx[i]] for a in w), gs, 4) for i in range(batch)])
    assert _ratio(out, ref) < 1.05
