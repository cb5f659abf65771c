"""Multi-row GEMV with an equal share of the weight rows per CU (qmv.hip, SHARE) at the edges of its tiles, against the oracle."""
import numpy as np
import pytest

from oracle import model
from tests.helpers import assert_close, make_weight, make_x, x_as_f64
from tests.test_gpu_precision import _ratio

pytestmark = pytest.mark.gpu


# On 256 CUs, shares of one row in the last tile and of whole tiles, two to four of them, the last workgroup with fewer rows or all of its own; one
# to four waves' tiles side by side, three and four slabs a wave; the row counts that begin and end each build (five to eight rows: up to three tiles).
@pytest.mark.parametrize("k,gs", [(4096, 64), (4096, 128), (3072, 64), (2048, 64), (1536, 128)])
@pytest.mark.parametrize("m,dtype", [(2, "f16"), (3, "bf16"), (4, "f16"), (5, "f16"), (8, "bf16")])
@pytest.mark.parametrize("share", [17, 32, 33, 48, 49, 64])
def test_shares(hip, k, gs, m, dtype, share):
    from rmlx_amd import ops, runtime as rt
    side = 1 if k >= 3072 else 2
    n = (256 * side * (share - 1) // 16 + 1) * 16 if share % 16 == 1 else 256 * side * share
    rng = np.random.default_rng(m + n + k)
    w = make_weight(rng, n, k, 4, gs)
    x = make_x(rng, m, k, dtype)
    xd = rt.DeviceBuffer.from_numpy(x, rt.BF16) if dtype == "bf16" else rt.DeviceBuffer.from_numpy(x)
    out = ops.affine_quantized_matmul_batched(xd, ops.QuantizedWeight.from_numpy(*w, gs, 4), kernel=rt.KERNEL_QMV_ROWS).numpy()
    rows = np.unique(np.concatenate([np.arange(200), np.arange(0, n, 61), np.arange(share - 2, n, 7 * share), np.arange(n - 200, n)]))
    ref = model.qmm(x_as_f64(x, dtype).astype(np.float16).astype(np.float64), *(a[rows] for a in w), gs, 4)
    assert_close(out[:, rows], ref)
    assert _ratio(out[:, rows], ref) < 1.05


# K of waves with fewer slabs than others, with none, that ends in the middle of a slab; one to four waves' tiles side by side; N of any kind
@pytest.mark.parametrize("k,gs", [(3968, 64), (3648, 64), (2880, 64), (2304, 128), (2176, 64), (1984, 64), (1088, 64), (896, 128)])
@pytest.mark.parametrize("m,dtype", [(3, "f16"), (4, "bf16"), (5, "bf16"), (8, "f16")])
@pytest.mark.parametrize("share,odd", [(17, 5), (32, 0), (33, 16), (48, 37), (49, 1), (64, 7)])
def test_guarded_shares(hip, k, gs, m, dtype, share, odd):
    from rmlx_amd import ops, runtime as rt
    side = 1 if k > 2048 else (2 if k > 1024 else 4)
    n = 256 * side * (share - 1) + 256 * side - odd if odd != 1 else 256 * side * (share - 1) + 1
    rng = np.random.default_rng(m + n + k)
    w = make_weight(rng, n, k, 4, gs)
    x = make_x(rng, m, k, dtype)
    xd = rt.DeviceBuffer.from_numpy(x, rt.BF16) if dtype == "bf16" else rt.DeviceBuffer.from_numpy(x)
    kernel = rt.KERNEL_QMV_ROWS if n % 16 == 0 and k % 128 == 0 else rt.KERNEL_QMV_RAGGED
    out = ops.affine_quantized_matmul_batched(xd, ops.QuantizedWeight.from_numpy(*w, gs, 4), kernel=kernel).numpy()
    rows = np.unique(np.concatenate([np.arange(200), np.arange(0, n, 61), np.arange(share - 2, n, 7 * share), np.arange(n - 200, n)]))
    ref = model.qmm(x_as_f64(x, dtype).astype(np.float16).astype(np.float64), *(a[rows] for a in w), gs, 4)
    assert_close(out[:, rows], ref)
    assert _ratio(out[:, rows], ref) < 1.05


def _builds():
    """(rows of x, K, group size, weight rows of a share, weight rows that the last one lacks): every build of the kernel, two waves' tiles beside each
    other (K up to 2048)."""
    whole = [(2, 4096, gs, s) for gs in (64, 128) for s in (17, 33, 49)] + [(4, 4096, gs, s) for gs in (64, 128) for s in (32, 48, 64)]
    whole += [(3, 3072, 64, s) for s in (17, 33, 49)] + [(8, k, gs, s) for k in (4096, 3072, 2048, 1536) for gs in (64, 128) for s in (17, 33)]
    guarded = [(4, 3968, gs, s) for gs in (64, 128) for s in (17, 33)] + [(3, k, gs, s) for k, gs in ((2880, 64), (2304, 128)) for s in (32, 36)]
    guarded += [(5, 3968, gs, s) for gs in (64, 128) for s in (32, 48)] + [(8, k, gs, s) for k, gs in ((2880, 64), (2304, 128), (1984, 64), (1088, 64)) for s in (17, 48)]
    return [b + (0,) for b in whole + guarded] + [b + (16,) for b in whole] + [b + (13,) for b in guarded]


# Selector 16 runs the shares or refuses: a rule that leaves a shape to another kernel fails here.
@pytest.mark.parametrize("m,k,gs,share,short", _builds())
def test_every_build(hip, m, k, gs, share, short):
    from rmlx_amd import ops, runtime as rt
    sides = 1 if k > 2048 else 2
    n = hip.device_info()["compute_units"] * sides * share - short
    rng = np.random.default_rng(m + n + k)
    w = make_weight(rng, n, k, 4, gs)
    dtype = "bf16" if (share + m) % 2 else "f16"
    x = make_x(rng, m, k, dtype)
    xd = rt.DeviceBuffer.from_numpy(x, rt.BF16) if dtype == "bf16" else rt.DeviceBuffer.from_numpy(x)
    out = ops.affine_quantized_matmul_batched(xd, ops.QuantizedWeight.from_numpy(*w, gs, 4), kernel=rt.KERNEL_QMV_SHARES).numpy()
    rows = np.unique(np.concatenate([np.arange(2 * share), np.arange(0, n, 61), np.arange(share - 1, n, 7 * share), np.arange(n - 2 * share, n)]))
    ref = model.qmm(x_as_f64(x, dtype).astype(np.float16).astype(np.float64), *(a[rows] for a in w), gs, 4)
    assert_close(out[:, rows], ref)
    assert _ratio(out[:, rows], ref) < 1.05


# eight rows of four tiles, seven slabs, two rows of K < 4096, one tile, two slots, more rows, other weights
@pytest.mark.parametrize("m,k,gs,share,bits", [(8, 4096, 64, 49, 4), (4, 896, 128, 17, 4), (2, 3072, 64, 33, 4), (4, 4096, 64, 16, 4), (4, 8192, 64, 33, 4),
                                               (9, 4096, 64, 33, 4), (1, 4096, 64, 33, 4), (4, 4096, 32, 33, 4), (4, 4096, 64, 33, 8), (3, 3200, 64, 48, 4)])
def test_shares_are_refused(hip, m, k, gs, share, bits):
    from rmlx_amd import ops, runtime as rt
    rng = np.random.default_rng(k)
    w = make_weight(rng, hip.device_info()["compute_units"] * share, k, bits, gs)
    with pytest.raises(rt.KernelError):
        ops.affine_quantized_matmul_batched(rt.DeviceBuffer.from_numpy(make_x(rng, m, k)), ops.QuantizedWeight.from_numpy(*w, gs, bits), kernel=rt.KERNEL_QMV_SHARES)


# f32 rows, 3 to 8 of them: read and rounded by the kernel itself on both sides of the line to the slot-streaming kernel, the builds of each form
@pytest.mark.parametrize("m,n,k,gs", [(8, 11008, 3840, 64), (6, 9216, 2880, 64), (5, 14336, 1984, 64), (7, 24001, 1984, 64), (3, 9001, 4096, 128), (4, 28672, 3328, 64),
                                      (4, 9216, 4096, 64), (2, 9216, 4096, 128), (8, 9216, 4096, 128), (3, 8448, 3072, 64), (8, 8704, 1536, 64), (4, 4608, 2304, 128)])
def test_f32_rows_take_no_scratch(hip, m, n, k, gs):
    from rmlx_amd import ops, runtime as rt
    rng = np.random.default_rng(m + n + k)
    w = make_weight(rng, n, k, 4, gs)
    wd = ops.QuantizedWeight.from_numpy(*w, gs, 4)
    x = make_x(rng, m, k, "f32")
    x16 = x.astype(np.float16)
    xd, xh = rt.DeviceBuffer.from_numpy(x), rt.DeviceBuffer.from_numpy(x16)
    stream = rt.Stream()
    before = rt.scratch_allocations()
    out = ops.affine_quantized_matmul_batched(xd, wd, stream=stream)
    stream.sync()
    assert rt.scratch_allocations() == before
    same = ops.affine_quantized_matmul_batched(xh, wd).numpy()
    assert np.array_equal(out.numpy().view(np.uint16), same.view(np.uint16))
    rows = np.unique(np.concatenate([np.arange(0, n, 61), np.arange(n - 40, n)]))
    assert_close(same[:, rows], model.qmm(x16.astype(np.float64), *(a[rows] for a in w), gs, 4))
