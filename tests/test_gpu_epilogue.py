"""Fused epilogues (residual add, SwiGLU gate) on the GPU: outputs written over the operand."""
import ctypes

import numpy as np
import pytest

from tests.helpers import assert_close, make_weight, make_x

pytestmark = pytest.mark.gpu


def _calls(rt):
    return {"residual": rt.lib().rmlx_hip_qmm_add_residual, "swiglu": rt.lib().rmlx_hip_qmm_swiglu}


def _in_place_equals_apart(rt, m, n, k, bits, gs=64, repeats=3):
    """out == operand gives the bits of an output of its own."""
    from rmlx_amd import ops
    from rmlx_amd.runtime import DeviceBuffer
    rng = np.random.default_rng(m + n + k + bits + gs)
    qw = ops.QuantizedWeight.from_numpy(*make_weight(rng, n, k, bits, gs), gs, bits)
    x = DeviceBuffer.from_numpy(make_x(rng, m, k))
    e = rng.standard_normal((m, n)).astype(np.float16)
    xa = x.array()
    for name, fn in _calls(rt).items():
        ed, apart = DeviceBuffer.from_numpy(e), DeviceBuffer((m, n), rt.F16)
        ea = ed.array()
        rt.check(fn(qw.handle, ctypes.byref(xa), ctypes.byref(ea), apart.ptr, apart.nbytes, None))
        want = apart.numpy()
        for _ in range(repeats):
            own = DeviceBuffer.from_numpy(e)
            oa = own.array()
            rt.check(fn(qw.handle, ctypes.byref(xa), ctypes.byref(oa), own.ptr, own.nbytes, None))
            assert np.array_equal(own.numpy().view(np.uint16), want.view(np.uint16)), f"{name} M={m} N={n} K={k} bits={bits} gs={gs}"


@pytest.mark.parametrize("m,n,k,bits", [(1, 12296, 4096, 4), (1, 33001, 4096, 4), (1, 33001, 1024, 8), (2, 12289, 512, 4), (1, 4104, 12288, 4),
                                        (1, 1023, 12288, 4), (1, 515, 16384, 8), (1, 9, 512, 4), (1, 112257, 1408, 4)])
def test_in_place_over_an_overlapping_last_block(hip, m, n, k, bits):
    """Single-row kernel, a number of weight rows that is no multiple of a block (of one and two rows per wave, of rows split over
    waves, of workgroups that walk several blocks): the rows that two blocks compute are stored by one of them."""
    _in_place_equals_apart(hip, m, n, k, bits)


@pytest.mark.parametrize("m,n,k,bits,gs", [(5, 4096, 4096, 4, 64), (12, 512, 1024, 8, 64), (3, 24576, 1024, 4, 32), (3, 5, 64, 4, 64), (3, 8, 32, 4, 32),
                                           (130, 192, 320, 4, 64), (130, 512, 1024, 4, 64), (600, 4096, 4096, 4, 64),
                                           (130, 4096, 8192, 4, 64), (600, 2051, 1088, 4, 64), (33, 130, 4160, 8, 64)])
def test_in_place_on_every_kernel(hip, m, n, k, bits, gs):
    """Streaming GEMVs, portable and LDS-staged kernels (the epilogue in a pass of its own) and the GEMMs that fuse it."""
    _in_place_equals_apart(hip, m, n, k, bits, gs, repeats=1)


def test_residual_over_more_than_two_gib_of_sums(hip):
    """256 rows x 2.2 million columns: offsets within a tile's rows pass 2 GiB where the sums are f32."""
    from oracle import model
    from rmlx_amd import ops
    from rmlx_amd.runtime import DeviceBuffer
    from tests.helpers import assert_close
    m, n, k = 256, 2_200_032, 64
    rng = np.random.default_rng(5)
    words, s, b = make_weight(rng, n, k)
    qw = ops.QuantizedWeight.from_numpy(words, s, b, 64, 4)
    x = make_x(rng, m, k)
    cols = np.unique(np.concatenate([np.arange(0, 300), rng.integers(0, n, 300), np.arange(n - 300, n)]))
    e = np.zeros((m, n), np.float16)
    e[:, cols] = rng.standard_normal((m, len(cols))).astype(np.float16)
    out = ops.qmm_add_residual(DeviceBuffer.from_numpy(x), qw, DeviceBuffer.from_numpy(e)).numpy()[:, cols]
    assert_close(out, model.qmm(x.astype(np.float64), words[cols], s[cols], b[cols], 64, 4) + e[:, cols].astype(np.float64), "residual")


@pytest.mark.parametrize("m,n,k,bits", [(2048, 4096, 4096, 4), (3001, 14336, 4096, 4), (512, 12288, 4096, 8), (128, 12288, 4096, 4)])
def test_fused_in_the_store_of_one_launch(hip, m, n, k, bits):
    """No block of the output's size is taken for an epilogue, and the result is the f32 sum rounded once: added to the plain
    product's f16 in 64 bits it differs by at most both roundings (2^-11 of either value)."""
    from rmlx_amd import ops
    from rmlx_amd.runtime import DeviceBuffer
    rng = np.random.default_rng(m + n)
    qw = ops.QuantizedWeight.from_numpy(*make_weight(rng, n, k, bits), 64, bits)
    x = DeviceBuffer.from_numpy(make_x(rng, m, k))
    e = rng.standard_normal((m, n)).astype(np.float16)
    ed, stream = DeviceBuffer.from_numpy(e), hip.Stream()
    plain = ops.affine_quantized_matmul_batched(x, qw, stream=stream)
    stream.sync()
    before = hip.scratch_allocations()
    out = ops.qmm_add_residual(x, qw, ed, stream=stream)
    stream.sync()
    assert hip.scratch_allocations() == before
    p, got = plain.numpy().astype(np.float64), out.numpy().astype(np.float64)
    assert np.all(np.abs(got - (p + e)) <= 2.0 ** -11 * (np.abs(p) + np.abs(got)) * 1.01 + 1e-7)


@pytest.mark.parametrize("m,n,k", [(6, 15680, 1088), (8, 15936, 1088), (5, 11968, 1472), (8, 12800, 1088), (6, 10496, 1472)])
def test_few_rows_keep_the_fused_epilogue(hip, m, n, k):
    """Shapes that a plain product takes as equal shares of the multi-row GEMV: an epilogue stays in the store of the tile GEMM, which needs no block for the
    product where the output is the operand."""
    from oracle import model
    from rmlx_amd import ops, runtime as rt
    rng = np.random.default_rng(m + n + k)
    w = make_weight(rng, n, k)
    qw = ops.QuantizedWeight.from_numpy(*w, 64, 4)
    x = make_x(rng, m, k)
    xd = rt.DeviceBuffer.from_numpy(x)
    plain, shares = (ops.affine_quantized_matmul_batched(xd, qw, kernel=q).numpy() for q in (0, rt.KERNEL_QMV_SHARES))
    assert np.array_equal(plain.view(np.uint16), shares.view(np.uint16))
    e = rng.standard_normal((m, n)).astype(np.float16)
    own, stream, xa = rt.DeviceBuffer.from_numpy(e), rt.Stream(), xd.array()
    oa, before = own.array(), rt.scratch_allocations()
    rt.check(_calls(rt)["residual"](qw.handle, ctypes.byref(xa), ctypes.byref(oa), own.ptr, own.nbytes, ops._h(stream)))
    stream.sync()
    assert rt.scratch_allocations() == before
    cols = np.arange(0, n, 61)
    assert_close(own.numpy()[:, cols], model.qmm(x.astype(np.float64), *(a[cols] for a in w), 64, 4) + e[:, cols].astype(np.float64))
