"""The slot-streaming GEMV (qmv_ring.hip) at the edges of its tiles, slots and splits, against the oracle."""
import numpy as np
import pytest

from oracle import model
from tests.helpers import assert_close, make_weight, make_x, x_as_f64
from tests.test_gpu_precision import _ratio

pytestmark = pytest.mark.gpu


# Every split of a row: one to eight parts of three and of four loads, the last one full, in part empty and (8-bit K = 2240, 4-bit K = 4608) all
# but empty, rows in two slots; 16-byte pieces of a row in multiples of 16, 8, 4 and 2; groups of a row in multiples of 32, even and odd.
@pytest.mark.parametrize("bits,gs,k", [(4, 64, 512), (4, 64, 704), (4, 64, 1024), (4, 64, 1088), (4, 64, 1536), (4, 64, 2048), (4, 64, 2880), (4, 64, 4032),
                                       (4, 64, 4096), (4, 64, 4608), (4, 64, 8128), (4, 64, 8192), (4, 32, 544), (4, 32, 1024), (4, 32, 2080), (4, 32, 2880),
                                       (4, 32, 4064), (4, 32, 4096), (4, 128, 512), (4, 128, 1408), (4, 128, 2944), (4, 128, 4096), (4, 128, 6144),
                                       (8, 64, 512), (8, 64, 1088), (8, 64, 1408), (8, 64, 2048), (8, 64, 2240), (8, 64, 4096), (8, 32, 544), (8, 32, 1504),
                                       (8, 32, 2016), (8, 32, 2880), (8, 32, 4096), (8, 128, 640), (8, 128, 2048), (8, 128, 2944), (8, 128, 4096)])
# fewer weight rows than workgroups and a tile's worth for each of a few, a little over one and two tiles a workgroup, many tiles with a ragged end
@pytest.mark.parametrize("m,n,dtype", [(1, 128, "f16"), (16, 257, "bf16"), (17, 4099, "f16"), (3, 8211, "f32"), (15, 28677, "bf16")])
def test_matrix(hip, bits, gs, k, m, n, dtype):
    from rmlx_amd import ops, runtime as rt
    rng = np.random.default_rng(m + n + k + bits + gs)
    w = make_weight(rng, n, k, bits, gs)
    x = make_x(rng, m, k, dtype)
    xd = rt.DeviceBuffer.from_numpy(x, rt.BF16) if dtype == "bf16" else rt.DeviceBuffer.from_numpy(x)
    out = ops.affine_quantized_matmul_batched(xd, ops.QuantizedWeight.from_numpy(*w, gs, bits), kernel=rt.KERNEL_QMV_RING).numpy()
    rows = np.unique(np.concatenate([np.arange(min(n, 300)), np.arange(0, n, 61), np.arange(max(0, n - 70), n)]))
    x64 = x_as_f64(x, dtype)
    ref = model.qmm(x64.astype(np.float16).astype(np.float64), *(a[rows] for a in w), gs, bits)
    assert_close(out[:, rows], ref)
    if out[:, rows].size > 500:
        assert _ratio(out[:, rows], ref) < 1.05


@pytest.mark.parametrize("bits,gs,hidden,inter", [(4, 64, 1024, 1088), (4, 64, 4608, 640), (4, 32, 1056, 576), (4, 128, 1408, 4096), (8, 64, 2240, 512), (8, 32, 544, 1504),
                                                  (8, 128, 640, 2176)])
@pytest.mark.parametrize("tokens,experts,fused,dtype", [(3, 5, True, "f16"), (40, 6, False, "bf16"), (90, 40, True, "f32")])
def test_routed_block(hip, bits, gs, hidden, inter, tokens, experts, fused, dtype):
    """Experts with no row, one chunk, a little over one and several; the entry point without allocations, which routes and groups up to 8
    tokens in one launch, returns the same bits."""
    from rmlx_amd import ops, runtime as rt
    rng = np.random.default_rng(tokens + hidden + inter + bits)
    gate, up = (make_weight(rng, inter, hidden, bits, gs, (experts,)) for _ in range(2))
    down = make_weight(rng, hidden, inter, bits, gs, (experts,))
    d = ops.QuantizedWeight.from_numpy(*down, gs, bits)
    if fused:
        g, u = ops.QuantizedWeight.from_numpy(*(np.concatenate(p, axis=1) for p in zip(gate, up)), gs, bits), None
    else:
        g, u = (ops.QuantizedWeight.from_numpy(*w, gs, bits) for w in (gate, up))
    x = make_x(rng, tokens, hidden, dtype)
    xd = rt.DeviceBuffer.from_numpy(x, rt.BF16) if dtype == "bf16" else rt.DeviceBuffer.from_numpy(x)
    logits = rng.standard_normal((tokens, experts)).astype(np.float32)
    logits[:, 1] -= 20.0  # no token's pick
    logits[:17, 2] += 20.0  # 17 rows, 16 of them in the first chunk
    logits[:, 3] += 10.0  # (nearly) every token's
    idx, w, counts, _ = model.topk_route(logits, 2)
    g.set_expert_stream_kernel(6)
    ld = rt.DeviceBuffer.from_numpy(logits)
    out = ops.moe_forward(g, u, d, xd, ld, 2).numpy()
    print(f"slot-streaming block Q{bits} gs={gs} {hidden}/{inter} rows per expert {counts.tolist()}", flush=True)
    x64 = x_as_f64(x, dtype).astype(np.float16)
    ref = model.moe_forward(x64, idx, w, gate, up, down, gs, 2, bits=bits)
    assert_close(out, ref)
    assert _ratio(out, ref) < 1.2  # (the hidden activations are rounded to f16: about 1.08)
    same = ops.moe_forward(g, u, d, xd, ld, 2, noalloc=True).numpy()
    assert np.array_equal(same.view(np.uint16), out.view(np.uint16))


@pytest.mark.parametrize("tokens,taken", [(18, False), (20, True), (52, True), (53, False)])
def test_library_takes_it_for_a_few_rows_per_expert(hip, tokens, taken):
    """Experts of 6 MB, on average 5 to 13 rows each; a threshold of the caller's for the grouped GEMM goes first."""
    from rmlx_amd import ops, runtime as rt
    rng = np.random.default_rng(tokens)
    experts, hidden = 8, 2048
    one = [make_weight(rng, n, hidden, 4, 64, (1,)) for n in (2 * hidden, hidden)]
    gate_up, down = (tuple(np.ascontiguousarray(np.broadcast_to(a, (experts,) + a.shape[1:])) for a in t) for t in one)
    g, d = (ops.QuantizedWeight.from_numpy(*w, 64, 4) for w in (gate_up, down))
    x = make_x(rng, tokens, hidden)
    logits = rng.standard_normal((tokens, experts)).astype(np.float32)
    xd, ld = rt.DeviceBuffer.from_numpy(x), rt.DeviceBuffer.from_numpy(logits)

    def run(kind, min_rows=None):
        g.set_expert_stream_kernel(kind)
        prev = g.set_expert_gemm_min_rows(min_rows) if min_rows is not None else None
        out = ops.moe_forward(g, None, d, xd, ld, 2).numpy()
        if prev is not None:
            g.set_expert_gemm_min_rows(prev)
        return out

    auto, forced = run(0), run(6)
    assert np.array_equal(auto.view(np.uint16), forced.view(np.uint16)) == taken
    assert not np.array_equal(run(0, 2), forced)
    idx, w, _, _ = model.topk_route(logits, 2)
    gate, up = tuple(a[:, :hidden] for a in gate_up), tuple(a[:, hidden:] for a in gate_up)
    assert_close(auto, model.moe_forward(x, idx, w, gate, up, down, 64, 2))


@pytest.mark.parametrize("gs,k,n", [(64, 512, 128), (64, 4096, 515), (64, 6208, 300), (32, 1056, 1001), (128, 2944, 4100)])
@pytest.mark.parametrize("batch,rows,experts,dtype", [(1, 1, 3, "f16"), (5, 16, 2, "f16"), (37, 3, 4, "f32"), (256, 1, 200, "f16"), (255, 5, 7, "f32"), (160, 13, 3, "f16"),
                                                      (129, 2, 1000, "f16")])
def test_gather(hip, gs, k, n, batch, rows, experts, dtype):
    """Entries of one expert share chunks of 16 rows: runs of one entry and of many, chunks that begin in the middle of an entry, from one
    chunk for the whole chip to about half a chunk for a workgroup; on a stream the rows of an index out of range are zero."""
    from rmlx_amd import ops, runtime as rt
    from rmlx_amd.runtime import DeviceBuffer
    rng = np.random.default_rng(batch + rows + n)
    stored = min(experts, 8)
    w = make_weight(rng, n, k, 4, gs, (experts,) if experts == stored else (stored,))
    if experts != stored:
        w = tuple(np.concatenate([a] * (experts // stored), axis=0) for a in w)
    experts = w[0].shape[0]
    idx = rng.integers(0, experts, size=batch).astype(np.uint32)
    bad = np.zeros(batch, bool)
    if batch > 30:
        bad[[3, 17, 29]] = True
        idx[bad] = experts, 0xFFFFFFFE, 0xFFFFFFFF
    x = make_x(rng, batch * rows, k, dtype).reshape(batch, rows, k)
    stream = rt.Stream()
    out = ops.gather_qmm(DeviceBuffer.from_numpy(x), *(DeviceBuffer.from_numpy(a) for a in w), DeviceBuffer.from_numpy(idx), batch, rows, n, k, experts, gs,
                         stream=stream, kernel=rt.GATHER_SLOTS)
    stream.sync()
    out = out.numpy().reshape(batch, rows, n)
    assert not out[bad].any()
    cols = np.unique(np.concatenate([np.arange(min(n, 100)), np.arange(0, n, 29), np.arange(n - 40, n)]))
    x64 = x.astype(np.float16).astype(np.float64)
    ref = np.zeros((batch, rows, cols.size))
    for e in range(stored):
        of = ~bad & (idx % stored == e)
        if of.any():
            ref[of] = model.qmm(x64[of].reshape(-1, k), *(a[e][cols] for a in w), gs, 4).reshape(-1, rows, cols.size)
    assert_close(out[..., cols], ref)
    assert _ratio(out[..., cols], ref) < 1.05


@pytest.mark.parametrize("batch,rows,experts,n,k,taken", [(144, 1, 8, 1536, 2048, True), (16, 1, 8, 512, 1024, False), (64, 4, 8, 3072, 4096, True),
                                                          (6, 16, 8, 1536, 2048, False), (8, 4, 8, 6400, 1984, True)])
def test_library_takes_it_for_gathers_of_many_weights(hip, batch, rows, experts, n, k, taken):
    from rmlx_amd import ops, runtime as rt
    from rmlx_amd.runtime import DeviceBuffer
    rng = np.random.default_rng(batch + n)
    one = make_weight(rng, n, k, 4, 64)
    w = [DeviceBuffer.from_numpy(np.ascontiguousarray(np.broadcast_to(a, (experts,) + a.shape))) for a in one]
    x = make_x(rng, batch * rows, k).reshape(batch, rows, k)
    xd, idx = DeviceBuffer.from_numpy(x), DeviceBuffer.from_numpy(rng.integers(0, experts, size=batch).astype(np.uint32))
    auto, forced = (ops.gather_qmm(xd, *w, idx, batch, rows, n, k, experts, 64, kernel=q).numpy() for q in (0, rt.GATHER_SLOTS))
    assert np.array_equal(auto.view(np.uint16), forced.view(np.uint16)) == taken
    cols = np.arange(0, n, 37)
    assert_close(auto.reshape(-1, n)[:, cols], model.qmm(x.reshape(-1, k).astype(np.float64), *(a[cols] for a in one), 64, 4))


# both sides of each line of the rule, one call of every kind that it takes over (odd height, ragged K, each row count class, f32 rows that it
# reads itself and that are cast first)
@pytest.mark.parametrize("m,n,k,bits,gs,dtype,taken", [(1, 50001, 1024, 4, 64, "f16", True), (1, 50000, 1024, 4, 64, "f16", False), (2, 33001, 2880, 4, 64, "bf16", True),
                                                       (2, 4096, 2880, 4, 64, "f16", False), (8, 9216, 2880, 4, 64, "f16", True), (8, 9216, 4096, 4, 64, "f16", False),
                                                       (4, 14336, 6400, 4, 64, "f16", False), (9, 9216, 2048, 4, 128, "bf16", True), (16, 4096, 4096, 4, 64, "f16", False),
                                                       (12, 14336, 4096, 4, 64, "f32", True), (3, 2304, 1728, 8, 64, "bf16", True), (3, 2304, 1536, 8, 64, "bf16", False),
                                                       (13, 4096, 4096, 8, 64, "f32", True), (5, 4096, 4096, 8, 32, "f32", True), (4, 4096, 1024, 4, 32, "f16", True),
                                                       (8, 4096, 1024, 4, 32, "f16", False), (16, 4096, 1152, 4, 32, "bf16", True), (17, 4096, 1152, 4, 32, "bf16", False),
                                                       (6, 8192, 2560, 8, 64, "f16", False), (7, 8192, 2816, 8, 64, "bf16", True), (6, 8256, 2560, 8, 64, "f32", True),
                                                       (3, 16384, 1024, 8, 64, "f16", False), (3, 16384, 1024, 8, 64, "f32", True), (8, 8192, 2304, 8, 64, "f32", False),
                                                       (8, 16384, 1024, 8, 64, "f16", True), (9, 8192, 2304, 8, 64, "f16", False), (10, 8192, 2304, 8, 64, "f16", True),
                                                       (9, 12288, 1024, 8, 64, "f16", False), (2, 14336, 3520, 4, 64, "f16", False), (2, 14345, 3520, 4, 64, "f16", True),
                                                       (4, 12288, 3264, 4, 64, "bf16", False), (3, 12289, 3264, 4, 64, "f16", True), (4, 8192, 2560, 8, 128, "f16", True)])
def test_library_takes_it_for_a_few_rows(hip, m, n, k, bits, gs, dtype, taken):
    from rmlx_amd import ops, runtime as rt
    rng = np.random.default_rng(m + n + k)
    w = make_weight(rng, n, k, bits, gs)
    x = make_x(rng, m, k, dtype)
    xd = rt.DeviceBuffer.from_numpy(x, rt.BF16) if dtype == "bf16" else rt.DeviceBuffer.from_numpy(x)
    wd = ops.QuantizedWeight.from_numpy(*w, gs, bits)
    auto, forced = (ops.affine_quantized_matmul_batched(xd, wd, kernel=q).numpy() for q in (0, rt.KERNEL_QMV_RING))
    assert np.array_equal(auto.view(np.uint16), forced.view(np.uint16)) == taken
    cols = np.unique(np.concatenate([np.arange(0, n, 41), np.arange(n - 20, n)]))
    x64 = x_as_f64(x, dtype).astype(np.float16).astype(np.float64)
    assert_close(auto[:, cols], model.qmm(x64, *(a[cols] for a in w), gs, bits))


def test_rows_with_infinities_leave_the_others_alone(hip):
    """A row's values meet only its own sums: not another row's through the shared operands, nor those of the rows that a chunk lacks."""
    from rmlx_amd import ops, runtime as rt
    rng = np.random.default_rng(9)
    for bits, k in ((4, 2880), (4, 6144), (8, 4096)):
        w = make_weight(rng, 515, k, bits, 64)
        wd = ops.QuantizedWeight.from_numpy(*w, 64, bits)
        x = make_x(rng, 13, k)
        clean = ops.affine_quantized_matmul_batched(rt.DeviceBuffer.from_numpy(x), wd, kernel=rt.KERNEL_QMV_RING).numpy()
        x[3, 7], x[3, k - 1], x[8, k // 2], x[12, 0] = np.inf, -np.inf, np.nan, np.inf
        out = ops.affine_quantized_matmul_batched(rt.DeviceBuffer.from_numpy(x), wd, kernel=rt.KERNEL_QMV_RING).numpy()
        rest = [i for i in range(13) if i not in (3, 8, 12)]
        assert np.array_equal(out[rest].view(np.uint16), clean[rest].view(np.uint16))
        assert np.isnan(out[8]).all() and not np.isfinite(out[3]).any() and not np.isfinite(out[12]).any()


def _unbounded(x, w, gs, bits):
    """Reference of rows with infinities: NaN, +-inf by the signs of the weights that they meet (others: any finite value)."""
    words, scales, biases = w
    q = (words[..., None] >> np.arange(0, 32, bits, dtype=np.uint32)) & np.uint32((1 << bits) - 1)
    q = q.reshape(words.shape[0], -1)
    wide = scales.astype(np.float64).repeat(gs, axis=1) * q + biases.astype(np.float64).repeat(gs, axis=1)
    odd = ~np.isfinite(x).all(axis=0)
    with np.errstate(invalid="ignore"):
        return sum((np.outer(x[:, k], wide[:, k]) for k in np.flatnonzero(odd)), np.zeros((x.shape[0], wide.shape[0])))


def _assert_same_class(out, ref):
    for of in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(of(out), of(ref)), (of.__name__, int(of(out).sum()), int(of(ref).sum()))


@pytest.mark.parametrize("bits,gs,n,k,dtype", [(4, 32, 515, 2880, "f16"), (4, 32, 515, 4096, "bf16"), (4, 64, 5003, 704, "f32"), (4, 64, 515, 4096, "f16"),
                                               (4, 64, 515, 6144, "bf16"), (4, 128, 5003, 1408, "f16"), (4, 128, 515, 8192, "f16"), (8, 32, 515, 1504, "f16"),
                                               (8, 32, 515, 4096, "f32"), (8, 64, 515, 2880, "bf16"), (8, 64, 5003, 512, "f16"), (8, 128, 515, 4096, "f16")])
@pytest.mark.parametrize("m", [13, 18])
def test_infinite_activations_of_a_matrix(hip, bits, gs, n, k, dtype, m):
    """A row with an infinite value, or one that f16 does not hold, is what the sum of its products is: an infinity of the weight's sign, a NaN
    where that is zero or where two of them cancel."""
    from rmlx_amd import ops, runtime as rt
    rng = np.random.default_rng(m + n + k)
    w = make_weight(rng, n, k, bits, gs)
    wd = ops.QuantizedWeight.from_numpy(*w, gs, bits)
    x = make_x(rng, m, k).astype(np.float32)
    x[3, 7] = x[12, 0] = x[m - 1, k - 1] = np.inf if dtype == "f16" else 1e6
    x[4, k // 2] = x[12, k // 3] = -np.inf
    x[8, 5] = np.nan
    x[8, 6] = np.inf
    raw = model.f32_to_bf16_bits(x) if dtype == "bf16" else x.astype(np.float16 if dtype == "f16" else np.float32)
    xd = rt.DeviceBuffer.from_numpy(raw, rt.BF16) if dtype == "bf16" else rt.DeviceBuffer.from_numpy(raw)
    with np.errstate(over="ignore"):
        x16 = x_as_f64(raw, dtype).astype(np.float16)
    odd = ~np.isfinite(x16).all(axis=1)
    out = ops.affine_quantized_matmul_batched(xd, wd, kernel=rt.KERNEL_QMV_RING).numpy()
    _assert_same_class(out, _unbounded(x16.astype(np.float64), w, gs, bits))
    assert_close(out[~odd], model.qmm(x16[~odd].astype(np.float64), *w, gs, bits))


@pytest.mark.parametrize("bits", [4, 8])
def test_infinite_scales_and_biases(hip, bits):
    from rmlx_amd import ops, runtime as rt
    rng = np.random.default_rng(bits)
    n, k = 515, 704
    words, scales, biases = make_weight(rng, n, k, bits, 64)
    words |= 0x11111111 if bits == 4 else 0x01010101  # (no value of zero)
    x = np.abs(make_x(rng, 5, k)) + np.float16(0.1)
    run = lambda s, b: ops.affine_quantized_matmul_batched(rt.DeviceBuffer.from_numpy(x), ops.QuantizedWeight.from_numpy(words, s, b, 64, bits),
                                                           kernel=rt.KERNEL_QMV_RING).numpy()
    clean = run(scales, biases)
    scales, biases = scales.copy(), biases.copy()
    scales[3, 2], scales[500, 0], biases[7, 1] = np.inf, -np.inf, -np.inf
    out = run(scales, biases)
    assert np.isposinf(out[:, 3]).all() and np.isneginf(out[:, 500]).all() and np.isneginf(out[:, 7]).all()
    rest = np.setdiff1d(np.arange(n), [3, 7, 500])
    assert np.array_equal(out[:, rest].view(np.uint16), clean[:, rest].view(np.uint16))


@pytest.mark.parametrize("gs,n,k,rows", [(64, 515, 4096, 3), (32, 300, 1056, 16), (128, 1001, 1408, 5)])
def test_infinite_activations_of_a_gather(hip, gs, n, k, rows):
    from rmlx_amd import ops, runtime as rt
    from rmlx_amd.runtime import DeviceBuffer
    rng = np.random.default_rng(n)
    batch, experts = 37, 4
    w = make_weight(rng, n, k, 4, gs, (experts,))
    idx = rng.integers(0, experts, size=batch).astype(np.uint32)
    idx[[3, 29]] = experts, 0xFFFFFFFF  # zeros, whatever their rows hold
    x = make_x(rng, batch * rows, k).reshape(batch, rows, k)
    x[3], x[0, 1, 9], x[11, 0, k - 1], x[36, rows - 1, 40] = np.inf, -np.inf, np.inf, np.inf
    stream = rt.Stream()
    out = ops.gather_qmm(DeviceBuffer.from_numpy(x), *(DeviceBuffer.from_numpy(a) for a in w), DeviceBuffer.from_numpy(idx), batch, rows, n, k, experts, gs,
                         stream=stream, kernel=rt.GATHER_SLOTS)
    stream.sync()
    out = out.numpy().reshape(batch, rows, n)
    assert not out[[3, 29]].any()
    for i in [i for i in range(batch) if i not in (3, 29)]:
        _assert_same_class(out[i], _unbounded(x[i].astype(np.float64), tuple(a[idx[i]] for a in w), gs, 4))


@pytest.mark.parametrize("bits,gs,hidden,inter,fused", [(4, 64, 1024, 1088, True), (4, 32, 1056, 576, False), (4, 128, 4224, 512, True), (8, 64, 576, 2240, False)])
def test_infinite_activations_of_a_routed_block(hip, bits, gs, hidden, inter, fused):
    """Positive gate and up weights make an infinite hidden row of an infinite activation, down weights of one sign a row infinities of that sign."""
    from rmlx_amd import ops, runtime as rt
    rng = np.random.default_rng(hidden)
    experts, tokens = 6, 40

    def weights(n, k):
        words, scales, _ = make_weight(rng, n, k, bits, gs, (experts,))
        return words, scales, scales.copy()

    gate, up, down = weights(inter, hidden), weights(inter, hidden), weights(hidden, inter)
    for a in down[1:]:
        a[:, 1::2] *= -1
    d = ops.QuantizedWeight.from_numpy(*down, gs, bits)
    if fused:
        g, u = ops.QuantizedWeight.from_numpy(*(np.concatenate(p, axis=1) for p in zip(gate, up)), gs, bits), None
    else:
        g, u = (ops.QuantizedWeight.from_numpy(*w, gs, bits) for w in (gate, up))
    g.set_expert_stream_kernel(6)
    x = (make_x(rng, tokens, hidden) * np.float16(0.01)).astype(np.float16)
    ld = rt.DeviceBuffer.from_numpy(rng.standard_normal((tokens, experts)).astype(np.float32))
    clean = ops.moe_forward(g, u, d, rt.DeviceBuffer.from_numpy(x), ld, 2).numpy()
    odd = [0, 17, tokens - 1]
    x[odd, [3, hidden // 2, hidden - 1]] = np.inf
    out = ops.moe_forward(g, u, d, rt.DeviceBuffer.from_numpy(x), ld, 2).numpy()
    rest = [t for t in range(tokens) if t not in odd]
    assert np.isfinite(clean).all() and np.array_equal(out[rest].view(np.uint16), clean[rest].view(np.uint16))
    assert np.isposinf(out[odd][:, 0::2]).all() and np.isneginf(out[odd][:, 1::2]).all()


@pytest.mark.parametrize("bits,gs,hidden,inter,experts,dtype", [(4, 64, 576, 512, 600, "f16"), (8, 64, 512, 640, 560, "bf16"), (4, 32, 544, 544, 300, "f32"),
                                                                (4, 64, 4608, 512, 540, "f16")])
def test_more_chunks_than_workgroups(hip, bits, gs, hidden, inter, experts, dtype):
    """A workgroup's share then holds whole chunks, one behind another, and begins and ends inside others: rings, sums and activations start over."""
    from rmlx_amd import ops, runtime as rt
    rng = np.random.default_rng(experts)
    tokens = experts * 3 // 2
    one = [make_weight(rng, n, k, bits, gs, (20,)) for n, k in ((inter, hidden), (inter, hidden), (hidden, inter))]
    gate, up, down = (tuple(np.ascontiguousarray(np.resize(a, (experts,) + a.shape[1:])) for a in t) for t in one)
    g, u, d = (ops.QuantizedWeight.from_numpy(*w, gs, bits) for w in (gate, up, down))
    g.set_expert_stream_kernel(6)
    x = make_x(rng, tokens, hidden, dtype)
    xd = rt.DeviceBuffer.from_numpy(x, rt.BF16) if dtype == "bf16" else rt.DeviceBuffer.from_numpy(x)
    idx = rng.integers(0, experts, size=(tokens, 2)).astype(np.uint32)
    idx[:, 0] = np.arange(tokens) % experts  # every expert one row or two and what it is picked by at random
    idx[7:40, 1], idx[60:77, 1] = 11, experts - 40  # three chunks, two
    w = rng.uniform(0.2, 0.8, size=(tokens, 2)).astype(np.float32)
    counts = np.bincount(idx.ravel(), minlength=experts)
    chunks = int(((counts + 15) // 16).sum())
    print(f"Q{bits} gs={gs} {hidden}/{inter}: {chunks} chunks, at most {counts.max()} rows", flush=True)
    assert chunks > 256 and (counts > 16).sum() >= 2 and (experts < 512 or chunks > 512)
    out = ops.moe_forward_grouped(g, u, d, xd, rt.DeviceBuffer.from_numpy(idx.ravel()), rt.DeviceBuffer.from_numpy(w.ravel()), 2).numpy()
    x16 = x_as_f64(x, dtype).astype(np.float16)
    assert_close(out, model.moe_forward(x16, idx.ravel(), w.ravel(), gate, up, down, gs, 2, bits=bits))


def test_pinned_block_keeps_the_callers_gemm_threshold(hip):
    """Pinned, it runs batches of every size; from a threshold of the caller's on the grouped GEMM does, as behind every other kernel."""
    from rmlx_amd import ops, runtime as rt
    rng = np.random.default_rng(13)
    experts, hidden, tokens = 8, 1024, 96
    g, d = (ops.QuantizedWeight.from_numpy(*make_weight(rng, n, hidden, 4, 64, (experts,)), 64, 4) for n in (2 * hidden, hidden))
    xd = rt.DeviceBuffer.from_numpy(make_x(rng, tokens, hidden))
    ld = rt.DeviceBuffer.from_numpy(rng.standard_normal((tokens, experts)).astype(np.float32))

    def run(kind, min_rows):
        g.set_expert_stream_kernel(kind)
        prev = g.set_expert_gemm_min_rows(min_rows) if min_rows is not None else None
        out = ops.moe_forward(g, None, d, xd, ld, 2).numpy().view(np.uint16)
        if prev is not None:
            g.set_expert_gemm_min_rows(prev)
        return out

    slots, gemm = run(6, 0), run(1, 24)
    assert not np.array_equal(slots, gemm)
    assert np.array_equal(run(6, 24), gemm)  # 24 rows per expert
    assert np.array_equal(run(6, 25), slots) and np.array_equal(run(6, None), slots)


def test_more_chunks_than_a_grid_has_rows(hip):
    """65552 chunks at most: their number is no grid dimension here."""
    from rmlx_amd import ops, runtime as rt
    rng = np.random.default_rng(14)
    hidden, inter, experts, tokens = 512, 512, 16, 131072
    gate, up, down = (make_weight(rng, n, 512, 4, 64, (experts,)) for n in (inter, inter, hidden))
    g, u, d = (ops.QuantizedWeight.from_numpy(*w, 64, 4) for w in (gate, up, down))
    g.set_expert_stream_kernel(6)
    x = make_x(rng, tokens, hidden)
    logits = rng.standard_normal((tokens, experts)).astype(np.float32)
    stream, out, xd, ld = rt.Stream(), rt.DeviceBuffer((tokens, hidden), rt.F16), rt.DeviceBuffer.from_numpy(x), rt.DeviceBuffer.from_numpy(logits)
    ops.moe_forward(g, u, d, xd, ld, 8, stream=stream, out=out)
    stream.sync()
    some = np.r_[np.arange(0, tokens, 5003), np.arange(tokens - 40, tokens)]
    idx, w, _, _ = model.topk_route(logits[some], 8)
    assert_close(out.numpy()[some], model.moe_forward(x[some], idx, w, gate, up, down, 64, 8))


def test_rows_beyond_a_gigabyte_of_activations(hip):
    """K = 2240 in two slots leaves a wave without k in the second: its loads stay outside the buffer wherever the row begins."""
    from rmlx_amd import ops, runtime as rt
    rng = np.random.default_rng(12)
    hidden, inter, experts, tokens = 2240, 512, 2, 239900
    assert tokens * hidden * 2 > 1 << 30
    gate, up = (make_weight(rng, inter, hidden, 8, 64, (experts,)) for _ in range(2))
    down = make_weight(rng, hidden, inter, 8, 64, (experts,))
    g, u, d = (ops.QuantizedWeight.from_numpy(*w, 64, 8) for w in (gate, up, down))
    g.set_expert_stream_kernel(6)
    x = np.resize(make_x(rng, 2000, hidden), (tokens, hidden))
    logits = rng.standard_normal((tokens, experts)).astype(np.float32)
    out = rt.DeviceBuffer((tokens, hidden), rt.F16)
    ops.moe_forward(g, u, d, rt.DeviceBuffer.from_numpy(x), rt.DeviceBuffer.from_numpy(logits), 1, out=out)
    some = np.r_[np.arange(0, tokens, 30011), np.arange(tokens - 250, tokens)]
    idx, w, _, _ = model.topk_route(logits[some], 1)
    ref = model.moe_forward(x[some], idx, w, gate, up, down, 64, 1, bits=8)
    assert_close(out.numpy()[some], ref)


@pytest.mark.parametrize("bits,gs,k,taken", [(4, 64, 8192, True), (4, 64, 8256, False), (4, 128, 8192, True), (4, 128, 8320, False), (4, 32, 4096, True), (4, 32, 4128, False),
                                             (8, 64, 4096, True), (8, 64, 4160, False), (8, 128, 512, True), (8, 128, 384, False)])
def test_refusals_name_the_limits_of_k(hip, bits, gs, k, taken):
    from rmlx_amd import ops, runtime as rt
    rng = np.random.default_rng(k)
    w, x = ops.QuantizedWeight.from_numpy(*make_weight(rng, 128, k, bits, gs), gs, bits), rt.DeviceBuffer.from_numpy(make_x(rng, 2, k))
    if taken:
        ops.affine_quantized_matmul_batched(x, w, kernel=rt.KERNEL_QMV_RING)
        return
    with pytest.raises(rt.KernelError, match=r"512 <= K <= 8192 \(8-bit weights and group size 32: 4096\)"):
        ops.affine_quantized_matmul_batched(x, w, kernel=rt.KERNEL_QMV_RING)


def test_recorded_calls_replay_bit_for_bit(hip):
    """A matrix, a gather and a routed block recorded into one graph, with eager work between the replays."""
    from rmlx_amd import ops, runtime as rt
    from rmlx_amd.runtime import DeviceBuffer
    rng = np.random.default_rng(10)
    n, k, experts, tokens = 520, 1088, 5, 40
    wd = ops.QuantizedWeight.from_numpy(*make_weight(rng, n, k, 4, 64), 64, 4)
    stacked = [DeviceBuffer.from_numpy(a) for a in make_weight(rng, n, k, 4, 64, (experts,))]
    gate_up, down = make_weight(rng, 1280, k, 4, 64, (experts,)), make_weight(rng, k, 640, 4, 64, (experts,))
    g, d = ops.QuantizedWeight.from_numpy(*gate_up, 64, 4), ops.QuantizedWeight.from_numpy(*down, 64, 4)
    g.set_expert_stream_kernel(6)
    x, rows = DeviceBuffer.from_numpy(make_x(rng, tokens, k)), DeviceBuffer.from_numpy(make_x(rng, 13, k))
    picks = DeviceBuffer.from_numpy(rng.integers(0, experts, size=20).astype(np.uint32))
    logits = DeviceBuffer.from_numpy(rng.standard_normal((tokens, experts)).astype(np.float32))
    stream = rt.Stream()
    outs = [DeviceBuffer(s, rt.F16) for s in ((13, n), (20, 2, n), (tokens, k))]

    def calls(outs):
        ops.affine_quantized_matmul_batched(rows, wd, stream=stream, kernel=rt.KERNEL_QMV_RING, out=outs[0])
        ops.gather_qmm(x, *stacked, picks, 20, 2, n, k, experts, 64, stream=stream, kernel=rt.GATHER_SLOTS, out=outs[1])
        ops.moe_forward(g, None, d, x, logits, 2, stream=stream, out=outs[2], noalloc=True)

    calls(outs)
    stream.sync()
    eager = [o.numpy().copy() for o in outs]
    with rt.Graph.record(stream) as graph:
        calls(outs)
    for _ in range(3):
        for o in outs:
            rt.check(rt.lib().rmlx_hip_memcpy_h2d(o.ptr, np.full(o.shape, np.nan, np.float16).ctypes.data, o.nbytes, None))
        graph.launch(stream)
        stream.sync()
        for o, e in zip(outs, eager):
            assert np.array_equal(o.numpy().view(np.uint16), e.view(np.uint16))
        calls(outs)
        stream.sync()


@pytest.mark.parametrize("bits,gs,n,k", [(8, 64, 32776, 4096), (8, 64, 33001, 4096), (8, 32, 33024, 4032), (4, 64, 33001, 8192), (4, 64, 132096, 4096)])
def test_shares_away_from_one_part_of_the_channels(hip, bits, gs, n, k):
    """One workgroup less or several: every row once, the same bits as in a matrix of a few rows."""
    from rmlx_amd import ops, runtime as rt
    rng = np.random.default_rng(n + k)
    base = 400
    w = make_weight(rng, base, k, bits, gs)
    x = make_x(rng, 3, k)
    xd = rt.DeviceBuffer.from_numpy(x)
    run = lambda t: ops.affine_quantized_matmul_batched(xd, ops.QuantizedWeight.from_numpy(*t, gs, bits), kernel=rt.KERNEL_QMV_RING).numpy()
    small, out = run(w), run(tuple(np.resize(a, (n,) + a.shape[1:]) for a in w))
    assert_close(small, model.qmm(x, *w, gs, bits))
    assert np.array_equal(out.view(np.uint16), np.resize(small.T, (n, 3)).T.view(np.uint16))
