"""GPU parity of the large-tile GEMM (kernel selector 12) against the float64 dequantize-then-matmul oracle."""
import numpy as np
import pytest

from oracle import model
from tests.helpers import assert_close, make_weight, make_x, x_as_f64

pytestmark = pytest.mark.gpu


def _run(words, scales, biases, x, bits, gs=64, dtype="f16"):
    from rmlx_amd import ops, runtime as rt
    from rmlx_amd.runtime import BF16, DeviceBuffer
    qw = ops.QuantizedWeight.from_numpy(words, scales, biases, gs, bits)
    xd = DeviceBuffer.from_numpy(x, BF16) if dtype == "bf16" else DeviceBuffer.from_numpy(x)
    return ops.affine_quantized_matmul_batched(xd, qw, kernel=rt.KERNEL_QMM_TILE).numpy()


@pytest.mark.parametrize("bits,gs", [(4, 64), (4, 32), (4, 128), (8, 64), (8, 32), (8, 128)])
@pytest.mark.parametrize("m,n,groups,dtype", [(1, 1, 8, "f16"), (31, 127, 9, "f16"), (33, 129, 8, "bf16"), (64, 64, 13, "f16"), (65, 7, 17, "f32"),
                                              (130, 257, 11, "f16"), (257, 300, 8, "bf16"), (96, 1000, 45, "f16"), (300, 2051, 8, "f16"),
                                              (40, 9, 1, "f16"), (70, 130, 2, "bf16"), (33, 3, 3, "f16"), (270, 521, 7, "f16"), (5, 2, 5, "f16")])
def test_large_tile_gemm(hip, bits, gs, m, n, groups, dtype):
    """Remainders in every dimension: rows and columns that are no whole tile (odd counts among them), K that is no whole
    128-wide round and no whole unit of eight groups or less than one, one row, one column."""
    k = groups * gs
    rng = np.random.default_rng(bits * 1000 + gs + m + n + k)
    words, s, b = make_weight(rng, n, k, bits, gs)
    x = make_x(rng, m, k, dtype)
    ref = model.qmm(x_as_f64(x, dtype), words, s, b, gs, bits)
    assert_close(_run(words, s, b, x, bits, gs, dtype), ref,
                 f"large-tile gemm M={m} N={n} K={k} bits={bits} gs={gs} {dtype}")


@pytest.mark.parametrize("m,n,k,bits", [(2085, 4128, 1088, 4), (1100, 4100, 576, 8), (700, 1030, 4160, 4), (160, 260, 8256, 4), (40, 20000, 640, 4),
                                      (70, 897, 5760, 4), (70, 5947, 576, 4), (7, 16459, 576, 4), (70, 10938, 1344, 4), (70, 5516, 512, 4),
                                      (7, 203, 3008, 8), (70, 901, 3008, 8), (7, 16439, 576, 8), (45, 8234, 3456, 8), (97, 2745, 9152, 8)])
def test_large_tile_gemm_plans_and_epilogues(hip, m, n, k, bits):
    """Sizes that the automatic choice sends to the different tiles and splits; fused epilogues."""
    from rmlx_amd import ops
    from rmlx_amd.runtime import DeviceBuffer
    rng = np.random.default_rng(m + n + k)
    words, s, b = make_weight(rng, n, k, bits)
    x = make_x(rng, m, k)
    rows = np.unique(np.concatenate([np.arange(0, m, 37), [m - 1]]))
    ref = model.qmm(x_as_f64(x[rows], "f16"), words, s, b, 64, bits)
    out = _run(words, s, b, x, bits)
    assert_close(out[rows], ref, f"large-tile gemm M={m} N={n} K={k} bits={bits}")
    qw = ops.QuantizedWeight.from_numpy(words, s, b, 64, bits)
    xd = DeviceBuffer.from_numpy(x)
    for edtype in (np.float16, np.float32):
        e = rng.standard_normal((m, n)).astype(edtype)
        ed = DeviceBuffer.from_numpy(e)
        assert_close(ops.qmm_add_residual(xd, qw, ed).numpy()[rows], ref + e[rows].astype(np.float64), "residual")
        assert_close(ops.qmm_swiglu(xd, qw, ed).numpy()[rows], model.silu(e[rows].astype(np.float64)) * ref, "swiglu")


@pytest.mark.parametrize("bits,gs", [(4, 64), (4, 32), (8, 64), (4, 128)])
@pytest.mark.parametrize("tokens,experts,top_k,hidden,inter,fused", [(600, 4, 2, 1088, 544, True), (150, 6, 3, 1024, 1056, False), (1100, 3, 1, 1280, 1024, True),
                                                                      (30, 8, 2, 1088, 544, True), (40, 5, 2, 1024, 1056, False),
                                                                      (80, 4, 2, 1088, 544, True), (80, 4, 2, 1280, 1024, False),
                                                                      (400, 4, 2, 1280, 1024, True), (900, 3, 2, 1088, 544, False)])
def test_routed_block_on_large_tiles(hip, bits, gs, tokens, experts, top_k, hidden, inter, fused):
    """Row tiles of 32 (8 and 16 rows per expert), 64 (40; 128 at group size 32), 128 (75, 300 and 366) and 256 rows (200 and 600) of one
    expert, reached through the token map; weights in two products (1088 x 544) and rounded (1280 x 1024); dimensions that are no whole tiles, gate / up stacked and apart; the packed
    outputs of ExpertGroup over the same experts, an item of one row and an empty one among them."""
    from rmlx_amd import ops
    from rmlx_amd.runtime import DeviceBuffer
    hidden, inter = max(hidden, 8 * gs) // gs * gs, max(inter, 8 * gs) // gs * gs
    rng = np.random.default_rng(bits + gs + tokens)
    gate, up = (make_weight(rng, inter, hidden, bits, gs, (experts,)) for _ in range(2))
    down = make_weight(rng, hidden, inter, bits, gs, (experts,))
    both = tuple(np.concatenate([a, b], axis=1) for a, b in zip(gate, up))
    g = ops.QuantizedWeight.from_numpy(*(both if fused else gate), gs, bits)
    u = None if fused else ops.QuantizedWeight.from_numpy(*up, gs, bits)
    d = ops.QuantizedWeight.from_numpy(*down, gs, bits)
    x = make_x(rng, tokens, hidden)
    logits = rng.standard_normal((tokens, experts)).astype(np.float32)
    out = ops.moe_forward(g, u, d, DeviceBuffer.from_numpy(x), DeviceBuffer.from_numpy(logits), top_k).numpy()
    idx, w, _, _ = model.topk_route(logits, top_k)
    rows = np.unique(np.concatenate([np.arange(0, tokens, 29), [tokens - 1]]))
    sel = (rows[:, None] * top_k + np.arange(top_k)[None, :]).reshape(-1)
    ref = model.moe_forward(x[rows], idx[sel], w[sel], gate, up, down, gs, top_k, bits=bits)
    assert_close(out[rows], ref, f"routed block T={tokens} E={experts} D={hidden} I={inter} bits={bits} gs={gs}")
    sizes = [1, 0, tokens // 2, 97]
    items = [(i % experts, DeviceBuffer.from_numpy(x[:n])) for i, n in enumerate(sizes)]
    for (e, y), n in zip(ops.ExpertGroup(g, u, d).grouped_forward(items), sizes):
        pick = slice(0, n, 17)
        ref = model.moe_forward(x[:n][pick], np.full(len(x[:n][pick]), e), np.ones(len(x[:n][pick]), np.float32), gate, up, down, gs, 1, bits=bits)
        if n:
            assert_close(y[pick], ref, f"ExpertGroup item of {n} rows")


@pytest.mark.parametrize("batch,rows,n,k,gs", [(3, 70, 130, 1056, 32), (5, 9, 129, 1088, 64), (2, 300, 260, 1024, 128), (40, 3, 72, 640, 64)])
def test_gather_on_small_tiles(hip, batch, rows, n, k, gs):
    """Few rows: tiles of 32 of one entry, and the single-row kernel."""
    _gather(batch, rows, n, k, gs)


# rows per entry -> row tiles of 64 (128 at group size 32), 128, 256 and again 128 rows, in equal shares; N in whole columns of a tile (K in whole
# slabs: the grouped GEMM's shapes) and off them
@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("batch,rows,n,k", [(45, 50, 448, 640), (45, 64, 450, 640), (45, 33, 512, 1024), (20, 100, 448, 640), (20, 128, 577, 640),
                                            (14, 200, 448, 640), (14, 256, 512, 1024), (8, 300, 514, 640), (5, 513, 512, 640)])
def test_gather_on_large_tiles(hip, batch, rows, n, k, gs):
    # (a third condition keeps small launches on tiles of 32 rows)
    assert batch * (-(-rows // 32)) * (-(-n // 64)) > 2 * hip.device_info()["compute_units"] and rows > 32
    _gather(batch, rows, n, k, gs)


def _gather(batch, rows, n, k, gs):
    from rmlx_amd import ops
    from rmlx_amd.runtime import DeviceBuffer
    rng = np.random.default_rng(batch + rows + n + k)
    words, s, b = make_weight(rng, n, k, 4, gs, (4,))
    idx = rng.integers(0, 4, size=batch).astype(np.uint32)
    x = make_x(rng, batch * rows, k).reshape(batch, rows, k)
    bufs = [DeviceBuffer.from_numpy(a) for a in (words, s, b)]
    out = ops.gather_qmm(DeviceBuffer.from_numpy(x), *bufs, DeviceBuffer.from_numpy(idx), batch, rows, n, k, 4, gs).numpy()
    for i in range(batch):
        ref = model.qmm(x[i].astype(np.float64), words[idx[i]], s[idx[i]], b[idx[i]], gs, 4)
        assert_close(out[i], ref, f"gather entry {i}")


def _block(rng, experts, hidden, inter, bits=4, gs=64):
    from rmlx_amd import ops
    gate, up = (make_weight(rng, inter, hidden, bits, gs, (experts,)) for _ in range(2))
    down = make_weight(rng, hidden, inter, bits, gs, (experts,))
    return (gate, up, down), tuple(ops.QuantizedWeight.from_numpy(*w, gs, bits) for w in (gate, up, down))


@pytest.mark.parametrize("m,n,k,bits,gs", [(1035, 7859, 160, 4, 32), (540, 18277, 160, 4, 32), (1424, 8708, 160, 4, 32), (519, 31005, 160, 4, 32),
                                         (550, 12011, 448, 4, 64), (1441, 6150, 384, 4, 128), (513, 3589, 160, 8, 32), (303, 3667, 5120, 8, 128),
                                         (780, 9275, 224, 8, 32), (543, 14190, 96, 8, 32), (2698, 4894, 96, 8, 32), (411, 22650, 96, 8, 32), (532, 23055, 192, 8, 64)])
def test_two_workgroups_per_cu(hip, m, n, k, bits, gs):
    """Sizes that the automatic choice sends to tiles of 128 and 256 columns of the GEMM with two workgroups per CU, at every height it has and
    with K split; K of half stages, columns and rows that are no whole tile.  Every output against the oracle's, plain and with a residual."""
    from rmlx_amd import ops
    from rmlx_amd.runtime import DeviceBuffer
    rng = np.random.default_rng(m + n + k)
    words, s, b = make_weight(rng, n, k, bits, gs)
    x = make_x(rng, m, k)
    ref = model.qmm(x_as_f64(x, "f16"), words, s, b, gs, bits)
    assert_close(_run(words, s, b, x, bits, gs), ref, f"M={m} N={n} K={k} bits={bits} gs={gs}")
    e = rng.standard_normal((m, n)).astype(np.float16)
    qw = ops.QuantizedWeight.from_numpy(words, s, b, gs, bits)
    assert_close(ops.qmm_add_residual(DeviceBuffer.from_numpy(x), qw, DeviceBuffer.from_numpy(e)).numpy(), ref + e.astype(np.float64), "residual")


@pytest.mark.parametrize("m,n,k,bits,gs", [(188, 62528, 512, 4, 128), (923, 12864, 512, 4, 64), (404, 32320, 512, 4, 32), (451, 18624, 512, 8, 64), (714, 14528, 512, 8, 128)])
def test_short_rows_of_bf16_stay_on_the_tile_gemm(hip, m, n, k, bits, gs):
    """Rows of up to 1024 values over wide matrices, where the estimate of the GEMM with two workgroups per CU lies below the line to the GEMMs of before."""
    from rmlx_amd import ops, runtime as rt
    rng = np.random.default_rng(m + n)
    w = make_weight(rng, n, k, bits, gs)
    x = make_x(rng, m, k, "bf16")
    xd, qw = rt.DeviceBuffer.from_numpy(x, rt.BF16), ops.QuantizedWeight.from_numpy(*w, gs, bits)
    auto, tile, other = (ops.affine_quantized_matmul_batched(xd, qw, kernel=q).numpy().view(np.uint16) for q in (0, rt.KERNEL_QMM_TILE, rt.KERNEL_QMM))
    assert np.array_equal(auto, tile) and not np.array_equal(auto, other)
    cols = np.arange(0, n, 97)
    assert_close(auto.view(np.float16)[:, cols], model.qmm(x_as_f64(x, "bf16"), *(a[cols] for a in w), gs, bits))


# Row tiles of one to seven fragments of 128 columns (8-bit too) and of one to five of 256 (8-bit: four), the last of them shorter; rows of several units
# of scales, the last one early, half a stage at the end; columns that are no whole tile.
@pytest.mark.parametrize("m,n,bits", [(5, 301, 4), (42, 1001, 4), (79, 300, 4), (301, 9001, 4), (153, 17001, 4), (190, 17000, 4), (1189, 5203, 4), (20, 110001, 4), (42, 33000, 4),
                                      (79, 33001, 4), (116, 33003, 4), (412, 33000, 4), (5, 301, 8), (42, 1001, 8), (116, 17003, 8), (412, 9001, 8), (486, 9001, 8),
                                      (1226, 5203, 8), (20, 70001, 8), (42, 70001, 8), (227, 33001, 8), (338, 33003, 8)])
@pytest.mark.parametrize("k,gs", [(2112, 64), (1056, 32), (1408, 128)])
def test_two_workgroups_at_every_height(hip, m, n, bits, k, gs):
    """Selector 17 runs the kernel whatever the estimate says."""
    from rmlx_amd import ops, runtime as rt
    rng = np.random.default_rng(m + n + k + bits)
    w = make_weight(rng, n, k, bits, gs)
    x = make_x(rng, m, k)
    out = ops.affine_quantized_matmul_batched(rt.DeviceBuffer.from_numpy(x), ops.QuantizedWeight.from_numpy(*w, gs, bits), kernel=rt.KERNEL_QMM_TWIN).numpy()
    cols = np.unique(np.concatenate([np.arange(0, n, 331), np.arange(max(0, n - 70), n)]))
    assert_close(out[:, cols], model.qmm(x_as_f64(x, "f16"), *(a[cols] for a in w), gs, bits), f"M={m} N={n} K={k} bits={bits} gs={gs}")


# The library's choice on both sides of its lines to that kernel, where the other plan splits K (over waves or workgroups, so its sums round differently): a few
# rows over short and long ones, 10432 values in three ranges.
@pytest.mark.parametrize("m,n,k,bits,gs,taken", [(30, 106240, 1024, 8, 128, True), (24, 130688, 1024, 4, 64, True), (9, 22016, 14336, 4, 64, False),
                                                 (21, 62144, 2048, 4, 64, False), (48, 32768, 4096, 8, 64, False), (2398, 896, 10432, 4, 64, False)])
def test_library_takes_two_workgroups(hip, m, n, k, bits, gs, taken):
    from rmlx_amd import ops, runtime as rt
    rng = np.random.default_rng(m + n + k)
    w = make_weight(rng, n, k, bits, gs)
    x = make_x(rng, m, k)
    xd, qw = rt.DeviceBuffer.from_numpy(x), ops.QuantizedWeight.from_numpy(*w, gs, bits)
    auto, tile, twin = (ops.affine_quantized_matmul_batched(xd, qw, kernel=q).numpy().view(np.uint16) for q in (0, rt.KERNEL_QMM_TILE, rt.KERNEL_QMM_TWIN))
    assert np.array_equal(auto, tile) and np.array_equal(auto, twin) == taken
    cols = np.arange(0, n, 331)
    rows = np.arange(0, m, 7)
    assert_close(auto.view(np.float16)[np.ix_(rows, cols)], model.qmm(x_as_f64(x, "f16")[rows], *(a[cols] for a in w), gs, bits))


@pytest.mark.parametrize("tokens,experts,hidden,inter,bits,gs,fused", [(1500, 32, 1088, 576, 4, 64, True), (3400, 32, 1056, 544, 4, 32, False), (5200, 32, 1088, 576, 4, 64, False),
                                                                      (1600, 40, 1024, 512, 4, 128, True), (3400, 40, 1088, 576, 8, 64, True), (5300, 40, 1056, 544, 8, 32, False)])
def test_routed_block_on_two_workgroups_per_cu(hip, tokens, experts, hidden, inter, bits, gs, fused):
    """Enough tiles for two workgroups on every CU: experts of a few rows to more than one row tile (160, 128 rows)."""
    from rmlx_amd import ops
    from rmlx_amd.runtime import DeviceBuffer
    rng = np.random.default_rng(bits + gs + tokens)
    gate, up = (make_weight(rng, inter, hidden, bits, gs, (experts,)) for _ in range(2))
    down = make_weight(rng, hidden, inter, bits, gs, (experts,))
    both = tuple(np.concatenate([a, b], axis=1) for a, b in zip(gate, up))
    g = ops.QuantizedWeight.from_numpy(*(both if fused else gate), gs, bits)
    u = None if fused else ops.QuantizedWeight.from_numpy(*up, gs, bits)
    d = ops.QuantizedWeight.from_numpy(*down, gs, bits)
    x = make_x(rng, tokens, hidden)
    logits = rng.standard_normal((tokens, experts)).astype(np.float32) + 1.5 * rng.standard_normal(experts).astype(np.float32)
    out = ops.moe_forward(g, u, d, DeviceBuffer.from_numpy(x), DeviceBuffer.from_numpy(logits), 1).numpy()
    idx, w, _, _ = model.topk_route(logits, 1)
    assert_close(out, model.moe_forward(x, idx, w, gate, up, down, gs, 1, bits=bits), f"E={experts} D={hidden} I={inter} T={tokens} bits={bits} gs={gs}")


# By the prices on 256 CUs: on two workgroups per CU, 4-bit at 130 rows an expert (group sizes 32 and 64) and 300 (128), 8-bit at 300 (32) and 90 (64), dimensions in
# multiples of 64, which round their weights; on the other tiles, 70 rows, 170 rows, 8-bit 110 rows.
@pytest.mark.parametrize("tokens,experts,hidden,inter,bits,gs,fused", [(4160, 32, 1088, 576, 4, 32, False), (4160, 32, 1088, 576, 4, 64, True), (7200, 24, 1152, 640, 4, 128, True),
                                                                      (7200, 24, 1088, 1152, 8, 32, False), (3600, 40, 1088, 576, 8, 64, False),
                                                                      (2240, 32, 1088, 1152, 4, 64, True), (5440, 32, 1088, 576, 4, 64, False), (4400, 40, 1088, 576, 8, 64, True)])
def test_routed_block_by_its_prices(hip, tokens, experts, hidden, inter, bits, gs, fused):
    test_routed_block_on_two_workgroups_per_cu(hip, tokens, experts, hidden, inter, bits, gs, fused)


@pytest.mark.parametrize("tokens,experts,top_k,hidden,inter", [(262200, 8, 8, 512, 512), (131100, 2, 1, 8192, 512)])
def test_routed_block_over_more_than_two_gib(hip, tokens, experts, top_k, hidden, inter):
    """Hidden activations, and activations reached through the token map, of more than 2 GiB; the last tokens, which lie beyond it."""
    from rmlx_amd import ops
    from rmlx_amd.runtime import DeviceBuffer
    rng = np.random.default_rng(tokens)
    host, dev = _block(rng, experts, hidden, inter)
    x = np.tile(make_x(rng, 600, hidden), (-(-tokens // 600), 1))[:tokens]
    assert max(x.nbytes, tokens * top_k * inter * 2) > 2 << 30
    logits = rng.standard_normal((tokens, experts)).astype(np.float32)
    out = ops.moe_forward(*dev, DeviceBuffer.from_numpy(x), DeviceBuffer.from_numpy(logits), top_k).numpy()
    rows = np.concatenate([np.arange(20), rng.integers(0, tokens, 20), np.arange(tokens - 20, tokens)])
    idx, w, _, _ = model.topk_route(logits[rows], top_k)
    assert_close(out[rows], model.moe_forward(x[rows], idx, w, *host, 64, top_k), f"T={tokens} D={hidden} I={inter}")


def test_routed_block_over_activations_off_16_bytes(hip):
    """bf16 and f32 activations are cast, so their alignment plays no part: the bits of the aligned call."""
    import ctypes
    from rmlx_amd import ops
    from rmlx_amd.runtime import BF16, DeviceBuffer
    rng = np.random.default_rng(4)
    _, dev = _block(rng, 4, 512, 512)
    logits = DeviceBuffer.from_numpy(rng.standard_normal((200, 4)).astype(np.float32))
    for dtype in ("bf16", "f32"):
        x = make_x(rng, 200, 512, dtype)
        kind = BF16 if dtype == "bf16" else None
        want = ops.moe_forward(*dev, DeviceBuffer.from_numpy(x, kind), logits, 2).numpy()
        off = DeviceBuffer.from_numpy(np.concatenate([x.reshape(-1)[:1], x.reshape(-1)]), kind)
        xa, la, out = off.array((200, 512), 1), logits.array(), DeviceBuffer((200, 512), hip.F16)
        hip.check(hip.lib().rmlx_hip_moe_forward(*(q.handle for q in dev), ctypes.byref(xa), ctypes.byref(la), 2, None, out.ptr, out.nbytes, None))
        assert np.array_equal(out.numpy().view(np.uint16), want.view(np.uint16)), dtype


def test_more_experts_than_the_grouping_kernel_sorts(hip):
    """Portable dimensions run without grouping, whatever the number of experts."""
    from rmlx_amd import ops
    from rmlx_amd.runtime import DeviceBuffer
    rng = np.random.default_rng(6)
    host, dev = _block(rng, 1100, 64, 64)
    x = make_x(rng, 3000, 64)
    idx = rng.integers(0, 1100, 3000).astype(np.uint32)
    w = rng.uniform(0.2, 1.0, 3000).astype(np.float32)
    out = ops.moe_forward_grouped(*dev, DeviceBuffer.from_numpy(x), DeviceBuffer.from_numpy(idx), DeviceBuffer.from_numpy(w), 1).numpy()
    assert_close(out[::17], model.moe_forward(x[::17], idx[::17], w[::17], *host, 64, 1))
