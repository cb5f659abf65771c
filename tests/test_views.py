"""The rmlx_array views that the hot calls keep on their buffers (CPU only: the library call is replaced)."""
import threading
import types
import weakref

import pytest

from rmlx_amd import ops, runtime as rt

CALLS = {
    "matmul": lambda x, q, out: ops.affine_quantized_matmul_batched(x, q, out=out),
    "gather_qmm": lambda x, q, out: ops.gather_qmm(x, out, out, out, x, 1, 1, 8, 64, 1, 64, out=out),
    "moe_forward_grouped": lambda x, q, out: ops.moe_forward_grouped(q, None, q, x, out, out, 1, out=out),
    "moe_forward": lambda x, q, out: ops.moe_forward(q, None, q, x, x, 1, expert_bias=x, out=out),
}


@pytest.mark.parametrize("name", sorted(CALLS))
def test_a_call_keeps_the_view_that_it_passes(monkeypatch, name):
    """Two threads make the first call on one buffer: the first is held while it builds the view, the second builds, keeps and passes
    its own, and the first replaces that one while the second call is still running.  No address may lead to a collected view."""
    dead, in_array, second_in_call, first_in_call = set(), threading.Event(), threading.Event(), threading.Event()
    bad = []

    class Buffer(rt.DeviceBuffer):
        def __init__(self):
            self.shape, self.dtype, self.nbytes, self.ptr = (1, 64), rt.F16, 128, 4096

        def free(self):
            self.ptr = None

        def array(self, *args, **kw):
            a = super().array(*args, **kw)
            at = rt.ctypes.addressof(a)
            dead.discard(at)
            weakref.finalize(a, dead.add, at)
            if threading.current_thread().name == "first" and not in_array.is_set():
                in_array.set()
                assert second_in_call.wait(20)
            return a

    x = Buffer()

    def entry(_name):
        def call(*args):
            if threading.current_thread().name == "second":
                second_in_call.set()
                assert first_in_call.wait(20)
            else:
                first_in_call.set()
            passed = [a for a in args if isinstance(a, int) and a > 1 << 20]
            assert passed
            bad.extend(a for a in passed if a in dead)
            return 0
        return call

    monkeypatch.setattr(ops, "_entry", entry)
    monkeypatch.setattr(rt, "check", lambda status: None)
    q, out = types.SimpleNamespace(handle=1, out_features=8), types.SimpleNamespace(ptr=2, nbytes=16)
    failed = []

    def body():
        try:
            CALLS[name](x, q, out)
        except BaseException as e:  # noqa: BLE001 (reported below)
            failed.append(e)

    first = threading.Thread(target=body, name="first")
    first.start()
    assert in_array.wait(20)
    second = threading.Thread(target=body, name="second")
    second.start()
    first.join(30), second.join(30)
    assert not failed and not first.is_alive() and not second.is_alive()
    assert not bad, "a call passed the address of a collected view"


def test_a_view_follows_its_buffer():
    x = rt.DeviceBuffer.__new__(rt.DeviceBuffer)
    x.ptr, x.shape, x.dtype = 4096, (3, 64), rt.F16
    address, v, _ = kept = x.view()
    assert x.view() is kept and address == rt.ctypes.addressof(v) and v.data == 4096 and list(v.shape[:2]) == [3, 64]
    x.shape = (6, 32)
    w = x.view()[1]
    assert w is not v and list(w.shape[:2]) == [6, 32] and list(v.shape[:2]) == [3, 64]
    x.ptr = None
