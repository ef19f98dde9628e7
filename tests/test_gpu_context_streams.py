"""A closed context's stream: memory that torch keeps under its handle (outputs that live
on, and what was dropped) must not come to a stream that is not ordered with the default
one, so its handle goes to later contexts only."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


def test_handle_of_a_closed_context():
    import torch
    from rt_entry_amd import Context
    torch.zeros(1, device="cuda")
    hip = C.CDLL("libamdhip64.so")
    a, b = Context(0), Context(0)
    closed = {a.stream, b.stream}
    a.close()
    b.close()
    others = []
    for _ in range(8):
        h = C.c_void_p()
        assert hip.hipStreamCreateWithFlags(C.byref(h), C.c_uint(1)) == 0  # non-blocking
        others.append(h)
    try:
        assert not closed & {h.value for h in others}
        ctxs = [Context(0) for _ in range(3)]
        assert closed <= {c.stream for c in ctxs}
        assert len({c.stream for c in ctxs}) == 3
        for c in ctxs:
            c.synchronize()
            c.close()
    finally:
        for h in others:
            hip.hipStreamDestroy(h)
