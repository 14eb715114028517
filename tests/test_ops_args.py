"""What the op layer takes for a stream and for device memory: an int handle, 0
or None; anything else is refused before the library is called. CPU only."""
import ctypes as C

import pytest

from peregrine_amd import ops
from peregrine_amd.ops import _dev, _s


@pytest.mark.parametrize("stream", ["stream", b"stream", C.c_void_p(64), 64.0, object()])
def test_stream_of_another_type_refused(monkeypatch, stream):
    called = []
    monkeypatch.setattr(ops, "call", lambda *a: called.append(a))
    with pytest.raises(TypeError):
        ops.rmsnorm(4096, 4096, 4096, 4096, stream=stream)
    assert not called


def test_stream_and_address_forms():
    assert _s(None) is None and _s(0) is None and _s(64) == 64
    assert _dev(None) is None and _dev(4096) == 4096
