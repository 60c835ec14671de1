"""Host threads that call the attention at the same time: the launches of one
call (attention, merge of its partial results) reach a stream together, since
the calls on a stream share a workspace.  The entry point is a host function
here, so that the enqueues' order is seen and nothing runs on the GPU."""
import ctypes
import threading
import time

import pytest
import torch

from taomate_amd import _native, kernels
from taomate_amd.kernels import KVSegment

pytestmark = pytest.mark.gpu


def _bind(**stubs):
    lib = _native.load()
    addr = {n: ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in _native.SIGNATURES}
    addr.update({n: ctypes.cast(f, ctypes.c_void_p).value for n, f in stubs.items()})
    _native.host().bind(addr, _native.NativeCallError)


@pytest.mark.parametrize("streams", [1, 2])
def test_calls_on_one_stream_take_turns(dev, streams):
    name = "ltx_flash_attn_fwd"
    events, both = [], threading.Barrier(2)

    @ctypes.CFUNCTYPE(ctypes.c_int, *_native.SIGNATURES[name])
    def enqueue(*args):
        ws, stream = args[-3], args[-1]
        events.append(("in", stream, ws))
        if streams == 2:
            both.wait(20)      # separate workspaces: the two calls are inside together
        else:
            time.sleep(0.2)    # long enough for the other thread to come in, were it let
        events.append(("out", stream, ws))
        return 0

    q = torch.zeros(1, 75, 8, 64, dtype=torch.bfloat16, device=dev)
    kv = torch.zeros(1, 1152, 8, 64, dtype=torch.bfloat16, device=dev)
    own = [torch.cuda.Stream() for _ in range(2)] if streams == 2 else [torch.cuda.current_stream()] * 2
    torch.cuda.synchronize()
    errors = []

    def thread(i):
        try:
            with torch.cuda.stream(own[i]):
                kernels.flash_attn(q, [KVSegment(kv, kv)], torch.empty_like(q))
        except BaseException as e:   # noqa: BLE001 (reported by the test)
            errors.append(e)
    _bind(**{name: enqueue})
    try:
        ts = [threading.Thread(target=thread, args=(i,)) for i in range(2)]
        for t in ts:
            t.start()
        for t in ts:
            t.join(60)
    finally:
        _bind()
    assert not errors and len(events) == 4 and all(ws for _, _, ws in events)
    if streams == 1:
        assert [e[0] for e in events] == ["in", "out", "in", "out"]
        assert len({e[2] for e in events}) == 1
    else:
        assert [e[0] for e in events] == ["in", "in", "out", "out"]
        assert len({e[2] for e in events}) == 2 and len({e[1] for e in events}) == 2
