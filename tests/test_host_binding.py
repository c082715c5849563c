"""The native call path's module on a machine without a GPU: what it leaves to
Python, and that other threads run while it works."""
import sys
import threading
import time

import pytest
import torch

from ironcore_amd import _lib, generation


def _calls():
    host, t = _lib.host(), torch.zeros(2, 1, 2, 64)
    return {
        "kv_append": lambda: host.kv_append(t, t, t, t, t, 0, 0),
        "paged_decode": lambda: host.paged_decode(t, t, t, t, t, 1, 1.0, None, 0, 1, None, 0, 0),
        "decode_step": lambda: host.decode_step(t, t, t, t, t, t, t, t, 1, 1.0, 1, None, None, None, None, 0, 0),
        "prefill_step": lambda: host.prefill_step(t, t, t, t, t, t, t, t, t, None, 1, 1.0, None, None, None, 0, 0),
        "dense": lambda: host.dense(t, t, t, False, None, None, 1, 1, 1.0, 0, 0),
        "linear_rows": lambda: host.linear_rows(t, t, None, 0, 0),
        "pack_mask": lambda: host.pack_mask(t, 0, 0),
    }


@pytest.mark.parametrize("name", ["kv_append", "paged_decode", "decode_step", "prefill_step", "dense", "linear_rows",
                                  "pack_mask"])
def test_other_threads_run_during_a_call(name):
    """With the interpreter's forced switches out of the way, another thread gets
    the GIL only while a call has given it up."""
    call, ran = _calls()[name], []
    assert not call()                       # tensors off the GPU are Python's to refuse
    switch = sys.getswitchinterval()
    ready = threading.Lock()
    ready.acquire()

    def other():
        ready.acquire()                     # (waits without the GIL)
        ran.append(True)

    thread = threading.Thread(target=other)
    thread.start()
    sys.setswitchinterval(1000)
    try:
        ready.release()
        end = time.monotonic() + 5
        while not ran and time.monotonic() < end:
            call()
        during = bool(ran)
    finally:
        sys.setswitchinterval(switch)
    thread.join()
    assert during


@pytest.mark.parametrize("bias", [False, True])
def test_linear_on_fake_tensors(bias):
    """Shapes worked out without a GPU, as torch's product does: nothing asks for the device."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode():
        x, w = torch.empty(4, 64, device="cuda"), torch.empty(64, 32, device="cuda")
        y = generation.linear(x, w, torch.empty(32, device="cuda") if bias else None)
        assert y.shape == (4, 32) and y.is_cuda
