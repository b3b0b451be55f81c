"""Two threads that need the workspace of one stream at a time: the address the extension is told stays that of a workspace that
is kept."""
import threading
import time
import types

import pytest
import torch

from gptq_triton_amd import _lib

WAIT = 0.5  # seconds a thread waits for the other one, which may be kept out on purpose


@pytest.mark.parametrize("needs", [(100, 100), (100, 300), (300, 100)])
@pytest.mark.parametrize("grown", [False, True])
def test_two_threads_make_the_workspace_of_a_stream(monkeypatch, needs, grown):
    told = {}
    both_allocate, both_stored = threading.Barrier(2), threading.Barrier(2)

    def meet(barrier):
        try:
            barrier.wait(WAIT)
        except threading.BrokenBarrierError:
            pass

    real = torch.zeros

    def zeros(*a, **k):
        out = real(*a, **k)
        meet(both_allocate)     # (the interpreter lock is given up while a tensor is made)
        if threading.current_thread().name == "early":
            time.sleep(0.1)     # (stores its workspace last and tells of it first)
        return out

    def set_workspace(index, stream, address, size):
        meet(both_stored)
        if threading.current_thread().name == "late":
            time.sleep(0.1)
        told[index, stream] = address, size

    monkeypatch.setattr(_lib, "_workspaces", {(0, 7): real(50, dtype=torch.uint8)} if grown else {})
    monkeypatch.setattr(_lib, "_outgrown", [])
    monkeypatch.setattr(_lib, "_WS_BYTES", 10)
    monkeypatch.setattr(_lib, "current_stream", lambda device: 7)
    monkeypatch.setattr(_lib, "host", lambda: types.SimpleNamespace(set_workspace=set_workspace))
    monkeypatch.setattr(_lib.torch, "zeros", lambda *a, device, **k: zeros(*a, **k))
    threads = [threading.Thread(target=_lib._workspace_of_current_stream, args=(0, need), name=name)
               for need, name in zip(needs, ("late", "early"))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    kept = {t.data_ptr(): t.numel() for t in list(_lib._workspaces.values()) + _lib._outgrown}
    address, size = told[0, 7]
    assert kept.get(address) == size >= 100
