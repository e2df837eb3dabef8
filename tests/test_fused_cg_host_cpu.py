"""Host side of the persistent CG with the engine's launch replaced by a stub that writes the control block:
buffers shared by threads."""
import ctypes
import importlib
import threading
import time

import pytest
import torch

import cola_amd._native as N

cgmod = importlib.import_module("cola_amd.linalg.cg")  # the package exports a function of that name


class Stream:
    """A stream of the stub device: a solve's results are there after a while."""
    cuda_stream = 0

    def synchronize(self):
        time.sleep(0.03)


@pytest.fixture
def engine(monkeypatch):
    """fused_solve on CPU tensors: a solve "takes" b[0] steps and ends with the status in b[1]."""
    empty, query = torch.empty, N.q

    def call(name, *a):
        assert name == "ck_cg_fused"
        b = (ctypes.c_float * 2).from_address(a[3].value)
        ints = (ctypes.c_int32 * 16).from_address(a[15].value)
        ints[0], ints[5] = int(b[0]), int(b[1])

    monkeypatch.setattr(torch, "empty", lambda *a, pin_memory=False, **k: empty(*a, **k).zero_())
    monkeypatch.setattr(torch.cuda, "current_stream", lambda dev=None: Stream())
    monkeypatch.setattr(N, "stream_ptr", lambda dev=None: None)
    monkeypatch.setattr(N, "call", call)
    monkeypatch.setattr(N, "q", lambda name, *a: N.CK_OK if name == "ck_cg_fused_supported" else query(name, *a))
    monkeypatch.setattr(cgmod, "lower", lambda A: (None, ))
    monkeypatch.setattr(cgmod, "_FUSED_BUFFERS", {})


def test_threads_on_one_stream(engine):
    """Threads that share a stream share a solve's buffers: each reads its own steps and status."""
    got, start = {}, threading.Barrier(4)

    def work(i):
        b = torch.zeros(64, 1)
        b[0], b[1] = 10 * (i + 1), N.CK_ERR_TIMEOUT if i == 3 else N.CK_OK
        start.wait()
        for _ in range(3):
            try:
                got.setdefault(i, []).append(cgmod.fused_solve(None, b, None, 100, 1e-6)[2])
            except N.KrylovError as e:
                got.setdefault(i, []).append(-e.status)

    ts = [threading.Thread(target=work, args=(i, )) for i in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert got == {0: [10] * 3, 1: [20] * 3, 2: [30] * 3, 3: [-N.CK_ERR_TIMEOUT] * 3}
