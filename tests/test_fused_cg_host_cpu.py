"""Host side of the persistent CG with the engine's launch replaced by a stub that writes the control block:
buffers shared by threads, the bound on workgroups in flight, the way out of a time-out."""
import ctypes
import importlib
import threading
import time

import pytest
import torch

import cola_amd._native as N

cgmod = importlib.import_module("cola_amd.linalg.cg")  # the package exports a function of that name


ENGINE = {}  # the stub: workgroups of a solve, of all solves in flight, the most there were
LOCK = threading.Lock()
BACKLOG, SOLVING = {}, set()  # by thread: seconds of earlier work on its stream; those with a solve in flight


def running(change):
    with LOCK:
        ENGINE["running"] += change
        ENGINE["most"] = max(ENGINE["most"], ENGINE["running"])


class Stream:
    """A stream of the stub device: a solve's results are there after a while."""

    def __init__(self):
        self.cuda_stream = threading.get_ident()

    def synchronize(self):
        me = threading.get_ident()
        time.sleep(BACKLOG.pop(me, 0.0))
        if me in SOLVING:
            SOLVING.remove(me)
            time.sleep(0.03)
            running(-ENGINE["workgroups"])


@pytest.fixture
def engine(monkeypatch):
    """fused_solve on CPU tensors: a solve "takes" b[0] steps and ends with the status in b[1]."""
    empty, query = torch.empty, N.q

    def call(name, *a):
        assert name == "ck_cg_fused"
        b = (ctypes.c_float * 2).from_address(a[3].value)
        ints = (ctypes.c_int32 * 16).from_address(a[15].value)
        ints[0], ints[5] = int(b[0]), int(b[1])
        SOLVING.add(threading.get_ident())
        running(ENGINE["workgroups"])

    monkeypatch.setattr(torch, "empty", lambda *a, pin_memory=False, **k: empty(*a, **k).zero_())
    monkeypatch.setattr(torch.cuda, "current_stream", lambda dev=None: Stream())
    monkeypatch.setattr(N, "stream_ptr", lambda dev=None: None)
    monkeypatch.setattr(N, "call", call)
    monkeypatch.setattr(N, "q", lambda name, *a: ENGINE["workgroups"]
                        if name == "ck_cg_fused_workgroups" else query(name, *a))
    monkeypatch.setattr(cgmod, "lower", lambda A: (None, ))
    monkeypatch.setattr(cgmod, "_WORKGROUPS", {None: cgmod._Workgroups(256)})
    ENGINE.update(workgroups=1, running=0, most=0)
    monkeypatch.setattr(cgmod, "_FUSED_BUFFERS", {})


def test_threads_on_one_stream(engine, monkeypatch):
    """Threads that share a stream share a solve's buffers: each reads its own steps and status."""
    got, start = {}, threading.Barrier(4)
    monkeypatch.setattr(Stream, "__init__", lambda self: setattr(self, "cuda_stream", 0))

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


@pytest.mark.parametrize("workgroups,cus,most", [(20, 256, 160), (100, 256, 200), (256, 256, 256), (20, 32, 20), (1, 4, 8)])
def test_solves_in_flight_fit_the_device(engine, workgroups, cus, most):
    """Eight threads with a stream each: as many solves at once as the device has CUs for; one workgroup
    waits for nobody and does not count."""
    cgmod._WORKGROUPS[None] = cgmod._Workgroups(cus)
    cgmod._WORKGROUPS[None].PATIENCE = 5.0
    ENGINE["workgroups"] = workgroups
    b, start = torch.ones(64, 1), threading.Barrier(8)

    def work():
        start.wait()
        assert cgmod.fused_solve(None, b, None, 100, 1e-6) is not None

    ts = [threading.Thread(target=work) for _ in range(8)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert ENGINE["most"] == most and cgmod._WORKGROUPS[None].used == 0


def test_earlier_work_of_a_stream_holds_up_nobody(engine):
    """A thread whose stream is busy for a second keeps the device's workgroups meanwhile: another's solve
    is told so after a moment and can take the chained launches."""
    ENGINE["workgroups"], b, done = 256, torch.ones(64, 1), {}

    def work(name, backlog):
        BACKLOG[threading.get_ident()] = backlog
        out = cgmod.fused_solve(None, b, None, 100, 1e-6)
        done[name] = time.monotonic(), out is not None

    t0, ts = time.monotonic(), [threading.Thread(target=work, args=a) for a in (("busy", 1.0), ("idle", 0.0))]
    ts[0].start()
    time.sleep(0.1)
    ts[1].start()
    [t.join() for t in ts]
    assert done["idle"][0] - t0 < 0.7 and not done["idle"][1]
    assert done["busy"][0] - t0 >= 1.0 and done["busy"][1] and cgmod._WORKGROUPS[None].used == 0


def test_devices_cus():
    assert N.q("ck_device_cus", -1) == 0 and N.q("ck_device_cus", 1000) == 0


def test_more_workgroups_than_the_device_has(engine):
    cgmod._WORKGROUPS[None] = cgmod._Workgroups(32)
    ENGINE["workgroups"] = 33
    assert cgmod.fused_solve(None, torch.ones(64, 1), None, 100, 1e-6) is None


def test_timeout_falls_back_to_chained_launches(engine, monkeypatch):
    b = torch.zeros(64, 1)
    b[0], b[1] = 5, N.CK_ERR_TIMEOUT
    monkeypatch.setattr(N, "require_device", lambda *a: None)
    monkeypatch.setattr(cgmod, "to_blocks", lambda t, ld: t)
    monkeypatch.setattr(cgmod, "from_blocks", lambda t, n: t)
    monkeypatch.setattr(cgmod, "cg_blocks", lambda *a: (7, True, {"status": "ok", "fused": False}))
    _, _, k, info = cgmod.run_batched_cg(None, b, None, 100, 1e-6)
    assert k == 7 and info == {"status": "ok", "fused": False, "fused_timeout": True}
    b[1] = N.CK_ERR_NAN  # any other status is the solve's own
    _, _, k, info = cgmod.run_batched_cg(None, b, None, 100, 1e-6)
    assert k == 5 and info["status"] == "nan" and "fused_timeout" not in info


@pytest.mark.parametrize("n,B,nblocks,offset,count", [(256, 1, 0, 0, 1), (257, 1, 0, 0, 1), (320, 1, 0, 0, 1), (321, 1, 0, 0, 21),
                                                      (300, 1, 0, 7, 19), (256, 4, 0, 0, 1), (257, 2, 0, 0, 17),
                                                      (64, 5, 0, 0, 4), (64, 1, 8, 0, 8), (3072, 4, 0, 0, 192),
                                                      (3584, 1, 0, 0, 180), (7168, 1, 0, 0, 256), (7169, 1, 0, 0, 0),
                                                      (64, 9, 0, 0, 0), (2049, 5, 0, 0, 0), (100, 1, 300, 0, 100)])
def test_planned_workgroups(n, B, nblocks, offset, count):
    op = N.CkOp()
    op.kind, op.n, op.lda, op.a = N.CK_OP_DENSE_F32, n, n, 4096
    assert N.q("ck_cg_fused_workgroups", op, None, B, nblocks, offset) == count
    assert (N.q("ck_cg_fused_supported", op, None, B) == N.CK_OK) == (count > 0)
