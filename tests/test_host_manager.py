"""CPU-only checks of ContextManager's host side: what its native calls may find, with a stand-in for the library."""
import ctypes
import threading
import time

import pytest
import torch

from infllm_amd._lib import ResidentCall
from infllm_amd.attention import ContextManager, context_manager


class Native:
    def __init__(self):
        self.open, self.overlaps, self.calls, self.guard = {}, 0, 0, threading.Lock()

    def infllm_resident_state(self, manager, wait, state):
        return 0

    def infllm_resident_destroy(self, manager):
        return 0

    def infllm_resident_append(self, manager, rc, stream):
        with self.guard:
            self.calls += 1
            key = rc._obj.d_q_loc
            self.overlaps += self.open.get(key, 0)
            self.open[key] = self.open.get(key, 0) + 1
        time.sleep(2e-3)                                   # (another thread runs, as while a native call is under way)
        with self.guard:
            self.open[key] -= 1
        return 0


def resident_manager(lib):
    """a manager of a small geometry as _init leaves it, without the library's own objects"""
    cm = ContextManager.__new__(ContextManager)
    cm.n_init, cm.n_local, cm.block_size, cm.topk, cm.exc_block_size, cm.cache_strategy = 4, 64, 16, 2, 32, "lru"
    cm.num_units, cm.unit_size, cm.unit_size_kv, cm.head_width, cm.dim_head = 1, 2, 1, 64, 64
    cm.length = cm.load_count = cm.num_global_block = 0
    cm._lib, cm._resident, cm._dev_index, cm.device, cm._layer = lib, cm, 0, torch.device("cpu"), None
    cm._chunk_units, cm._local_group, cm._part_rows2, cm._chunks, cm._call_scores, cm._call_stream = 4, 1, 64, [], None, None
    cm._streams, cm.reps = set(), torch.empty((1, 16, 128), dtype=torch.bfloat16)
    cm._rc = ResidentCall()
    cm._rc.max_tokens = 64
    cm._rc_ref = ctypes.byref(cm._rc)
    return cm


@pytest.fixture
def one_stream(monkeypatch):
    monkeypatch.setattr(context_manager, "current_stream", lambda: 7)


def test_calls_of_two_threads_on_one_stream_are_enqueued_one_after_the_other(one_stream):
    """Both managers' launches write the same workspaces; interleaved, one call's prologue would overwrite the queries that
    the other's attention has yet to read."""
    lib = Native()
    managers = [resident_manager(lib) for _ in range(2)]
    row = lambda h: torch.zeros((1, h, 1, 64), dtype=torch.bfloat16)

    def steps(cm):
        for _ in range(20):
            cm._append_resident(row(2), row(1), row(1), 1)

    [cm._append_resident(row(2), row(1), row(1), 1) for cm in managers]          # binds them to the stream's workspaces
    threads = [threading.Thread(target=steps, args=(cm,)) for cm in managers]
    [t.start() for t in threads]
    [t.join() for t in threads]
    shared = managers[0]._rc.d_q_loc == managers[1]._rc.d_q_loc
    for cm in managers:
        cm._resident = None                                # (nothing to give back)
    assert shared and lib.calls == 42 and lib.overlaps == 0


def test_a_manager_may_be_collected_while_the_budget_is_looked_at():
    """The interpreter runs a collected object's destructor wherever it allocates, also inside the budget's own sections."""
    units, done = context_manager._Units, threading.Event()

    def inside():
        with units.lock:
            units.give(99, 5)
        done.set()

    thread = threading.Thread(target=inside, daemon=True)
    assert units.take(99, 5, 5) and not units.take(99, 1, 5)
    thread.start()
    assert done.wait(5) and units.used.pop(99) == 0


@pytest.mark.parametrize("streams,waits", [({1}, False), ({1, 2}, True)])
def test_a_log_is_handed_on_when_every_stream_is_done_with_it(streams, waits, monkeypatch):
    """With two streams the newest selection may have arrived while an older one is still to be written."""
    order = []
    monkeypatch.setattr(torch.cuda, "synchronize", lambda dev=None: order.append("wait"))
    monkeypatch.setattr(context_manager._Units, "give_log", lambda dev, log, seq: order.append((log, seq)))
    cm = resident_manager(Native())
    cm._streams, cm._chunk_bytes, cm._log, cm._state = streams, 0, "log", [0] * 9 + [12]
    cm._drop_resident()
    assert order == (["wait"] if waits else []) + [("log", 12)] and cm._log is None and cm._resident is None


def test_a_log_that_cannot_be_waited_for_is_not_handed_on(monkeypatch):
    def fails(dev=None):
        raise RuntimeError("a capture is under way")

    monkeypatch.setattr(torch.cuda, "synchronize", fails)
    monkeypatch.setattr(context_manager._Units, "give_log", lambda *a: pytest.fail("handed on"))
    monkeypatch.setattr(context_manager._Units, "lost", [])
    cm = resident_manager(Native())
    cm._streams, cm._chunk_bytes, cm._log, cm._state = {1, 2}, 0, "log", [0] * 9 + [12]
    with pytest.raises(RuntimeError):
        cm._drop_resident()
    assert context_manager._Units.lost == ["log"] and cm._resident is None


@pytest.mark.parametrize("free,reserved,allocated,budget,fits", [
    (100, 0, 0, None, True), (12, 0, 0, None, False),              # of 100 chunks' memory: enough, and the last eighth of it
    (2, 30, 5, None, True),                                        # ... with what the allocator holds and does not use
    (2, 0, 0, 10, True),                                           # a budget of the caller's is taken at its word
])
def test_units_leave_memory_to_the_other_users_of_the_device(free, reserved, allocated, budget, fits, monkeypatch):
    cm = resident_manager(Native())
    cm._chunk_units, cm._chunk_bytes, cm.resident_bytes = 4, 4 * 2 * 16 * 64 * 2, budget
    cm._chunk_host, cm._chunk_dev = (ctypes.c_uint64 * 16)(), torch.zeros((16,), dtype=torch.int64)
    mem = cm._chunk_bytes
    monkeypatch.setattr(context_manager._Units, "used", {})
    monkeypatch.setattr(context_manager._Units, "asked", {})
    monkeypatch.setattr(ContextManager, "_resident_limit", lambda self: 10 * mem)
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda dev: (free * mem, 100 * mem))
    monkeypatch.setattr(torch.cuda, "memory_reserved", lambda dev: reserved * mem)
    monkeypatch.setattr(torch.cuda, "memory_allocated", lambda dev: allocated * mem)
    assert cm._add_chunks(7) == fits
    assert len(cm._chunks) == (2 if fits else 0)
    assert context_manager._Units.used.get(0, 0) == len(cm._chunks) * mem
    cm._resident = None


def test_the_driver_is_asked_again_when_what_it_granted_is_used_up(monkeypatch):
    cm, asked = resident_manager(Native()), []
    monkeypatch.setattr(context_manager._Units, "asked", {})
    monkeypatch.setattr(context_manager, "_ASK_BYTES", 100)
    left = [1000, 1000, 200, 120]

    def info(dev):
        asked.append(dev)
        return left[len(asked) - 1], 800                            # an eighth: 100

    monkeypatch.setattr(torch.cuda, "mem_get_info", info)
    monkeypatch.setattr(torch.cuda, "memory_reserved", lambda dev: 0)
    monkeypatch.setattr(torch.cuda, "memory_allocated", lambda dev: 0)
    cm.resident_bytes, cm._resident = None, None
    assert [cm._leaves_room(40) for _ in range(9)] == [True] * 8 + [False]      # asked at the 1st, 4th, 7th (60 to spare) and 9th
    assert len(asked) == 4


def test_a_batch_takes_its_memory_in_smaller_steps():
    unit = 2 * 8 * 128 * 128 * 2                                    # one row's unit of the reference's geometry: 512 KiB
    steps = {b: ContextManager._units_per_chunk(b * unit) for b in (1, 2, 8, 64, 1024)}
    assert steps == {1: 64, 2: 64, 8: 16, 64: 4, 1024: 4}


def test_replaced_buffers_wait_for_the_stream_that_uses_them(one_stream, monkeypatch):
    """A manager that has moved to another stream: the allocator would hand a replaced buffer out again in the order of the
    stream it was made on, while launches of the other one still read it."""
    class Buffer:
        is_cuda, device, streams = True, "cuda:0", None

        def __init__(self, *shape):
            self.t, self.shape = torch.zeros(shape, dtype=torch.bfloat16), torch.Size(shape)

        def __getitem__(self, i):
            return self.t[i]

        def record_stream(self, stream):
            self.streams = stream

    monkeypatch.setattr(torch.cuda, "current_stream", lambda dev=None: "the call's stream")
    cm = resident_manager(Native())
    monkeypatch.setattr(cm, "_add_chunks", lambda n: True)
    cm.length, cm.reps, cm.unit_scores, cm._call_scores = 400, Buffer(1, 16, 128), Buffer(1, 16), Buffer(1, 1, 8)
    old = cm.reps, cm.unit_scores, cm._call_scores
    row = lambda h: torch.zeros((1, h, 2, 64), dtype=torch.bfloat16)
    cm._append_resident(row(2), row(1), row(1), 2)
    assert cm.reps.shape[1] >= 21 and [b.streams for b in old] == ["the call's stream"] * 3
    cm._resident = None


@pytest.mark.parametrize("k,v,error", [
    (((1, 2, 5, 128), torch.half, "cpu"), ((1, 2, 5, 128), torch.half, "cpu"), TypeError),
    (((1, 2, 5, 128), torch.bfloat16, "cpu"), ((1, 2, 5, 128), torch.float8_e4m3fn, "cpu"), TypeError),
    (((1, 2, 5, 128), torch.bfloat16, "meta"), ((1, 2, 5, 128), torch.bfloat16, "cpu"), ValueError),
    (((1, 2, 5, 128), torch.bfloat16, "cpu"), ((1, 1, 5, 128), torch.bfloat16, "cpu"), AssertionError),
])
def test_keys_and_values_that_would_be_read_out_of_range_are_refused(k, v, error, monkeypatch):
    """another type, device or head count than the queries and keys have (before anything is set up or launched)"""
    cm = ContextManager.__new__(ContextManager)
    cm.perhead, cm.initialized = False, False
    monkeypatch.setattr(ContextManager, "_init", lambda *a: pytest.fail("accepted"))
    q = torch.zeros((1, 4, 5, 128), dtype=torch.bfloat16)
    k, v = (torch.zeros(shape, dtype=dtype, device=device) for shape, dtype, device in (k, v))
    with pytest.raises(error, match=None if error is not AssertionError else "shape"):
        cm.append(q, k, v, q, k, v)
