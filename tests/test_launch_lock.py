"""Host threads that share a stream: a call of several launches over the
stream's buffer is enqueued as a whole, on the CPU against a stand-in library
whose calls are a main launch and a merge."""
import threading
import time

import pytest
import torch

from nano_qwen_amd import kernels


class Library:
    """Every entry asks for a buffer once, then records the two launches."""

    def __init__(self):
        self.log, self.inside, self.most = [], 0, 0
        self.guard = threading.Lock()

    def nq_prefill_workspace_bytes(self):
        return 256

    def launches(self, buffer, nbytes, need):
        if buffer is None or nbytes < 64:
            need.value = 64
            return 1
        with self.guard:
            self.inside += 1
            self.most = max(self.most, self.inside)
            self.log.append(("main", threading.get_ident(), buffer))
        time.sleep(0.01)    # as ctypes: other threads run meanwhile
        with self.guard:
            self.inside -= 1
            self.log.append(("merge", threading.get_ident(), buffer))
        return 0

    def nq_varlen_prefill_split(self, *a):
        return self.launches(*a[-4:-1])

    def nq_gdn_prefill_split(self, *a):
        return self.launches(*a[-4:-1])

    def nq_paged_decode_auto(self, *a):
        return self.launches(a[25], a[26], a[-2])


def prefill():
    q, k = torch.zeros(4, 4, 128), torch.zeros(4, 1, 128)
    cu = torch.tensor([0, 4], dtype=torch.int32)
    kernels.varlen_prefill(q.bfloat16(), k.bfloat16(), k.bfloat16(), cu, cu, 4, 4, 1.0)


def gdn_prefill():
    x, ab = torch.zeros(4, 2, 128).bfloat16(), torch.zeros(4, 2).bfloat16()
    cu = torch.tensor([0, 4], dtype=torch.int32)
    kernels.gdn_prefill(x, x, x, ab, ab, torch.zeros(2), torch.zeros(2), cu, torch.zeros(1, 2, 128, 128),
                        torch.zeros(1, dtype=torch.int32))


def decode():
    q, c = torch.zeros(1, 4, 128).bfloat16(), torch.zeros(1, 128, 1, 128).bfloat16()
    kernels.paged_decode(q, c, c, torch.ones(1, dtype=torch.int32), torch.zeros(1, 1, dtype=torch.int32), 1.0)


@pytest.fixture
def library(monkeypatch):
    fake, stream = Library(), threading.local()
    monkeypatch.setattr(kernels, "lib", lambda: fake)
    monkeypatch.setattr(kernels, "require_cuda", lambda *a, **k: None)
    monkeypatch.setattr(kernels, "_key", lambda device: (0, getattr(stream, "handle", 0)))
    monkeypatch.setattr(kernels, "_capturing", lambda key: False)
    monkeypatch.setattr(kernels, "_decode_counter_slot", lambda key: None)
    for table in ("_workspaces", "_prefill_queues", "_prefill_parts", "_gdn_segments"):
        monkeypatch.setattr(kernels, table, {})
    monkeypatch.setattr(kernels, "_retired", [])
    fake.stream = stream
    return fake


def _threads(n, f):
    fails = []

    def body(i):
        try:
            f(i)
        except BaseException as e:
            fails.append(e)
    ts = [threading.Thread(target=body, args=(i,)) for i in range(n)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not fails, fails


@pytest.mark.parametrize("call", [prefill, gdn_prefill, decode])
def test_threads_of_one_stream_take_turns(library, call):
    start = threading.Barrier(4)

    def body(i):
        start.wait()
        for _ in range(5):
            call()
    _threads(4, body)
    assert len(library.log) == 40
    for main, merge in zip(library.log[::2], library.log[1::2]):
        assert main[0] == "main" and merge[0] == "merge" and main[1:] == merge[1:]
    assert len({entry[2] for entry in library.log}) == 1    # one buffer, and none replaced
    assert not kernels._retired


@pytest.mark.parametrize("call", [prefill, gdn_prefill, decode])
def test_streams_do_not_wait_for_each_other(library, call):
    start = threading.Barrier(4)

    def body(i):
        library.stream.handle = i + 1
        start.wait()
        for _ in range(10):
            call()
    _threads(4, body)
    assert library.most > 1
