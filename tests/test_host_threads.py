"""Host threads that call on one stream: a call's launches are enqueued without another thread's in between, since calls on a
stream share its workspace and the library lets go of the interpreter while it enqueues.  And a captured call's workspace, which
is the graph's own.  On the CPU, with the library's entry points replaced by ones that take a while."""

import contextlib
import threading
import time

import pytest
import torch

from evox_amd import ops, runtime


def _plain(op):
    return getattr(op, "_init_fn", op)


_F, _X = torch.rand(300, 3), torch.rand(300, 5)
CALLS = {
    "rank": lambda: _plain(ops.nd_rank)(_F),
    "rank_until": lambda: _plain(ops.nd_rank_until)(_F, 100),
    "first_front": lambda: _plain(ops.nd_first_front)(_F),
    "crowding": lambda: _plain(ops.crowding)(_F, None),
    "crowding_wide": lambda: _plain(ops.crowding_wide)(_F.double(), None),
    "select": lambda: _plain(ops.nd_select)(_X, _F, 100),
    "select_batch": lambda: _plain(ops.nd_select)(torch.stack([_X, _X]), torch.stack([_F, _F]), 100),
    "select_two_part": lambda: _plain(ops.nd_select_two_part)(_X[:150], _F[:150], _X[150:], _F[150:], 100),
    "select_wide": lambda: _plain(ops.nd_select_wide)(_X, _F.double(), 100),
    "select_wide_batch": lambda: _plain(ops.nd_select_wide)(torch.stack([_X, _X]), torch.stack([_F, _F]).double(), 100),
    "argsort_step": lambda: _plain(ops.stable_argsort_step)(_F[:, 0].contiguous(), 0, None),
    "argsort_rows": lambda: _plain(ops.stable_argsort_rows)(_F.t().contiguous(), 0, None),
}


@pytest.fixture
def device_on_the_cpu(monkeypatch):
    """The host side of the calls as on a GPU, on CPU tensors; the result lists the calls that overlapped on a workspace."""
    inside, overlaps, guard = {}, [], threading.Lock()

    def call(name, *args):
        with guard:
            inside[name, threading.get_ident()] = True
            if len(inside) > 1 and not name.endswith("dense_rank_rows"):
                overlaps.append(sorted(n for n, _ in inside))
        time.sleep(0.003)
        with guard:
            del inside[name, threading.get_ident()]

    class Library:
        def __getattr__(self, name):
            return lambda *a: 1 if "per_launch" in name or "max_rows" in name else 4096

    monkeypatch.setattr(ops._lib, "call", call)
    monkeypatch.setattr(ops._lib, "lib", lambda: Library())
    monkeypatch.setattr(ops, "_on", lambda device: contextlib.nullcontext())
    monkeypatch.setattr(ops, "_at", lambda here: here.turn)
    monkeypatch.setattr(ops, "_current_device", lambda: None)
    monkeypatch.setattr(runtime, "require_gpu_tensor", lambda t, what: None)
    monkeypatch.setattr(runtime, "stream_handle", lambda device: 7)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(runtime, "_capturing", lambda: False)
    empty = torch.empty

    def aligned(*size, **kw):  # (as the allocator of a GPU gives it)
        if kw.get("dtype") is not torch.uint8:
            return empty(*size, **kw)
        whole = empty(size[0] + 256, **kw)
        return whole[-whole.data_ptr() % 256:][:size[0]]

    monkeypatch.setattr(torch, "empty", aligned)
    for cache in ("_places", "_workspace_need", "_batched_max_rows"):
        monkeypatch.setattr(runtime, cache, {})
    yield overlaps


@pytest.mark.parametrize("name", CALLS)
def test_calls_of_two_threads_on_a_stream_take_turns(name, device_on_the_cpu):
    errors = []

    def work(mine):
        try:
            for _ in range(6):
                CALLS[mine]()
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(n,)) for n in (name, "rank")]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    assert device_on_the_cpu == []


def test_a_call_on_another_device_holds_the_lock_inside_its_guard(monkeypatch):
    inside = []

    @contextlib.contextmanager
    def guard(device):
        inside.append(device)
        try:
            yield
        finally:
            inside.remove(device)

    monkeypatch.setattr(torch.cuda, "device", guard)
    here = runtime.Place(torch.device("cuda", 1), 7)
    monkeypatch.setattr(ops, "_current_device", lambda: 0)
    with pytest.raises(KeyError):
        with ops._at(here):
            assert inside == [here.device]
            other = threading.Thread(target=lambda: inside.append(here.turn.acquire(blocking=False)))
            other.start()
            other.join()
            assert inside.pop() is False
            raise KeyError
    assert not inside and here.turn.acquire(blocking=False)
    here.turn.release()
    monkeypatch.setattr(ops, "_current_device", lambda: 1)
    assert ops._at(here) is here.turn


def test_a_captured_call_keeps_no_buffer_that_later_calls_replace(device_on_the_cpu, monkeypatch):
    """A replay works on the memory that the call was captured with: the stream's buffer, which a larger call replaces, would go
    back to the allocator under it."""
    device = torch.device("cpu")
    here = runtime.place(device)
    eager = runtime.workspace(300, 3, here)
    monkeypatch.setattr(runtime, "_capturing", lambda: True)
    captured = runtime.workspace(300, 3, here)
    assert captured.data_ptr() != eager.data_ptr() and here.kept is eager
    monkeypatch.setattr(runtime, "_capturing", lambda: False)
    assert runtime.workspace(300, 3, here) is eager
