"""Host-side plumbing between torch tensors and the C ABI: workspaces, streams, status."""

import contextlib
import ctypes
import threading
import os
from typing import Dict, Optional, Tuple

import torch

from . import _lib

_last: Optional[Tuple[torch.Tensor, int, int, int]] = None  # (workspace, stream handle, copies, their step) of the latest call

CHECK_STATUS = os.environ.get("EVOX_AMD_CHECK_STATUS", "0") not in ("", "0")

# Populations of at most evox_hip_batched_max_rows(m) rows can run in the one-workgroup-per-population kernels, larger
# ones need a workspace.  None = choose by size.  Three to eight objectives: up to 256 rows always.  Above, one population is faster in
# the two launches whose first one spreads the matrix over the whole device (selection of half the rows, us on the device, two launches
# against one workgroup: 300 x 3 12.5 / 16, 1000 x 3 21 / 28, 1000 x 8 47 / 60); two to 31 only from a size on that shrinks as the objectives
# grow, since that call costs the host 29 us against 18 (in a loop of calls, 2 to 16 populations: 512 x 3 29 / 19, 777 x 3 29 / 29, 1000 x 3
# 29 / 32, 512 x 5 29 / 26, 1000 x 5 31 / 41, 300 x 8 32 / 30, 777 x 8 42 / 52); from 32 populations on never (32 of 1000 x 3 32 / 30, of
# 1000 x 8 70 / 61, 64 of 300 x 3 33 / 17).  Other numbers of objectives: a lone population is faster in the
# pipeline from a size on that shrinks as the objectives grow (16 objectives 67 / 77 at 128 rows, 119 / 101 at 256), two or
# three from twice that size on, four or more never.  True / False force the choice where it is possible (tests use that to drive small
# inputs through both).
use_small_population_kernel = None


def _lone_population_limit(m: int) -> int:
    return 896 if m <= 2 else 160  # (three to eight objectives have a rule of their own)


_batched_max_rows = {}  # objectives -> rows that the one-workgroup kernel takes (asked of the library once)


def small_population_kernel_fits(n: int, m: int, batch: int) -> bool:
    if use_small_population_kernel is False:
        return False
    if m == 2:
        # (two objectives have a one-workgroup kernel of their own, which takes up to 4096 rows and beats the pipeline
        # at every size; a tunable switches it off, so the library is asked every time)
        most = int(_lib.lib().evox_hip_batched_max_rows(m))
        return 1 <= n <= most and (most > 1024 or use_small_population_kernel is True or batch >= 4
                                   or n <= _lone_population_limit(m) * (1 if batch == 1 else 2))
    most = _batched_max_rows.get(m)
    if most is None:
        most = _batched_max_rows[m] = int(_lib.lib().evox_hip_batched_max_rows(m))
    if not 1 <= n <= most:
        return False
    if use_small_population_kernel is True:
        return True
    if 3 <= m <= 8:
        return n <= 256 or batch >= 32 or (batch >= 2 and n <= (832 if m == 3 else 576 if m <= 5 else 320))
    if batch >= 4:
        return True
    return n <= _lone_population_limit(m) * (1 if batch == 1 else 2)


def require_gpu_tensor(t: torch.Tensor, what: str) -> None:
    if not isinstance(t, torch.Tensor):
        raise TypeError(f"{what} must be a torch.Tensor")
    if not t.is_cuda:
        raise RuntimeError(
            f"{what} is on {t.device}: evox_amd runs on an AMD GPU only (HIP kernels, no CPU fallback); "
            "move the tensors to the 'cuda' device"
        )


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def stream_handle(device: torch.device) -> int:
    """The hipStream_t of torch's current stream on ``device`` (asked of torch directly where it offers that: the
    Stream object costs 1.5 us more to build)."""
    if _raw_stream is not None and device.index is not None:
        return _raw_stream(device.index)
    return int(torch.cuda.current_stream(device).cuda_stream)


class Place:
    """A stream of a device: its handle, the workspace that calls on it share, and the lock under which they use it.

    A call works on the workspace from the first of its launches to the last, and the library lets go of the interpreter while
    it enqueues them: a thread holds ``turn`` from before it takes the workspace until the library has returned, so that no
    other thread's launches come in between."""

    __slots__ = ("device", "handle", "turn", "kept")

    def __init__(self, device: torch.device, handle: int):
        self.device, self.handle, self.turn, self.kept = device, handle, threading.RLock(), None

    def buffer(self, need: int) -> torch.Tensor:
        """At least ``need`` bytes: the stream's buffer, made anew where it holds less.  A call that is being captured gets one of
        its own, from the graph's memory: a replay works on it whatever later calls do to the stream's buffer (a larger one
        replaces it, and other streams' calls may run beside the replay)."""
        if _capturing():
            return torch.empty(need, dtype=torch.uint8, device=self.device)
        ws = self.kept
        if ws is None or ws.numel() < need:
            self.kept = ws = None
            ws = torch.empty(need, dtype=torch.uint8, device=self.device)
            assert ws.data_ptr() % 256 == 0
            self.kept = ws
        return ws


_capturing = torch.cuda.is_current_stream_capturing
_places: Dict[Tuple[int, int], Place] = {}


def place(device: torch.device) -> Place:
    """The current stream of ``device``."""
    handle = stream_handle(device)
    index = device.index
    key = (index if index is not None else torch.cuda.current_device(), handle)
    here = _places.get(key)
    return here if here is not None else _places.setdefault(key, Place(device, handle))


def _buffer(need: int, where) -> torch.Tensor:
    return (where if type(where) is Place else place(where)).buffer(need)


_workspace_need = {}  # (rows, objectives, with the matrix), or the length of a sort -> bytes (asked of the library once per shape)


def workspace(n: int, m: int, where, with_matrix: bool = True) -> torch.Tensor:
    """A uint8 tensor of at least evox_hip_workspace_bytes(n, m) bytes, cached per (device, stream) -- ``where`` is a ``Place``,
    or a device for its current stream: calls on one stream are ordered, so they can share it.  ``with_matrix=False`` asks
    only for the bytes that the entry points without a dominance matrix need."""
    need = _workspace_need.get((n, m, with_matrix))
    if need is None:
        query = _lib.lib().evox_hip_workspace_bytes if with_matrix else _lib.lib().evox_hip_first_front_workspace_bytes
        need = int(query(n, m))
        if need == 0:
            raise ValueError(f"unsupported population shape n={n}, m={m}")
        if len(_workspace_need) < 4096:
            _workspace_need[(n, m, with_matrix)] = need
    return _buffer(need, where)


def sort_workspace(n: int, where) -> torch.Tensor:
    """Workspace of the standalone stable argsort; shares the per-(device, stream) buffer of `workspace`
    (every call initialises the parts it uses)."""
    need = _workspace_need.get(n)
    if need is None:
        need = int(_lib.lib().evox_hip_argsort_workspace_bytes(n))
        if need == 0:
            raise ValueError(f"unsupported sort length n={n}")
        if len(_workspace_need) < 4096:
            _workspace_need[n] = need
    return _buffer(need, where)


def wide_workspace(n: int, m: int, where, copies: int = 1) -> torch.Tensor:
    """Workspace of the entry points for 8-byte fitness (`copies` of it, each rounded up to 256 bytes, for as many
    populations in the same launches); shares the per-(device, stream) buffer of `workspace`."""
    need = int(_lib.lib().evox_hip_wide_workspace_bytes(n, m))
    if need == 0:
        raise ValueError(f"unsupported population shape n={n}, m={m}")
    if copies > 1:
        need = ((need + 255) // 256 * 256) * copies
    return _buffer(need, where)


def sized_workspace(need: int, where) -> torch.Tensor:
    """The per-(device, stream) buffer of `workspace`, at least `need` bytes."""
    if need <= 0:
        raise ValueError("unsupported population shape")
    return _buffer(need, where)


def many_workspace(batch: int, n: int, m: int, stop_count: int, where):
    """Workspace of the entry points that take many populations of one shape: (tensor, populations per launch, bytes
    from one population's copy of the workspace to the next); shares the per-(device, stream) buffer of `workspace`.
    Asked anew at every call: the answer depends on the tunables in use."""
    lib = _lib.lib()
    need = int(lib.evox_hip_many_workspace_bytes(batch, n, m, stop_count))
    per_launch = int(lib.evox_hip_many_populations_per_launch(batch, n, m, stop_count))
    if need == 0 or per_launch < 1:
        raise ValueError(f"unsupported population shape n={n}, m={m}")
    return _buffer(need, where), per_launch, need // per_launch


def release_workspaces() -> None:
    for here in list(_places.values()):
        here.kept = None


def note_call(ws: torch.Tensor, stream: int, copies: int = 1, step: int = 0) -> None:
    """copies, step: the call used that many copies of the workspace, `step` bytes apart, each with a control block."""
    global _last
    _last = (ws, stream, copies, step)
    if CHECK_STATUS:
        _status(ws, stream, copies, step)  # (not that of _last: another thread may have noted a call of its own)


# With status checking on, a ranking or selection whose device-side wait ran out (the persistent kernels need all
# their workgroups resident at once: another kernel may hold the compute units) is issued once more through the
# kernels that never wait for each other (tunable peel_stepped), instead of raising.
RETRY_WITHOUT_CORESIDENCY = True


def checked(issue) -> None:
    """``issue()`` enqueues one library call and notes it (``note_call``)."""
    try:
        issue()
    except _lib.EvoxHipError as e:
        if e.code != _lib.E_BARRIER_TIMEOUT or not RETRY_WITHOUT_CORESIDENCY or current_option("peel_stepped", 0):
            raise
        with options(peel_stepped=1):
            issue()


def note_small_kernel_call() -> None:
    """The one-workgroup-per-population kernel has no control block and no device-side waits."""
    global _last
    _last = None


def last_status() -> dict:
    """Waits for the latest call and returns its control block; raises if the device reported an error.
    Calls served by the small-population kernel have no control block: {"error": 0}."""
    last = _last
    return {"error": 0} if last is None else _status(*last)


def _status(ws: torch.Tensor, stream: int, copies: int, step: int) -> dict:
    out = (ctypes.c_int32 * 8)()
    for b in reversed(range(copies)):  # (the control block reported is that of the first copy)
        code = _lib.lib().evox_hip_read_status(ws.data_ptr() + b * step, stream, out)
        if code != 0:
            raise _lib.EvoxHipError("evox_hip_read_status", code)
    keys = ("error", "fronts", "worst_rank", "better_rows", "last_front_size", "taken_from_last", "passes")
    return dict(zip(keys, list(out)[:7]))


_process_options: Dict[str, int] = {}  # what set_option has changed (the library holds the values themselves)


def set_option(name: str, value: int) -> None:
    """Changes a process-wide tunable (configuration at start-up; see ``options`` for a scoped change)."""
    _lib.call("evox_hip_set_option", name.encode(), int(value))
    _process_options[name] = int(value)


_options_in_use = threading.local()


def current_option(name: str, default: int) -> int:
    """The value of a tunable as the calls of this thread see it, where this module has set it (else ``default``,
    which must be the library's own default)."""
    stack = getattr(_options_in_use, "stack", None)
    if stack and name in stack[-1][1]:
        return stack[-1][1][name]
    return _process_options.get(name, default)


@contextlib.contextmanager
def options(**tunables):
    """Tunables for the library calls that this thread makes inside the ``with`` block (the process-wide ones,
    with the given changes); other threads and the process-wide values are left alone."""
    lib = _lib.lib()
    handle = lib.evox_hip_options_create()
    if not handle:
        raise MemoryError("evox_hip_options_create")
    stack = getattr(_options_in_use, "stack", None)
    if stack is None:
        stack = _options_in_use.stack = []
    try:
        if stack:  # start from the enclosing block's values, not from the process-wide ones
            for name, value in stack[-1][1].items():
                _lib.call("evox_hip_options_set", handle, name.encode(), int(value))
        merged = dict(stack[-1][1]) if stack else {}
        for name, value in tunables.items():
            _lib.call("evox_hip_options_set", handle, name.encode(), int(value))
            merged[name] = int(value)
        stack.append((handle, merged))
        _lib.call("evox_hip_options_use", handle)
        try:
            yield
        finally:
            stack.pop()
            _lib.call("evox_hip_options_use", stack[-1][0] if stack else None)
    finally:
        lib.evox_hip_options_destroy(handle)


def workspace_views(ws: torch.Tensor, n: int, m: int) -> dict:
    """Typed views of the workspace regions (for tests and tools)."""
    out = (ctypes.c_int64 * 11)()
    _lib.call("evox_hip_workspace_layout", n, m, out)
    dom_off, wstride, nwords, count, rank, dist, perm, fstart, order, ctrl, orig_of = list(out)

    def view(off, count_, dtype):
        size = torch.empty((), dtype=dtype).element_size()
        return ws[off: off + count_ * size].view(dtype)

    sort = (ctypes.c_int64 * 6)()
    _lib.call("evox_hip_slot_sort_layout", n, m, sort)
    npad = sort[4]
    return {
        "key_sorted": view(sort[0], npad, torch.int64),
        "kid_sorted": view(sort[1], npad, torch.int32),
        "xs_sorted": view(sort[2], m * npad, torch.float32).view(m, npad),
        "xs": view(sort[3], m * npad, torch.float32).view(m, npad),
        "slot_of": view(sort[5], n, torch.int32),
        "dom": view(dom_off, n * wstride, torch.int64).view(n, wstride),
        "nwords": nwords,
        "count": view(count, n, torch.int32),
        "rank": view(rank, n, torch.int32),
        "dist": view(dist, n, torch.float32),
        "perm": view(perm, n, torch.int32),
        "fstart": view(fstart, n + 2, torch.int32),
        "order": view(order, n, torch.int32),
        "ctrl": view(ctrl, 16, torch.int32),
        "orig_of": view(orig_of, n, torch.int32),
        "orig_of_padded": view(orig_of, npad, torch.int32),
    }
