"""One helper thread on which all device work of the planner runs.

The planner is usually called while a graph-capture context keeps a FakeTensorMode (or
another dispatch mode) active in the caller's thread (the reference builds its optimizer
inside ``AutoParallel.__enter__``, api.py:273-282): a tensor made there would be a fake one
and an operator would be handed fakes.  torch keeps its dispatch modes per thread, so code
that runs on a thread of its own sees none of them and its tensors are real allocations,
without reaching into torch's private mode stack.  The caller's current stream (also
per-thread state) is carried over, so "the current stream" keeps meaning the caller's.

Calls are serialised (one worker), nested calls run in place, exceptions come back to the
caller unchanged.

A call costs its two hand-overs between the threads: a queue of the interpreter's own (no Python
code between put and get) one way, a lock the caller waits on the other.  (With an executor's
futures, and the stream context entered for every call, 40 us a call; so 14 - 20.)
"""

from __future__ import annotations

import _thread
import atexit
import functools
import os
import queue
import threading
from concurrent.futures import Future

_lock = threading.RLock()
_tasks: queue.SimpleQueue | None = None
_worker: threading.Thread | None = None
_worker_ident: int | None = None
_closed = False


class _Call:
    """One call: what to run, the caller's stream, and the outcome."""

    __slots__ = ("fn", "args", "kwargs", "stream", "done", "result", "error")

    def __init__(self, fn, args, kwargs, stream):
        self.fn, self.args, self.kwargs, self.stream = fn, args, kwargs, stream
        self.result = self.error = None
        self.done = _thread.allocate_lock()
        self.done.acquire()

    def run(self):
        try:
            _stand_on(self.stream)
            self.result = self.fn(*self.args, **self.kwargs)
        except BaseException as e:  # noqa: BLE001 (raised again in the caller)
            self.error = e
            _raised()
        self.done.release()


class _Submitted:
    """Work that nobody waits for here: the outcome goes to a future."""

    __slots__ = ("fn", "args", "kwargs", "future")

    def __init__(self, fn, args, kwargs, future):
        self.fn, self.args, self.kwargs, self.future = fn, args, kwargs, future

    def run(self):
        if not self.future.set_running_or_notify_cancel():
            return
        try:
            _stand_on(None)
            result = self.fn(*self.args, **self.kwargs)
        except BaseException as e:  # noqa: BLE001 (the future's holder sees it)
            _raised()
            self.future.set_exception(e)
        else:
            self.future.set_result(result)


_UNKNOWN = object()
_stands_on = None  # the stream the worker stands on; None: its own default


def _stand_on(stream):
    """Makes ``stream`` the worker's current one; None: the default stream of the device a thread starts on.  Part of the
    call, so that a stream torch refuses is the caller's exception and not the end of the worker.  (Compared with the stream
    set last: what runs here puts a stream it changes back.  Asking torch for the current one costs 3 us a call on the
    worker, on which the caller's wait can grow by 30.)"""
    global _stands_on
    if stream == _stands_on:
        return
    import torch

    torch.cuda.set_stream(torch.cuda.default_stream(0) if stream is None else stream)  # (sets the stream's device as well)
    _stands_on = stream


def _raised():
    # (a graph capture that fails, for one, leaves its stream behind)
    global _stands_on
    import torch

    if torch.cuda.is_initialized():
        _stands_on = _UNKNOWN


def _work(tasks):
    global _worker_ident
    _worker_ident = threading.get_ident()
    while True:
        task = tasks.get()
        if task is None:
            return
        task.run()
        del task  # (nothing of a call outlives it here)


def _put(task):
    """Queues ``task``; the worker starts with the first one."""
    global _tasks, _worker
    with _lock:  # (nothing may come behind the None that ends the worker: its caller would wait for ever)
        if _closed:
            raise RuntimeError("apcost: no device work can start any more, the interpreter is shutting down")
        if _tasks is None:
            tasks = queue.SimpleQueue()
            worker = threading.Thread(target=_work, args=(tasks,), name="apcost-device_0", daemon=True)
            worker.start()
            _tasks, _worker = tasks, worker
        _tasks.put(task)


def _finish():
    """What has been queued is finished before the interpreter ends (submitted work has nobody else who waits for it, and
    an interpreter torn down under a thread inside a HIP call can crash)."""
    global _closed
    with _lock:
        _closed = True
        worker = _worker
        if _tasks is not None:
            _tasks.put(None)
    if worker is not None:
        worker.join()


# (before the functions of ``atexit``, as the executors of concurrent.futures do, and in the children of
# multiprocessing, which end without those)
getattr(threading, "_register_atexit", atexit.register)(_finish)


def _forget_thread():
    # a forked child has the parent's queue but not its thread
    global _tasks, _worker, _worker_ident, _lock, _stands_on
    _tasks = None
    _worker = None
    _worker_ident = None
    _stands_on = None
    _lock = threading.RLock()


os.register_at_fork(after_in_child=_forget_thread)


def _callers_stream():
    """The caller's current stream, None on a machine without a GPU.  A child forked from a
    process that had already initialised the GPU cannot use the device at all (torch refuses
    to initialise it a second time): that is reported as what it is, not as a torch internal."""
    import torch

    if not torch.cuda.is_available():
        return None
    try:
        return torch.cuda.current_stream()
    except RuntimeError as e:
        if "fork" in str(e):
            raise RuntimeError("apcost: this process was forked from one that had initialised the GPU; a forked child "
                               "cannot do device work (start workers with the 'spawn' method, or fork before the "
                               "parent touches the GPU)") from e
        raise


def call(fn, *args, **kwargs):
    """``fn(*args, **kwargs)`` on the device thread; the result (or the exception) of the call.
    In a forked child the parent's thread is gone and the first call starts a new one; device
    work there needs a parent that had not initialised the GPU before the fork."""
    if threading.get_ident() == _worker_ident:
        return fn(*args, **kwargs)
    task = _Call(fn, args, kwargs, _callers_stream())
    _put(task)
    task.done.acquire()
    if task.error is not None:
        try:
            raise task.error
        finally:
            task.error = None  # (the traceback holds this frame: no cycle)
    return task.result


def submit(fn, *args, **kwargs):
    """Queues ``fn(*args, **kwargs)`` on the device thread and returns its future without
    waiting (work that may overlap the caller's: the device's first-use costs)."""
    future = Future()
    _put(_Submitted(fn, args, kwargs, future))
    return future


def on_device_thread(fn):
    """Decorator form of ``call``."""

    @functools.wraps(fn)
    def wrapper(*args, **kwargs):
        return call(fn, *args, **kwargs)

    return wrapper
