"""The native tensor checks behind cgpt_amd/ops.py (host code, no GPU needed)."""
import ctypes
import subprocess
import sys
import threading

import torch

from cgpt_amd import _dispatch, ops


def test_tensors_declines_what_the_library_does_not_take():
    assert _dispatch.tensors(torch.zeros(4)) is None                  # not on a device
    assert _dispatch.tensors(1.0) is None
    assert _dispatch.tensors(None) == (-1, 0)
    assert _dispatch.same_shape(torch.zeros(2, 3), torch.ones(2, 3))
    assert not _dispatch.same_shape(torch.zeros(2, 3), torch.ones(3, 2))
    assert not _dispatch.same_shape(torch.zeros(2), None)


_REFUSING = r"""
import torch
from cgpt_amd import _dispatch
nested = torch.nested.nested_tensor([torch.zeros(2), torch.zeros(3)])
try:
    _dispatch.same_shape(nested, nested)
except RuntimeError:
    print("raised")
"""


def test_a_tensor_without_sizes_raises_instead_of_ending_the_process():
    """A nested tensor throws in C++ when asked for its sizes. In a process of its own, which an exception that leaves the C
    entry ends."""
    proc = subprocess.run([sys.executable, "-c", _REFUSING], capture_output=True, text=True, timeout=120)
    assert proc.returncode == 0 and proc.stdout.strip() == "raised", (proc.returncode, proc.stderr[-2000:])


class _Parameter:
    """What adamw_step_many_async asks of a device tensor, on a machine without one."""

    def __init__(self, address, dtype=torch.float32):
        self.address, self.dtype, self.shape, self.device = address, dtype, (4,), torch.device("cuda:0")

    def data_ptr(self):
        return self.address

    def numel(self):
        return 4


def test_two_threads_on_one_adamw_workspace_pass_their_own_entries(monkeypatch):
    """The library reads the entries without the interpreter's lock: a second call that starts meanwhile must not change
    them."""
    options, workspace = ops.AdamWOptions(), object.__new__(ops.AdamWWorkspace)
    workspace._handle, workspace._states = None, None
    state = ops.AdamWState(_Parameter(1), _Parameter(2), _Parameter(3))
    inside, resume, seen = threading.Event(), threading.Event(), {}

    def call(name, handle, array, count, *rest):
        if threading.current_thread().name == "first":
            inside.set()
            assert resume.wait(60)
        seen[threading.current_thread().name] = [array[i].gradient for i in range(count)]

    def step(gradient):
        ops.adamw_step_many_async([ops.AdamWBatchEntry(_Parameter(10), _Parameter(gradient), state)], options, workspace, 0)

    monkeypatch.setattr(ops.capi, "call", call)
    step(5)  # binds the workspace
    first, second = threading.Thread(target=step, args=(20,), name="first"), threading.Thread(target=step, args=(30,), name="second")
    first.start()
    assert inside.wait(60)
    second.start()
    second.join(60)
    resume.set()
    first.join(60)
    assert seen["first"] == [20] and seen["second"] == [30]
