"""The native tensor checks behind cgpt_amd/ops.py (host code, no GPU needed)."""
import subprocess
import sys

import torch

from cgpt_amd import _dispatch


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
