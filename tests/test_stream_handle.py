"""The current stream's handle that calls pass on: through torch's private
calls where it has them, through its public one in a torch without them."""
import os
import subprocess
import sys

import pytest

PKG = os.path.join(os.path.dirname(__file__), "..", "needle-rs_amd")

CODE = """
import sys
import torch

class Stream:
    cuda_stream = 77

if {without}:
    del torch._C._cuda_getCurrentRawStream
    torch.cuda.current_stream = Stream
else:
    torch._C._cuda_getDevice = lambda: 3
    torch._C._cuda_getCurrentRawStream = lambda d: 74 + d
sys.path.insert(0, {pkg!r})
import needle_hip as nh
assert nh._stream() == 77, nh._stream()
s = Stream()
s.cuda_stream = 5
assert nh._stream(s) == 5
"""


@pytest.mark.parametrize("without", [False, True])
def test_current_stream(without):
    r = subprocess.run([sys.executable, "-c", CODE.format(without=without, pkg=PKG)], capture_output=True, text=True,
                       timeout=110)
    assert r.returncode == 0, r.stderr
