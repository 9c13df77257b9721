"""A process whose plan cache holds plans that several streams have used ends normally."""
import os
import subprocess
import sys

import pytest

from conftest import PKG

pytestmark = pytest.mark.gpu

PROGRAM = """
import torch
import _spherical_distortion_ext._ops as ops
m = torch.rand(40, 80, 9, 2, device="cuda") * 39
x, w = torch.rand(1, 40, 40, 80, device="cuda"), torch.rand(66, 40, 9, device="cuda")
b, g = torch.zeros(66, device="cuda"), torch.rand(1, 66, 40, 80, device="cuda")
for stream in (torch.cuda.current_stream(), torch.cuda.Stream(), torch.cuda.Stream()):
    with torch.cuda.stream(stream):
        ops.ops.mapped_conv_backward(g, m, None, x, w, b, 9, 1)
        ops.ops.resample_to_map(x, m[:, :, 0].contiguous(), None, 40, 80, 1)
torch.cuda.synchronize()
assert ops.plan_cache_size() >= 2
print("done", flush=True)
"""


def test_process_ends_with_plans_in_the_cache():
    env = dict(os.environ, PYTHONPATH=PKG)
    r = subprocess.run([sys.executable, "-c", PROGRAM], env=env, timeout=100, capture_output=True,
                       text=True)
    assert "done" in r.stdout, r.stderr[-2000:]
    assert r.returncode == 0, r.stderr[-2000:]
