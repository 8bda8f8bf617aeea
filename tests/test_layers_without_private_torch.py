"""The layers work on a torch without the private check for hooks of all modules."""
import subprocess
import sys

CODE = """
import torch.nn.modules.module as m
del m._has_any_global_hook
import torch
from sortnet_amd.layers import MeanShiftDropout, NormDist
layer = NormDist(8, 6, bias=True).eval()
x = torch.randn(2, 8, 1)
with torch.no_grad():
    assert layer._evaluation_shift(x, None, None) is None      # the mean shift as a step of its own
print("fine")
"""


def test_import_and_evaluation():
    out = subprocess.run([sys.executable, "-c", CODE], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.strip().endswith("fine"), out.stderr
