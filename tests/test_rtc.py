"""Kernels are compiled by the library's own ROCm also in a process that has loaded another one's compiler (PyTorch's
wheel brings one): the child process that then compiles them returns the code object that hiprtc gives in a process
without it."""
import subprocess
import sys

import pytest

from _loader import ROOT

SCRIPT = """
import sys
%s
sys.path.insert(0, "tests")
from _loader import load_pkg, load_programs
rx, P = load_pkg(), load_programs()
print(rx.compile_offline(P.mlp(256, (128, 256, 256, 128))).split("code object:")[1])
"""


def _code_size(first_line):
    r = subprocess.run([sys.executable, "-c", SCRIPT % first_line], cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    return r.stdout.strip(), r.stderr


def test_another_rocm_in_the_process_does_not_compile_the_kernels():
    torch = pytest.importorskip("torch")
    if not torch.version.hip:
        pytest.skip("this torch brings no ROCm")
    want, _ = _code_size("")
    got, err = _code_size("import torch")
    assert "rx_rtc_worker" not in err
    assert got == want
