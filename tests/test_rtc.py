"""Kernels are compiled by the library's own ROCm also in a process that has loaded another one's compiler (PyTorch's
wheel brings one): the child process that then compiles them returns the code object that hiprtc gives in a process
without it."""
import os
import shutil
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
rx.compile_offline(P.mlp(256, (128, 256, 256, 128)))
"""


def _code(tmp_path, first_line, **env):
    """The code object, and what was written to standard error."""
    out = tmp_path / "code"
    r = subprocess.run([sys.executable, "-c", SCRIPT % first_line], cwd=ROOT, capture_output=True, text=True, timeout=300,
                       env=dict(os.environ, RX_DUMP_CODE_OBJECT=str(out), **env))
    assert r.returncode == 0, r.stderr[-2000:]
    return out.read_bytes(), r.stderr


@pytest.fixture(scope="module")
def want(tmp_path_factory):
    torch = pytest.importorskip("torch")
    if not torch.version.hip:
        pytest.skip("this torch brings no ROCm")
    code, _ = _code(tmp_path_factory.mktemp("rtc"), "")
    assert code[:4] == b"\x7fELF"
    return code


def test_another_rocm_in_the_process_does_not_compile_the_kernels(tmp_path, want):
    got, err = _code(tmp_path, "import torch")
    assert "rx_rtc_worker" not in err
    assert got == want


def test_a_preloaded_library_that_prints(tmp_path, want):
    cc = shutil.which("cc") or shutil.which("gcc")
    if not cc:
        pytest.skip("no C compiler")
    src, lib = tmp_path / "p.c", tmp_path / "libp.so"
    src.write_text('#include <stdio.h>\n__attribute__((constructor)) static void f(void) { puts("hello"); fflush(stdout); }\n')
    subprocess.run([cc, "-shared", "-fPIC", "-o", str(lib), str(src)], check=True)
    got, err = _code(tmp_path, "import torch", LD_PRELOAD=":".join([str(lib)] + os.environ.get("LD_PRELOAD", "").split()))
    assert "rx_rtc_worker" not in err
    assert got == want


def test_a_process_that_ignores_its_children(tmp_path, want):
    got, err = _code(tmp_path, "import torch, signal; signal.signal(signal.SIGCHLD, signal.SIG_IGN)")
    assert "rx_rtc_worker" not in err
    assert got == want


@pytest.mark.parametrize("how", ["LD_PRELOAD", "LD_LIBRARY_PATH"])
def test_another_compiler_in_the_environment(tmp_path, want, how):
    """The child compiles with neither (with that comgr the code object is another one)."""
    import torch
    lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    value = [os.path.join(lib, "libamd_comgr.so")] if how == "LD_PRELOAD" else [lib]
    if not os.path.exists(os.path.join(lib, "libamd_comgr.so")):
        pytest.skip("this torch brings no comgr")
    got, err = _code(tmp_path, "import torch", **{how: ":".join(value + os.environ.get(how, "").split(":")).rstrip(":")})
    assert "rx_rtc_worker" not in err
    assert got == want
