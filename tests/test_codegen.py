"""Properties of the kernels' machine code that their times hang on."""
import os
import subprocess

import pytest

from _loader import load_pkg, load_programs

rx, P = load_pkg(), load_programs()
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
@pytest.mark.parametrize("dt", ["f32", "f64"])
def test_sine_of_one_element_at_a_time_skips_the_large_arguments_path(tmp_path, monkeypatch, dt):
    """An odd number of elements is read one by one, four per thread: every sine has a branch around each of its two paths."""
    out = tmp_path / "code"
    monkeypatch.setenv("RX_DUMP_CODE_OBJECT", str(out))
    rx.compile_offline(P.sinsum_add(10379445, dt))
    text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(out)], check=True, capture_output=True, text=True).stdout
    kernel = text[text.index("k0_reduce>:"):text.index("k0_reduce_final>:")]
    # three branches per element (bounds, large, small) where both paths are kept apart, one where they are selected from
    assert kernel.count("s_cbranch") >= 10, kernel.count("s_cbranch")
