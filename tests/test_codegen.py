"""The compiler's part: texts that it has to take, and properties of the machine code that times hang on."""
import os
import subprocess
import sys

import pytest

from _loader import load_pkg, load_programs, ROOT

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


@pytest.mark.parametrize("op", ["%0 = stablehlo.negate %a : (T) -> T", "%c = stablehlo.constant dense<-1.0> : T\n  %0 = stablehlo.multiply %a, %c : (T, T) -> T"])
@pytest.mark.parametrize("dt", ["bf16", "f16", "f8E4M3FN"])
def test_negated_narrow_floats_compile(op, dt):
    """In a process of its own: the compiler ends the process that it fails in (and kernels are compiled in this one otherwise)."""
    t = "tensor<656x1024x%s>" % dt
    text = "module {\n func.func @main(%a: T) -> T {\n  OP\n  return %0 : T\n }\n}\n".replace("OP", op).replace("T", t)
    r = subprocess.run([sys.executable, "-c", "import sys; sys.path.insert(0, 'tests')\nfrom _loader import load_pkg\nprint(load_pkg().compile_offline(sys.stdin.read()))"],
                       input=text, cwd=ROOT, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "code object:" in r.stdout, r.stderr[-500:]
