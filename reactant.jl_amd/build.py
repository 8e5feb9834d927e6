"""Build libreactant_mi355x.so in-tree with hipcc for gfx950.

    python reactant.jl_amd/build.py            # rebuild what is out of date
    python reactant.jl_amd/build.py --force    # rebuild everything

Steps: (1) the device headers under csrc/kernels/ are embedded as string
constants (csrc/rx_embedded.inc) so that hiprtc can include them at run time;
(2) every csrc/*.cpp is compiled (rx_api.cpp as HIP: it holds the AOT copy
kernel); (3) the GEMM skeletons are compiled once ahead of time with a plain
epilogue (csrc/kernels/rx_gemm_check.hip) as a device-code build check; (4) link the library and the compiler's process (rx_rtc_worker.so).

    python reactant.jl_amd/build.py --sanitize   # host-only program of the importer / planner under ASan + UBSan
"""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(CSRC, "build")
LIB = os.path.join(HERE, "libreactant_mi355x.so")
WORKER = os.path.join(HERE, "rx_rtc_worker.so")   # a program: named so that it travels wherever the library does
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ROCM_LIB = "/opt/rocm/lib"
ARCH = "gfx950"
PACKED = ["-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
COMMON = ["-std=c++17", "-O2", "-fPIC", "-fvisibility=hidden", "-Wall", "-Wno-unused-function",
          "-Wno-unused-command-line-argument", "-Wno-unknown-attributes"]


def _run(cmd):
    print("+", " ".join(cmd), flush=True)
    subprocess.check_call(cmd)


def _embed():
    out = os.path.join(CSRC, "rx_embedded.inc")
    parts = ["// generated by build.py from csrc/kernels/*.h -- do not edit\n"]
    for var, fname in (("kRxPreambleSrc", "rx_preamble.h"), ("kRxGemmKernelsSrc", "rx_gemm_kernels.h")):
        with open(os.path.join(CSRC, "kernels", fname)) as f:
            text = f.read()
        assert ')RXSRC"' not in text
        # string literals are limited in length by some compilers: split into chunks
        chunks = [text[i:i + 12000] for i in range(0, len(text), 12000)] or [""]
        parts.append("static const char %s[] =\n" % var +
                     "\n".join('R"RXSRC(%s)RXSRC"' % c for c in chunks) + ";\n")
    new = "".join(parts)
    old = open(out).read() if os.path.exists(out) else None
    if new != old:
        with open(out, "w") as f:
            f.write(new)
    return out


def _stale(target, deps):
    if not os.path.exists(target):
        return True
    t = os.path.getmtime(target)
    return any(os.path.getmtime(d) > t for d in deps)


def build_library(force=False, verbose=True):
    os.makedirs(OBJ, exist_ok=True)
    inc = _embed()
    headers = [os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".h")] + [inc]
    headers += [os.path.join(CSRC, "kernels", f) for f in os.listdir(os.path.join(CSRC, "kernels"))]
    headers.append(os.path.join(HERE, "..", "include", "reactant_mi355x.h"))
    objs = []
    for f in sorted(os.listdir(CSRC)):
        if not f.endswith(".cpp") or f in ("rx_hostcheck.cpp", "rx_rtc_worker.cpp"):   # programs of their own
            continue
        src = os.path.join(CSRC, f)
        obj = os.path.join(OBJ, f[:-4] + ".o")
        objs.append(obj)
        if force or _stale(obj, [src] + headers):
            cmd = [HIPCC] + COMMON
            if f == "rx_api.cpp":
                cmd += ["-x", "hip", "--offload-arch=" + ARCH] + PACKED
            else:
                cmd += ["-x", "c++", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", '-DRX_ROCM_LIB="%s"' % ROCM_LIB]   # host code only: no device pass
            _run(cmd + ["-c", src, "-o", obj])
    chk_src = os.path.join(CSRC, "kernels", "rx_gemm_check.hip")
    if os.path.exists(chk_src):
        chk_obj = os.path.join(OBJ, "rx_gemm_check.o")
        if force or _stale(chk_obj, [chk_src] + headers):
            _run([HIPCC, "-std=c++17", "-O3", "--offload-arch=" + ARCH, "-ffp-contract=off"] + PACKED +
                 ["-Wno-unused-command-line-argument", "-c", chk_src, "-o", chk_obj])
    if force or _stale(LIB, objs):
        _run([HIPCC, "-shared", "-fPIC", "--offload-arch=" + ARCH, "-o", LIB] + objs +
             ["-L" + ROCM_LIB, "-lhiprtc", "-ldl", "-Wl,-rpath," + ROCM_LIB])
    # the compiler's process (csrc/rx_rtc_worker.cpp): its hiprtc comes from ROCM_LIB whatever the environment's library path says
    src = os.path.join(CSRC, "rx_rtc_worker.cpp")
    if force or _stale(WORKER, [src] + headers):
        _run([os.environ.get("CXX", "/opt/rocm/lib/llvm/bin/clang++"), "-std=c++17", "-O2", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
              '-DRX_ROCM_LIB="%s"' % ROCM_LIB, src,
              "-o", WORKER, "-L" + ROCM_LIB, "-lhiprtc", "-Wl,--disable-new-dtags,-rpath," + ROCM_LIB])
    return LIB


HOSTCHECK = os.path.join(OBJ, "rx_hostcheck_asan")


def build_hostcheck():
    """The importer, planner, code generator and GEMM chooser as a host-only program under AddressSanitizer and
    UndefinedBehaviorSanitizer (csrc/rx_hostcheck.cpp; tests/test_host_sanitizers.py runs it over the module texts
    of the program builders).  No device code, no HIP runtime: ROCm's clang++ as a plain host compiler (the sources use
    _Float16, which the image's g++ 11 does not have in C++), sanitizer runtimes linked statically."""
    os.makedirs(OBJ, exist_ok=True)
    srcs = [os.path.join(CSRC, f) for f in ("rx_hostcheck.cpp", "rx_parse.cpp", "rx_plan.cpp", "rx_emit.cpp", "rx_gemm.cpp")]
    headers = [os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".h")]
    if _stale(HOSTCHECK, srcs + headers):
        _run([os.environ.get("CXX", "/opt/rocm/lib/llvm/bin/clang++"), "-std=c++17", "-O1", "-g", "-fno-omit-frame-pointer",
              "-fsanitize=address,undefined", "-fno-sanitize-recover=undefined", "-o", HOSTCHECK] + srcs)
    return HOSTCHECK


if __name__ == "__main__":
    if "--sanitize" in sys.argv:
        print(build_hostcheck())
    else:
        build_library(force="--force" in sys.argv)
        print(LIB)
