"""The persistent kernels re-read their arguments stage by stage from the kernel-argument
memory (csrc/k2_persistent.hip).  Outside a kernel's own body the builtin that names it is
0 until the function is inlined into one, which no flag promises: the front end's code, ahead
of every optimization, takes it in kernels alone."""

import subprocess

import pytest


def test_argument_memory_is_taken_in_kernels_alone(tmp_path):
    from sgl_amd_mono import _build

    try:
        cxx = _build.hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    out = tmp_path / "k2.ll"
    subprocess.run([cxx, *_build.HIPCC_FLAGS, "-I", str(_build.INCLUDE), "-I", str(_build.CSRC), "--cuda-device-only", "-S",
                    "-emit-llvm", "-Xclang", "-disable-llvm-passes", str(_build.CSRC / "k2_persistent.hip"), "-o", str(out)],
                   check=True, capture_output=True)
    inside, takers = "", set()
    for line in out.read_text().splitlines():
        if line.startswith("define "):
            inside = line
        elif "call " in line and "@llvm.amdgcn.kernarg.segment.ptr" in line:
            takers.add(inside)
    assert takers
    for f in takers:
        assert " amdgpu_kernel " in f, f
