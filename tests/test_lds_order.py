"""The dense-restore kernels pass values between the lanes of a wave through LDS.  What
makes that safe is in the code the compiler is given, not in what one compiler version
does with it: every exchange is fenced, and a 16-bit store into a staged 16-byte vector
may alias it.  Read from the unoptimised IR of the sources, so no GPU is needed."""
import re
import subprocess

import pytest

from marlin_style_fluxbin_amd import build as b


def _ir(unit: str) -> str:
    try:
        compiler = b.hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    done = subprocess.run([compiler, *b.HIPCC_FLAGS, "--cuda-device-only", "-S", "-emit-llvm", "-Xclang",
                           "-disable-llvm-passes", "-I", str(b.PACKAGE.parent / "include"), str(b.CSRC / unit), "-o",
                           "-"], capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, done.stderr
    return done.stdout


@pytest.mark.parametrize("unit", ["hybrid_restore.hip", "w3_restore.hip"])
def test_wave_exchanges_are_fenced(unit):
    lines = [line.strip() for line in _ir(unit).splitlines()]
    barriers = [i for i, line in enumerate(lines) if "call void @llvm.amdgcn.wave.barrier()" in line]
    assert barriers
    for i in barriers:
        assert lines[i - 1] == 'fence syncscope("wavefront") release'
        assert lines[i + 1] == 'fence syncscope("wavefront") acquire'


def test_patched_columns_may_alias_the_staged_vectors():
    ir = _ir("hybrid_restore.hip")
    kernels = re.findall(r"^define [^\n]*amdgpu_kernel [^\n]*hybrid_restore_kernelILi[12].*?^}", ir, flags=re.M | re.S)
    tags = [t for k in kernels for t in re.findall(r"store i16 .*!tbaa (!\d+)", k)]
    assert len(kernels) == 2 and len(tags) == 2
    nodes = dict(re.findall(r"^(!\d+) = !\{(.*)\}$", ir, flags=re.M))
    for tag in tags:
        access = nodes[tag].split(",")[0]
        assert nodes[access].startswith('!"omnipotent char"')
