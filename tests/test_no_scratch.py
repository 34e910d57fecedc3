"""Every kernel of the library keeps its registers: none spills to scratch memory (a spilled value's
reload waits for every vector-memory access in flight, the row gathers among them), and the 128-head
kernels, whose code about fills the instruction cache, lie at multiples of 64 KB and the combine
kernels at multiples of 16 KB, whatever precedes them.  The device code of each source is compiled with the build's own flags, and the compiler's
report and assembly are read."""
import re
import subprocess

import pytest

from opfoundry_amd import build


@pytest.mark.parametrize("src", build.SRCS, ids=lambda s: s.rsplit("/", 1)[-1])
def test_no_kernel_uses_scratch(src):
    flags = [f for f in build.HIPCC_FLAGS if f not in ("-shared", "-fPIC")]
    res = subprocess.run([build.hipcc(), *flags, f"-I{build.INCLUDE}", "-S", "--cuda-device-only", src, "-o", "-",
                          "-Rpass-analysis=kernel-resource-usage"], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    names = re.findall(r"Function Name: (\S+)", res.stderr)
    sizes = [int(n) for n in re.findall(r"ScratchSize \[bytes/lane\]: (\d+)", res.stderr)]
    assert len(names) == len(sizes) > 0
    assert {n: s for n, s in zip(names, sizes) if s} == {}
    if src.endswith("dsa_mla.hip"):
        wide = re.findall(r"\.p2align\s+(\d+)[^\n]*\n\s*\.type\s+(\S*dsa_mla_fwd_kernelILi\d\S*),@function", res.stdout)
        assert len(wide) == 5 and {a for a, _ in wide} == {"16"}
        after = re.findall(r"\.p2align\s+(\d+)[^\n]*\n\s*\.type\s+(\S*dsa_mla_combine_\S*),@function", res.stdout)
        assert len(after) == 2 and {a for a, _ in after} == {"14"}
