"""Build-time guard for kernels that live off their registers (CPU only).

The row kernels hold whole rows or tiles in VGPRs; past the limit that their
launch bounds leave, the compiler spills to scratch memory without a word, and
the kernel loses what it was built for (a LayerNorm backward that spilled 107
registers took 183 us where it takes 39).  Each source is compiled to gfx950
device assembly with the library's own flags, and the resource report of its
kernels is held to the most that was measured to be harmless.
"""
import os
import re
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(REPO, "thot_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"

# source: (pattern of the kernels' names, spilled registers allowed)
LIMITS = {
    "layernorm.hip": [(r"ln_(fwd|bwd)_kernel", 0)],
    "attention.hip": [(r"attn_(fwd32|dq32|dkdv32)_kernel", 2)],
}


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
@pytest.mark.parametrize("src", sorted(LIMITS))
def test_spilled_registers(src, tmp_path):
    from thot_amd.build import HIP_FLAGS
    asm = tmp_path / (src + ".s")
    r = subprocess.run([HIPCC, *[f for f in HIP_FLAGS if f != "-fPIC"], "--cuda-device-only", "-S",
                        os.path.join(CSRC, src), "-o", str(asm)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    kernels = re.findall(r"\.name:\s+(\S+).*?\.vgpr_spill_count:\s+(\d+)", asm.read_text().split(".amdgpu_metadata")[1],
                         re.S)
    for pattern, most in LIMITS[src]:
        mine = {name: int(n) for name, n in kernels if re.search(pattern, name)}
        assert mine, f"{src}: no kernel matches {pattern}"
        over = {name: n for name, n in mine.items() if n > most}
        assert not over, f"{src}: spilled registers {over} (at most {most})"
