"""What the kernels' sources have to say for themselves, read as text: facts that no run on the hardware shows."""
import os
import re

import inferllm_amd

CSRC = os.path.join(os.path.dirname(inferllm_amd.__file__), "csrc")
SOURCES = {f: open(os.path.join(CSRC, f)).read() for f in sorted(os.listdir(CSRC)) if f.endswith((".hip", ".h"))}


def test_dynamic_lds_is_declared_on_16_bytes():
    """An array of dynamic LDS stands behind the kernel's other LDS at the alignment it declares: read or
    written 16 bytes at a time, it has to declare 16, whatever the hardware would take."""
    found = 0
    for name, text in SOURCES.items():
        for line in re.findall(r"extern __shared__[^;]*;", text):
            found += 1
            assert "__attribute__((aligned(16)))" in line, (name, line)
    assert found >= 20
