"""What the kernels' sources have to say for themselves, read as text: facts that no run on the hardware shows."""
import os
import re
import subprocess

import inferllm_amd
from inferllm_amd.kernels import build

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


def test_the_float32_parts_loads_are_issued_in_the_order_their_waits_count(tmp_path):
    """The product in bfloat16 parts waits for "all but the youngest n" loads before other waves read what a wave brought
    into LDS: in the compiled code W's loads (registers) and X's (LDS) stand stage by stage, and no load moves
    from one turn to another."""
    out = str(tmp_path / "parts.s")
    subprocess.run([build._hipcc()] + build.HIPCC_FLAGS + ["--offload-device-only", "-S", "-o", out,
                                                           os.path.join(CSRC, "gemm_f32_split.hip")], check=True,
                   stderr=subprocess.DEVNULL)
    kernels = re.findall(r"^_Z\w*gemm_f32_split_kernelILi(\d+)ELi(\d+)ELi(\d+)ELb[01]ELi(\d+)E\w*:(.*?)\.Lfunc_end", open(out).read(),
                         re.S | re.M)
    assert len(kernels) >= 15
    for *sizes, body in kernels:
        mt, nt, ns, waves = map(int, sizes)
        x, w = "X" * -(-3 * mt // waves), "W" * (2 * nt)
        stages = []
        for part in body.split("s_barrier")[:4]:
            loads = [line for line in part.splitlines() if re.search(r"\b(buffer|global)_load", line)]
            stages.append("".join("X" if "lds" in line else "W" for line in loads))
        # ahead of the first wait ns - 1 stages and W of one more; then a stage a turn
        assert stages[0] == (w + x) * (ns - 1) + w, (mt, nt, ns, stages[0])
        assert stages[1:] == [x + w] * 3, (mt, nt, ns, stages)
        counts = re.findall(r"s_waitcnt vmcnt\((\d+)\) lgkmcnt\(0\)\s*\n\s*s_barrier", body)
        assert counts and set(counts) == {str((ns - 2) * len(x + w))}, (mt, nt, ns, counts)


def test_what_lanes_of_a_wave_hand_each_other_through_lds_is_fenced_for_the_compiler():
    """The softmax's weights go from some lanes of a wave to all of them, with no barrier: the compiler, to which a lane's
    loads are its own, is told by a fence before a round's stores and another between them and the loads."""
    body = re.search(r"^attn_cap_decode_keys16_kernel\(.*?^}", SOURCES["attention_capped.hip"], re.S | re.M).group(0)
    fence = re.search(r"auto (\w+) = \[\]\(\)[^{]*{([^}]*)}", body)
    assert '__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront")' in fence.group(2)
    assert "__builtin_amdgcn_wave_barrier()" in fence.group(2)
    uses = re.findall(r"weights\[w\][^;=]*(=?)|" + fence.group(1) + r"(\(\));", body[fence.end():])
    assert "".join("S" if store else "F" if call else "L" for store, call in uses) == "FSSFLL"
