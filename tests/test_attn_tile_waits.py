"""The attention tile kernel's waits, in the assembly that hipcc makes of it.

The kernel copies a key block into the LDS buffer that its waves read one block
earlier. Before the barrier that opens a block every wave has to have waited
for its own copies (vmcnt) and for its LDS reads of that buffer (lgkmcnt); a
wave whose last reads were still in flight could see the next block's keys.
"""
import os
import re
import shutil
import subprocess

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen-mlx_amd")


@pytest.mark.skipif(shutil.which("make") is None or not os.path.exists("/opt/rocm/bin/hipcc"),
                    reason="needs make and hipcc")
@pytest.mark.parametrize("G", [4, 8])
def test_tile_kernel_waits_for_copies_and_reads_before_each_barrier(tmp_path, G):
    line = subprocess.run(["make", "-s", "-n", "-B", "-C", PKG, "_obj/gdn_attn.hip.o"], check=True,
                          capture_output=True, text=True).stdout
    cmd = next(ln for ln in line.splitlines() if "-c -o" in ln).split()
    cmd[cmd.index("-o") + 1] = str(tmp_path / "attn.s")
    cmd[cmd.index("-c")] = "-S"
    subprocess.run([*cmd, "--cuda-device-only"], check=True, cwd=PKG, capture_output=True)
    text = (tmp_path / "attn.s").read_text()
    body = re.search(rf"^_ZN3gdn16attn_tile_kernelILi{G}E[^:\n]*:[^\n]*\n(.*?)s_endpgm", text,
                     re.S | re.M).group(1)
    code = [ln.split(";")[0].strip() for ln in body.splitlines()]
    code = [ln for ln in code if ln and not ln.startswith(".")]
    barriers = [i for i, ln in enumerate(code) if ln.startswith("s_barrier")]
    assert len(barriers) >= 2  # the two buffers' blocks
    for i in barriers:
        pending = {"vmcnt(0)", "lgkmcnt(0)"}
        for ln in reversed(code[:i]):
            if ln.startswith("s_waitcnt"):
                pending -= set(re.findall(r"\w+\(\d+\)", ln))
            elif ln.startswith("ds_"):
                assert "lgkmcnt(0)" not in pending, f"LDS access not waited for before: {ln}"
            elif re.match(r"(global|buffer)_load", ln):
                assert "vmcnt(0)" not in pending, f"copy not waited for before: {ln}"
            if not pending:
                break
        assert not pending
