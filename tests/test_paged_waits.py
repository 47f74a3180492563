"""The waits in the tile loops of the paged kernels, read in the generated code: below 4 GB of K cache (SMALL) a tile's K transfers have landed
before its operands are read, and the next tile's stay in flight."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def test_the_next_tile_stays_in_flight(tmp_path):
    if shutil.which(HIPCC) is None and not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    from inference_lib_amd import build
    asm = tmp_path / "paged.s"
    cmd = [HIPCC, f"--offload-arch={build.ARCH}", "-O3", "-std=c++17", "-fno-gpu-rdc", "-munsafe-fp-atomics", "--cuda-device-only",
           *build.DEVICE_FLAGS, "-I", os.path.join(ROOT, "include"), "-S", os.path.join(build.CSRC, "hogwild_paged.hip"), "-o", str(asm)]
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=900)
    assert r.returncode == 0, r.stderr[-3000:]
    text = asm.read_text()
    # paged_attention_kernel<DT, E, EV, RB, MINW, SMALL, KEEP>
    kernels = re.findall(r"^(_ZN2hw22paged_attention_kernelINS_(\d)(\w+?)ELi(\d+)ELi\d+ELi\d+ELi\d+ELb1ELb\S*):", text, re.M)
    assert len(kernels) >= 12
    for name, _, dtype, e in kernels:
        size = 4 if dtype == "F32" else 2
        transfers = 32 * int(e) * size // 1024                   # 1 KB each
        loads = 8 * max(1, int(e) * size // 256)                 # of a tile's V rows
        body = text[text.index(name + ":"):]
        body = body[:body.index("; -- End function")]
        assert re.search(r"scratch_(load|store)", body) is None, name
        checked = 0
        for block in re.split(r"\n\.LBB\d+_\d+:", body)[1:]:
            if "Depth=2" not in block or len(re.findall(r"buffer_load_dwordx4[^\n]*\blds\b", block)) < transfers:
                continue
            wait, issued = None, 0
            for line in block.splitlines():
                if re.search(r"buffer_load_dwordx4[^\n]*\blds\b", line):
                    issued += 1
                elif re.search(r"s_waitcnt[^\n]*vmcnt\((\d+)\)", line):
                    n = int(re.search(r"vmcnt\((\d+)\)", line).group(1))
                    assert n >= transfers, f"{name}: {line.strip()} leaves less than a tile's K transfers in flight"
                    if issued == transfers:
                        wait = n
                elif issued == transfers and "ds_read_b128" in line:
                    # behind the tile's K: its V loads, a table entry, the next tile's transfers and V loads
                    assert wait is not None and wait <= 2 * loads + transfers + 1, f"{name}: operands read behind a wait for {wait}"
                    checked += 1
                    break
        assert checked >= 2, name
