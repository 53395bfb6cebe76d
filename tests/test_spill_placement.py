"""Register spills of the batched LU kernels (batched_lu.hip, the only ones
that spill more than a word).  The compiler can place a spill or a reload at
the head of the block that ends a divergent branch, before exec is restored:
then only the branch's lanes are saved or loaded and the others go on with
stale values, which no diagnostic shows.  Checks the assembly of the kernels as built."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "rust-la_amd", "csrc")


def misplaced(asm):
    """Spills and reloads between a block's label and its restore of exec (a
    block that does vector work first is a branch's body, which ends there)."""
    found, kernel, head = [], None, None
    for line in asm.splitlines():
        m = re.match(r"(_Z\w+):", line)
        if m:
            kernel, head = m.group(1), None
        elif re.match(r"\.LBB|; %bb", line):
            head = []
        elif head is not None:
            if re.match(r"\s+s_or_b64 exec, exec", line):
                found += [(kernel, h) for h in head]
                head = None
            elif re.match(r"\s+scratch_(store.*Spill|load.*Reload)", line):
                head.append(line.strip())
            elif re.match(r"\s+(s_c?branch|v_|ds_|global_|scratch_|flat_)", line) and \
                    not re.match(r"\s+v_(readlane|writelane|mov)_b", line):
                head = None
    return found


def test_finds_a_planted_one():
    good = "_Zk:\n.LBB0_1:\n\ts_or_b64 exec, exec, s[0:1]\n\tscratch_store_dword off, v1, off ; 4-byte Folded Spill\n"
    bad = "_Zk:\n.LBB0_1:\n\ts_mov_b32 s1, s2\n\tscratch_store_dword off, v1, off ; 4-byte Folded Spill\n\ts_or_b64 exec, exec, s[0:1]\n"
    assert misplaced(good) == [] and len(misplaced(bad)) == 1


def test_batched_lu():
    make = subprocess.run(["make", "-n", "-B", "-C", CSRC, "_build/batched_lu.hip.o"],
                          capture_output=True, text=True).stdout
    line = next((l for l in make.splitlines() if "batched_lu.hip" in l and " -c " in l), None)
    if line is None or shutil.which(line.split()[0]) is None:
        pytest.skip("no HIP compiler")
    args = line.split(" -o ")[0].split()
    args.remove("-c")
    asm = subprocess.run(args + ["--cuda-device-only", "-S", "-o", "-"], cwd=CSRC, check=True,
                         capture_output=True, text=True).stdout
    assert "k_lu_ir_batched" in asm
    assert misplaced(asm) == []
