"""A product whose rows of x come as parts copies them to LDS by instructions that the compiler does not count.  A step ends with a wait for all but 16 of
its requests, those of W, which follow the copies: the built code is looked at for whether they do."""
import re
import shutil
import subprocess

import pytest

import shainet_amd as sa

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.mark.skipif(shutil.which(OBJDUMP) is None, reason="no disassembler")
def test_sixteen_loads_follow_the_copies_of_a_step(tmp_path):
    lib = shutil.copy(sa.library_path(), tmp_path)
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, stdout=subprocess.DEVNULL, cwd=tmp_path)
    found = 0
    for code in tmp_path.glob("*gfx950*"):
        symbols = subprocess.run([OBJDUMP, "-t", str(code)], check=True, capture_output=True, text=True).stdout
        names = {w for w in symbols.split() if w.startswith("_Z") and "sgemm_wide_kernel" in w and "Lb1EEE" in w and "." not in w}
        for name in sorted(names):
            text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--disassemble-symbols=" + name, str(code)], check=True, capture_output=True, text=True).stdout
            ops = [line.split("//")[0].strip() for line in text.splitlines()]
            steps = []
            for at, op in enumerate(ops):
                if not re.match(r"s_waitcnt vmcnt\(16\)", op) or "s_barrier" not in ops[at + 1:at + 4]:
                    continue  # (the compiler's own)
                behind = 0
                for before in reversed(ops[:at]):
                    if before.startswith("global_load_lds"):
                        break
                    behind += before.startswith(("global_load", "global_store", "buffer_", "scratch_"))
                    assert not before.startswith(("s_branch", "s_cbranch", "s_barrier")), (name, before)  # (one block from the copies to the wait)
                steps.append(behind)
            # (none behind the last step of a tile, whose copies are nobody's)
            assert any(n == 16 for n in steps) and all(n >= 16 or n == 0 for n in steps), (name, steps)
            found += 1
    assert found >= 4, found
