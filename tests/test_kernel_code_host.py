"""What the compiler is told where results cannot show a mistake: inline assembly that writes a register must say so."""

import glob
import os
import re

from ampere_kv_engine_amd.csrc import build


def test_inline_assembly_that_writes_m0_says_so():
    blocks = []
    for path in sorted(glob.glob(os.path.join(build.HERE, "*.hip")) + glob.glob(os.path.join(build.HERE, "*.h"))):
        with open(path) as handle:
            blocks += [(os.path.basename(path), block) for block in re.findall(r"\basm volatile\((.*?)\);", handle.read(), re.S)]
    writers = [(name, block) for name, block in blocks if re.search(r"s_mov_b32 m0", block)]
    assert writers, "no block writes m0 any more: this test can go"
    for name, block in writers:
        assert block.count(":") == 3 and '"m0"' in block.split(":")[3], f"{name}: {block}"
