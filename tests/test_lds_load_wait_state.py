"""The instruction set asks for one wait state between a scalar write of M0 and
a load to LDS; the compiler does not look into inline assembly for it."""

import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flex_shard_amd", "csrc")


def test_every_load_to_lds_waits_for_m0():
    loads = 0
    for name in sorted(os.listdir(CSRC)):
        if not name.endswith((".hip", ".hpp")):
            continue
        text = open(os.path.join(CSRC, name)).read()
        for block in re.findall(r'asm volatile\(\s*"((?:[^"\\]|\\.)*)"', text):
            lines = [line.strip() for line in re.split(r"\\n|\\t", block) if line.strip()]
            for i, line in enumerate(lines):
                if line.startswith(("global_load_lds", "buffer_load")):
                    loads += 1
                    assert i >= 2 and re.match(r"s_\w+ m0,", lines[i - 2]) and lines[i - 1] == "s_nop 0", (name, block)
    assert loads >= 3  # 16 bytes per lane by offset and by address, 4 by offset
