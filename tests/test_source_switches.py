"""What the native sources look at besides their arguments: the trace build's
macros, and inside it the address of the trace buffer."""

import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flex_shard_amd", "csrc")
MACROS = {"FSH_TRACE", "FSH_TRACE_NODRAIN"}


def test_only_the_trace_build_changes_the_library():
    environment = []
    for name in sorted(os.listdir(CSRC)):
        if not name.endswith((".hip", ".hpp")):
            continue
        enclosing = []  # the conditions that a line is under
        for line in open(os.path.join(CSRC, name)):
            directive = re.match(r"\s*#\s*(if|ifdef|ifndef|elif|endif)\b(.*)", line)
            if directive and directive[1] == "endif":
                enclosing.pop()
            elif directive:
                macros = set(re.findall(r"\b[A-Z_][A-Z0-9_]*\b", directive[2]))
                assert macros and macros <= MACROS, (name, line)
                if directive[1] == "elif":
                    enclosing.pop()
                enclosing.append(directive[0].split())
            for variable in re.findall(r'getenv\((.*?)\)', line):
                assert ["#ifdef", "FSH_TRACE"] in enclosing, (name, line)
                environment.append(variable)
    assert set(environment) == {'"FSH_GEMM_TRACE"'}
