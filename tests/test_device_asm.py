"""The device code's inline assembly: an instruction that reads or writes
memory names memory as clobbered, so that the compiler keeps it in order with
the accesses around it, and a load waits for its result in the same statement
(the compiler counts neither)."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hvm-64_amd", "csrc")


def statements():
    for path in sorted(glob.glob(os.path.join(CSRC, "*"))):
        text = open(path).read()
        for m in re.finditer(r"\basm\s+volatile\s*\(", text):
            depth, i = 1, m.end()
            while depth:
                depth += {"(": 1, ")": -1}.get(text[i], 0)
                i += 1
            yield os.path.basename(path), re.sub(r"\s+", " ", text[m.end():i - 1])


def test_memory_instructions_clobber_memory_and_loads_wait():
    memory = 0
    for where, s in statements():
        if re.search(r"(global|flat|buffer|ds)_(load|store|atomic|read|write)|s_waitcnt", s):
            memory += 1
            assert s.rstrip().endswith('"memory"'), (where, s)
        if re.search(r"_load_", s):
            assert "s_waitcnt vmcnt(0)" in s, (where, s)
    assert memory >= 4
