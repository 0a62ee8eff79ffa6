"""Hand-written loads straight into LDS keep the wait state that their address in m0 wants."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llmserver_amd", "csrc")


def test_a_load_into_lds_waits_a_state_behind_the_write_of_its_address():
    """The scalar instruction that writes m0 and a load that takes its LDS address from m0 stand in one asm block, into which the compiler does
    not look: between them stands at least one instruction, as the compiler itself places it."""
    found = 0
    for name in sorted(os.listdir(CSRC)):
        with open(os.path.join(CSRC, name)) as handle:
            blocks = re.findall(r'asm volatile\(\s*((?:"[^"]*"\s*)+)', handle.read())
        for block in blocks:
            lines = [line.strip() for piece in re.findall(r'"([^"]*)"', block) for line in re.split(r"\\n|\\t|;", piece) if line.strip()]
            for at, line in enumerate(lines):
                if re.match(r"(global|buffer|scratch)_load_(lds_)?\w+", line) and "lds" in line:
                    found += 1
                    writes = [i for i in range(at) if re.match(r"s_\w+\s+m0\b", lines[i])]
                    assert writes and at - writes[-1] >= 2, f"{name}: {lines}"
    assert found
