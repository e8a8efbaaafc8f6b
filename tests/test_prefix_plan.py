"""The prefix sort's arithmetic that needs no device (sadcs_amd/csrc/prefix_plan.h), compiled here and
compared with Python's integers."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sadcs_amd", "csrc")


def run_cpp(tmp_path, body, lines):
    """Output lines of a program whose main is `body`, given `lines` on its standard input."""
    source = tmp_path / "main.cpp"
    source.write_text('#include <cstdio>\n#include "prefix_plan.h"\nusing namespace sadcs;\nint main() {\n' + body + "\n}\n")
    subprocess.run(["g++", "-std=c++20", "-O1", "-Wall", f"-I{CSRC}", str(source), "-o", str(tmp_path / "main")], check=True)
    return subprocess.run([str(tmp_path / "main")], input="\n".join(lines) + "\n", text=True, check=True, capture_output=True).stdout.split()


@pytest.mark.parametrize("bits", range(1, 10))
def test_held_bits(tmp_path, bits):
    """Where remaining * bits passes a multiple of 2^32, too, up to the longest text there is."""
    near = [k * 2**32 // bits + d for k in range(bits) for d in range(-2, 130)]
    cases = sorted({r for r in list(range(300)) + near + [2**31 - 1, 2**30, 2**31 - 257] if 0 <= r < 2**31})
    got = run_cpp(tmp_path, 'unsigned r; while (scanf("%u", &r) == 1) printf("%u\\n", heldBits(r, ' + str(bits) + "));", map(str, cases))
    assert [int(x) for x in got] == [min(r * bits, 128) for r in cases]
