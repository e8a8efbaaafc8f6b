"""The prefix sort's arithmetic that needs no device (sadcs_amd/csrc/prefix_plan.h), compiled here and
compared with Python's integers."""
import os
import random
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


def test_large_tie_rows(tmp_path):
    """Groups of every size up to 100 rows, among them those around 24, at every place in a word."""
    rng = random.Random(3)
    bits, want = [], 0
    for size in list(range(1, 101)) * 4 + [24, 25, 26] * 40 + [1] * 31 + [700, 65, 64, 33, 32]:
        bits += [0] + [1] * (size - 1)
        want += size if size > 24 else 0
        gap = rng.randrange(0, 40)
        bits += [0] * gap
    bits += [0] * (32 - len(bits) % 32) + [0] * 32
    words = [sum(b << r for r, b in enumerate(bits[w:w + 32])) for w in range(0, len(bits), 32)]
    got = run_cpp(tmp_path, 'unsigned a, b, sum = 0; while (scanf("%u %u", &a, &b) == 2) sum += largeTieRows(a, b); printf("%u\\n", sum);',
                  [f"{a} {b}" for a, b in zip(words, words[1:] + [0])])
    assert int(got[0]) == want


@pytest.mark.parametrize("density", [1 / 32, 1 / 96])
def test_tie_estimate(tmp_path, density):
    """Counts that a sample of this density has on average where a share of the rows lies in groups of one
    size. A row meets the others of its group with a binomial number, of which the estimate makes a Poisson
    number: of g rows it sees between g - 1 and g, and the share larger by as much."""
    cases, lines = [(g, share) for g in (2, 3, 6, 12, 25, 64, 300) for share in (0.1, 0.5, 1.0)], []
    for g, share in cases:
        alone = (1 - density) ** (g - 1)
        one = (g - 1) * density * (1 - density) ** (g - 2)
        lines.append(f"1e6 {1e6 * share * (1 - alone)!r} {1e6 * share * max(0.0, 1 - alone - one)!r} {density!r}")
    lines += [f"1000 0 0 {density!r}", f"0 0 0 {density!r}", f"1000 900 900 {density!r}"]
    got = run_cpp(tmp_path, 'double s, r, u, d; while (scanf("%lf %lf %lf %lf", &s, &r, &u, &d) == 4) { TieEstimate e = estimateTies(s, r, u, d); '
                  'printf("%.9f %.9f\\n", e.share, e.groupRows); }', lines)
    got = list(zip(map(float, got[::2]), map(float, got[1::2])))
    for (g, share), (got_share, rows) in zip(cases, got):
        assert 0.95 * max(2, g - 1) <= rows <= 1.05 * g, (g, share)
        assert 0.95 * share <= got_share <= min(1.0, 1.05 * share * (g - 1) / max(1, g - 2)), (g, share)
    assert got[-3:-1] == [(0, 1), (0, 1)]
    assert got[-1][0] == pytest.approx(0.9, rel=1e-4) and got[-1][1] == pytest.approx(1 + 12 / density, rel=1e-6)
