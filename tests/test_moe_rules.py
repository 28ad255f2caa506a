"""CPU: the arithmetic by which the few-token expert kernels are cut into workgroups."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "leviathan_amd", "csrc")

PROGRAM = """
#include "moe_split.hpp"
#include <cstdio>
int main() {
    unsigned cus, hidden, inter, pairs, per_cu;
    while (std::scanf("%u %u %u %u %u", &cus, &hidden, &inter, &pairs, &per_cu) == 5)
        std::printf("%u\\n", moe_gate_up_rows(cus, hidden, inter, pairs, per_cu));
}
"""


@pytest.fixture(scope="module")
def rows_of(tmp_path_factory):
    cxx = os.environ.get("CXX") or shutil.which("g++")
    if not cxx:
        pytest.skip("no C++ compiler")
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.cpp").write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-Wall", "-Werror", f"-I{CSRC}", str(d / "rules.cpp"), "-o", str(d / "rules")], check=True)

    def run(cases):
        text = "\n".join(" ".join(map(str, c)) for c in cases)
        out = subprocess.run([str(d / "rules")], input=text, check=True, capture_output=True, text=True).stdout.split()
        assert len(out) == len(cases)
        return [int(v) for v in out]
    return run


@pytest.mark.parametrize("hidden,inter,top_k,want", [(2048, 768, 8, (24, 12, 6)), (2816, 704, 8, (22, 11, 6))])
def test_gate_up_candidates_are_different_launches(rows_of, hidden, inter, top_k, want):
    """Schedule fields 1, 2 (the built-in rule) and 4: one, two and four workgroups a CU at one token."""
    assert tuple(rows_of([(256, hidden, inter, top_k, f) for f in (1, 2, 4)])) == want


def test_gate_up_rows_cover_every_shape(rows_of):
    cases = [(cus, h, i, k * t, f) for cus in (256, 304) for h in (64, 2048, 2112, 4096) for i in (64, 704, 1536, 4096)
             for k in (1, 2, 8, 16) for t in (1, 2, 4, 15) for f in (1, 2, 4)]
    for (cus, h, i, pairs, f), rows in zip(cases, rows_of(cases)):
        assert 1 <= rows <= i
        assert f != 2 or rows <= 16 or rows % 16 == 0 or rows == i
