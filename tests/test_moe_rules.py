"""CPU: the arithmetic by which the few-token expert kernels are cut into workgroups."""
import itertools
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


PLAN_PROGRAM = """
#include "moe_prefill_plan.hpp"
#include <cstdio>
int main() {
    unsigned cus, hidden, inter, experts, top_k, tokens;
    while (std::scanf("%u %u %u %u %u %u", &cus, &hidden, &inter, &experts, &top_k, &tokens) == 6) {
        const pf_plan p = pf_plan_of(pf_shape{cus, hidden, inter, experts, top_k, tokens});
        std::printf("%u %u %u\\n", p.cols, (unsigned)p.gate_up, (unsigned)p.down);
    }
}
"""


def test_prompt_product_forms(tmp_path):
    """Every form of the grouped product is reached by a shape of tests/test_gpu_moe_prefill.py, the narrow one (4) only where
    items are cut to 32 pairs, the folded ones (1 to 4) exactly where a row has more than 32 blocks."""
    from tests.test_gpu_moe_prefill import FORMS
    cxx = os.environ.get("CXX") or shutil.which("g++")
    if not cxx:
        pytest.skip("no C++ compiler")
    (tmp_path / "plan.cpp").write_text(PLAN_PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-Wall", "-Werror", f"-I{CSRC}", str(tmp_path / "plan.cpp"), "-o", str(tmp_path / "plan")], check=True)
    cases = [(256, h, i, e, 1, t) for h, i, e, t, _ in FORMS]
    cases += list(itertools.product((64, 256), (64, 1024, 1088, 4160), (64, 704, 1088), (1, 32, 128, 4096), (1, 8), (1, 300, 1000, 20000)))
    text = "\n".join(" ".join(map(str, c)) for c in cases)
    out = subprocess.run([str(tmp_path / "plan")], input=text, check=True, capture_output=True, text=True).stdout.split()
    plans = [tuple(map(int, out[k:k + 3])) for k in range(0, len(out), 3)]
    assert len(plans) == len(cases)
    assert [p for p in plans[:len(FORMS)]] == [f[4] for f in FORMS]
    assert {p[1] for p in plans[:len(FORMS)]} == {0, 1, 2, 3, 4} == {p[2] for p in plans[:len(FORMS)]}
    for (cus, hidden, inter, *_), (cols, gate_up, down) in zip(cases, plans):
        assert cols == (32 if 4 in (gate_up, down) else 64)
        assert (gate_up == 0) == (hidden <= 1024) and (down == 0) == (inter <= 1024)


RANK_PROGRAM = """
#include "moe_prefill_plan.hpp"
#include <cstdio>
int main() {
    unsigned experts, top_k, k0;
    int own[8], good[8];
    while (std::scanf("%u %u %u", &experts, &top_k, &k0) == 3) {
        bool ok[8];
        for (int u = 0; u < 8; ++u) {
            if (std::scanf("%d %d", own + u, good + u) != 2) return 1;
            ok[u] = good[u] != 0;
        }
        int rank[8], adds = 0;
        pf_rank_pairs(own, ok, k0, top_k, experts, [&](uint32_t word) { std::printf("%u ", word); return 100 + adds++; }, rank);
        std::printf("|");
        for (int r : rank) std::printf(" %d", r);
        std::printf("\\n");
    }
}
"""


def test_prompt_grouping_adds_once_a_pair(tmp_path):
    """A slot past top_k adds to no word of the counts (lanes that add to one word take the LDS a turn each); a pair adds to its
    expert's word, a dropped one to the word behind the lists, and gets no rank."""
    cxx = os.environ.get("CXX") or shutil.which("g++")
    if not cxx:
        pytest.skip("no C++ compiler")
    (tmp_path / "rank.cpp").write_text(RANK_PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-Wall", "-Werror", f"-I{CSRC}", str(tmp_path / "rank.cpp"),
                    "-o", str(tmp_path / "rank")], check=True)
    cases = [(60, top_k, k0, dropped) for top_k in range(1, 20) for k0 in range(0, top_k, 8) for dropped in ((), (0,), (1, 6))]
    lines = []
    for experts, top_k, k0, dropped in cases:
        ok = [k0 + u < top_k and u not in dropped for u in range(8)]
        lines.append(f"{experts} {top_k} {k0} " + " ".join(f"{7 * u if good else -5} {int(good)}" for u, good in enumerate(ok)))
    out = subprocess.run([str(tmp_path / "rank")], input="\n".join(lines), check=True, capture_output=True, text=True).stdout.splitlines()
    assert len(out) == len(cases)
    for (experts, top_k, k0, dropped), line in zip(cases, out):
        words, ranks = (list(map(int, part.split())) for part in line.split("|"))
        pairs = min(8, top_k - k0)
        assert words == [2 * experts if u in dropped else 7 * u for u in range(pairs)], (top_k, k0)
        assert ranks == [100 + u if u < pairs and u not in dropped else -1 for u in range(8)], (top_k, k0)
