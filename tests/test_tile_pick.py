"""CPU test of the rule on tile shapes (hy-mt-rs_amd/csrc/hyq_tile_pick.hpp,
host code compiled here with g++): the products that the GPU tests run for each
shape (tests/tile_cases.py) are the ones the rule sends there, so that another
rule cannot leave a shape untested."""
import os
import subprocess

import tile_cases

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "hy-mt-rs_amd", "csrc", "hyq_tile_pick.hpp")

PROGRAM = r'''
#include "HEADER"
#include <cstdio>
int main() {
    const char *names[] = {"T256", "T256R96", "T192", "T128", "T64"};
    static_assert(hyq::T256 == 0 && hyq::T256R96 == 1 && hyq::T192 == 2 && hyq::T128 == 3 &&
                  hyq::T64 == 4, "names");
    int gate_up, rows, tokens;
    while (std::scanf("%d %d %d", &gate_up, &rows, &tokens) == 3)
        std::puts(names[hyq::pick_tile(tokens, 1, !gate_up, [&](int r) {
            return gate_up ? hyq::gate_up_row_tiles(rows, r) : hyq::matmul_row_tiles(rows, r);
        })]);
}
'''


def test_cases_reach_their_shapes(tmp_path):
    src, exe = tmp_path / "pick.cpp", tmp_path / "pick"
    src.write_text(PROGRAM.replace("HEADER", HEADER))
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", str(src), "-o", str(exe)], check=True)
    cases = [(0, c) for c in tile_cases.MATMUL] + [(1, c) for c in tile_cases.GATE_UP]
    text = "".join(f"{g} {rows} {tokens}\n" for g, (_, rows, tokens) in cases)
    out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True)
    assert out.stdout.split() == [shape for _, (shape, _, _) in cases]
    for cases in (tile_cases.MATMUL, tile_cases.GATE_UP):
        assert len({shape for shape, _, _ in cases}) == len(cases)
