"""The parts of the fixed-length K = 256 forward (csrc/gdn_plan.hpp), compiled for the host."""
import subprocess
from pathlib import Path

import pytest

HEADER = Path(__file__).resolve().parents[1] / "kairos-sensenova_amd" / "csrc" / "gdn_plan.hpp"
MAIN = r"""
#include <cstdio>
#include <cstdlib>
#include "%s"
int main(int, char** v) {
  const kgdn::PipePlan p = kgdn::wide_pipe_plan(atoi(v[1]), atoi(v[2]), atoi(v[3]), 256, atoi(v[4]) & 1, atoi(v[4]) & 2);
  printf("%%d %%.1f", p.parts, p.growth);
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "main.cpp").write_text(MAIN % HEADER)
    subprocess.run(["g++", "-std=c++17", "-O1", "-o", str(d / "main"), str(d / "main.cpp")], check=True)

    def run(*args):
        return subprocess.run([str(d / "main"), *map(str, args)], check=True, capture_output=True, text=True).stdout
    return run


# chunks, (sequence, head) pairs, value tiles: the form that measured fastest, or within 1% of it
@pytest.mark.parametrize("nt,heads,tiles,want", [
    (25, 20, 8, "1 1.4"), (64, 20, 8, "1 1.4"), (256, 20, 8, "2 1.4"), (512, 20, 8, "4 1.4"), (512, 24, 8, "4 1.4"),
    (256, 28, 8, "1 1.0"), (256, 32, 8, "1 1.0"), (512, 36, 8, "4 1.4"), (128, 40, 8, "2 1.4"), (512, 40, 8, "4 1.4"),
    (256, 48, 8, "1 1.0"), (128, 60, 8, "1 1.0"), (256, 64, 8, "1 1.0"), (128, 80, 8, "1 1.0"),
    (64, 5, 8, "1 3.0"), (512, 5, 8, "2 3.0"), (512, 10, 8, "2 3.0"), (64, 20, 4, "1 3.0"), (128, 20, 4, "2 3.0"),
    (512, 5, 1, "4 1.4"), (256, 10, 1, "4 1.4"), (128, 20, 2, "4 1.4"), (64, 20, 1, "1 3.0"), (32, 40, 2, "1 1.4"),
    (64, 40, 2, "2 1.4"), (64, 40, 1, "4 1.4"), (47, 64, 1, "2 1.4"),
    (256, 16, 8, "2 1.4"), (512, 14, 8, "2 3.0"), (375, 20, 4, "2 3.0"), (256, 32, 4, "4 1.4"), (512, 32, 4, "4 1.4"),
])
def test_fastest_measured_form(plan, nt, heads, tiles, want):
    assert plan(nt, heads, tiles, 0) == want


@pytest.mark.parametrize("nt,heads,tiles,want", [(128, 20, 8, "1 1.4"), (256, 20, 8, "4 1.4"), (375, 20, 8, "4 1.4"),
                                                 (512, 20, 8, "4 1.4"), (128, 40, 8, "2 1.4"), (512, 10, 8, "2 3.0"),
                                                 (256, 20, 4, "2 3.0"), (256, 32, 8, "1 1.0"),
                                                 (512, 16, 8, "4 1.4"), (256, 32, 4, "4 1.4")])
def test_fastest_measured_form_with_the_norm_by_parts(plan, nt, heads, tiles, want):
    assert plan(nt, heads, tiles, 1) == want


@pytest.mark.parametrize("nt,heads,tiles,want", [(188, 16, 8, "2 1.4"), (375, 16, 8, "4 1.4"), (188, 20, 4, "4 1.4"),
                                                 (375, 12, 8, "4 1.4"), (375, 10, 8, "2 3.0"), (375, 20, 8, "2 1.4"),
                                                 (94, 20, 8, "1 1.4"), (375, 5, 8, "2 3.0")])
def test_fastest_measured_form_with_the_convolution(plan, nt, heads, tiles, want):
    assert plan(nt, heads, tiles, 2) == want
