"""The order of workgroups over the XCDs (csrc/gdn_order.hpp), compiled for the host."""
import subprocess
from collections import Counter
from pathlib import Path

import pytest

HEADER = Path(__file__).resolve().parents[1] / "kairos-sensenova_amd" / "csrc" / "gdn_order.hpp"
MAIN = r"""
#include <cstdio>
#include <cstdlib>
#include "%s"
using namespace kgdn;
int main(int, char** v) {
  const int N = atoi(v[1]), H = atoi(v[2]), S = atoi(v[3]);
  const bool whole = atoi(v[4]) < 0 ? whole_heads(N, H, S, 256, atoi(v[4]) == -2) : atoi(v[4]) != 0;
  printf("%%d\n", whole ? 1 : 0);
  for (int b = 0; b < unit_grid(N, H, S, whole); ++b) {
    const WgUnit u = unit_of(b, N, H, S, whole);
    if (u.ok) printf("%%d %%d %%d %%d\n", b, u.seq, u.head, u.slice);
  }
}
"""


@pytest.fixture(scope="module")
def order(tmp_path_factory):
    d = tmp_path_factory.mktemp("order")
    (d / "main.cpp").write_text(MAIN % HEADER)
    subprocess.run(["g++", "-std=c++17", "-O1", "-o", str(d / "main"), str(d / "main.cpp")], check=True)

    def run(N, H, S, whole=-1):
        out = subprocess.run([str(d / "main"), *map(str, (N, H, S, whole))], check=True, capture_output=True, text=True)
        flag, *rows = out.stdout.splitlines()
        return flag == "1", [tuple(map(int, r.split())) for r in rows]
    return run


# (sequences, heads, slices): the layer's head dims with one sequence and batches, few heads, narrow values
SHAPES = [(1, 20, 8), (2, 20, 8), (4, 10, 8), (8, 5, 8), (1, 5, 8), (20, 1, 8), (200, 1, 1), (3, 7, 4), (2, 20, 4),
          (1, 1, 1), (1, 20, 12), (2, 21, 12), (1, 50, 5)]


@pytest.mark.parametrize("N,H,S", SHAPES)
@pytest.mark.parametrize("whole", [-1, 0, 1])
def test_every_unit_once(order, N, H, S, whole):
    _, rows = order(N, H, S, whole)
    assert sorted(r[1:] for r in rows) == [(n, h, s) for n in range(N) for h in range(H) for s in range(S)]


@pytest.mark.parametrize("N,H,S", SHAPES)
def test_a_head_stays_on_one_xcd(order, N, H, S):
    """Its slices follow each other there, no XCD has more than one head above another, and a
    sequence's heads lie on as many XCDs as they can."""
    _, rows = order(N, H, S, 1)
    at = {}
    for b, n, h, s in rows:
        at.setdefault((n, h), []).append((b % 8, b // 8, s))
    for v in at.values():
        assert len({x for x, _, _ in v}) == 1 and [(j - v[0][1], s) for _, j, s in v] == [(i, i) for i in range(S)]
    load = Counter(v[0][0] for v in at.values())
    assert max(load.values()) - min(load[x] for x in range(8)) <= 1
    for n in range(N):
        assert len({at[n, h][0][0] for h in range(H)}) == min(H, 8)


def test_whole_heads_unless_they_take_another_round(order):
    for N, H, S in [(2, 20, 8), (4, 10, 8), (8, 5, 8), (20, 1, 8), (200, 1, 1), (2, 20, 6), (2, 20, 12), (2, 10, 8)]:
        assert order(N, H, S)[0], (N, H, S)
    # one sequence; 72 and 36 workgroups on some XCDs of 32 CUs against 64 and 30 in equal runs
    for N, H, S in [(1, 20, 8), (1, 33, 8), (2, 21, 12), (2, 10, 12)]:
        assert not order(N, H, S)[0], (N, H, S)


def test_equal_runs_beside_another_kernel(order):
    """Of 20 heads three lie on some XCDs and two on others, while their workgroups take 160 of 256 CUs."""
    for N, H, S, whole in [(2, 10, 8, False), (5, 4, 8, False), (2, 12, 8, True), (3, 5, 8, True), (3, 20, 8, True)]:
        assert order(N, H, S, -2)[0] == whole, (N, H, S)
