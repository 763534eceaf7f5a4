"""The workspace of ffmi_linear (runtime/graph_workspace.h) with an allocator that
records: what a captured call was given is never freed, whatever is asked for later,
everything else is, and what is kept stays below the current block."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include "runtime/graph_workspace.h"
// arguments: sizes, 'g' before those of captured calls; prints every call's block and
// its size, what was freed, and what is kept
int main(int argc, char **argv) {
  ffmi::GraphWorkspace ws;
  long next = 0;
  for (int i = 1; i < argc; ++i) {
    const bool graph = argv[i][0] == 'g';
    long freed = 0;
    void *p = ws.get(
        (size_t)atol(argv[i] + graph), graph, [&](size_t n) { return n > 5000 ? nullptr : (void *)++next; },
        [&](void *q) { return freed = (long)q, true; });
    printf("%ld %zu %ld %zu\n", (long)p, ws.bytes(), freed, ws.kept());
  }
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("ws")
    (d / "p.cc").write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "flexflow_amd", "csrc"),
                           str(d / "p.cc"), "-o", str(d / "p")])

    def run(*calls):
        out = subprocess.run([str(d / "p"), *map(str, calls)], capture_output=True, text=True, check=True).stdout
        return [tuple(map(int, line.split())) for line in out.splitlines()]
    return run


def test_without_graphs_one_block(program):
    # (block, bytes, freed, kept)
    assert program(0, 100, 50, 100, 300, 10) == [(0, 0, 0, 0), (1, 100, 0, 0), (1, 100, 0, 0), (1, 100, 0, 0),
                                                 (2, 300, 1, 0), (2, 300, 0, 0)]


def test_a_captured_call_then_the_same_eagerly(program):
    assert program("g22", 26, 22) == [(1, 22, 0, 0), (2, 44, 0, 22), (2, 44, 0, 22)]


def test_an_eager_call_then_captured_then_a_larger_one(program):
    assert program(22, "g20", 34, 500) == [(1, 22, 0, 0), (1, 22, 0, 0), (2, 44, 0, 22), (3, 500, 2, 22)]


def test_a_captured_call_that_needs_more_frees_nothing(program):
    assert program(10, "g30", "g70") == [(1, 10, 0, 0), (2, 30, 0, 10), (3, 70, 0, 40)]


def test_no_memory(program):
    # the block in a graph stays, another one was given back
    assert program("g10", 6000, 10) == [(1, 10, 0, 0), (0, 10, 0, 0), (1, 10, 0, 0)]
    assert program(10, 6000, 10) == [(1, 10, 0, 0), (0, 0, 1, 0), (2, 10, 0, 0)]


@pytest.mark.parametrize("seed", range(20))
def test_any_order(program, seed):
    import random
    rng = random.Random(seed)
    calls = [("g" if rng.random() < 0.3 else "") + str(rng.randint(1, 2000)) for _ in range(60)]
    in_graph = set()
    for call, (p, n, freed, kept) in zip(calls, program(*calls)):
        assert p and n >= int(call.lstrip("g")) and kept <= n and freed not in in_graph
        if call[0] == "g":
            in_graph.add(p)
