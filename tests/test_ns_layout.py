"""Where the entries of non-symmetric trees stand (ns_layout.h), walked as EvalNonSymmetricLdsKernel walks them."""
import os
import random
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SMALL = 64  # items of a tree whose leaves have one place each


@pytest.fixture(scope="module")
def lay_out(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("ns") / "ns_layout_main")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", os.path.join(ROOT, "tests", "ns_layout_main.cpp"), "-o", out])

    def run(trees):
        text = "".join(" ".join(map(str, tree)) + "\n" for tree in trees)
        layouts = []
        for line in subprocess.check_output([out], input=text, text=True).splitlines():
            numbers = list(map(int, line.split()))
            layouts.append((numbers[0], numbers[1:8], numbers[8::2], numbers[9::2]))
        assert len(layouts) == len(trees)
        return layouts
    return run


def _tree(rng, depth, p_leaf, shape=None):
    """Breadth first, the left child's item of every item (-1: a leaf). shape: "left" or "right", a chain to that side."""
    left, level, on_chain = [None], [0], [True]
    at = 0
    while at < len(left):
        if level[at] == depth or (shape and not on_chain[at]) or (not shape and rng.random() < p_leaf):
            left[at] = -1
        else:
            left[at] = len(left)
            left += [None, None]
            level += [level[at] + 1] * 2
            on_chain += [shape == "left", shape == "right"]
        at += 1
    return left


def _trees():
    rng = random.Random(1)
    trees = [_tree(rng, depth, 0.0) for depth in range(9)]
    trees += [_tree(rng, depth, 0.0, side) for depth in (1, 2, 3, 4, 9, 200) for side in ("left", "right")]
    trees += [_tree(rng, rng.randint(1, 8), rng.choice([0.1, 0.3, 0.5])) for _ in range(300)]
    # pairs that two items name, as behind a one-hot split: of leaves, and of items with children
    trees += [[1, 3, 5, -1, -1, 7, 3, -1, -1], [1, 3, 5, 9, -1, 7, 3, -1, -1, -1, -1], [1, 3, 5, 9, 11, 7, 3, -1, -1, -1, -1, 13, -1, -1, -1]]
    return trees


def test_walks_end_at_the_leaf_that_the_decisions_lead_to(lay_out):
    rng = random.Random(2)
    trees = _trees()
    for left, (steps, top, items, following) in zip(trees, lay_out(trees)):
        assert max(following) < len(items)
        for _ in range(40):
            decisions = {}  # of an item, whichever way it is met
            side = lambda item: decisions.setdefault(item, rng.randrange(2))  # noqa: E731
            at = 0
            while left[at] != -1:
                at = left[at] + side(at)
            node = 0
            path = 0
            for _ in range(3):
                bit = side(top[node]) if top[node] != -1 else 0  # a node that is not there is false
                path, node = 2 * path + bit, 2 * node + 1 + bit
            place = path
            for _ in range(steps):
                item = items[place]
                place = following[place] + (side(item) if left[item] != -1 else 0)
            if left[items[place]] == -1:
                place = following[place]  # with no steps an exit names the place itself
            assert left[items[place]] == -1 and items[place] == at and following[place] == place


def test_leaves_of_small_trees_have_one_place(lay_out):
    """Leaf values are read by place: leaves above the third level, which several exits hold, stand behind each other."""
    trees = _trees()
    seen = 0
    for left, (_, _, items, following) in zip(trees, lay_out(trees)):
        shared = [exit for exit in range(8) if items[:8].count(items[exit]) > 1]
        places = sorted({following[exit] for exit in shared})
        if len(left) <= SMALL:
            seen += bool(shared)
            assert len(places) == len({items[exit] for exit in shared})
            assert places == list(range(len(items) - len(places), len(items)))
        else:
            assert places == shared and len(items) <= len(left) + 1
    assert seen > 100


def test_rows_of_leaf_values(tmp_path):
    """One dimension reads a region's zeros behind the last entry; several read the range's trees alone, and nothing lies behind theirs."""
    source = tmp_path / "rows.cpp"
    source.write_text('#include "ns_layout.h"\n'
                      "static_assert(cbamd::NsSliceRows(1000, 1, 2048) == 3048);\n"
                      "static_assert(cbamd::NsSliceRows(1000, 2, 2048) == 1000 && cbamd::NsSliceRows(1000, 4, 1024) == 1000);\n"
                      "int main() {}\n")
    subprocess.check_call(["g++", "-std=c++17", "-I", os.path.join(ROOT, "catboost_amd", "csrc"), "-fsyntax-only", str(source)])
    with open(os.path.join(ROOT, "catboost_amd", "csrc", "hip_evaluator.hip")) as f:
        assert "sliceRows = NsSliceRows(entries.size(), dims, m.NsLdsShape.Entries)" in f.read()


def test_rows_of_trees_that_end_at_their_exits(tmp_path):
    """Units without a step: every exit names a row with its own leaf's value, the rows of a unit's trees lie behind each other from the
    first on, one per leaf that an exit holds, and their entries read as the kernel reads them."""
    source = tmp_path / "exits.cpp"
    source.write_text(r'''
#include "ns_layout.h"
#include <cstdio>
int main() {
    for (unsigned seed = 1; seed < 2000; ++seed) {
        unsigned state = seed * 2654435761u;
        const auto draw = [&](unsigned n) { state = state * 1664525u + 1013904223u; return (state >> 10) % n; };
        std::vector<uint32_t> from;
        size_t rows = 0;
        for (unsigned tree = 0, trees = 1 + draw(3); tree < trees; ++tree) {
            const unsigned start = 16 * tree, leaves = 1 + draw(8);
            uint32_t exits[8], places[8];
            bool held[16] = {};
            for (unsigned exit = 0; exit < 8; ++exit) {
                places[exit] = start + draw(leaves) * 2 % 16 + (leaves > 4 ? draw(2) : 0);
                held[places[exit] - start] = true;
                exits[exit] = cbamd::NsTerminalEntry(places[exit]);
            }
            cbamd::CompactNsExits(exits, &from);
            for (bool h : held) {
                rows += h;
            }
            if (from.size() != rows) {
                return 1;
            }
            for (unsigned exit = 0; exit < 8; ++exit) {
                const uint32_t row = ((exits[exit] >> 18) | (~exits[exit] & 8u)) / 8;
                if (row >= rows || from[row] != places[exit] || (exits[exit] & 0x1fff00u) != 0) {
                    return 2;
                }
            }
        }
    }
    return 0;
}
''')
    program = str(tmp_path / "exits")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "catboost_amd", "csrc"), str(source), "-o", program])
    subprocess.check_call([program])
