"""Which rows and which KV head a workgroup of the prompt attention takes: every group of every head once, a head's workgroups nkv apart
(eight heads: one to an XCD), the longest rows first, and with two workgroups to a compute unit the second half from the short end."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "turbospark_amd", "csrc")
PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "prompt_place.h"
int main(int, char** v) {
    const int grid = atoi(v[1]), nkv = atoi(v[2]);
    for (int b = 0; b < grid; b++) {
        const tsv::PromptAttnPlace p = tsv::prompt_attn_place(b, grid, nkv, v[3][0] == '1');
        printf("%d %d\n", p.head, p.group);
    }
}
"""


@pytest.fixture(scope="module")
def place(tmp_path_factory):
    d = tmp_path_factory.mktemp("place")
    (d / "t.cpp").write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-I", CSRC, str(d / "t.cpp"), "-o", str(d / "t")])
    return lambda *a: [tuple(map(int, line.split())) for line in subprocess.check_output([str(d / "t"), *map(str, a)], text=True).splitlines()]


@pytest.mark.parametrize("nkv", [1, 2, 3, 4, 8, 16])
@pytest.mark.parametrize("groups", [1, 5, 31, 32, 33, 64, 65, 100, 256, 257, 512])
def test_every_group_of_every_head_once(place, nkv, groups):
    grid = nkv * groups
    for whole in (0, 1):
        got = place(grid, nkv, whole)
        assert sorted(got) == [(h, g) for h in range(nkv) for g in range(groups)]
        assert [h for h, _ in got] == [b % nkv for b in range(grid)]        # a head stays on its XCDs
        order = [g for _, g in got][::nkv]
        turned = 256 // nkv if whole and 256 < grid <= 512 else groups
        assert order[:turned] == sorted(order[:turned], reverse=True) and order[turned:] == sorted(order[turned:])
