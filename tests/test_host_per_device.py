"""What is done once on every device (the permission for a kernel's dynamic LDS): kept by device, and nowhere in a flag of the process."""
import os
import re
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "turbospark_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <thread>
#include <vector>
#include "per_device.h"
int main() {
    tsv::OncePerDevice a, b;
    std::vector<std::thread> all;
    for (int d : {0, 3, 63, 64, -1}) all.emplace_back([&a, d] { a.note(d); });
    for (auto& t : all) t.join();
    for (int d = -1; d <= 128; d++) printf("%d%d", a.needed(d), b.needed(d));
}
"""


def test_a_device_does_not_stand_for_another(tmp_path):
    src = tmp_path / "t.cpp"
    src.write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-pthread", "-I", CSRC, str(src), "-o", str(tmp_path / "t")])
    out = subprocess.check_output([str(tmp_path / "t")], text=True)
    got = [out[2 * i] for i in range(130)]
    assert [d - 1 for d in range(130) if got[d] == "0"] == [0, 3, 63]      # beyond 64 devices: asked for every time
    assert set(out[1::2]) == {"1"}                                         # another kernel's record is another one


def test_every_permission_is_asked_for_by_device():
    places = {name: len(re.findall(r"hipFuncSetAttribute", open(os.path.join(CSRC, name)).read())) for name in os.listdir(CSRC)
              if name.endswith((".hip", ".h"))}
    assert {n: c for n, c in places.items() if c} == {"tsv_internal.h": 1}
