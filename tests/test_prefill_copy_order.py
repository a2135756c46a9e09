"""The copy schedule of the 64-rows-per-wave prefill kernel with four key parts
(csrc/rows64_copies.hpp, whose constants the kernel issues and waits by), walked on
the CPU: every unit of K and V has landed when it is read."""
import pathlib
import subprocess

CSRC = pathlib.Path(__file__).resolve().parents[1] / "llm-inference_amd" / "csrc"

PROGRAM = r"""
#include "rows64_copies.hpp"
#include <cstdio>
using namespace rows64;
int main() {
    for (int units = 1; units <= 56; ++units)
        if (!copies_ok(kFirst, kLeftFirst, kLeftK, kLeftV, units)) {
            std::printf("schedule reads a unit in flight at %d units\n", units);
            return 1;
        }
    // the model sees K 1 in flight when V 0 stands before it, unless the wait
    // covers it, and waits that are one unit short
    constexpr First v_early = {{true, false, true, true}};
    if (copies_ok(v_early, 3, 3, 1, 1) || !copies_ok(v_early, 3, 2, 1, 8)) return 2;
    if (copies_ok(kFirst, 4, 3, 1, 1) || copies_ok(kFirst, 3, 4, 1, 8) ||
        copies_ok(kFirst, 3, 3, 2, 8))
        return 3;
    return 0;
}
"""


def test_every_unit_has_landed_when_read(tmp_path):
    src, exe = tmp_path / "order.cpp", tmp_path / "order"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++20", "-Wall", "-Werror", f"-I{CSRC}", str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    kernel = (CSRC / "prefill_rows64.hip").read_text()
    for name in ("kFirst.k[", "kLeftFirst * NI", "kLeftK * NI", "kLeftV * NI"):
        assert f"rows64::{name}" in kernel, name
