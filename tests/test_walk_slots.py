"""The slot a lane of the group walk takes from its list of 64: the lowest set
bit, and a slot of the stage where the list is empty (lists of one wave differ
in length, so empty ones are met in every draw).  The expression itself is
compiled for the CPU, where a count of zeros that the language leaves undefined
ends the program."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = os.path.join(ROOT, "rust-softrender_amd", "csrc", "sr_raster_common.hpp")


def test_slot_of_every_list(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host compiler")
    text = open(SOURCE).read()
    slot = re.findall(r"^\s*(const uint32_t k = .*\bleft\b.*;)$", text[text.index("void walk_groups("):], re.M)
    assert len(slot) == 1, slot
    (tmp_path / "slot.cpp").write_text(f"""#include <cstdint>
#include <initializer_list>
__attribute__((noinline)) uint32_t slot(uint64_t left) {{ {slot[0]} return k; }}
int main() {{
    if (slot(0) > 63u) return 1;
    for (uint32_t b = 0; b < 64; b++)
        for (uint64_t above : {{0ull, ~0ull, 0x8000000000000001ull, 0x5555555555555555ull}})
            if (slot(1ull << b | (b < 63 ? above >> (b + 1) << (b + 1) : 0)) != b) return 2;
    return 0;
}}
""")
    subprocess.run([cxx, "-std=c++17", "-O1", "-fsanitize=builtin", "-fsanitize-undefined-trap-on-error", "-o",
                    str(tmp_path / "slot"), str(tmp_path / "slot.cpp")], check=True)
    assert subprocess.run([str(tmp_path / "slot")]).returncode == 0
