"""unorm8 and quant8_unit as sr_device.hpp defines them, compiled for the CPU:
unorm8 is the table's i / 255.0f for all 256 bytes, quant8_unit is quant8 on
[0, 1 + 2^-20], and each byte comes back."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = os.path.join(ROOT, "rust-softrender_amd", "csrc", "sr_device.hpp")


def test_float_forms_of_a_byte(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host compiler")
    text = open(SOURCE).read()
    bodies = []
    for name in ("clampf", "quant8", "unorm8", "quant8_unit"):
        m = re.search(r"^__device__ __forceinline__ \w+ %s\(.*?\)\s*\{.*?\}$" % name, text, re.M | re.S)
        assert m, name
        bodies.append(m.group(0))
    (tmp_path / "unorm.cpp").write_text("""#include <cmath>
#include <cstdint>
#include <cstring>
#define __device__
#define __forceinline__ inline
""" + "\n".join(bodies) + """
static float bits(uint32_t b) { float f; memcpy(&f, &b, 4); return f; }
int main() {
    for (int i = 0; i < 256; i++) {
        if (unorm8((float)i) != (float)i / 255.0f) return 1;
        if (quant8_unit(unorm8((float)i)) != (float)i) return 2;
    }
    for (uint32_t b = 0; b <= 0x3F800008u; b += b < 0x38000000u ? 65537u : 61u)
        if (quant8_unit(bits(b)) != (float)quant8(bits(b))) return 3;
    return 0;
}
""")
    subprocess.run([cxx, "-std=c++17", "-O1", "-ffp-contract=off", "-o", str(tmp_path / "unorm"),
                    str(tmp_path / "unorm.cpp")], check=True)
    assert subprocess.run([str(tmp_path / "unorm")]).returncode == 0
