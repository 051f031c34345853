"""round_quotient_fast (blink_divrn.hpp) on products that no int holds, under the undefined
behaviour sanitizer (host code, no GPU)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = """
#include <cmath>
#include <cstdio>
#include "imager_amd/csrc/blink_divrn.hpp"
int main() {
    const double refused[] = {NAN, INFINITY, -INFINITY, 1e300, -1e300, 0x1p29, -0x1p29, 0x1p31, -0x1p31,
                              0x1p63, 0.5, -0.5, 1.5, 2.5 + 1e-7, 0x1p28 + 0.5};
    for (double p : refused) {
        int out = 7;
        if (blink::round_quotient_fast(p, 1.0, out)) return std::printf("%g taken\\n", p), 1;
    }
    const double taken[] = {0.0, -0.0, 0.25, -0.75, 3.0, -1e6 + 0.3, 0x1p29 - 1.0, 1.0 - 0x1p29};
    for (double p : taken) {
        int out = 7;
        if (!blink::round_quotient_fast(p, 1.0, out) || out != (int)std::round(p))
            return std::printf("%g: %d\\n", p, out), 1;
    }
    return 0;
}
"""


def test_no_cast_out_of_range(tmp_path):
    src, exe = tmp_path / "rounding.cpp", tmp_path / "rounding"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=gnu++17", "-O1", "-I", ROOT, "-fsanitize=undefined,float-cast-overflow",
                    "-fno-sanitize-recover=all", "-o", str(exe), str(src)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
