"""Arithmetic of launch shapes (csrc/launch_shape.h), compiled for the host."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "turbulence_tracing_amd", "csrc")


def run(tmp_path, body):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host compiler")
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text('#include <cstdio>\n#include "launch_shape.h"\nint main() {\n' + body + "\n}\n")
    subprocess.run([cxx, "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    return [tuple(int(v) for v in line.split()) for line in
            subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.splitlines()]


def test_blocks_resident_on_a_cu(tmp_path):
    got = run(tmp_path, 'for (int b = 1; b <= 64; ++b) std::printf("%d %d\\n", b, tt::lds_for_residency(b));')
    assert [b for b, _ in got] == list(range(1, 65))
    units = 160 * 1024 // 1280
    for blocks, lds in got:
        assert 0 < lds <= 160 * 1024
        fit = units // -(-lds // 1280)  # a request takes whole units
        best = max(units // u for u in range(1, units + 1) if units // u <= blocks)
        assert fit == best, (blocks, lds)
    assert [units // (lds // 1280) for _, lds in got[:12]] == list(range(1, 13))


def test_blocks_beyond_one_axis_of_a_grid(tmp_path):
    cases = [(b, t) for t in (64, 256, 512) for top in [(1 << 32) // t]
             for b in (1, 2, top - 2, top - 1, top, top + 1, 2 * top - 2, 2 * top, 5 * top + 3, 1 << 30)]
    body = "".join(f'{{ auto g = tt::spread({b}ll, {t}); std::printf("%u %u\\n", g.x, g.y); }}\n' for b, t in cases)
    for (b, t), (x, y) in zip(cases, run(tmp_path, body), strict=True):
        assert x * t < 1 << 32 and 1 <= y <= 65535
        assert b <= x * y < b + y  # every block, and fewer spare ones than rows
        assert (y == 1) == (b * t < 1 << 32)
