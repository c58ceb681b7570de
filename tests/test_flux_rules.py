"""The flux kernel's rules (cgenie_amd/csrc/flux_rules.h), compiled for the CPU
and gone through over their whole range."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")


def run(tmp_path, body):
    src, exe = tmp_path / "rules.cpp", tmp_path / "rules"
    src.write_text('#include <cstdio>\n#include "flux_rules.h"\nusing namespace cgo;\nint main() {\n' + body + "\nreturn 0;\n}\n")
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "cgenie_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    return subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout


def test_staged_slots_hold_the_members_tracers(tmp_path):
    """Every block of every tracer count, tile and coefficient mode stages its
    own tracers, T and S where it needs them, and no plane past the state."""
    out = run(tmp_path, """
    for (int L = 2; L <= 256; L++)
        for (int LB = 2; LB <= 8; LB += 2)
            for (int im = 0; im <= 2; im++)
                for (int l0 = 0; l0 < (im == 1 ? 1 : L); l0 += LB) {
                    const int nl = L - l0 < LB ? L - l0 : LB;
                    bool T = false, S = false;
                    int own = 0;
                    for (int q = 0; q < (im == 0 ? LB + 2 : LB); q++) {
                        if (!flux_staged(q, l0, nl, LB, im)) continue;
                        const int t = flux_slot_tracer(q, l0, LB);
                        if (t < 0 || t >= L) std::printf("L %d LB %d im %d l0 %d slot %d: tracer %d\\n", L, LB, im, l0, q, t);
                        T = T || t == 0;
                        S = S || t == 1;
                        own += t == l0 + q && q < nl;
                    }
                    if (own != nl || (im == 0 && !(T && S))) std::printf("L %d LB %d im %d l0 %d: incomplete\\n", L, LB, im, l0);
                }""")
    assert out == "", out[:2000]
