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


def test_split_by_levels_over_its_range(tmp_path):
    """The split's levels per block for every batch size and depth: at least
    two, chunks that cover the column and fill the chip no more than once, none
    past the sizes where whole columns are faster nor with a workspace above
    its bound."""
    out = run(tmp_path, """
    for (int p = 0; p < 2; p++)
        for (int mix = 0; mix < 2; mix++)
            for (int bgc = 0; bgc < 2; bgc++)
                for (int maxk = 2; maxk <= 48; maxk++)
                    for (int nb = 1; nb <= 1000; nb++)
                        for (int cols = 16; cols <= 200000; cols *= 5) {
                            const int kc = flux_split_levels(nb, cols, maxk, p, mix, bgc, FLUX_NV_MAX);
                            bool ok = kc == 0 || (kc >= 2 && kc <= maxk);
                            if (kc) ok = ok && ((maxk + kc - 1) / kc == 1 || (long long)nb * ((maxk + kc - 1) / kc) <= 768);
                            ok = ok && !(nb > 832 && kc) && !(nb <= 192 && maxk >= 8 && mix && cols <= 1000 && !kc);
                            ok = ok && flux_split_levels(nb, cols, maxk, p, mix, bgc, FLUX_NV_MAX + 1) == 0;
                            if (!ok) std::printf("p %d mix %d bgc %d maxk %d nb %d cols %d: %d\\n", p, mix, bgc, maxk, nb, cols, kc);
                        }
    // nb, columns, levels, precision, mixing, BIOGEM: on either side of the line, where both were measured
    const int at[][6] = {{48, 907, 16, 0, 1, 1}, {480, 27210, 16, 0, 1, 1}, {768, 14512, 16, 0, 1, 1}, {816, 43548, 32, 0, 1, 1},
                         {224, 12698, 16, 1, 1, 1}, {384, 7256, 16, 1, 1, 1}, {768, 43536, 16, 1, 1, 0}, {480, 9070, 16, 0, 0, 0},
                         {192, 3628, 8, 0, 0, 0}, {408, 21774, 32, 0, 0, 0}, {384, 7256, 16, 1, 0, 0}, {272, 14516, 32, 1, 0, 0}};
    const int no[][6] = {{576, 32652, 16, 0, 1, 1}, {576, 32688, 8, 0, 1, 1}, {864, 16326, 16, 0, 1, 1}, {1152, 21768, 16, 0, 1, 1},
                         {320, 18140, 16, 1, 1, 1}, {480, 9070, 16, 1, 1, 1}, {769, 9000, 16, 1, 1, 0}, {576, 10884, 16, 0, 0, 0},
                         {384, 7256, 8, 0, 0, 0}, {544, 29032, 32, 0, 0, 0}, {480, 9070, 16, 1, 0, 0}, {408, 21774, 32, 1, 0, 0}};
    for (auto& a : at) if (!flux_split_levels(a[0], a[1], a[2], a[3], a[4], a[5], 0)) std::printf("no split %d %d\\n", a[0], a[1]);
    for (auto& a : no) if (flux_split_levels(a[0], a[1], a[2], a[3], a[4], a[5], 0)) std::printf("split %d %d\\n", a[0], a[1]);""")
    assert out == "", out[:2000]
