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
            for (int maxk = 2; maxk <= 48; maxk++)
                for (int nb = 1; nb <= 2000; nb++) {
                    const int kc = flux_split_levels(nb, maxk, p, mix, FLUX_NV_MAX);
                    bool ok = kc == 0 || (kc >= 2 && kc <= maxk);
                    if (kc) ok = ok && (kc == maxk || (long long)nb * ((maxk + kc - 1) / kc) <= 768);
                    ok = ok && (kc != 0) <= (flux_split_levels(1, maxk, p, mix, 0) != 0) && !(nb > 1152 && kc);
                    ok = ok && flux_split_levels(nb, maxk, p, mix, FLUX_NV_MAX + 1) == 0;
                    ok = ok && !(kc && !flux_split_levels(nb, maxk, p, true, 0));
                    if (!ok) std::printf("p %d mix %d maxk %d nb %d: %d\\n", p, mix, maxk, nb, kc);
                }
    // where it was measured
    const int at[][4] = {{0, 1, 16, 48}, {0, 1, 16, 1152}, {1, 1, 16, 768}, {0, 0, 16, 480}, {0, 0, 8, 192}, {0, 0, 32, 384},
                         {1, 0, 16, 384}, {1, 0, 32, 256}};
    const int no[][4] = {{0, 1, 16, 1153}, {1, 1, 16, 769}, {0, 0, 16, 576}, {0, 0, 8, 384}, {0, 0, 32, 512}, {1, 0, 16, 480},
                         {1, 0, 32, 384}};
    for (auto& a : at) if (!flux_split_levels(a[3], a[2], a[0], a[1], 0)) std::printf("no split %d %d\\n", a[2], a[3]);
    for (auto& a : no) if (flux_split_levels(a[3], a[2], a[0], a[1], 0)) std::printf("split %d %d\\n", a[2], a[3]);""")
    assert out == "", out[:2000]
