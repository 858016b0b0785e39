"""CPU test of the column pass's choice of form (mc_cols_form.h): at every even
size from 64 to 8192 and every box up to 256 the chosen radix divides the size,
its tiles hold the box, and the workgroup fits the kernel's launch bound and the
160 KB of LDS of a CU."""
import os
import subprocess

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_every_form_fits(tmp_path):
    src = tmp_path / "form.cpp"
    src.write_text(
        '#include "mc_cols_form.h"\n#include <cstdio>\n'
        "int main() {\n"
        "  for (int n = 64; n <= 8192; n += 2)\n"
        "    for (int box = 1; box <= 256 && box <= n; box++) {\n"
        "      int t = 0;\n"
        "      const int r = mc::cols_radix(n, box, &t);\n"
        "      if (r) printf(\"%d %d %d %d %d %zu\\n\", n, box, r, t, mc::cols_r_waves(n, r),\n"
        "                    mc::cols_r_lds(n, r, t));\n"
        "    }\n}\n")
    exe = tmp_path / "form"
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "motioncorr1exp_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True, timeout=120)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=120).stdout
    n, box, r, t, nw, lds = np.array(out.split(), int).reshape(-1, 6).T
    assert (n % r == 0).all() and (8 * r * t >= box).all()
    assert (nw * 64 >= n // r).all() and (nw <= np.where((t == 1) | (r <= 8), 16, 8)).all()
    assert lds.max() <= 160 * 1024
    # sixteen waves of three tiles do not fit; fifteen do
    assert not ((n == 5766) & (box == 128)).any() and not ((n == 8184) & (box == 192)).any()
    assert ((n == 7672) & (box == 144) & (r == 8) & (t == 3) & (nw == 15)).any()
