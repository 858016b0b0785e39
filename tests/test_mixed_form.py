"""CPU test of the choice between the mixed-factor and the chirp-z transforms
(mc_mixed_form.h): at every even canvas the factors multiply to the length and
lie in 2..127, lengths with a larger prime have none, and the choice is the one
measured: chirp-z for few transforms of a short length with a large factor, mixed
factors for many, for lengths above 1024 and for factors up to 16 (lengths of 129
to 256 forward only for many)."""
import os
import subprocess

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _largest_prime(n):
    p, q = 1, 2
    while q * q <= n:
        while n % q == 0:
            n //= q
            p = q
        q += 1
    return max(p, n)


def test_factors_and_choice(tmp_path):
    src = tmp_path / "form.cpp"
    src.write_text(
        '#include "mc_mixed_form.h"\n#include <cstdio>\n'
        "int main() {\n"
        "  for (int n = 32; n <= 8192; n += n < 4096 ? 1 : 2) {\n"
        "    int f[4] = {1, 1, 1, 1};\n"
        "    const int m = mc::mix_factors(n, f);\n"
        '    printf("%d %d %d %d %d %d %d %d %d\\n", n, m, f[0], f[1], f[2], f[3], (int)mc::mix_use(n, n / 2 + 1, true),\n'
        "           (int)mc::mix_use(n, 24LL * (n / 2 + 1), true), (int)mc::mix_use(n, n / 2 + 1, false));\n"
        "  }\n}\n")
    exe = tmp_path / "form"
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "motioncorr1exp_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True, timeout=120)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=120).stdout
    t = np.array(out.split(), int).reshape(-1, 9)
    few, many = {}, {}
    for n, m, a, b, c, d, u1, u24, back in t:
        few[n], many[n] = u1, u24
        assert (m == 0) == (_largest_prime(n) > 127 or _largest_prime(n) == n), n
        if m:
            assert a * b * c * d == n and min(a, b) >= 2 and max(a, b, c, d) <= 127, n
            if max(a, b, c, d) <= 16 or n > 1024:
                # forward, few: not where the convolution of 512 is the faster
                assert back and u24 and u1 == (not 128 < n <= 256), n
        else:
            assert not u1 and not u24 and not back, n
    # one image: the columns at which the chirp-z transform was the faster, and not
    assert not any(few[n] for n in (134, 254, 412, 508, 762, 1010, 1016))
    assert all(few[n] for n in (310, 374, 530, 590, 708, 890, 976, 1026, 1090, 1854))
    # 24 frames
    assert all(many[n] for n in (186, 212, 340, 412, 508, 762, 1016)) and not many[254]
