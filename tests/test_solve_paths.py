"""How the field solve of a grid runs: the radices of its axes (fft_lines.h on
the host) and the kernels that it launches."""
import os
import shutil
import subprocess

import fake_hip
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include "fft_lines.h"
#include <cstdio>
int main() {
  for (int n = 1; n <= 512; n++) {
    emg::FftAxis a;
    const bool ok = emg::fft_axis(n, 211, &a);
    std::printf("%d %d", n, (int)ok);
    for (int p = 0; p < a.npass; p++) std::printf(" %d", a.r[p]);
    std::printf("\n");
  }
}
"""


def test_axes_split_into_small_radices_and_large_primes(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not found")
    (tmp_path / "drv.cpp").write_text(DRIVER)
    exe = str(tmp_path / "drv")
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-I",
                    os.path.join(ROOT, "ctca_amd", "csrc"), str(tmp_path / "drv.cpp"), "-o", exe],
                   check=True, capture_output=True, text=True)
    primes = [p for p in range(2, 512) if all(p % d for d in range(2, p))]
    small = (2, 3, 4, 5, 7, 8, 11, 13)
    for line in subprocess.run([exe], check=True, capture_output=True, text=True).stdout.split("\n"):
        if not line:
            continue
        n, ok, *radices = (int(v) for v in line.split())
        factors = [p for p in primes if n % p == 0]
        assert ok == all(p <= 211 for p in factors), n
        if not ok:
            continue
        product = 1
        for r in radices:
            assert r in small or (r in primes and r <= 211), (n, radices)
            product *= r
        assert product == n, (n, radices)
        # a large prime's pass has no twiddles if it is the first one
        large = [r for r in radices if r > 13]
        assert radices[:len(large)] == large, (n, radices)


@pytest.mark.parametrize("path,sizes", [
    ("planes", [(16, 16, 16), (45, 45, 45), (49, 50, 63), (90, 70, 51), (77, 77, 60), (98, 98, 48),
                (96, 96, 96), (31, 31, 31), (62, 62, 62), (72, 72, 4), (9, 9, 211), (512, 9, 2)]),
    ("lines", [(95, 66, 40), (114, 95, 133), (199, 40, 40), (62, 127, 9), (105, 100, 100),
               (125, 125, 125), (225, 64, 64), (99, 121, 98), (90, 100, 47), (60, 140, 4),
               (100, 100, 16), (100, 100, 100), (128, 128, 128), (400, 40, 40)]),
    ("library", [(150, 150, 150), (200, 200, 60), (180, 150, 170), (128, 126, 135),
                 (256, 256, 64), (110, 121, 100), (112, 112, 112), (512, 64, 64), (8, 223, 8),
                 (6, 10, 640)]),
])
def test_grids_take_the_path_that_was_measured_for_them(tmp_path, path, sizes):
    fake_hip.run(tmp_path, f"""
        for n in {sizes}:
            with emg.Context(n, [1.0], [1.0], [1.0], (10,)) as c:
                c.upload(records(10, n), (10,))
                c.deposit_rho(0)
                c.solve_es(0.0)
                k = launches(c.solve_es, 0.0)
                got = "library" if "hipfftExecD2Z" in k else \\
                    {{3: "planes", 5: "lines"}}[sum(v.startswith(("k_plane", "k_columns")) for v in k)]
                assert got == "{path}", (n, got)
    """)
